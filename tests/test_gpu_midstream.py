"""The grouped product for a few tokens per expert (moe_midstream.hip), which
launch_grouped_mxfp4 takes up to 1800 rows and 50 rows per expert.  Its chain
of matrix-core products is grouped_mfma_kernel's, so the same rows give the
same bits in a larger call that takes that kernel: the cases append filler rows
until the call leaves the range, and compare the original rows.  Against fp64
the result is one bf16 rounding away."""
import numpy as np
import pytest
import torch

import gptoss_moe as g
import moe_data
import moe_oracle as orc

pytestmark = pytest.mark.gpu


def _dev(a):
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16)).view(torch.bfloat16).cuda()
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _tiled(w, E, N, K):
    nb, sb = g.tiled_size(N, K)
    out = torch.empty(E * nb, dtype=torch.uint8, device="cuda"), torch.empty(E * sb, dtype=torch.uint8, device="cuda")
    for e in range(E):
        g.pack_tiled(_dev(w[0][e]), _dev(w[1][e]), N, K, out[0][e * nb:(e + 1) * nb], out[1][e * sb:(e + 1) * sb])
    return out


# K / 32 = 10 (one block into the second phase), 16, 18, 33 (ragged phases), 90;
# N / 64 with 1 .. 4 live waves in the last group
@pytest.mark.parametrize("N,K", [(64, 320), (320, 512), (128, 576), (448, 1056), (256, 2880)])
@pytest.mark.parametrize("counts", [(1,), (16, 0, 17), (48, 64, 1), (65, 0, 128, 3), (2, 33, 49, 63)])
@pytest.mark.parametrize("special", [False, True])
def test_mid_stream_rows(N, K, counts, special):
    E = len(counts) + 1
    rng = np.random.default_rng([N, K, len(counts)])
    packed = rng.integers(0, 256, (E, N, K // 2), dtype=np.uint8)
    scales = rng.integers(119, 124, (E, N, K // 32), dtype=np.uint8)
    if special:
        scales[0, N // 2, -1], scales[len(counts) - 1, 0, 0] = 255, 0
    bias = moe_data.bf16(rng.normal(0.0, 0.5, (E, N)))
    S = sum(counts)
    fill = 1801
    x = moe_data.bf16(rng.normal(0.0, 1.0, (S + fill, K)))
    tn, ts = _tiled((packed, scales), E, N, K)
    offs = np.concatenate([[0], np.cumsum(counts)])
    small = _dev(np.append(offs, S).astype(np.int32))          # the last expert has no rows
    large = _dev(np.append(offs, S + fill).astype(np.int32))   # and here it has the filler's
    tx, tb = _dev(x), _dev(bias)
    for swiglu in (False, True):
        got = g.grouped_mxfp4_gemm(tx[:S].contiguous(), small, tn, ts, N, K, S, bias=tb, swiglu=swiglu)
        ref = g.grouped_mxfp4_gemm(tx, large, tn, ts, N, K, S + fill, bias=tb, swiglu=swiglu)
        assert torch.equal(got.view(torch.int16), ref[:S].view(torch.int16))
    if special:
        return
    y = g.grouped_mxfp4_gemm(tx[:S].contiguous(), small, tn, ts, N, K, S, bias=tb).float().cpu().numpy()
    xf = orc.bf16_to_f32(x[:S]).astype(np.float64)
    for e, c in enumerate(counts):
        w = _dequant(packed[e], scales[e])
        r = slice(offs[e], offs[e] + c)
        want = xf[r] @ w.T + orc.bf16_to_f32(bias[e]).astype(np.float64)
        # fp32 sums of K products, then one rounding to bf16: 8 significant
        # bits, so half a step is at most 2^-8 of the value
        bound = 2.0 ** -8 * np.abs(want) + (K + 2) * 2.0 ** -24 * (np.abs(xf[r]) @ np.abs(w).T + 1.0)
        assert (np.abs(y[r] - want) <= bound).all()


def _nan_behind(a):
    """The rows of a on the device, followed by NaN."""
    t = _dev(a)
    buf = torch.full((t.numel() + 8192,), float("nan"), dtype=torch.bfloat16, device="cuda")
    v = buf[:t.numel()].view(t.shape)
    v.copy_(t)
    return v


# One row of x: a phase's loads of K blocks past the last must not reach
# behind the row, where NaN would survive the zero weights.
@pytest.mark.parametrize("K", [320, 352, 416, 576, 1024, 1056])
def test_mid_stream_one_row_of_x(K):
    E, N = 2, 128
    rng = np.random.default_rng(K)
    packed = rng.integers(0, 256, (E, N, K // 2), dtype=np.uint8)
    scales = rng.integers(119, 124, (E, N, K // 32), dtype=np.uint8)
    x = moe_data.bf16(rng.normal(0.0, 1.0, (1, K)))
    tn, ts = _tiled((packed, scales), E, N, K)
    offs = torch.tensor([0, 0, 1], dtype=torch.int32, device="cuda")
    y = g.grouped_mxfp4_gemm(_nan_behind(x), offs, tn, ts, N, K, 1).float().cpu().numpy()
    xf = orc.bf16_to_f32(x).astype(np.float64)
    w = _dequant(packed[1], scales[1])
    bound = 2.0 ** -8 * np.abs(xf @ w.T) + (K + 2) * 2.0 ** -24 * (np.abs(xf) @ np.abs(w).T + 1.0)
    assert (np.abs(y - xf @ w.T) <= bound).all()


# The same through the layer, which gathers its one token for every expert.
def test_mid_stream_one_token_layer():
    E, k, H, I = 8, 4, 320, 448
    w = moe_data.make_layer(3, E, H, I, bias="random")
    x, res = moe_data.make_tokens(1, 1, H)
    cfg = g.default_config(E, 1, prefill_min_tokens=1)
    cfg.hidden_size, cfg.intermediate_size, cfg.top_k = H, I, k
    t = {n: _dev(v) for n, v in w.items()}
    layer = g.MoELayer().init(cfg, 0, t["router_w"], t["router_b"], t["w1_bias"], t["w2_bias"],
                              mlp1=([t["w1_packed"][e] for e in range(E)], [t["w1_scales"][e] for e in range(E)]),
                              mlp2=([t["w2_packed"][e] for e in range(E)], [t["w2_scales"][e] for e in range(E)]))
    idx = torch.tensor([[5, 0, 7, 2]], dtype=torch.int32, device="cuda")
    wts = torch.tensor([[0.4, 0.3, 0.2, 0.1]], device="cuda")
    a = layer.forward_routed(_dev(x), idx, wts, residual=_dev(res))
    b = layer.forward_routed(_nan_behind(x), idx, wts, residual=_dev(res))
    assert torch.isfinite(a.float()).all() and torch.equal(a.view(torch.int16), b.view(torch.int16))
    layer.destroy()


def _random_tiled(E, N, K, special, seed):
    """Uniform codes and scales, made on the device; special: codes 0 and 255
    in the scales of every fifth expert."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    nb, sb = g.tiled_size(N, K)
    out = torch.empty(E * nb, dtype=torch.uint8, device="cuda"), torch.empty(E * sb, dtype=torch.uint8, device="cuda")
    for e in range(E):
        q = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device="cuda", generator=gen)
        s = torch.randint(119, 124, (N, K // 32), dtype=torch.uint8, device="cuda", generator=gen)
        if special and e % 5 == 0:
            s[e % N, -1], s[(7 * e + 70) % N, e % (K // 32)] = 0, 255
        g.pack_tiled(q, s, N, K, out[0][e * nb:(e + 1) * nb], out[1][e * sb:(e + 1) * sb])
    return out


# Several items per work-group (about 130 chunks x 8 groups of tiles on 512
# work-groups: full rounds and a partial one), and fewer items than
# work-groups; phases of 8 (K / 32 = 16, 22) and 9 blocks (18, 26), two and
# three of them; chunks of 1 to 64 rows next to each other
@pytest.mark.parametrize("K", [512, 576, 704, 832])
@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("routing", ["ragged", "few"])
def test_mid_stream_many_items(K, special, routing):
    E, N = 96, 2048
    rng = np.random.default_rng([K, special])
    counts = np.zeros(E, dtype=np.int64)
    if routing == "ragged":
        counts[:] = rng.choice([0, 1, 5, 8, 16, 17, 31, 33], E, p=[.15, .15, .15, .15, .12, .12, .08, .08])
        counts[rng.choice(E, 6, replace=False)] = [47, 49, 63, 64, 65, 100]
    else:
        counts[rng.choice(E, 4, replace=False)] = [50, 50, 16, 129]
    S = int(counts.sum())
    assert S <= 1800
    tn, ts = _random_tiled(E + 1, N, K, special, K)
    gen = torch.Generator(device="cuda").manual_seed(K + 1)
    x = torch.randn((S + 1801, K), device="cuda", generator=gen).to(torch.bfloat16)
    bias = (0.5 * torch.randn((E + 1, N), device="cuda", generator=gen)).to(torch.bfloat16)
    offs = np.concatenate([[0], np.cumsum(counts)])
    small, large = _dev(np.append(offs, S).astype(np.int32)), _dev(np.append(offs, S + 1801).astype(np.int32))
    for swiglu, b in ((False, bias), (True, bias), (True, None)):
        gu = [torch.zeros((n, N), dtype=torch.bfloat16, device="cuda") if swiglu else None for n in (S, S + 1801)]
        got = g.grouped_mxfp4_gemm(x[:S], small, tn, ts, N, K, S, bias=b, swiglu=swiglu, gate_up=gu[0])
        ref = g.grouped_mxfp4_gemm(x, large, tn, ts, N, K, S + 1801, bias=b, swiglu=swiglu, gate_up=gu[1])
        assert torch.equal(got.view(torch.int16), ref[:S].view(torch.int16))
        if swiglu:
            assert torch.equal(gu[0].view(torch.int16), gu[1][:S].view(torch.int16))


# The most chunks a call can have: 1800 rows, 255 of 256 experts with one each
def test_mid_stream_most_chunks():
    E, N, K, S = 256, 64, 320, 1800
    tn, ts = _random_tiled(E, N, K, False, 9)
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn((S + 128, K), device="cuda", generator=gen).to(torch.bfloat16)
    for big in (0, 100, 255):
        counts = np.ones(E, dtype=np.int64)
        counts[big] = S - (E - 1)
        offs = np.concatenate([[0], np.cumsum(counts)])
        got = g.grouped_mxfp4_gemm(x[:S], _dev(offs.astype(np.int32)), tn, ts, N, K, S)
        ref = g.grouped_mxfp4_gemm(x, _dev(offs.astype(np.int32)), tn, ts, N, K, S + 128)
        assert torch.equal(got.view(torch.int16), ref[:S].view(torch.int16))


# The layer's products: rows gathered through the plan, the gate_up trace,
# scale codes 0 and 255, with and without biases.  The first T tokens of a
# larger forward (more than 1800 rows) take the other kernel: the same bits.
@pytest.mark.parametrize("H,I", [(512, 576), (832, 704)])
@pytest.mark.parametrize("T", [130, 450])
@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("bias", [True, False])
def test_mid_stream_layer(H, I, T, special, bias):
    E, k, fill = 64, 4, 460
    tiled = (*_random_tiled(E, 2 * I, H, special, 1), *_random_tiled(E, H, I, special, 2))
    gen = torch.Generator(device="cuda").manual_seed(T)

    def randn(*shape, scale=1.0):
        return (scale * torch.randn(shape, device="cuda", generator=gen)).to(torch.bfloat16)

    rw, rb = randn(E, H, scale=0.02), randn(E, scale=0.02)
    b1, b2 = (randn(E, 2 * I, scale=0.5), randn(E, H, scale=0.5)) if bias else (None, None)
    cfg = g.default_config(E, T + fill)
    cfg.hidden_size, cfg.intermediate_size, cfg.top_k = H, I, k
    layer = g.MoELayer().init(cfg, 0, rw, rb, b1, b2, tiled=tiled)
    layer.set_trace_gate_up(True)
    x, res = randn(T + fill, H), randn(T + fill, H)
    # expert popularity by a power law, so that chunks of all heights occur
    logp = -1.1 * torch.log(torch.arange(E, device="cuda") + 1.0)
    noise = -torch.log(-torch.log(torch.rand((T + fill, E), device="cuda", generator=gen).clamp_(1e-6, 1 - 1e-6)))
    idx = (logp + noise).topk(k, dim=1).indices.to(torch.int32).contiguous()
    wts = torch.softmax(torch.randn((T + fill, k), device="cuda", generator=gen), dim=1).contiguous()

    def stages(n):
        out = layer.forward_routed(x[:n], idx[:n], wts[:n], residual=res[:n])
        torch.cuda.synchronize()
        tr, S = layer.trace(), n * k
        gm = g.copy_device_to_tensor(tr.gather_map, S * 4, torch.int32)[:T * k].long()
        rows = [g.copy_device_to_tensor(p, S * w * 2, torch.int16).view(S, w)[gm]
                for p, w in ((tr.gate_up, 2 * I), (tr.act, I), (tr.expert_out, H))]
        return [*rows, out[:T].view(torch.int16)]

    for what, a, b in zip(("gate_up", "activations", "expert outputs", "out"), stages(T), stages(T + fill)):
        assert torch.equal(a, b), what
    layer.destroy()


# What the grouped product refuses (an expert's nibbles of 2 GiB or more) it
# refuses at every row count.  The buffers are real: nothing would be read out
# of range if a call were taken.
@pytest.mark.parametrize("rows", [1, 40, 1801])
def test_matrix_too_large_is_refused(rows):
    N, K = 1398144, 3072
    nb, sb = g.tiled_size(N, K)
    assert nb >= 2 ** 31
    nib, sc = (torch.zeros(n, dtype=torch.uint8, device="cuda") for n in (nb, sb))
    x = torch.zeros((rows, K), dtype=torch.bfloat16, device="cuda")
    offs = torch.zeros(2, dtype=torch.int32, device="cuda")
    with pytest.raises(g.GptossError, match="grouped gemm launch"):
        g.grouped_mxfp4_gemm(x, offs, nib, sc, N, K, rows)


def _dequant(packed, scales):
    lut = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6])
    v = np.stack([lut[packed & 15], lut[packed >> 4]], axis=-1).reshape(packed.shape[0], -1)
    return v * np.repeat(2.0 ** (scales.astype(np.float64) - 127.0), 32, axis=1)
