"""The grouped product for a few tokens per expert (moe_midstream.hip), which
launch_grouped_mxfp4 takes up to 1800 rows and 50 rows per expert.  Its chain
of matrix-core products is grouped_mfma_kernel's, so the same rows give the
same bits in a larger call that takes that kernel: every case appends filler
rows on one more expert until the call leaves the range, and compares the
original rows.  Against fp64 the result is one bf16 rounding away."""
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
