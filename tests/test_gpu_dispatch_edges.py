"""Sizes at the edges of the dispatch rules, against the oracle or a plain
restatement: the dense GEMV's rows per work-group, unaligned inputs and scale
codes 0 and 255; the layer's routing plan around the sizes where its launches
change; the exact decode's steps under skewed routing; the stage
combine's 16-byte form and its fallback."""
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


def _bits(t):
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


# one, two and four rows per work-group (tiles x M up to 1024, 2560, above);
# 1, 2, 5, 15 and 16 blocks per K-part; x on 16 or 2 bytes
@pytest.mark.parametrize("N,K", [(64, 32), (128, 320), (192, 960), (2880, 2880), (512, 2048)])
@pytest.mark.parametrize("M", [1, 7, 23, 57, 130])
@pytest.mark.parametrize("shift", [0, 1])
def test_gemv_rows(N, K, M, shift):
    rng = np.random.default_rng([N, K, M])
    x = moe_data.bf16(rng.normal(0, 1, (M, K)))
    packed = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    scales = rng.integers(119, 124, (N, K // 32), dtype=np.uint8)
    scales[5, -1], scales[N - 1, 0] = 0, 255
    packed[N - 1, :16] = 0x22  # times +inf: no 0 * inf
    bias = moe_data.bf16(rng.normal(0, 0.5, N))
    nib, sc = g.pack_tiled(_dev(packed), _dev(scales), N, K)
    buf = torch.zeros(M * K + 8, dtype=torch.bfloat16, device="cuda")
    xs = buf[shift:shift + M * K].view(M, K)
    xs.copy_(_dev(x))
    y = _bits(g.mxfp4_gemv(xs, nib, sc, _dev(bias), N, K))
    ref = orc.mxfp4_gemv(x, packed, scales, bias, N, K)
    nan = np.isnan(orc.bf16_to_f32(ref))
    assert np.array_equal(np.isnan(orc.bf16_to_f32(y)), nan)
    assert np.array_equal(y[~nan], ref[~nan])


# scales off a dword (no alignment is asked of them), with x on and off one
@pytest.mark.parametrize("N,K", [(64, 96), (128, 960), (64, 2048)])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_gemv_scales_unaligned(N, K, off):
    rng = np.random.default_rng([N, K])
    M = 5
    x = moe_data.bf16(rng.normal(0, 1, (M, K)))
    packed = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    scales = rng.integers(119, 124, (N, K // 32), dtype=np.uint8)
    nib, sc = g.pack_tiled(_dev(packed), _dev(scales), N, K)
    moved = torch.zeros(sc.numel() + 8, dtype=torch.uint8, device="cuda")[off:off + sc.numel()]
    moved.copy_(sc.flatten())
    ref = orc.mxfp4_gemv(x, packed, scales, None, N, K)
    for shift in (0, 1):
        assert np.array_equal(_bits(g.mxfp4_gemv(_shifted(x, shift), nib, moved, None, N, K)), ref)


# top-k and plan in one launch up to 64 tokens, plan in one work-group up to
# 4096 slots, over the chip above
@pytest.mark.parametrize("E,k", [(30, 4), (64, 8), (128, 4)])
@pytest.mark.parametrize("T", [63, 64, 65, 255, 257, 512, 513, 1024, 1025])
def test_layer_plan(E, k, T):
    H = I = 128
    w = moe_data.make_layer(3, E, H, I, bias="random")
    x, res = moe_data.make_tokens(T, T, H)
    cfg = g.default_config(E, T)
    cfg.hidden_size, cfg.intermediate_size, cfg.top_k = H, I, k
    t = {n: _dev(v) for n, v in w.items()}
    layer = g.MoELayer().init(cfg, 0, t["router_w"], t["router_b"], t["w1_bias"], t["w2_bias"],
                              mlp1=([t["w1_packed"][e] for e in range(E)], [t["w1_scales"][e] for e in range(E)]),
                              mlp2=([t["w2_packed"][e] for e in range(E)], [t["w2_scales"][e] for e in range(E)]))
    layer.forward_prenormed(_dev(x), _dev(res))
    torch.cuda.synchronize()
    tr = layer.trace()

    def read(p, n, dt=torch.int32):
        return g.copy_device_to_tensor(p, n * 4, dt).cpu().numpy()

    S = T * k
    idx = read(tr.expert_indices, S).reshape(T, k)
    logits = g.copy_device_to_tensor(tr.logits, T * E * 2, torch.bfloat16).view(T, E)
    ri, rw = g.topk_softmax(logits, k)
    assert np.array_equal(idx, ri.cpu().numpy())
    assert np.array_equal(read(tr.expert_weights, S), rw.cpu().view(torch.int32).numpy().ravel())
    order = np.argsort(idx.ravel(), kind="stable")
    counts = np.bincount(idx.ravel(), minlength=E)
    gmap = np.empty(S, np.int32)
    gmap[order] = np.arange(S)
    act = np.flatnonzero(counts)
    assert np.array_equal(read(tr.expert_counts, E), counts)
    assert np.array_equal(read(tr.expert_offsets, E + 1), np.concatenate([[0], np.cumsum(counts)]))
    assert np.array_equal(read(tr.gather_map, S), gmap)
    assert np.array_equal(read(tr.perm_token, S), order // k)
    assert read(tr.n_active, 1)[0] == act.size and np.array_equal(read(tr.active_experts, E)[:act.size], act)
    layer.destroy()


# a plan's tensors are a caller's to write, resize and index with: they share
# neither memory nor a version counter
def test_plan_tensors_are_separate():
    idx = torch.randint(0, 30, (7, 4), dtype=torch.int32, device="cuda")
    p = g.permute_plan(idx, 30)
    assert len({t.untyped_storage().data_ptr() for t in p.values()}) == len(p)
    x = torch.randn((7, 8), device="cuda", requires_grad=True)
    rows = x[p["perm_token"]]
    p["active"].fill_(0)
    rows.sum().backward()
    assert torch.equal(x.grad, torch.full_like(x, 4.0))


# exact decode under skewed routing, token for token the bits of a batch of
# one: K-parts of an odd and an even number of blocks, one to six of them; one
# row per lane or two; experts from one token to all of them, more records than
# one wave holds
@pytest.mark.parametrize("E,k,H,I", [(1, 1, 128, 64), (30, 4, 448, 192), (200, 4, 128, 64), (8, 2, 2880, 960)])
@pytest.mark.parametrize("T", [1, 2, 3, 17, 64, 150])
def test_exact_steps(E, k, H, I, T):
    w = moe_data.make_layer(3, E, H, I, bias="random")
    x, res = moe_data.make_tokens(T, T, H)
    cfg = g.default_config(E, T, decode_exact=True, prefill_min_tokens=0)
    cfg.hidden_size, cfg.intermediate_size, cfg.top_k = H, I, k
    t = {n: _dev(v) for n, v in w.items()}
    layer = g.MoELayer().init(cfg, 0, t["router_w"], t["router_b"], t["w1_bias"], t["w2_bias"],
                              mlp1=([t["w1_packed"][e] for e in range(E)], [t["w1_scales"][e] for e in range(E)]),
                              mlp2=([t["w2_packed"][e] for e in range(E)], [t["w2_scales"][e] for e in range(E)]))
    rng = np.random.default_rng([E, T])
    # expert 0 of every token, the others by a steep law
    p = 1.0 / np.arange(1, E) ** 1.3
    rest = [rng.choice(np.arange(1, E), k - 1, replace=False, p=p / p.sum()) if k > 1 else [] for _ in range(T)]
    idx = _dev(np.array([[0, *r] for r in rest], dtype=np.int32))
    wts = _dev(rng.dirichlet(np.ones(k), T).astype(np.float32))
    dx, dr = _dev(x), _dev(res)
    got = _bits(layer.forward_routed(dx, idx, wts, residual=dr))
    for i in range(T):
        one = layer.forward_routed(dx[i:i + 1].contiguous(), idx[i:i + 1].contiguous(), wts[i:i + 1].contiguous(),
                                   residual=dr[i:i + 1].contiguous())
        assert np.array_equal(_bits(one)[0], got[i]), i
    layer.destroy()


# The same against the oracle: one row per lane (few slots, or all steps
# resident) and two; more first chunks than work-groups in both (64 experts, 8
# and 40 tokens at top-8); parts of 16, 8, 4, 3 and 2 blocks
@pytest.mark.parametrize("E,k,H,I", [(64, 8, 1024, 768), (6, 2, 2048, 576), (12, 4, 640, 384)])
@pytest.mark.parametrize("T", [1, 3, 8, 9, 40])
def test_exact_steps_oracle(E, k, H, I, T):
    w = moe_data.make_layer(5, E, H, I, bias="random")
    x, res = moe_data.make_tokens(T, T, H)
    idx, wts = moe_data.zipf_routing(T, T, E, k, s=0.2)
    cfg = g.default_config(E, T, decode_exact=True, prefill_min_tokens=0)
    cfg.hidden_size, cfg.intermediate_size, cfg.top_k = H, I, k
    t = {n: _dev(v) for n, v in w.items()}
    layer = g.MoELayer().init(cfg, 0, t["router_w"], t["router_b"], t["w1_bias"], t["w2_bias"],
                              mlp1=([t["w1_packed"][e] for e in range(E)], [t["w1_scales"][e] for e in range(E)]),
                              mlp2=([t["w2_packed"][e] for e in range(E)], [t["w2_scales"][e] for e in range(E)]))
    got = _bits(layer.forward_routed(_dev(x), _dev(idx), _dev(wts), residual=_dev(res)))
    assert np.array_equal(got, orc.moe_forward_routed(w, x, res, idx, wts, E, k, H, I))
    layer.destroy()


def _shifted(a, shift):
    """The rows of a on the device, `shift` elements past a 16-byte boundary."""
    t = _dev(a)
    buf = torch.zeros(t.numel() + 16, dtype=t.dtype, device="cuda")
    v = buf[shift:shift + t.numel()].view(t.shape)
    v.copy_(t)
    return v


# 16-byte pieces or one output per thread; dropped slots; every top-k
@pytest.mark.parametrize("T,H,k", [(1, 8, 1), (5, 20, 3), (33, 64, 8), (257, 2888, 4)])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("residual", [True, False])
def test_combine_forms(T, H, k, shift, residual):
    rng = np.random.default_rng([T, H, k])
    S = T * k
    y, res = moe_data.bf16(rng.normal(0, 1, (S, H))), moe_data.bf16(rng.normal(0, 1, (T, H)))
    gm = rng.permutation(S).astype(np.int32)
    if S > 4:
        gm[rng.choice(S, S // 5, replace=False)] = -1
    w = rng.dirichlet(np.ones(k), T).astype(np.float32)
    got = _bits(g.combine(_shifted(y, shift), _dev(gm), _dev(w), _dev(res) if residual else None, T, H, k))
    assert np.array_equal(got, orc.combine(y, gm, w, res if residual else None, T, k, H))
