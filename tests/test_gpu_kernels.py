"""Per-kernel parity on the GPU: each C-ABI entry point against the CPU oracle.

Integer outputs (router ids, counts, offsets, permutations, fp8 bytes) must be
bit-exact.  GEMM outputs are compared with the oracle's fp32 math on the same
bf16 inputs; the tolerance covers bf16 storage of the result (2^-8 relative) and
fp32 accumulation-order differences.
"""
import math

import numpy as np
import pytest
import torch

import oracle
from easyinfra_amd import ops

pytestmark = pytest.mark.gpu


def cpu(t):
    return t.detach().cpu()


def _distinct_ids(T, E, k, gen, weights=None):
    if weights is None:
        return torch.rand(T, E, generator=gen).argsort(dim=1)[:, :k].to(torch.int32)
    return torch.multinomial(weights.expand(T, E), k, replacement=False, generator=gen).to(torch.int32)


# --------------------------------------------------------------------------- router
@pytest.mark.parametrize("T,E,k,renorm", [
    (1, 8, 2, True), (37, 8, 2, True), (512, 8, 2, True), (257, 64, 6, False), (100, 128, 8, True),
    (64, 16, 4, True), (33, 32, 3, False), (10, 256, 8, True), (5, 512, 32, True), (3, 5, 5, True),
    (300, 100, 1, False),
])
def test_router_topk_matches_oracle(dev, T, E, k, renorm):
    g = torch.Generator().manual_seed(T * 1000 + E)
    logits = torch.randn(T, E, generator=g) * 2.0
    ids, w = ops.router_topk(logits.to(dev), k, renorm)
    rid, rw = oracle.route_topk(logits, k, renorm)
    assert torch.equal(cpu(ids), rid)
    torch.testing.assert_close(cpu(w), rw, rtol=3e-6, atol=1e-7)


def test_router_ties_go_to_lower_expert(dev):
    logits = torch.tensor([[1., 1., 1., 1., 0., 0., 0., 0.],
                           [0., 2., 2., 0., 2., 0., 0., 0.],
                           [-1., -1., -1., -1., -1., -1., -1., -1.],
                           [0., 0., 0., 0., 0., 0., 3., 3.]])
    ids, w = ops.router_topk(logits.to(dev), 3, True)
    assert cpu(ids).tolist() == [[0, 1, 2], [1, 2, 4], [0, 1, 2], [6, 7, 0]]
    rid, rw = oracle.route_topk(logits, 3, True)
    assert torch.equal(cpu(ids), rid)
    torch.testing.assert_close(cpu(w), rw, rtol=3e-6, atol=1e-7)


def test_router_empty(dev):
    ids, w = ops.router_topk(torch.empty(0, 8, device=dev), 2)
    assert ids.shape == (0, 2) and w.shape == (0, 2)


# --------------------------------------------------------------------------- DeepSeek-V3 gate
@pytest.mark.parametrize("T,E,k,ng,tg,norm,scale,use_bias", [
    (1, 256, 8, 8, 4, True, 2.5, True), (300, 256, 8, 8, 4, True, 2.5, True), (257, 64, 6, 1, 1, True, 2.446, False),
    (33, 512, 32, 256, 16, True, 1.5, True), (5, 16, 3, 4, 2, False, 2.5, True), (40, 100, 6, 10, 3, True, 1.0, True),
    (7, 8, 8, 4, 4, True, 1.0, False)])
def test_router_grouped_matches_oracle(dev, T, E, k, ng, tg, norm, scale, use_bias):
    g = torch.Generator().manual_seed(T * 7 + E)
    logits = torch.randn(T, E, generator=g) * 2.0
    bias = torch.randn(E, generator=g) * 0.1 if use_bias else None
    ids, w = ops.router_grouped_topk(logits.to(dev), k, ng, tg, None if bias is None else bias.to(dev), norm, scale)
    rid, rw = oracle.route_grouped_topk(logits, k, ng, tg, bias, norm, scale)
    assert torch.equal(cpu(ids), rid)
    torch.testing.assert_close(cpu(w), rw, rtol=2e-6, atol=1e-7)


def test_router_grouped_ties_and_masked_zeros(dev):
    # integer logits: equal scores everywhere (ties to the lower group / expert); the second
    # row makes every kept score negative so experts masked to 0.0 are picked
    logits = torch.tensor([[1., 1., 2., 2., 1., 1., 2., 2., 0., 0., 0., 0., 2., 2., 1., 1.],
                           [-4.] * 16])
    bias = torch.cat([torch.zeros(16)]) - 0.5
    for ng, tg, k in [(4, 2, 3), (8, 1, 5), (2, 1, 4)]:
        ids, w = ops.router_grouped_topk(logits.to(dev), k, ng, tg, bias.to(dev), True, 1.0)
        rid, rw = oracle.route_grouped_topk(logits, k, ng, tg, bias, True, 1.0)
        assert torch.equal(cpu(ids), rid), (ng, tg, k)
        torch.testing.assert_close(cpu(w), rw, rtol=2e-6, atol=1e-7)


# The token-per-row kernel (64, 128 or 256 experts in up to 16 groups, a power of two, 16-byte aligned
# logits) against the wave-wide one, which takes the same logits off alignment: bit for bit, with ties,
# infinities and NaN, ragged token counts, every group count and both pick slots.
@pytest.mark.parametrize("E", [64, 128, 256])
@pytest.mark.parametrize("ng", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("T,k,norm,use_bias", [(1, 1, True, True), (67, 16, False, False), (1024, 8, True, True),
                                               (1027, 32, True, True)])
def test_router_grouped_row_kernel_bit_identical(dev, E, ng, T, k, norm, use_bias):
    g = torch.Generator().manual_seed(E + ng + T)
    logits = torch.randn(T, E, generator=g) * 2.0
    logits[T // 2] = torch.randint(-2, 3, (E,), generator=g).float()
    logits[T - 1, ::7] = float("inf")
    logits[0, 1::5] = -float("inf")
    if T > 3:
        logits[2, ::3] = float("nan")
        logits[3] = float("nan")
    bias = (torch.randn(E, generator=g) * 0.1).to(dev) if use_bias else None
    buf = torch.empty(T * E + 1, device=dev)
    buf[1:] = logits.reshape(-1).to(dev)
    tg = max(1, ng // 2)
    ids0, w0 = ops.router_grouped_topk(buf[1:].view(T, E), k, ng, tg, bias, norm, 2.5)
    ids1, w1 = ops.router_grouped_topk(logits.to(dev), k, ng, tg, bias, norm, 2.5)
    assert torch.equal(cpu(ids0), cpu(ids1))
    assert torch.equal(cpu(w0).view(torch.int32), cpu(w1).view(torch.int32))


def test_router_grouped_empty(dev):
    ids, w = ops.router_grouped_topk(torch.empty(0, 64, device=dev), 6, 8, 4)
    assert ids.shape == (0, 6)


# --------------------------------------------------------------------------- EPLB replica map
@pytest.mark.parametrize("L,ep,P,T,k", [(8, 2, 5, 3, 2), (64, 4, 20, 500, 6), (256, 8, 40, 1000, 8), (128, 1, 128, 7, 8)])
def test_eplb_map_matches_oracle(dev, L, ep, P, T, k):
    _, log2phy, count = ops.eplb_default_layout(L, ep, P)
    g = torch.Generator().manual_seed(L + T)
    ids = torch.randint(0, L, (T, k), generator=g, dtype=torch.int32)
    ids[0, 0] = -1                                   # out of range -> -1
    ids[-1, -1] = L
    want = oracle.eplb_map(ids, log2phy, count)
    got = ops.eplb_map(ids.to(dev), log2phy.to(dev), count.to(dev))
    assert torch.equal(cpu(got), want)
    inplace = ids.to(dev)
    ops.eplb_map(inplace, log2phy.to(dev), count.to(dev), out=inplace)
    assert torch.equal(cpu(inplace), want)


# --------------------------------------------------------------------------- MoE prologue
# One pass for small routers (gate staged in LDS; the 8 x 7168 gate is 114 KiB), the MFMA
# router GEMM for E a multiple of 64 (Qwen3 128, DeepSeek-V3 256), its H split into 1-8 fp32
# planes (4096 x 256: 8 planes; 257 x 256 in 16 x 64 tiles: 8; 16384 x 128: 4; 4100 x 192: none).
@pytest.mark.parametrize("T,H,E,lbf16", [(1, 4096, 8, True), (300, 4096, 8, True), (257, 2048, 16, True),
                                         (64, 7168, 8, False), (33, 64, 32, True), (100, 2048, 128, True),
                                         (257, 7168, 256, False), (1, 4096, 64, True), (4096, 7168, 256, False),
                                         (16384, 2048, 128, True), (8192, 4096, 8, True), (4100, 1024, 192, False)])
def test_moe_prologue_matches_oracle(dev, T, H, E, lbf16):
    g = torch.Generator().manual_seed(T + H + E)
    hid = (torch.randn(T, H, generator=g) * 2).to(torch.bfloat16)
    res = (torch.randn(T, H, generator=g) * 3).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16)
    gw = (0.05 * torch.randn(E, H, generator=g)).to(torch.bfloat16)
    r, normed, logits = ops.moe_prologue(hid.to(dev), res.to(dev), w.to(dev), 1e-6, gw.to(dev), lbf16)
    rr, rn, rl = oracle.moe_prologue(hid, res, w, 1e-6, gw, lbf16)
    assert torch.equal(cpu(r), rr)                                   # the bf16 add is exact
    # the fp32 mean of squares sums in another order: bf16(r * rsqrt) may flip by one ulp, and
    # that ulp carried through the second rounding, bf16(w * t), is at most two ulps of normed
    n, ref = cpu(normed).float(), rn.float()
    assert (n == ref).float().mean() > 0.995
    assert bool(((n - ref).abs() <= ref.abs() * 2.0 ** -6 + 1e-30).all())
    # the router dots are checked on the kernel's own normed rows (float64 reference), so the
    # normed rounding differences above do not leak into this comparison
    l64 = cpu(normed).double() @ gw.double().T
    lg = cpu(logits).double()
    if lbf16:
        exact = l64.float().to(torch.bfloat16).double()
        assert (lg == exact).float().mean() > 0.98
        assert bool(((lg - exact).abs() <= exact.abs() * 2.0 ** -7 + 1e-6).all())
    else:
        torch.testing.assert_close(lg, l64, rtol=1e-5, atol=1e-5)
    assert rl.shape == lg.shape


def test_moe_prologue_in_place_residual(dev):
    g = torch.Generator().manual_seed(9)
    hid = torch.randn(40, 512, generator=g).to(torch.bfloat16).to(dev)
    res = torch.randn(40, 512, generator=g).to(torch.bfloat16).to(dev)
    w = torch.ones(512, dtype=torch.bfloat16, device=dev)
    gw = (0.1 * torch.randn(8, 512, generator=g)).to(torch.bfloat16).to(dev)
    want = ops.moe_prologue(hid, res, w, 1e-6, gw)
    r, n, l = ops.moe_prologue(hid, res, w, 1e-6, gw, residual_out=res)   # residual updated in place
    assert r.data_ptr() == res.data_ptr()
    assert torch.equal(res, want[0]) and torch.equal(n, want[1]) and torch.equal(l, want[2])


# --------------------------------------------------------------------------- align
@pytest.mark.parametrize("T,k,E,e_lo,n_loc,skew", [
    (1, 2, 8, 0, 8, False), (512, 2, 8, 0, 8, False), (8192, 2, 8, 0, 8, False), (4096, 6, 64, 0, 64, True),
    (2048, 8, 128, 0, 32, True), (2048, 8, 128, 32, 32, False), (1000, 8, 128, 96, 32, False), (7, 3, 5, 1, 3, False),
    (3, 1, 1, 0, 1, False), (16384, 8, 512, 0, 512, False),
])
def test_align_bit_exact(dev, T, k, E, e_lo, n_loc, skew):
    g = torch.Generator().manual_seed(T + 7 * E + e_lo)
    wts = (1.0 / torch.arange(1, E + 1, dtype=torch.float32) ** 1.2) if skew else None
    ids = _distinct_ids(T, E, k, g, wts)
    got = ops.align(ids.to(dev), n_loc, e_lo)
    ref = oracle.align(ids.numpy(), n_loc, e_lo)
    A = int(ref["offsets"][-1])
    assert np.array_equal(cpu(got["counts"]).numpy(), ref["counts"])
    assert np.array_equal(cpu(got["offsets"]).numpy(), ref["offsets"])
    assert np.array_equal(cpu(got["sorted_flat"])[:A].numpy(), ref["sorted_flat"])
    assert np.array_equal(cpu(got["sorted_tok"])[:A].numpy(), ref["sorted_tok"])
    assert np.array_equal(cpu(got["pos"]).numpy(), ref["pos"])


# From 4096 routed pairs the sort runs over many workgroups (chunk counts, then placement);
# it must equal the one-workgroup kernel and the oracle bit for bit, including chunks that
# end mid-row, every id on one expert, window filtering and the largest expert count.
@pytest.mark.parametrize("T,k,E,e_lo,n_loc,mode", [
    (4096, 1, 8, 0, 8, "uniform"), (4097, 1, 16, 0, 16, "uniform"), (2731, 3, 64, 16, 32, "uniform"),
    (3000, 8, 128, 0, 32, "one"), (16384, 8, 512, 0, 512, "uniform"), (65536, 2, 8, 0, 8, "skew"),
    (5000, 6, 64, 0, 64, "skew"),
])
def test_align_many_workgroups_bit_exact(dev, T, k, E, e_lo, n_loc, mode):
    g = torch.Generator().manual_seed(T + k)
    if mode == "one":
        ids = torch.full((T, k), e_lo + 3, dtype=torch.int32)
        ids[:, 1:] = torch.arange(1, k, dtype=torch.int32) + E // 2   # the other slots: distinct, off-window
    else:
        wts = (1.0 / torch.arange(1, E + 1, dtype=torch.float32) ** 1.2) if mode == "skew" else None
        ids = _distinct_ids(T, E, k, g, wts)
    many = ops.align(ids.to(dev), n_loc, e_lo)
    one = ops.align(ids.to(dev), n_loc, e_lo, one_workgroup=True)
    ref = oracle.align(ids.numpy(), n_loc, e_lo)
    A = int(ref["offsets"][-1])
    for got in (many, one):
        assert np.array_equal(cpu(got["counts"]).numpy(), ref["counts"])
        assert np.array_equal(cpu(got["offsets"]).numpy(), ref["offsets"])
        assert np.array_equal(cpu(got["sorted_flat"])[:A].numpy(), ref["sorted_flat"])
        assert np.array_equal(cpu(got["sorted_tok"])[:A].numpy(), ref["sorted_tok"])
        assert np.array_equal(cpu(got["pos"]).numpy(), ref["pos"])


def test_align_all_to_one_expert_and_repeats(dev):
    ids = torch.full((300, 4), 3, dtype=torch.int32)
    ids[::7, 1] = 0
    got = ops.align(ids.to(dev), 5, 0)
    ref = oracle.align(ids.numpy(), 5, 0)
    A = int(ref["offsets"][-1])
    for key in ("counts", "offsets", "pos"):
        assert np.array_equal(cpu(got[key]).numpy(), ref[key]), key
    assert np.array_equal(cpu(got["sorted_flat"])[:A].numpy(), ref["sorted_flat"])


def test_align_out_of_window_ids_dropped(dev):
    ids = torch.tensor([[0, 9], [5, 2], [7, 8]], dtype=torch.int32)
    got = ops.align(ids.to(dev), 4, 2)
    ref = oracle.align(ids.numpy(), 4, 2)
    # window [2,6): id 2 -> local 0 (flat 3), id 5 -> local 3 (flat 2)
    assert cpu(got["counts"]).tolist() == [1, 0, 0, 1] == ref["counts"].tolist()
    assert cpu(got["pos"]).tolist() == [-1, -1, 1, 0, -1, -1]


# --------------------------------------------------------------------------- route + align
# Batches small enough for the one-workgroup kernel (up to 2 routing steps of 16 waves:
# 256 tokens at E <= 8, 128 at E <= 128, 64 at E <= 256) and ones just past it (two kernels).
@pytest.mark.parametrize("T,E,k,e_lo,n_loc,renorm", [
    (1, 8, 2, 0, 8, True), (64, 8, 2, 0, 8, True), (256, 8, 2, 0, 8, True), (257, 8, 2, 0, 8, True),
    (32, 128, 8, 0, 32, True), (128, 128, 8, 32, 32, True), (129, 128, 8, 0, 32, True), (60, 64, 6, 0, 64, False),
    (7, 256, 16, 50, 100, True), (64, 200, 20, 0, 200, False), (3, 300, 4, 0, 300, True), (5, 16, 1, 3, 1, True),
    # at most 64 routed pairs: the one-wave sort
    (1, 128, 8, 0, 32, True), (8, 128, 8, 32, 32, True), (3, 256, 8, 0, 256, False), (5, 64, 6, 16, 16, True),
    (32, 8, 2, 0, 8, True), (1, 8, 2, 6, 2, False), (4, 256, 16, 0, 256, True),
    # larger batches: the router, then the one-workgroup align (this entry takes no workspace; the
    # layer's many-workgroup paths are checked through its routing ids and outputs)
    (600, 128, 8, 0, 32, True), (8192, 8, 2, 0, 8, True), (1536, 128, 8, 32, 32, True),
    (2048, 128, 8, 0, 32, True), (2040, 128, 8, 96, 32, False),
])
def test_route_align_bit_exact(dev, T, E, k, e_lo, n_loc, renorm):
    g = torch.Generator().manual_seed(T * 31 + E)
    logits = torch.randn(T, E, generator=g) * 2.0
    logits[0, :4] = 1.5                                    # ties go to the lower id
    ids, w, got = ops.route_align(logits.to(dev), k, n_loc, e_lo, renorm)
    rid, rw = oracle.route_topk(logits, k, renorm)
    assert torch.equal(cpu(ids), rid)
    torch.testing.assert_close(cpu(w), rw, rtol=3e-6, atol=1e-7)
    ref = oracle.align(rid.numpy(), n_loc, e_lo)
    A = int(ref["offsets"][-1])
    for key in ("counts", "offsets", "pos"):
        assert np.array_equal(cpu(got[key]).numpy(), ref[key]), key
    assert np.array_equal(cpu(got["sorted_flat"])[:A].numpy(), ref["sorted_flat"])
    assert np.array_equal(cpu(got["sorted_tok"])[:A].numpy(), ref["sorted_tok"])


# A token or two over 16+ experts (T*E <= 256) route by rank inside the route+align kernel: each
# value's pick slot is the number of values beating it.  Same ids in the same order as the
# router's k argmax rounds, on rows full of ties, +-inf and NaN (NaN never picked; slots past a
# row's non-NaN values hold 0x7fffffff), and bit-identical weights up to 128 experts (the same
# 16-lane summation); above, within the router tests' tolerance.
@pytest.mark.parametrize("T,E,k,renorm", [(1, 128, 8, True), (2, 128, 8, False), (1, 128, 8, False),
                                          (4, 64, 6, True), (16, 16, 4, False), (1, 256, 8, True),
                                          (2, 32, 32, True), (8, 32, 4, True)])
def test_route_align_rank_selection_matches_router(dev, T, E, k, renorm):
    g = torch.Generator().manual_seed(T * 7 + E)
    logits = torch.round(torch.randn(T, E, generator=g) * 2.0)   # a handful of distinct values per row
    logits[1::3, ::7] = float("inf")
    logits[2::3, 3::11] = -float("inf")
    if T > 1:
        logits[1, : E - 3] = float("nan")                         # fewer than k non-NaN values
    ids, w, _ = ops.route_align(logits.to(dev), k, E, 0, renorm)
    rid, rw = ops.router_topk(logits.to(dev), k, renorm)
    assert torch.equal(cpu(ids), cpu(rid))
    if E <= 128:
        torch.testing.assert_close(cpu(w), cpu(rw), rtol=0, atol=0, equal_nan=True)
    fin = torch.isfinite(logits).all(dim=1)
    if bool(fin.any()):
        oid, ow = oracle.route_topk(logits[fin], k, renorm)
        assert torch.equal(cpu(ids)[fin], oid)


def test_route_align_empty(dev):
    ids, w, got = ops.route_align(torch.empty(0, 8, device=dev), 2, 8)
    assert ids.shape == (0, 2) and cpu(got["offsets"]).tolist() == [0] * 9


# --------------------------------------------------------------------------- gather / combine
def test_gather_rows(dev):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(50, 256, generator=g).to(torch.bfloat16)
    rows = torch.randint(0, 50, (70,), generator=g, dtype=torch.int32)
    n = torch.tensor([61], dtype=torch.int32)
    xs = ops.gather(x.to(dev), rows.to(dev), n.to(dev), 70)
    assert torch.equal(cpu(xs)[:61], x[rows[:61].long()])


@pytest.mark.parametrize("y_dtype,out_dtype,n_split", [(torch.float32, torch.float32, 1), (torch.bfloat16, torch.bfloat16, 1),
                                                        (torch.float32, torch.bfloat16, 3)])
def test_combine_matches_index_add(dev, y_dtype, out_dtype, n_split):
    g = torch.Generator().manual_seed(11)
    T, k, E, H = 97, 3, 6, 128
    ids = _distinct_ids(T, E, k, g)
    al = oracle.align(ids.numpy(), 4, 1)           # experts 1..4 local: some slots dropped
    A = int(al["offsets"][-1])
    w = torch.rand(T, k, generator=g)
    y = torch.randn(n_split, A, H, generator=g).to(y_dtype)
    sh = torch.randn(T, H, generator=g)
    got = ops.combine(y.to(dev), torch.as_tensor(al["pos"]).to(dev), w.to(dev), shared_y=sh.to(dev),
                      out_dtype=out_dtype)
    tok = torch.as_tensor(al["sorted_tok"]).long()
    slot = torch.as_tensor(al["sorted_slot"]).long()
    ref = torch.zeros(T, H)
    ref.index_add_(0, tok, y.float().sum(0) * w[tok, slot][:, None])
    ref += sh
    tol = 1e-5 if out_dtype == torch.float32 else 8e-3
    torch.testing.assert_close(cpu(got).float(), ref, rtol=tol, atol=tol)


# Batches of up to 512 tokens with slot and split counts up to 8 loads per output vector take a kernel
# with both fixed (all of a token's loads in flight at once); others the general loop.  Same sums in the same order: a third
# plane of zeros sends the two-plane case through the general kernel, bit for bit the same output
# (top-1, 2, 4, 6, 8 with 1 or 2 planes, with and without shared-expert planes, fp32 and bf16 out).
@pytest.mark.parametrize("k,n_split", [(1, 1), (2, 1), (2, 2), (4, 2), (6, 1), (8, 1)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_combine_fixed_counts_bit_exact_with_general_loop(dev, k, n_split, out_dtype):
    g = torch.Generator().manual_seed(100 * k + n_split)
    T, E, H = 301, 12, 256
    ids = _distinct_ids(T, E, k, g)
    al = oracle.align(ids.numpy(), 9, 2)            # experts 2..10 local: some slots dropped
    A = int(al["offsets"][-1])
    w = torch.rand(T, k, generator=g)
    y = torch.randn(n_split, A, H, generator=g)
    pos = torch.as_tensor(al["pos"]).to(dev)
    for sh in (None, torch.randn(T, H, generator=g).to(dev)):
        fixed = ops.combine(y.to(dev), pos, w.to(dev), shared_y=sh, out_dtype=out_dtype)
        y3 = torch.cat([y, torch.zeros(3 - n_split if n_split < 3 else 1, A, H)]).to(dev)
        general = ops.combine(y3, pos, w.to(dev), shared_y=sh, out_dtype=out_dtype)
        assert torch.equal(cpu(fixed), cpu(general))


# --------------------------------------------------------------------------- GEMMs
def _segments(counts):
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    return off, torch.as_tensor(off)


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("counts", [[0, 5, 300, 1, 64], [17], [0, 0, 3]])
def test_gate_up_silu(dev, tile, counts):
    g = torch.Generator().manual_seed(sum(counts) + tile)
    H, I = 256, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 40
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (max(rows, 1),), generator=g, dtype=torch.int32)
    w = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    h = ops.gemm_gate_up_silu(x.to(dev), w.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev), tile=tile)
    h = cpu(h).float()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        xs = x[a_rows[a:b].long()].float()
        gu = xs @ w[e].float().T
        ref = oracle.silu(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], ref, rtol=1e-2, atol=1e-2)


# silu(g) = g * rcp(1 + exp(-g)) in the epilogues (the hardware reciprocal): gate values where
# exp(-g) overflows (g <= -89: rcp(inf) = 0, h = -0), where the reciprocal is subnormal (g = -88),
# and where it is 1 (large g).  x rows are one-hot scalings, so g is an exact product of bf16
# values; h is compared with the float64 silu on those g (bf16 output rounding, tiny values
# flushed to zero allowed).
@pytest.mark.parametrize("tile", [1, 2, 5])
def test_gate_up_silu_extreme_gates(dev, tile):
    gates = [-200.0, -100.0, -90.0, -88.0, -20.0, -1.0, -1e-3, 0.0, 1e-3, 1.0, 20.0, 88.0, 90.0, 100.0, 200.0, 3.0]
    H, I, R = 64, 256, 40
    w = torch.zeros(1, 2 * I, H)
    for n in range(I):
        w[0, n, 0] = gates[n % len(gates)]
        w[0, I + n, 0] = 1.0 + (n % 3)
    scales = [1.0, 0.5, 2.0, -1.0]
    x = torch.zeros(R, H)
    for r in range(R):
        x[r, 0] = scales[r % len(scales)]
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    off_t = torch.tensor([0, R], dtype=torch.int32)
    h = ops.gemm_gate_up_silu(x.to(dev), w.to(dev), off_t.to(dev), R, tile=tile)
    h = cpu(h).double()
    gu = x.double() @ w[0].double().T
    g, u = gu[:, :I], gu[:, I:]
    ref = g * torch.sigmoid(g) * u
    assert torch.isfinite(h).all()
    assert ((h - ref).abs() <= 1e-2 * ref.abs() + 1e-6).all(), (h - ref).abs().max()


@pytest.mark.parametrize("tile,k_split", [(1, 1), (2, 1), (3, 1), (4, 1), (3, 2), (4, 4), (5, 1), (5, 2), (5, 8),
                                          (6, 1), (6, 2)])
def test_down_gemm(dev, tile, k_split):
    g = torch.Generator().manual_seed(31 + tile * 7 + k_split)
    H, I = 256, 512
    counts = [3, 0, 257, 40]
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    h = torch.randn(rows, I, generator=g).to(torch.bfloat16)
    w = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16)
    y = ops.gemm_down(h.to(dev), w.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, k_split=k_split, tile=tile)
    y = cpu(y).sum(0)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        ref = h[a:b].float() @ w[e].float().T
        torch.testing.assert_close(y[a:b], ref, rtol=1e-4, atol=1e-4)


# The 256x256 GEMM runs as a persistent kernel for launches of at most 64 segments and as one
# tile per workgroup beyond that.  Padding the same segments with empty ones switches kernels
# without changing any tile (empty segments own no tiles), so the two must agree bit for bit:
# full, half (129 rows) and quarter (1, 44, 64 rows) height tiles, gathered rows, split K, and
# enough tiles that every persistent workgroup walks several.
@pytest.mark.parametrize("w8a8,n_seg", [(False, 8), (True, 8), (False, 64), (True, 64)])
def test_persistent_gemm_bit_exact_with_one_tile_kernel(dev, w8a8, n_seg):
    g = torch.Generator().manual_seed(77 + w8a8 + n_seg)
    H, I, T = 512, 512, 600   # down K split 2 keeps whole 128-byte e4m3 slabs
    if n_seg == 8:
        counts = [300, 0, 1, 513, 64, 129, 700, 44]
    else:   # exactly 64 segments, the persistent kernel's limit (one per lane of its schedule)
        counts = torch.randint(0, 300, (n_seg,), generator=g).tolist()
        counts[5] = 0
        counts[63] = 257
    E = len(counts)
    off, off_t = _segments(counts)
    off_pad = np.concatenate([off, np.full(65 - E if E == 64 else 64, off[-1], dtype=np.int32)])
    assert len(off_pad) - 1 > 64
    off_t, off_pad_t = off_t.to(dev), torch.as_tensor(off_pad).to(dev)
    rows = int(off[-1])
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32).to(dev)
    w_gu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    w_d = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    hs = torch.randn(rows, I, generator=g).to(torch.bfloat16).to(dev)
    if w8a8:
        xq, sx = ops.quantize_rows_fp8(x)
        qgu, sgu = ops.quantize_weights_fp8(w_gu)
        qd, sd = ops.quantize_weights_fp8(w_d)
        hq, sh = ops.quantize_rows_fp8(hs)
        gu = lambda o: ops.gemm_gate_up_silu_w8a8(xq, sx, qgu, sgu, o, rows, a_rows=a_rows, e_mod=E, tile=1)
        dn = lambda o, ks: ops.gemm_down_w8a8(hq, sh, qd, sd, o, rows, k_split=ks, e_mod=E, tile=1)
    else:
        gu = lambda o: ops.gemm_gate_up_silu(x, w_gu, o, rows, a_rows=a_rows, e_mod=E, tile=1)
        dn = lambda o, ks: ops.gemm_down(hs, w_d, o, rows, out_dtype=torch.float32, k_split=ks, e_mod=E, tile=1)
    assert torch.equal(cpu(gu(off_t)), cpu(gu(off_pad_t)))
    for ks in (1, 2):
        assert torch.equal(cpu(dn(off_t, ks)), cpu(dn(off_pad_t, ks)))


def _carve_above_bit31(dev, tensors):
    """Copies of `tensors` inside one device allocation, at addresses with bit 31 set and no 4 GiB
    boundary inside the block: a slice of a plain allocation a little over 2 GiB always holds such a
    window.  Returns (the allocation, the copies)."""
    sizes = [(t.numel() * t.element_size() + 255) // 256 * 256 for t in tensors]
    need = sum(sizes)
    big = torch.empty(2 ** 31 + 2 * need + 512, dtype=torch.uint8, device=dev)
    base = big.data_ptr()
    c = (base + 255) // 256 * 256
    while not ((c >> 31) & 1 and (c % 2 ** 32) + need <= 2 ** 32):
        c = (c | (2 ** 31 - 1)) + 1 if not (c >> 31) & 1 else (c | (2 ** 32 - 1)) + 1 + 2 ** 31
    assert c + need <= base + big.numel()
    out, o = [], c - base
    for t, n in zip(tensors, sizes):
        v = big[o:o + t.numel() * t.element_size()].view(t.dtype).view(t.shape)
        v.copy_(t)
        assert (v.data_ptr() >> 31) & 1
        out.append(v)
        o += n
    return big, out


# Operands whose base address has bit 31 set, on the persistent 256x256 kernel: it takes its buffer
# bases from the first lane as two 32-bit halves, and a sign-extended low half would turn such a
# base into 0xffffffff........  The same GEMMs on ordinary buffers must match bit for bit.
@pytest.mark.parametrize("w8a8", [False, True])
def test_persistent_gemm_operands_with_address_bit31(dev, w8a8):
    g = torch.Generator().manual_seed(41 + w8a8)
    H, I, T = 512, 512, 600
    counts = [300, 1, 513, 129, 64]
    E = len(counts)
    off, off_t = _segments(counts)
    off_t = off_t.to(dev)
    rows = int(off[-1])
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32).to(dev)
    w_gu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    w_d = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    hs = torch.randn(rows, I, generator=g).to(torch.bfloat16).to(dev)
    if w8a8:
        xq, sx = ops.quantize_rows_fp8(x)
        qgu, sgu = ops.quantize_weights_fp8(w_gu)
        qd, sd = ops.quantize_weights_fp8(w_d)
        hq, sh = ops.quantize_rows_fp8(hs)
        operands = [xq, sx, a_rows, qgu, sgu, hq, sh, qd, sd]

        def run(xq, sx, a_rows, qgu, sgu, hq, sh, qd, sd):
            return (ops.gemm_gate_up_silu_w8a8(xq, sx, qgu, sgu, off_t, rows, a_rows=a_rows, tile=1),
                    ops.gemm_down_w8a8(hq, sh, qd, sd, off_t, rows, k_split=2, tile=1))
    else:
        operands = [x, a_rows, w_gu, hs, w_d]

        def run(x, a_rows, w_gu, hs, w_d):
            return (ops.gemm_gate_up_silu(x, w_gu, off_t, rows, a_rows=a_rows, tile=1),
                    ops.gemm_down(hs, w_d, off_t, rows, out_dtype=torch.float32, k_split=2, tile=1))
    want = [cpu(t) for t in run(*operands)]
    big, high = _carve_above_bit31(dev, operands)
    got = [cpu(t) for t in run(*high)]
    torch.cuda.synchronize()
    del big, high
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# The weight-streaming kernel (tile 5) picks its column width (8/4/2 fragments), its K split
# over waves and its register ring depth (2 or 1) from the shapes, or, for grids this small,
# the short-stream mode (K split over 4 or 8 waves, at most 4 k-steps each, all in flight:
# K = 256, 512, 768, 1024, 1536, 2048 here); these cases reach every combination, rows past
# 32 per segment (several row chunks), empty and one-row segments.  Nd is the down
# projection's output width (0: not run).
@pytest.mark.parametrize("H,I,Nd", [(256, 256, 256), (192, 32, 0), (512, 96, 0), (64, 32, 0), (1408, 128, 1408),
                                    (128, 320, 64), (256, 512, 192), (2048, 768, 2048), (1024, 1536, 256)])
def test_stream_gemms_shapes(dev, H, I, Nd):
    g = torch.Generator().manual_seed(H + I + Nd)
    counts = [1, 0, 40, 7, 70]
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 50
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    h = ops.gemm_gate_up_silu(x.to(dev), wgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev), tile=5)
    if Nd:
        wd = (torch.randn(E, Nd, I, generator=g) * 0.05).to(torch.bfloat16)
        y = cpu(ops.gemm_down(h, wd.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, tile=5)).sum(0)
    h = cpu(h).float()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = x[a_rows[a:b].long()].float() @ wgu[e].float().T
        torch.testing.assert_close(h[a:b], oracle.silu(gu[:, :I]) * gu[:, I:], rtol=1e-2, atol=1e-2)
        if Nd:
            torch.testing.assert_close(y[a:b], h[a:b] @ wd[e].float().T, rtol=1e-4, atol=1e-4)


def test_grouped_gemm_single_contract(dev):
    g = torch.Generator().manual_seed(3)
    K, N = 192, 320
    blocks = [10, 0, 33, 128]
    a = torch.randn(sum(blocks), K, generator=g).to(torch.bfloat16)
    b = (torch.randn(len(blocks), N, K, generator=g) * 0.1).to(torch.bfloat16)
    off, off_t = _segments(blocks)
    c = ops.grouped_gemm(a.to(dev), b.to(dev), off_t.to(dev), sum(blocks), out_dtype=torch.float32, tile=4)
    ref = oracle.grouped_gemm(a, list(b), blocks)
    torch.testing.assert_close(cpu(c), ref, rtol=1e-4, atol=1e-4)


def test_gemm_rejects_bad_shapes(dev):
    from easyinfra_amd._lib import EimoeError
    a = torch.zeros(4, 100, dtype=torch.bfloat16, device=dev)
    w = torch.zeros(1, 64, 100, dtype=torch.bfloat16, device=dev)
    off = torch.tensor([0, 4], dtype=torch.int32, device=dev)
    with pytest.raises(EimoeError):
        ops.gemm_gate_up_silu(a, w, off, 4)


# --------------------------------------------------------------------------- fp8
@pytest.mark.parametrize("shape,dtype", [((7, 1000), torch.float32), ((64, 4096), torch.bfloat16),
                                         ((3, 5), torch.float32), ((2, 16, 96), torch.bfloat16),
                                         ((128, 14336), torch.bfloat16), ((5, 8192), torch.float32),
                                         ((9, 2052), torch.float32), ((3, 20000), torch.bfloat16),
                                         ((4, 100), torch.bfloat16)])
def test_quantize_rows_fp8_bit_exact(dev, shape, dtype):
    g = torch.Generator().manual_seed(shape[0])
    x = (torch.randn(*shape, generator=g) * 0.3).to(dtype)
    x.view(-1, shape[-1])[0, :] = 0.0                      # an all-zero row -> scale 1
    q, s = ops.quantize_rows_fp8(x.to(dev))
    rq, rs = oracle.quantize_rows_fp8(x.reshape(-1, shape[-1]))
    assert torch.equal(cpu(s).reshape(-1), rs)
    assert torch.equal(cpu(q).reshape(-1, shape[-1]).view(torch.uint8), rq.view(torch.uint8))


# W8A16 on the LDS tiles that widen e4m3 weights through registers; the small counts put each
# segment in one m-tile, so the weight DMA carries the non-temporal hint.
@pytest.mark.parametrize("tile,counts", [(2, [20, 0, 70]), (3, [20, 0, 70]), (4, [20, 0, 70]), (2, [5, 0, 12]),
                                         (3, [5, 0, 12]), (4, [5, 0, 12]), (6, [20, 0, 70]), (6, [5, 0, 12])])
def test_fp8_weight_gemms(dev, tile, counts):
    g = torch.Generator().manual_seed(tile + len(counts) * counts[0])
    H, I = 256, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    x = torch.randn(rows, H, generator=g).to(torch.bfloat16)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.02
    wd = torch.randn(E, H, I, generator=g) * 0.02
    qgu, sgu = oracle.quantize_weights_fp8(wgu)
    qd, sd = oracle.quantize_weights_fp8(wd)
    h = ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, w_scale=sgu.to(dev), tile=tile)
    y = ops.gemm_down(h, qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), tile=tile)
    h, y = cpu(h).float(), cpu(y)[0]
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = (x[a:b].float() @ qgu[e].float().T) * sgu[e]
        href = oracle.silu(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], href, rtol=1e-2, atol=1e-2)
        yref = (h[a:b] @ qd[e].float().T) * sd[e]
        torch.testing.assert_close(y[a:b], yref, rtol=1e-3, atol=1e-3)


# W8A16 on the weight-streaming kernel (tile 5): e4m3 weights widened to bf16 in registers against
# bf16 activations, 128 k per step.  The shapes reach its short-stream mode (H 256; the 1024-wide
# down projection), the 2- and 4-wave K splits with a 2-deep register ring (H 4096, 8192) and the
# unsplit ring (the 256-wide down projection); gathered rows, row chunks past 32, empty and one-row
# segments.
@pytest.mark.parametrize("H,I,counts", [(256, 256, [20, 0, 70, 1]), (4096, 1024, [40, 3, 0, 90]),
                                        (8192, 256, [33, 1, 64, 0, 7])])
def test_fp8_weight_stream_gemms(dev, H, I, counts):
    g = torch.Generator().manual_seed(H + I)
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 50
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.02
    wd = torch.randn(E, H, I, generator=g) * 0.02
    qgu, sgu = oracle.quantize_weights_fp8(wgu)
    qd, sd = oracle.quantize_weights_fp8(wd)
    h = ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev), w_scale=sgu.to(dev),
                              tile=5)
    y = ops.gemm_down(h, qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), tile=5)
    h, y = cpu(h).float(), cpu(y)[0]
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = (x[a_rows[a:b].long()].float() @ qgu[e].float().T) * sgu[e]
        href = oracle.silu(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], href, rtol=1e-2, atol=1e-2)
        yref = (h[a:b] @ qd[e].float().T) * sd[e]
        torch.testing.assert_close(y[a:b], yref, rtol=1e-3, atol=1e-3)


# W8A16 on the 256x256 ping-pong tile (e4m3 weights DMA'd to LDS, 128 k per stage, widened at
# fragment reads): quarter, half and full-height tiles and several m-tiles per segment, gathered
# rows, K of one 128-k weight chunk (H 128), of exactly one unrolled loop (6 slabs: H 384, the down
# projection's 768 split in two) and not a multiple of it (H 1024: 16 slabs; 768 unsplit: 12).
@pytest.mark.parametrize("H,I,k_split", [(128, 256, 1), (384, 256, 1), (1024, 256, 1), (512, 768, 1),
                                         (512, 768, 2)])
def test_fp8_weight_pingpong_gemms(dev, H, I, k_split):
    g = torch.Generator().manual_seed(H + I + k_split)
    counts = [257, 320, 63, 0, 129, 2 * 256 + 2, 64]
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 300
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.02
    wd = torch.randn(E, H, I, generator=g) * 0.02
    qgu, sgu = oracle.quantize_weights_fp8(wgu)
    qd, sd = oracle.quantize_weights_fp8(wd)
    hs = (torch.randn(rows, I, generator=g) * 0.5).to(torch.bfloat16)
    h = cpu(ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev),
                                  w_scale=sgu.to(dev), tile=1)).float()
    down = H % 256 == 0   # the 256x256 down tile writes 256 output columns
    if down:
        y = cpu(ops.gemm_down(hs.to(dev), qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), k_split=k_split,
                              tile=1)).sum(0)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = (x[a_rows[a:b].long()].float() @ qgu[e].float().T) * sgu[e]
        href = oracle.silu(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], href, rtol=1e-2, atol=1e-2)
        if down:
            yref = (hs[a:b].float() @ qd[e].float().T) * sd[e]
            torch.testing.assert_close(y[a:b], yref, rtol=1e-3, atol=1e-3)


# W8A16 launches that the persistent ping-pong kernel does not take (more than 64 segments: its
# schedule holds one segment per lane; K not a multiple of its 128-k weight stage) run the
# lock-step 256x256 kernel that widens the e4m3 weights through registers: 70 segments with empty
# ones and every remainder height, and K = 192 on 7 segments, against the oracle's e4m3 GEMMs (the
# down projection where its 256-column tile divides H).
@pytest.mark.parametrize("n_seg,H", [(70, 256), (7, 192)])
def test_fp8_weight_256_tile_lockstep_fallback(dev, n_seg, H):
    g = torch.Generator().manual_seed(1000 + n_seg + H)
    I = 256
    counts = torch.randint(0, 300, (n_seg,), generator=g).tolist()
    counts[3], counts[-3], counts[-1] = 0, 64, 257
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 400
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.02
    wd = torch.randn(E, H, I, generator=g) * 0.02
    qgu, sgu = oracle.quantize_weights_fp8(wgu)
    qd, sd = oracle.quantize_weights_fp8(wd)
    hs = (torch.randn(rows, I, generator=g) * 0.5).to(torch.bfloat16)
    h = cpu(ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev),
                                  w_scale=sgu.to(dev), tile=1)).float()
    down = H % 256 == 0
    if down:
        y = cpu(ops.gemm_down(hs.to(dev), qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), tile=1)).sum(0)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = (x[a_rows[a:b].long()].float() @ qgu[e].float().T) * sgu[e]
        torch.testing.assert_close(h[a:b], oracle.silu(gu[:, :I]) * gu[:, I:], rtol=1e-2, atol=1e-2)
        if down:
            yref = (hs[a:b].float() @ qd[e].float().T) * sd[e]
            torch.testing.assert_close(y[a:b], yref, rtol=1e-3, atol=1e-3)


# Segment remainders of every height class: a segment's last tile is a quarter, half or full
# tile (256x256: 64 / 128 / 256 rows; 128x128: 32 / 64 / 128; 64x128, whose two wave rows of
# 32 have no quarter: 32 / 64), and the last m-tile group of a long segment takes the leftover
# tiles (10 m-tiles of 256 rows: groups of 4 and 6; 12 of 64 rows: groups of 4, 4 and 4).
REMAINDER_COUNTS = {1: [257, 320, 321, 128, 129, 712, 63, 9 * 256 + 2, 0],
                    2: [33, 32, 64, 65, 129, 127, 11 * 128 + 7, 0, 1],
                    6: [33, 32, 64, 65, 97, 127, 11 * 64 + 7, 0, 1, 9 * 64 + 40]}


@pytest.mark.parametrize("tile", [1, 2, 6])
@pytest.mark.parametrize("k_split", [1, 2])
def test_gemms_remainder_tile_heights(dev, tile, k_split):
    counts = REMAINDER_COUNTS[tile]
    g = torch.Generator().manual_seed(77 + tile + k_split)
    H, I = 256, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 300
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16)
    h = ops.gemm_gate_up_silu(x.to(dev), wgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev), tile=tile)
    y = cpu(ops.gemm_down(h, wd.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, k_split=k_split,
                          tile=tile)).sum(0)
    h = cpu(h).float()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = x[a_rows[a:b].long()].float() @ wgu[e].float().T
        torch.testing.assert_close(h[a:b], oracle.silu(gu[:, :I]) * gu[:, I:], rtol=1e-2, atol=1e-2)
        torch.testing.assert_close(y[a:b], h[a:b] @ wd[e].float().T, rtol=1e-4, atol=1e-4)


# Every LDS tile adds the K slabs of a row in the same order on the same MFMA, so the 64x128,
# 128x128 and 32x128 tiles (and the 256x256 tile where it divides the output) agree bit for bit
# on the same segments: gathered rows, remainder heights, empty segments, K split planes.
@pytest.mark.parametrize("k_split", [1, 2])
def test_lds_tiles_bit_identical(dev, k_split):
    counts = [33, 0, 64, 65, 97, 300, 1, 7 * 64 + 5]
    g = torch.Generator().manual_seed(123 + k_split)
    H, I = 512, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 200
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32).to(dev)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    off_t = off_t.to(dev)
    hs = {t: cpu(ops.gemm_gate_up_silu(x, wgu, off_t, rows, a_rows=a_rows, tile=t)) for t in (1, 2, 3, 6)}
    for t in (1, 3, 6):
        assert torch.equal(hs[t], hs[2]), t
    h = hs[2].to(dev)
    ys = {t: cpu(ops.gemm_down(h, wd, off_t, rows, out_dtype=torch.float32, k_split=k_split, tile=t))
          for t in (1, 2, 3, 6)}
    for t in (1, 3, 6):
        assert torch.equal(ys[t], ys[2]), t


# W8A16 with K not a multiple of 128 (one 64-k weight slab left over): the LDS tiles widen the
# weights through registers instead (gate/up K = H = 192, down K = I = 192).
@pytest.mark.parametrize("tile", [2, 3, 4, 6])
def test_w8a16_lds_tiles_k_not_multiple_of_128(dev, tile):
    counts = [20, 0, 70, 5]
    g = torch.Generator().manual_seed(40 + tile)
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    Hg, Ig = 192, 256   # gate/up: K = 192
    Hd, Id = 256, 192   # down: K = 192
    x = torch.randn(rows, Hg, generator=g).to(torch.bfloat16)
    qgu, sgu = oracle.quantize_weights_fp8(torch.randn(E, 2 * Ig, Hg, generator=g) * 0.02)
    qd, sd = oracle.quantize_weights_fp8(torch.randn(E, Hd, Id, generator=g) * 0.02)
    hin = torch.randn(rows, Id, generator=g).to(torch.bfloat16)
    h = cpu(ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, w_scale=sgu.to(dev), tile=tile)).float()
    y = cpu(ops.gemm_down(hin.to(dev), qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), tile=tile))[0]
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = (x[a:b].float() @ qgu[e].float().T) * sgu[e]
        torch.testing.assert_close(h[a:b], oracle.silu(gu[:, :Ig]) * gu[:, Ig:], rtol=1e-2, atol=1e-2)
        torch.testing.assert_close(y[a:b], (hin[a:b].float() @ qd[e].float().T) * sd[e], rtol=1e-3, atol=1e-3)


# W8A16 (e4m3 weights, bf16 activations): the LDS tiles DMA the weight bytes and widen them at the
# fragment reads with the k assignment of the 256x256 ping-pong W8A16 tile, so all of them agree
# with it bit for bit (K a multiple of 128; K split planes of 128).
@pytest.mark.parametrize("k_split", [1, 2])
def test_w8a16_lds_tiles_bit_identical(dev, k_split):
    counts = [33, 0, 64, 65, 97, 300, 1, 7 * 64 + 5]
    g = torch.Generator().manual_seed(321 + k_split)
    H, I = 512, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 200
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32).to(dev)
    qgu, sgu = oracle.quantize_weights_fp8(torch.randn(E, 2 * I, H, generator=g) * 0.02)
    qd, sd = oracle.quantize_weights_fp8(torch.randn(E, H, I, generator=g) * 0.02)
    qgu, sgu, qd, sd, off_t = qgu.to(dev), sgu.to(dev), qd.to(dev), sd.to(dev), off_t.to(dev)
    hs = {t: cpu(ops.gemm_gate_up_silu(x, qgu, off_t, rows, a_rows=a_rows, w_scale=sgu, tile=t)) for t in (1, 2, 3, 4, 6)}
    for t in (2, 3, 4, 6):
        assert torch.equal(hs[t], hs[1]), t
    h = hs[1].to(dev)
    ys = {t: cpu(ops.gemm_down(h, qd, off_t, rows, w_scale=sd, k_split=k_split, tile=t)) for t in (1, 2, 3, 4, 6)}
    for t in (2, 3, 4, 6):
        assert torch.equal(ys[t], ys[1]), t


@pytest.mark.parametrize("tile", [1, 2, 6])
def test_fp8_gemms_remainder_tile_heights(dev, tile):
    """The same segment layouts on the W8A8 (fp8 x fp8) and W8A16 (fp8 weights) kernels."""
    counts = REMAINDER_COUNTS[tile]
    g = torch.Generator().manual_seed(91 + tile)
    H, I = 256, 256
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 300
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    qgu, sgu = oracle.quantize_weights_fp8(torch.randn(E, 2 * I, H, generator=g) * 0.02)
    qd, sd = oracle.quantize_weights_fp8(torch.randn(E, H, I, generator=g) * 0.02)
    xq, sx = oracle.quantize_rows_fp8(x)
    h8 = cpu(ops.gemm_gate_up_silu_w8a8(xq.to(dev), sx.to(dev), qgu.to(dev), sgu.to(dev), off_t.to(dev), rows,
                                        a_rows=a_rows.to(dev), tile=tile)).float()
    h16 = ops.gemm_gate_up_silu(x.to(dev), qgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev),
                                w_scale=sgu.to(dev), tile=tile)
    hq, sh = oracle.quantize_rows_fp8(h8)
    y8 = cpu(ops.gemm_down_w8a8(hq.to(dev), sh.to(dev), qd.to(dev), sd.to(dev), off_t.to(dev), rows,
                                tile=tile)).sum(0)
    y16 = cpu(ops.gemm_down(h16, qd.to(dev), off_t.to(dev), rows, w_scale=sd.to(dev), tile=tile)).sum(0)
    h16 = cpu(h16).float()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        tok = a_rows[a:b].long()
        gu8 = (xq[tok].float() @ qgu[e].float().T) * sx[tok][:, None] * sgu[e][None, :]
        torch.testing.assert_close(h8[a:b], oracle.silu(gu8[:, :I]) * gu8[:, I:], rtol=1e-2, atol=1e-2)
        gu16 = (x[tok].float() @ qgu[e].float().T) * sgu[e][None, :]
        torch.testing.assert_close(h16[a:b], oracle.silu(gu16[:, :I]) * gu16[:, I:], rtol=1e-2, atol=1e-2)
        torch.testing.assert_close(y8[a:b], (hq[a:b].float() @ qd[e].float().T) * sh[a:b][:, None] * sd[e][None, :],
                                   rtol=1e-4, atol=1e-4)
        torch.testing.assert_close(y16[a:b], (h16[a:b] @ qd[e].float().T) * sd[e][None, :], rtol=1e-3, atol=1e-3)


# fp32 operands on the fp32 MFMA (the fp32 layer): every LDS tile, remainder heights of the 128x128
# tile, K split planes; against float64 with only the summation order left to differ.
@pytest.mark.parametrize("tile", [0, 2, 3, 4, 6])
@pytest.mark.parametrize("k_split", [1, 2])
def test_fp32_gemms(dev, tile, k_split):
    counts = [33, 0, 64, 65, 129, 7, 300]
    g = torch.Generator().manual_seed(5 + tile + k_split)
    H, I = 256, 128
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    T = 90
    x = torch.randn(T, H, generator=g)
    a_rows = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.05
    wd = torch.randn(E, H, I, generator=g) * 0.05
    h = ops.gemm_gate_up_silu(x.to(dev), wgu.to(dev), off_t.to(dev), rows, a_rows=a_rows.to(dev), tile=tile)
    assert h.dtype == torch.float32
    y = cpu(ops.gemm_down(h, wd.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, k_split=k_split,
                          tile=tile)).sum(0).double()
    h = cpu(h).double()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        if b == a:
            continue
        gu = x[a_rows[a:b].long()].double() @ wgu[e].double().T
        href = gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], href, rtol=2e-5, atol=2e-6)
        torch.testing.assert_close(y[a:b], h[a:b] @ wd[e].double().T, rtol=2e-5, atol=2e-6)


# The streaming tile has no fp32 kernel: an explicit request runs on the LDS tiles, stepping down
# until the tile's output columns divide N.  Its host check admits any multiple of its own 16 SiLU
# / 32 output columns, so gate/up with I = 96 (not a multiple of the 128x128 tile's 64 SiLU
# columns) and the down / grouped GEMM with N = 192 (not a multiple of 128) must still write every
# column.
@pytest.mark.parametrize("tile", [5])
def test_fp32_gemms_explicit_tile_narrow_columns(dev, tile):
    counts = [40, 3, 77]
    g = torch.Generator().manual_seed(31 + tile)
    H, I, Id = 192, 96, 128
    E = len(counts)
    off, off_t = _segments(counts)
    rows = int(off[-1])
    x = torch.randn(rows, H, generator=g)
    wgu = torch.randn(E, 2 * I, H, generator=g) * 0.05
    hd = torch.randn(rows, Id, generator=g)
    wd = torch.randn(E, H, Id, generator=g) * 0.05
    h = cpu(ops.gemm_gate_up_silu(x.to(dev), wgu.to(dev), off_t.to(dev), rows, tile=tile)).double()
    y = cpu(ops.gemm_down(hd.to(dev), wd.to(dev), off_t.to(dev), rows, out_dtype=torch.float32,
                          tile=tile)).sum(0).double()
    c = cpu(ops.grouped_gemm(hd.to(dev), wd.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, tile=tile)).double()
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        gu = x[a:b].double() @ wgu[e].double().T
        href = gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]
        torch.testing.assert_close(h[a:b], href, rtol=2e-5, atol=2e-6)
        yref = hd[a:b].double() @ wd[e].double().T
        torch.testing.assert_close(y[a:b], yref, rtol=2e-5, atol=2e-6)
        torch.testing.assert_close(c[a:b], yref, rtol=2e-5, atol=2e-6)


# The LDS tiles of up to 64 rows (bf16, W8A16 and W8A8) run on a three-stage ring (grouped_gemm_ring_kernel,
# grouped_gemm_w8a16_ring_kernel, grouped_gemm_fp8_ring_kernel) unless the two-stage kernel would hold a
# launch's estimated tiles in one round and the ring would not; with no expected rows given the
# estimate takes the row bound.  The same segments under two row bounds, one in each regime (the rule
# restated below), must agree bit for bit: gathered rows, remainder heights, empty segments, K split
# planes.
def _lds_tile_wgs(stage_bytes, stages):
    kib = -(-(stages * stage_bytes + 1025 * 4) // 1024)
    return 160 // kib


def _ring_taken(bm, stage_bytes, S, max_rows, n_tiles, ks):
    est = S * math.ceil(max_rows / S / bm) * n_tiles * ks
    return est > _lds_tile_wgs(stage_bytes, 2) * 256 or est * 1.3 <= _lds_tile_wgs(stage_bytes, 3) * 256


def _two_stage_bound(bm, stage_bytes, S, n_tiles, ks):
    for m in range(1, 200):
        if not _ring_taken(bm, stage_bytes, S, S * bm * m, n_tiles, ks):
            return S * bm * m
    raise AssertionError("no row bound in the two-stage band")


@pytest.mark.parametrize("mode", ["bf16", "w8a16", "w8a8"])
@pytest.mark.parametrize("tile,bm,bn", [(3, 32, 128), (6, 64, 128), (4, 16, 64)])
def test_ring_lds_tiles_bit_identical_with_two_stage(dev, tile, bm, bn, mode):
    counts = [40, 0, 3, 70, 17, 33, 1, 64]
    S, rows = len(counts), sum(counts)
    g = torch.Generator().manual_seed(300 + tile + 10 * len(mode))
    H, I, T = 256, 256, 97
    off_t = _segments(counts)[1].to(dev)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    wgu = (torch.randn(S, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    wd = (torch.randn(S, H, I, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    sgu = sd = None
    if mode != "bf16":
        wgu, sgu = ops.quantize_weights_fp8(wgu)
        wd, sd = ops.quantize_weights_fp8(wd)
    stage = (2 * bm + bn) * 128 if mode == "w8a16" else (bm + bn) * 128
    nt_gu, nt_dn = I // (bn // 2), H // bn
    bounds = {"gu": _two_stage_bound(bm, stage, S, nt_gu, 1), "dn1": _two_stage_bound(bm, stage, S, nt_dn, 1),
              "dn2": _two_stage_bound(bm, stage, S, nt_dn, 2)}
    big = max(bounds.values())
    a_rows = torch.zeros(big, dtype=torch.int32)
    a_rows[:rows] = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32)
    a_rows = a_rows.to(dev)
    hs = torch.zeros(big, I, dtype=torch.bfloat16)
    hs[:rows] = torch.randn(rows, I, generator=g).to(torch.bfloat16)
    hs = hs.to(dev)
    assert _ring_taken(bm, stage, S, rows, nt_gu, 1) and _ring_taken(bm, stage, S, rows, nt_dn, 2)
    if mode == "w8a8":
        xq, sx = ops.quantize_rows_fp8(x)
        hq, sh = ops.quantize_rows_fp8(hs)
        gu = lambda mr: cpu(ops.gemm_gate_up_silu_w8a8(xq, sx, wgu, sgu, off_t, mr, a_rows=a_rows[:mr],
                                                       tile=tile))[:rows]
        dn = lambda mr, ks: cpu(ops.gemm_down_w8a8(hq[:mr], sh[:mr], wd, sd, off_t, mr, k_split=ks,
                                                   tile=tile))[:, :rows]
    else:
        gu = lambda mr: cpu(ops.gemm_gate_up_silu(x, wgu, off_t, mr, a_rows=a_rows[:mr], w_scale=sgu,
                                                  tile=tile))[:rows]
        dn = lambda mr, ks: cpu(ops.gemm_down(hs[:mr], wd, off_t, mr, out_dtype=torch.float32, k_split=ks,
                                              w_scale=sd, tile=tile))[:, :rows]
    assert torch.equal(gu(rows), gu(bounds["gu"]))
    for ks in (1, 2):
        assert torch.equal(dn(rows, ks), dn(bounds[f"dn{ks}"], ks))


# The fp32 tiles of 32 rows and more multiply three bf16 terms per operand on the bf16 MFMA; a tile with an
# operand that the terms do not hold, or with sums that are not finite, is computed again on the fp32 MFMA.  Every tile, on the
# two-stage kernel and on the ring (row bounds in both regimes), against float64: ordinary values,
# infinities, NaN, zero rows and the largest finite values, and operands near the smallest normal.
# Bound: K rounded additions of partial sums below the norm n of the products, of rms 2^-24 n sqrt(K/2)
# when taken as independent, six times that; the products left out are below 2^-24 each.  (A missing
# term, or one cut at the smallest bf16, is 2^-16 n, three times the bound.)
@pytest.mark.parametrize("tile", [2, 3, 6])
@pytest.mark.parametrize("counts", [[33, 0, 70, 1], [400, 129, 700, 260]])
@pytest.mark.parametrize("values", ["ordinary", "special", "tiny"])
def test_fp32_split_terms(dev, tile, counts, values):
    g = torch.Generator().manual_seed(101 + tile)
    E, N, K = len(counts), 256, 320
    off, off_t = _segments(counts)
    rows = int(off[-1])
    a = torch.randn(rows, K, generator=g)
    b = torch.randn(E, N, K, generator=g)
    if values == "special":
        a[3, 7] = float("inf")
        a[5, 0] = float("nan")
        a[20] = 0.0
        a[21] = 3.4e38
        b[2, 9, 11] = -float("inf")
        b[2, 40, 3] = 3.4028234663852886e38
    elif values == "tiny":
        a *= 2.0 ** -118
        b *= 2.0 ** 30
    c = cpu(ops.grouped_gemm(a.to(dev), b.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, tile=tile))
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        x, w = a[lo:hi].double(), b[e].double()
        ref = x @ w.T
        got = c[lo:hi].double()
        fin = torch.isfinite(ref) & (ref.abs() < 3.4e38)
        if values == "special":
            # a sum past fp32 in the middle of a row may end infinite or NaN: only rows and columns
            # without the largest values are compared value by value
            plain = (x.abs().amax(1) < 1e30)[:, None] & (w.abs().amax(1) < 1e30)[None, :]
            special = ~torch.isfinite(x).all(1)[:, None] | ~torch.isfinite(w).all(1)[None, :]
            assert torch.equal(torch.isnan(got)[special], torch.isnan(ref)[special])
            assert torch.equal(got[special & torch.isinf(ref)], ref[special & torch.isinf(ref)])
            assert not torch.isfinite(got[~(ref.abs() <= 3.4029e38)]).any()   # past the largest fp32
            fin &= plain
        norm = ((x[:, None, :] * w[None, :, :]) ** 2).sum(-1).sqrt()
        err = (got - ref).abs()
        assert (err[fin] <= 6 * math.sqrt(K / 2) * 2.0 ** -24 * norm[fin]).all()


# Operands whose last bits lie below the smallest bf16 (2^-133), times large ones so that the sums are
# ordinary: all of them, or one row or weight row among ordinary values, which sit in the same tile.  Same
# bound as above; the fp32 MFMA multiplies subnormal operands as they are.
@pytest.mark.parametrize("tile", [2, 3, 6])
@pytest.mark.parametrize("counts", [[33, 0, 70, 1], [400, 129, 700, 260]])
@pytest.mark.parametrize("ea,eb,only", [(-118, 100, None), (-122, 90, None), (-125, 80, None), (-140, 90, None),
                                        (90, -140, None), (-125, 80, "row"), (-140, 40, "row"), (80, -125, "weight")])
def test_fp32_small_operands_keep_their_bits(dev, tile, counts, ea, eb, only):
    g = torch.Generator().manual_seed(7 + tile)
    E, N, K = len(counts), 256, 320
    off, off_t = _segments(counts)
    rows = int(off[-1])
    a = torch.randn(rows, K, generator=g)
    b = torch.randn(E, N, K, generator=g)
    sa, sb = torch.ones(rows, 1), torch.ones(E, N, 1)
    sa[[5, rows - 1] if only == "row" else slice(None)] = 2.0 ** ea
    sb[:, [17, 200] if only == "weight" else slice(None)] = 2.0 ** eb
    a, b = a * sa, b * sb
    c = cpu(ops.grouped_gemm(a.to(dev), b.to(dev), off_t.to(dev), rows, out_dtype=torch.float32, tile=tile))
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        x, w = a[lo:hi].double(), b[e].double()
        norm = (x ** 2 @ (w ** 2).T).sqrt()
        err = (c[lo:hi].double() - x @ w.T).abs()
        assert (err <= 6 * math.sqrt(K / 2) * 2.0 ** -24 * norm).all()


# Operands of one sign, where what each addition drops adds up instead of averaging, and one repeated value
# whose terms are all at their largest (1 + 2^-7 - 2^-23).  Bound: the rms of a sum of K products in K / 4
# rounded additions, as the fp32 MFMA adds them, each off by at most half a unit of a partial sum that grows
# evenly: 2^-24 sqrt(K / 12).
@pytest.mark.parametrize("tile", [2, 3, 6])
@pytest.mark.parametrize("values,K", [("normal", 2816), ("uniform", 2816), ("uniform", 14336), ("repeated", 64)])
def test_fp32_sums_of_one_sign(dev, tile, values, K):
    g = torch.Generator().manual_seed(K)
    rows, N = 129, 256
    draw = {"normal": lambda *s: torch.randn(*s, generator=g).abs(), "uniform": lambda *s: torch.rand(*s, generator=g),
            "repeated": lambda *s: torch.full(s, 1 + 2.0 ** -7 - 2.0 ** -23)}[values]
    a, b = draw(rows, K), draw(1, N, K)
    off = torch.tensor([0, rows], dtype=torch.int32)
    c = cpu(ops.grouped_gemm(a.to(dev), b.to(dev), off.to(dev), rows, out_dtype=torch.float32, tile=tile)).double()
    ref = a.double() @ b[0].double().T
    assert float((c - ref).norm() / ref.norm()) <= 2.0 ** -24 * math.sqrt(K / 12)
