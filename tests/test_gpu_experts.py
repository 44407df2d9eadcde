"""The experts' MLP on pre-grouped rows (eimoe_experts): rows of one expert from several source ranks
computed as one segment, written back in their own order, against the oracle per segment."""
import pytest
import torch

import oracle
from easyinfra_amd import _lib, ops


def test_experts_validation():
    f = _lib.lib().eimoe_experts
    ok = dict(x=1, M=8, H=128, I=128, Ho=128, gu=1, d=1, dt=_lib.BF16, sg=None, sd=None, c=1, S=8, E=4, y=1, ws=1,
              wsb=1 << 30, st=None)
    rc = lambda **kw: f(*dict(ok, **kw).values())
    assert rc(S=6) == _lib.ERR_SHAPE                      # segments not a multiple of the experts
    assert rc(S=2000, E=2) == _lib.ERR_SHAPE              # too many segments
    assert rc(H=100) == _lib.ERR_ALIGN and rc(I=96) == _lib.ERR_ALIGN and rc(Ho=32) == _lib.ERR_ALIGN
    assert rc(dt=7) == _lib.ERR_DTYPE
    assert rc(dt=_lib.FP8) == _lib.ERR_NULL               # fp8 without scales
    assert rc(c=None) == _lib.ERR_NULL
    assert rc(wsb=16) == _lib.ERR_WORKSPACE
    assert rc(M=1 << 20, H=1024) == _lib.ERR_SHAPE        # x: 2 GiB
    assert rc(M=0, x=None) == _lib.EIMOE_OK


# (experts, ranks, H, I, counts): one row, empty segments and ranks, tile edges (16, 32, 64, 128, 256
# rows and one past), one hot expert, more segments than the register tile schedule holds (64 experts
# on one rank against 65), and an expert of 32 MiB (K split planes).
def _counts(E, ep, pattern, seed):
    g = torch.Generator().manual_seed(seed)
    c = torch.zeros(ep, E, dtype=torch.int64)
    if pattern == "one":
        c[ep - 1, E // 2] = 1
    elif pattern == "edges":
        v = [0, 1, 15, 16, 17, 31, 33, 64, 65, 0, 127, 129]
        for i in range(ep * E):
            c.view(-1)[i] = v[i % len(v)]
    elif pattern == "hot":
        c[:, 0] = 300
        c[0, E - 1] = 2
    else:
        c = torch.randint(0, 12, (ep, E), generator=g)
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("E,ep,H,I,pattern", [(4, 1, 128, 128, "edges"), (4, 2, 128, 192, "one"), (5, 3, 192, 128, "edges"),
                                              (3, 4, 256, 256, "hot"), (1, 8, 128, 128, "edges"), (65, 2, 128, 64, "few"),
                                              (64, 16, 64, 64, "few"), (2, 2, 1024, 16384, "few")])
@pytest.mark.parametrize("mode", ["bf16", "w8a16", "fp32"])
def test_experts_match_oracle_per_segment(dev, E, ep, H, I, pattern, mode):
    g = torch.Generator().manual_seed(E * ep + I)
    counts = _counts(E, ep, pattern, E)
    M = int(counts.sum())
    dt = torch.float32 if mode == "fp32" else torch.bfloat16
    x = torch.randn(M, H, generator=g).to(dt)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dt)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(dt)
    ref_gu, ref_d, scales = wgu.float(), wd.float(), None
    if mode == "w8a16":
        (wgu, sgu), (wd, sd) = oracle.quantize_weights_fp8(wgu.float()), oracle.quantize_weights_fp8(wd.float())
        ref_gu, ref_d = wgu.float() * sgu[..., None], wd.float() * sd[..., None]
        scales = (sgu.to(dev), sd.to(dev))
    print("CASE", dict(E=E, ep=ep, H=H, I=I, pattern=pattern, mode=mode, M=M), flush=True)
    y = ops.experts(x.to(dev), wgu.to(dev), wd.to(dev), counts.reshape(-1).to(torch.int32).to(dev), E, scales)
    assert y.shape == (M, H) and y.dtype == dt
    ref, r = torch.empty(M, H), 0
    for s, c in enumerate(counts.reshape(-1).tolist()):
        ref[r:r + c] = oracle.expert_mlp(x[r:r + c].float(), ref_gu[s % E], ref_d[s % E], round_h_bf16=mode != "fp32")
        r += c
    # one bf16 rounding of the output (at most 2^-9 of each value) and h values whose bf16 rounding
    # flips with the order of the fp32 sums (far fewer); W8A16 forms the oracle's products with the
    # scale applied to the sum instead of the weight (fp32 rounding).  fp32: sums of up to 16384 terms.
    assert oracle.rel_l2(y.cpu().float(), ref) <= (2e-5 if mode == "fp32" else 2.0 ** -8)


def test_grouped_gemm_blocks_validation():
    f = _lib.lib().eimoe_grouped_gemm_blocks
    ok = dict(a=1, M=8, lda=128, b=1, n_b=4, N=128, K=128, c=1, S=8, out=1, ws=1, wsb=1 << 30, st=None)
    rc = lambda **kw: f(*dict(ok, **kw).values())
    assert rc(S=6) == _lib.ERR_SHAPE                      # blocks not a multiple of the weights
    assert rc(S=2000, n_b=2) == _lib.ERR_SHAPE and rc(lda=64) == _lib.ERR_SHAPE
    assert rc(K=100) == _lib.ERR_ALIGN and rc(N=96) == _lib.ERR_ALIGN
    assert rc(c=None) == _lib.ERR_NULL and rc(a=None) == _lib.ERR_NULL
    assert rc(wsb=16) == _lib.ERR_WORKSPACE
    assert rc(M=1 << 23) == _lib.ERR_SHAPE                # A: 2 GiB
    assert rc(M=0, a=None) == _lib.EIMOE_OK


# The op point on lists that repeat their weights (blocks of one weight multiplied as one segment) against
# the oracle per block.
@pytest.mark.gpu
@pytest.mark.parametrize("E,ep,K,N,pattern", [(4, 2, 128, 192, "one"), (5, 3, 192, 128, "edges"), (3, 4, 256, 256, "hot"),
                                              (1, 8, 128, 128, "edges"), (65, 2, 64, 64, "few"),
                                              (2, 3, 4096, 4096, "edges")])
def test_op_point_merges_repeated_weights(dev, E, ep, K, N, pattern):
    import easyinfra_amd.torch_ops  # noqa: F401
    g = torch.Generator().manual_seed(E * ep + N)
    blocks = [int(v) for v in _counts(E, ep, pattern, E).reshape(-1)]
    a = torch.randn(sum(blocks), K, generator=g).to(torch.bfloat16)
    w = [(torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16) for _ in range(E)]
    print("CASE", dict(E=E, ep=ep, K=K, N=N, pattern=pattern), flush=True)
    out = torch.ops.ops.hip_grouped_gemm_single(a.to(dev), [b.to(dev) for b in w] * ep, blocks)
    ref = oracle.grouped_gemm(a, w * ep, blocks)
    # one bf16 rounding of the output, at most 2^-9 of each value; fp32 sums of up to 4096 terms
    assert oracle.rel_l2(out.cpu().float(), ref) <= 2.0 ** -8


# One or two experts of 32 MiB and more, whose down projection splits K over the idle CUs: both sides of
# each tile and split bound (32, 36, 64, 192 rows; 8, 4 and 2 splits), and routed small experts at the
# bounds of the 64x128 and 256x256 tiles.
@pytest.mark.gpu
@pytest.mark.parametrize("E,H,I,rows", [(1, 1024, 16384, r) for r in (1, 32, 33, 36, 37, 64, 65, 128, 192, 193, 257, 600)]
                         + [(2, 1024, 16384, r) for r in (1, 49, 130, 400)]
                         + [(16, 512, 1024, r) for r in (127, 128, 256, 639, 641, 3199, 3201)])
@pytest.mark.parametrize("mode", ["bf16", "w8a16"])
def test_experts_tile_bounds(dev, E, H, I, rows, mode):
    g = torch.Generator().manual_seed(rows)
    counts = torch.bincount(torch.randint(0, E, (rows,), generator=g), minlength=E)
    x = torch.randn(rows, H, generator=g).to(torch.bfloat16)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16)
    ref_gu, ref_d, scales = wgu.float(), wd.float(), None
    if mode == "w8a16":
        (wgu, sgu), (wd, sd) = oracle.quantize_weights_fp8(wgu.float()), oracle.quantize_weights_fp8(wd.float())
        ref_gu, ref_d = wgu.float() * sgu[..., None], wd.float() * sd[..., None]
        scales = (sgu.to(dev), sd.to(dev))
    print("CASE", dict(E=E, H=H, I=I, rows=rows, mode=mode), flush=True)
    y = ops.experts(x.to(dev), wgu.to(dev), wd.to(dev), counts.to(torch.int32).to(dev), E, scales)
    xd, rgu, rd = x.to(dev).float(), ref_gu.to(dev), ref_d.to(dev)
    ref, r = torch.empty(rows, H, device=dev), 0
    for e, c in enumerate(counts.tolist()):
        gu = xd[r:r + c] @ rgu[e].T
        h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]).to(torch.bfloat16).float()
        ref[r:r + c] = h @ rd[e].T
        r += c
    # one bf16 rounding of the output and of h, each at most 2^-9 of a value
    assert oracle.rel_l2(y.cpu().float(), ref.cpu()) <= 2.0 ** -8


# Counts that come to fewer rows than x has, to more, or that are negative (empty segments), on each route:
# rows straight to their places from one rank and from several, fp32 planes, K split planes.  Every row of
# y is defined: its segment's product, or zeros past the last segment.
@pytest.mark.gpu
@pytest.mark.parametrize("E,ep,H,I", [(4, 1, 128, 128), (4, 2, 128, 128), (2, 2, 1024, 16384), (1, 1, 1024, 16384)])
@pytest.mark.parametrize("kind", ["short", "empty", "over", "negative"])
@pytest.mark.parametrize("mode", ["bf16", "fp32"])
def test_experts_counts_off_the_rows(dev, E, ep, H, I, kind, mode):
    M = 120
    g = torch.Generator().manual_seed(E * ep)
    S = E * ep
    counts = torch.full((S,), {"short": 90 // S, "empty": 0, "over": 150 // S, "negative": 60 // S}[kind])
    if kind == "over":
        counts[0] = 2 ** 31 - 1 if S == 1 else counts[0]
        counts[-1] = 2 ** 31 - 1
    if kind == "negative":
        counts[S // 2] = -10 if S > 2 else counts[S // 2]
        counts[S - 1] = -(2 ** 31)
    dt = torch.float32 if mode == "fp32" else torch.bfloat16
    x = torch.randn(M, H, generator=g).to(dt)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dt)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(dt)
    print("CASE", dict(E=E, ep=ep, H=H, I=I, kind=kind, mode=mode), flush=True)
    y = ops.experts(x.to(dev), wgu.to(dev), wd.to(dev), counts.to(torch.int32).to(dev), E)
    ref, r = torch.zeros(M, H), 0
    for s, c in enumerate(counts.tolist()):
        n = min(max(c, 0), M - r)
        ref[r:r + n] = oracle.expert_mlp(x[r:r + n].float(), wgu[s % E].float(), wd[s % E].float(),
                                         round_h_bf16=mode != "fp32")
        r += n
    got = y.cpu().float()
    assert not got[r:].any()
    # the bounds of test_experts_match_oracle_per_segment
    assert float((got - ref).norm()) <= (2e-5 if mode == "fp32" else 2.0 ** -8) * float(ref.norm())


L, M, S, XS, STREAM, MS = 1, 2, 3, 4, 5, 6   # EIMOE_TILE_*


def _mapped_rows(E, ep, rows, seed):
    """Rows of (source rank, expert), uneven, so that tiles end in remainders on every expert."""
    g = torch.Generator().manual_seed(seed)
    return torch.bincount(torch.randint(0, E * ep, (rows,), generator=g), minlength=E * ep)


# Every kernel that stores rows through the map of merged ranks, with remainder tiles: the down projection on
# each tile (in one round and past it, where ring and two-stage kernels meet; up to 64 experts and beyond,
# where the 256x256 kernels change; W8A16 with K a multiple of 128 and not).  The tile is asserted, so that a
# change of the rules moves the sizes here too.
@pytest.mark.gpu
@pytest.mark.parametrize("E,H,I,per,mode,tile", [
    (16, 2048, 256, 0.5, "bf16", STREAM), (16, 2048, 256, 5, "bf16", XS), (4, 512, 256, 40, "bf16", S),
    (16, 2048, 256, 30, "bf16", MS), (32, 2048, 256, 35, "bf16", MS), (16, 1024, 256, 90, "bf16", M),
    (20, 2048, 256, 60, "bf16", L), (16, 2048, 256, 300, "bf16", L), (70, 1024, 256, 210, "bf16", L),
    (16, 2048, 256, 0.5, "w8a16", STREAM), (16, 2048, 256, 1.5, "w8a16", XS), (16, 2048, 256, 15, "w8a16", S),
    (16, 2048, 256, 45, "w8a16", MS), (32, 2048, 256, 60, "w8a16", MS), (16, 2048, 256, 120, "w8a16", M),
    (16, 2048, 256, 270, "w8a16", L), (70, 1024, 256, 400, "w8a16", L), (16, 2048, 192, 15, "w8a16", S),
    (16, 2048, 192, 120, "w8a16", M)])
def test_experts_store_through_the_map(dev, E, H, I, per, mode, tile):
    ep, rows = 2, int(per * E)
    dt = _lib.FP8 if mode == "w8a16" else _lib.BF16
    assert _lib.lib().eimoe_gemm_tile(rows, E, H, I, dt, 0, 1) == tile
    g = torch.Generator().manual_seed(E + rows)
    counts = _mapped_rows(E, ep, rows, E + rows)
    x = torch.randn(rows, H, generator=g).to(torch.bfloat16)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(E, H, I, generator=g) * 0.05).to(torch.bfloat16)
    ref_gu, ref_d, scales = wgu.float(), wd.float(), None
    if mode == "w8a16":
        (wgu, sgu), (wd, sd) = oracle.quantize_weights_fp8(wgu.float()), oracle.quantize_weights_fp8(wd.float())
        ref_gu, ref_d = wgu.float() * sgu[..., None], wd.float() * sd[..., None]
        scales = (sgu.to(dev), sd.to(dev))
    print("CASE", dict(E=E, H=H, I=I, rows=rows, mode=mode, tile=tile), flush=True)
    y = ops.experts(x.to(dev), wgu.to(dev), wd.to(dev), counts.to(torch.int32).to(dev), E, scales)
    xd, rgu, rd = x.to(dev).float(), ref_gu.to(dev), ref_d.to(dev)
    ref, r = torch.empty(rows, H, device=dev), 0
    for s, c in enumerate(counts.tolist()):
        gu = xd[r:r + c] @ rgu[s % E].T
        h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]).to(torch.bfloat16).float()
        ref[r:r + c] = h @ rd[s % E].T
        r += c
    # as test_experts_tile_bounds, and row by row: a row in another's place is off by its whole size (a bf16
    # rounding of one value is at most 2^-8 of it; h flips and the rest are far below)
    err = (y.float() - ref).norm(dim=1)
    assert bool((err <= 2.0 ** -7 * ref.norm(dim=1)).all())
    assert oracle.rel_l2(y.cpu().float(), ref.cpu()) <= 2.0 ** -8


# The op point on weights of 32 MiB over two ranks, both sides of each of its rule's bounds (56 and 62 rows per
# weight), which are also the tiles that store through the map there.
@pytest.mark.gpu
@pytest.mark.parametrize("rows,tile", [(240, MS), (447, MS), (448, M), (495, M), (496, L), (1500, L)])
def test_op_point_large_weights_store_through_the_map(dev, rows, tile):
    import easyinfra_amd.torch_ops  # noqa: F401
    E, ep, N, K = 8, 2, 16384, 1024
    assert _lib.lib().eimoe_gemm_tile(rows, E, N, K, _lib.BF16, 0, 1) == tile
    g = torch.Generator().manual_seed(rows)
    blocks = _mapped_rows(E, ep, rows, rows).tolist()
    a = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(dev)
    w = [(torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16).to(dev) for _ in range(E)]
    print("CASE", dict(rows=rows, tile=tile), flush=True)
    out = torch.ops.ops.hip_grouped_gemm_single(a, w * ep, blocks)
    r = 0
    for s, c in enumerate(blocks):
        ref = a[r:r + c].float() @ w[s % E].float().T
        # one bf16 rounding, at most 2^-9 of each value; fp32 sums of 1024 terms
        assert bool(((out[r:r + c].float() - ref).norm(dim=1) <= 2.0 ** -8 * ref.norm(dim=1)).all())
        r += c
