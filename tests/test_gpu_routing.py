"""Routing at the edges of its kernels' ranges: pick order on zeros of both signs and infinities, and
layers whose routing spans the many-workgroup kernels."""
import pytest
import torch

import oracle
from easyinfra_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k", [(8, 2), (8, 8), (16, 3), (32, 32), (64, 6), (128, 8), (256, 8), (300, 9)])
def test_router_orders_zeros_and_infinities_as_the_oracle(dev, E, k):
    g = torch.Generator().manual_seed(E + k)
    vals = torch.tensor([-float("inf"), -1.0, -0.0, 0.0, 1e-40, -1e-40, 2.5])
    logits = vals[torch.randint(0, len(vals), (70, E), generator=g)]
    logits[:, 0] = 3.0                                   # a finite maximum, so that the weights are numbers
    ids, w = ops.router_topk(logits.to(dev), k, True)
    rid, rw = oracle.route_topk(logits, k, True)
    assert torch.equal(ids.cpu(), rid)
    torch.testing.assert_close(w.cpu(), rw, rtol=3e-6, atol=1e-7)


# One routing workgroup (its waves' rows of 64 ids full, and one past), then workgroups of 4, 8 and 16
# waves, then the separate histogram; experts in number a power of two and not.
@pytest.mark.parametrize("E,k,lo,hi,T", [(32, 8, 0, 32, 8), (32, 8, 0, 32, 9), (128, 8, 0, 32, 127), (128, 8, 0, 32, 128),
                                         (128, 8, 64, 96, 129), (64, 6, 0, 64, 511), (64, 6, 0, 64, 1024),
                                         (64, 6, 0, 64, 2047), (64, 6, 0, 64, 4096), (64, 6, 0, 64, 4097),
                                         (96, 5, 3, 80, 1500), (300, 4, 0, 300, 100)])
def test_layer_routing_permutation(dev, E, k, lo, hi, T):
    H = I = 64
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, generator=g) * 2.0
    wgu = (torch.randn(hi - lo, 2 * I, H, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(hi - lo, H, I, generator=g) * 0.05).to(torch.bfloat16)
    print("CASE", dict(E=E, k=k, lo=lo, hi=hi, T=T), flush=True)
    out, ids, w = ops.fused_moe(x.to(dev), logits.to(dev), k, wgu.to(dev), wd.to(dev), expert_range=(lo, hi),
                                out_dtype=torch.float32, return_routing=True)
    rid, rw = oracle.route_topk(logits, k, True)
    assert torch.equal(ids.cpu(), rid)
    torch.testing.assert_close(w.cpu(), rw, rtol=3e-6, atol=1e-7)
    ref = torch.zeros(T, H)
    for e in range(lo, hi):
        t, s = torch.nonzero(rid == e, as_tuple=True)
        ref.index_add_(0, t, oracle.expert_mlp(x[t].float(), wgu[e - lo].float(), wd[e - lo].float()) * rw[t, s][:, None])
    # h rounded to bf16, at most 2^-9 of each value; the rest are fp32 sums
    assert oracle.rel_l2(out.cpu(), ref) <= 2.0 ** -8
