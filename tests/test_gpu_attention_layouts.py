"""Attention at the grids where the launch changes kernel, against float64: the smallest grid on
64-query workgroups, just under one per CU, three products past one per CU (two of them share a
CU), and causal grids, whose query tiles are dealt longest first, on the split kernel."""
import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def reference(q, k, v, nh, nkv, causal, off):
    B, Tq, _ = q.shape
    Tk = k.shape[1]
    out = torch.empty(B, Tq, nh * 64, dtype=torch.float64)
    mask = torch.arange(Tk)[None, :] > torch.arange(Tq)[:, None] + off if causal else None
    for b in range(B):
        for h in range(nh):
            g = h // (nh // nkv)
            s = q[b, :, h * 64:h * 64 + 64] @ k[b, :, g * 64:g * 64 + 64].t().contiguous() / 8.0
            if causal:
                s = s.masked_fill(mask, -np.inf)
            out[b, :, h * 64:h * 64 + 64] = torch.softmax(s, -1) @ v[b, :, g * 64:g * 64 + 64]
    return out


# error bounds: fp32 level (six products, the fp32 kernel) or two 8-bit parts per operand
@pytest.mark.parametrize("B,T,nh,nkv,products,causal,off,tol", [
    (2, 256, 16, 16, 3, False, 0, 2e-6), (2, 257, 16, 16, 3, False, 0, 2e-6),
    (2, 449, 16, 16, 6, False, 0, 2e-6), (2, 513, 16, 16, 3, False, 0, 1.5e-5),
    (1, 1055, 16, 4, 3, False, 0, 1.5e-5), (1, 769, 14, 2, 6, True, 0, 2e-6),
    (1, 1217, 14, 2, 6, True, 0, 2e-6), (1, 1217, 14, 2, 3, True, 0, 1.5e-5),
    (1, 1217, 14, 2, 6, True, 37, 2e-6),
])
def test_attention_layouts(gpu, B, T, nh, nkv, products, causal, off, tol):
    from larynx_amd import ops
    announce(f"attention layout B={B} T={T} heads={nh}/{nkv} products={products} causal={causal}")
    g = torch.Generator().manual_seed(T + products)
    q = torch.randn(B, T, nh * 64, generator=g)
    k, v = (torch.randn(B, T + off, nkv * 64, generator=g) for _ in range(2))
    o = ops.attention(q.to(gpu), k.to(gpu), v.to(gpu), nh, nkv, causal=causal, q_offset=off,
                      products=products).cpu().double()
    ref = reference(q.double(), k.double(), v.double(), nh, nkv, causal, off)
    err = ((o - ref).norm() / ref.norm()).item()
    assert err < tol, err


@pytest.mark.parametrize("B,T,nh,nkv,products,causal", [
    (2, 300, 16, 16, 3, False), (2, 300, 16, 16, 6, False), (1, 800, 14, 2, 6, True),
])
def test_attention_nonfinite_where_six_products_replace_fp32(gpu, B, T, nh, nkv, products, causal):
    """Grids under one 64-query workgroup per CU that run six products whatever the caller asks
    for: an infinite q element makes its query NaN, an infinite k or v element every query that
    sees its key (a later key's v also queries before it, undefined), as on the larger grids of
    that kernel; the rest stays finite."""
    from larynx_amd import ops
    announce(f"attention non-finite B={B} T={T} products={products} causal={causal}")
    g = torch.Generator().manual_seed(T)
    q = torch.randn(B, T, nh, 64, generator=g)
    k, v = (torch.randn(B, T, nkv, 64, generator=g) for _ in range(2))
    q[0, 10, nh - 2, 5] = np.inf
    k[B - 1, 20, nkv - 1, 7] = np.inf
    v[0, 40, 0, 9] = -np.inf
    rep = nh // nkv
    hit, free = torch.zeros(B, T, nh, dtype=torch.bool), torch.zeros(B, T, nh, dtype=torch.bool)
    hit[0, 10, nh - 2] = True
    hit[B - 1, (20 if causal else 0):, nh - rep:] = True
    vhit = torch.zeros(B, T, nh, 64, dtype=torch.bool)
    vhit[0, (40 if causal else 0):, :rep, 9] = True
    free[0, :, :rep] = True
    o = ops.attention(*(x.flatten(2).to(gpu) for x in (q, k, v)), nh, nkv, causal=causal,
                      products=products).cpu().view(B, T, nh, 64)
    assert o[hit].isnan().all() and o[vhit].isnan().all()
    assert o[~hit & ~free].isfinite().all()
