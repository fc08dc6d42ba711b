"""The projections on fragment-order activations (lx_gemm_fs.hip, lx_gemm_ft.hip) through the
estimator and the Qwen2 prefill, against the oracle at the row counts where a launch changes
its tiles: part of one 32-row block, whole blocks and one row past them, the last row count of
the 32 x 32 and 64 x 64 tiles, the tiled kernel's three tile shapes, and the first row past the
fragment-order block."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def dit_vs_oracle(gpu, cfg, B, T, products):
    """One evaluation with O(1) modulation, so that every projection carries weight in the
    result.  Tolerance: the two-part operands' 2^-16 per element, some ten roundings deep."""
    from larynx_amd.flow import DiTEstimator, dit_param_shapes
    announce(f"dit F={cfg.ff_inner} B={B} T={T} products={products}")
    params = orc.make_params(dit_param_shapes(cfg), 29)
    dparams = {k: torch.from_numpy(v).to(gpu) for k, v in params.items()}
    est = DiTEstimator(dparams, cfg, B=B, max_T=max(T, 64))
    est.set_products(products)
    x, mu, cond = (orc.normal((B, 80, T), 31 + T, s) for s in (1, 2, 3))
    spks = orc.normal((B, 80), 31, 4, 1.0 / np.sqrt(80.0))
    t = np.linspace(0.2, 0.7, B).astype(np.float32)
    dphi = est.forward(*(torch.from_numpy(a).to(gpu) for a in (x, mu, cond, spks, t)))
    torch.cuda.synchronize()
    est.close()
    ref = orc.Dit(params, depth=cfg.depth, ff_inner=cfg.ff_inner).forward(x, mu, cond, spks, t)
    err = orc.rel_err(dphi.cpu().numpy(), ref)
    assert err < (1e-4 if products == 3 else 2e-5), err


@pytest.mark.parametrize("B,T,products", [
    (1, 5, 3), (2, 16, 3), (2, 17, 6), (2, 32, 3), (2, 33, 3), (1, 65, 3), (2, 80, 3), (3, 41, 3),
    (2, 128, 3), (2, 83, 6), (1, 161, 3), (2, 160, 6),
    (2, 161, 6), (2, 255, 3), (2, 257, 3),
])
def test_dit_projection_tiles_vs_oracle(gpu, B, T, products):
    from larynx_amd.flow import DiTConfig
    dit_vs_oracle(gpu, DiTConfig(depth=2), B, T, products)


@pytest.mark.parametrize("F,B,T,products", [
    (4096, 2, 37, 6), (4096, 1, 320, 3), (4096, 1, 321, 3), (4096, 2, 128, 6), (4096, 1, 257, 6), (3072, 1, 320, 6),
    (8192, 1, 149, 3), (8192, 1, 289, 3), (8192, 2, 75, 6),
])
def test_dit_wide_mlp_vs_oracle(gpu, F, B, T, products):
    """MLPs whose FF0 outgrows one round of the few-row tiles: both tile widths of the tiled
    kernel's GELU (three products; 128 x 64 and, from 150 tiles, 128 x 128), the few-row kernel
    past one tile per CU (six), and the first row past the fragment-order block."""
    from larynx_amd.flow import DiTConfig
    dit_vs_oracle(gpu, DiTConfig(depth=1, ff_inner=F), B, T, products)


def make_lm(gpu, n_layers, max_ctx):
    from larynx_amd.llm import Qwen2Config, Qwen2LM, qwen2_param_shapes
    cfg = Qwen2Config(n_layers=n_layers, text_vocab=2000)
    params = orc.make_params(qwen2_param_shapes(cfg), 78)
    for k in params:
        if k.endswith("layernorm.weight") or k == "norm.weight":
            params[k] = (params[k] + 1.0).astype(np.float32)
    lm = Qwen2LM({k: torch.from_numpy(v).to(gpu) for k, v in params.items()}, cfg, max_ctx=max_ctx)
    return cfg, params, lm


@pytest.fixture(scope="module")
def qwen2(gpu):
    cfg, params, lm = make_lm(gpu, 2, 1100)
    yield cfg, params, lm
    lm.close()


@pytest.fixture(scope="module")
def qwen2_long(gpu):
    cfg, params, lm = make_lm(gpu, 1, 2750)
    yield cfg, params, lm
    lm.close()


def prefill_vs_oracle(gpu, model, L, products):
    cfg, params, lm = model
    announce(f"qwen2 prefill L={L} products={products}")
    lm.set_products(products)
    lm_in = torch.from_numpy(orc.normal((L, cfg.hidden), 500 + L, 1, 0.5)).to(gpu)
    logits, hidden, final = lm.prefill(lm_in, capture=True)
    torch.cuda.synchronize()
    o = orc.Qwen2(params, cfg, cap=L)
    rl, rh, rf = o.prefill(lm_in.cpu().numpy(), capture=True)
    tol = 5e-5 if products == 3 else 1e-5
    for layer in range(cfg.n_layers):
        assert orc.rel_err(hidden[layer].cpu().numpy(), rh[layer]) < tol, layer
        k, v = lm.cache_views(layer)
        assert orc.rel_err(k[:L].cpu().numpy(), o.k_cache[layer, :L]) < tol, layer
        assert orc.rel_err(v[:L].cpu().numpy(), o.v_cache[layer, :L]) < tol, layer
    assert orc.rel_err(logits.cpu().numpy(), rl) < tol


@pytest.mark.parametrize("L,products", [
    (1, 6), (31, 3), (32, 3), (33, 6), (65, 3), (129, 3), (129, 6), (256, 6), (385, 3), (545, 3), (640, 3),
    (1089, 3),
])
def test_prefill_projection_tiles_vs_oracle(gpu, qwen2, L, products):
    """q|k|v with the rotary and cache append in its epilogue, o_proj's residual epilogue,
    gate/up with SwiGLU in fragment order and down_proj's K slices."""
    prefill_vs_oracle(gpu, qwen2, L, products)


@pytest.mark.parametrize("L", [1152, 1153, 2435, 2689, 2750])
def test_prefill_long_tiles_vs_oracle(gpu, qwen2_long, L):
    """The last length of o_proj on the few-row kernel, its 128 x 64 (1153-2688 rows) and 128 x
    128 tiles, and down_proj whole in K on 128 x 64 (2305-2688 rows) and 128 x 128 ones."""
    prefill_vs_oracle(gpu, qwen2_long, L, 3)


@pytest.mark.parametrize("M,N,K,products,lda", [
    (1, 1024, 1024, 3, 0), (33, 1024, 2048, 6, 0), (85, 3072, 1024, 3, 0), (86, 3072, 1024, 3, 12),
    (256, 1024, 1024, 3, 0), (257, 1024, 1024, 6, 4), (512, 1024, 64, 3, 0), (31, 128, 64, 6, 0),
    (160, 3072, 128, 6, 0), (256, 3072, 128, 6, 0), (700, 3072, 128, 3, 0), (768, 3072, 64, 6, 4), (1040, 2048, 128, 3, 0),
])
def test_linear_bx_few_rows(gpu, M, N, K, products, lda):
    """lx_linear_bx on fp32 rows at the row counts of the few-row kernel (row strides past K
    among them) and of the 96-row tiles, against float64: each operand is its two or three bf16 parts (2^-17 or 2^-25
    of it at most, signs at random), the rest fp32 sums."""
    from larynx_amd import ops
    announce(f"linear_bx few rows M={M} N={N} K={K} products={products}")
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + lda, generator=g)[:, :K]
    W, b = torch.randn(N, K, generator=g) / K ** 0.5, torch.randn(N, generator=g)
    h = torch.randn(M, N, generator=g)
    xd = torch.zeros(M, K + lda, device=gpu)
    xd[:, :K] = x.to(gpu)
    wf = ops.wfrag_pack(W.to(gpu))
    y0 = x.double() @ W.double().t() + b.double()
    tol = 1e-5 if products == 3 else 1e-6
    cases = ((None, y0, None), (ops.LX_EPI_RESID, h.double() + y0, h),
             (ops.LX_EPI_GELU_TANH, torch.nn.functional.gelu(y0, approximate="tanh"), None))
    for kind, ref, init in cases:
        ep = ops.Epilogue(kind=kind) if kind is not None else None
        out = init.to(gpu) if init is not None else None
        y = ops.linear_bx(xd[:, :K], wf, N, b.to(gpu), ep, out=out, bm=64, products=products)
        err = ((y.cpu().double() - ref).norm() / ref.norm()).item()
        assert err < tol, (kind, err)
