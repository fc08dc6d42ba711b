"""Decode over short caches, where attention is formed inside the o_proj launch: one key, the
last and first positions of the one-tile (64 keys) and the merged form, against
the oracle, with the rows past the cache holding NaN."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def short_lm(gpu):
    from larynx_amd.llm import Qwen2Config, Qwen2LM, qwen2_param_shapes
    cfg = Qwen2Config(n_layers=2, text_vocab=2000)
    params = orc.make_params(qwen2_param_shapes(cfg), 79)
    for k in params:
        if k.endswith("layernorm.weight") or k == "norm.weight":
            params[k] = (params[k] + 1.0).astype(np.float32)
    lm = Qwen2LM({k: torch.from_numpy(v).to(gpu) for k, v in params.items()}, cfg, max_ctx=160)
    yield cfg, params, lm
    lm.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("n", [1, 2, 3, 33, 62, 63, 64])
def test_decode_short_cache_vs_oracle(gpu, short_lm, n, graph):
    """Keys and values of unit size, so that the softmax is far from uniform; fp32 sums over
    at most 65 keys and 4864 products per row."""
    cfg, params, lm = short_lm
    announce(f"decode short cache n={n} graph={graph}")
    lm.set_decode_graph(graph)
    o = orc.Qwen2(params, cfg, cap=160)
    for layer in range(cfg.n_layers):
        kd, vd = lm.cache_views(layer)
        kd.fill_(float("nan"))
        vd.fill_(float("nan"))
        for cache, dev, part in ((o.k_cache, kd, 1), (o.v_cache, vd, 2)):
            c = orc.normal((n, 128), 600 + layer, part, 1.0)
            cache[layer, :n] = c
            dev[:n].copy_(torch.from_numpy(c))
    o.cache_len = n
    lm.set_cache_len(n)
    lg, fn = lm.decode(4321, final_norm=True)
    torch.cuda.synchronize()
    rlg, rfn = o.decode(4321)
    assert orc.rel_err(fn.cpu().numpy(), rfn) < 1e-5
    assert orc.rel_err(lg.cpu().numpy(), rlg) < 1e-5
