"""The fused prefill layer at many rows per expert, on the row tiles (few tiles
of the grouped GEMM for the CUs) and on the grouped GEMM (both products; with
f16 x act goes between them as int8 limbs and down runs on the int8 matrix
cores), against the CPU oracle: on every token, or on those at the edges of row
tiles and a spread of others. The GEMM's shapes exercise its tiling: partial
64-row blocks, a last N-tile narrower than 512 columns, experts with no rows, a
hot expert, K with an odd number of step pairs, and the f16 hi + lo pairs form
that f32 x and I not a multiple of 64 take.

Bar: expert ids bit-exact, outputs within 2e-3 + 1e-2·|want| of the oracle."""
import numpy as np
import pytest
import torch

import runntime_amd as rt
from oracle import ref
from runntime_amd.synth import MoeConfig, make_inputs
from tests.helpers import assert_close, expert_tiles
from tests.test_gpu_parity import _edge_tokens

pytestmark = pytest.mark.gpu

SHAPES = [  # rows per tile; name, T, d, E, k, I, x
    (16, MoeConfig("p_small", 512, 1024, 8, 2, 1024, "f16")),
    (16, MoeConfig("p_ragged", 300, 640, 6, 4, 384, "f16")),
    (16, MoeConfig("p_oddpairs", 384, 640, 5, 2, 448, "f16")),
    (16, MoeConfig("p_skew", 512, 640, 16, 2, 384, "f16", zipf=1.2, hot_share=0.5, empty=2)),
    (16, MoeConfig("p_f32x", 512, 1024, 8, 2, 1024, "f32")),
    (16, MoeConfig("p_i1056", 512, 1024, 8, 2, 1056, "f16")),
    (128, MoeConfig("g_small", 1024, 1024, 8, 2, 1024, "f16")),
    (128, MoeConfig("g_ragged", 900, 640, 6, 4, 1152, "f16")),      # d = 640: N-tile of 128 columns
    (128, MoeConfig("g_oddpairs", 1200, 640, 12, 2, 1088, "f16")),  # 17 step pairs
    (128, MoeConfig("g_skew", 2048, 640, 16, 2, 1152, "f16", zipf=1.2, hot_share=0.5, empty=2)),
    # the layer's other prefill forms: f32 x (act as f16 hi + lo pairs, down
    # on the f16 matrix cores), and f16 x with I not a multiple of 64 (the
    # same pairs form: int8 limbs need whole step pairs)
    (128, MoeConfig("g_f32x", 1536, 1024, 8, 2, 1024, "f32")),
    (128, MoeConfig("g_i1056", 1024, 1024, 8, 2, 1056, "f16")),
]


def _oracle(inp, cfg, tokens):
    x = inp.x[tokens].float().cpu().numpy()
    logits = ref.router_logits(x, inp.router_w.cpu().numpy(), inp.router_b.cpu().numpy())
    route = ref.topk(logits, cfg.k)
    pk = {n: ref.pack_ekn(inp.q[n].numpy(), 8) for n in ("glu", "lin", "down")}
    w = {n: (pk[n], getattr(inp, n).scales.cpu().numpy(), getattr(inp, n).bias.cpu().numpy())
         for n in ("glu", "lin", "down")}
    act = ref.moe_up(x, route, w["glu"], w["lin"], 8, cfg.d, cfg.E)
    out = ref.moe_down(act, route, w["down"], inp.residual[tokens].cpu().numpy(), 8, cfg.I,
                       cfg.E)
    return route, out


@pytest.mark.parametrize("rows,cfg", SHAPES, ids=[c.name for _, c in SHAPES])
def test_prefill_layer_int8_limbs(rows, cfg):
    print(f"prefill layer {cfg}", flush=True)
    assert expert_tiles("layer", cfg.T, cfg.d, cfg.I, cfg.E, cfg.k, cfg.x_dtype) == (rows, rows)
    inp = make_inputs(cfg, seed=11, keep_q=True, bias_rand=True)
    g = torch.Generator().manual_seed(5)
    inp.residual.copy_(torch.randn(tuple(inp.residual.shape), generator=g))
    out, route = rt.moe_layer(inp.x, inp.router_w, inp.router_b, inp.glu, inp.lin, inp.down,
                              inp.residual, cfg.k, return_route=True)
    torch.cuda.synchronize()
    got_route, got = route.cpu().numpy(), out.cpu().numpy()
    k = cfg.k
    t = np.arange(cfg.T)
    if rows == 128:
        t = np.array(sorted(set(t[::16].tolist()) | _edge_tokens(got_route[:, :k], cfg.E, k)))
    want_route, want = _oracle(inp, cfg, t)
    assert np.array_equal(got_route[t, :k], want_route[:, :k]), "expert ids differ"
    counts = np.bincount(got_route[:, :k].astype(np.int64).ravel(), minlength=cfg.E)
    print(f"  rows per expert {counts.tolist()}, {len(t)} tokens checked", flush=True)
    if cfg.zipf:
        assert (counts == 0).any(), "the skewed shape should leave an expert without rows"
    assert_close(got[t], want, what=f"{cfg.name} output")


@pytest.mark.parametrize("cfg", [MoeConfig("e_f32x", 1536, 1024, 8, 2, 1024, "f32"),
                                 MoeConfig("e_i1056", 1024, 1024, 8, 2, 1056, "f16")],
                         ids=lambda c: c.name)
def test_prefill_act_pairs_keep_f32(cfg):
    """act as f16 hi + lo pairs between the products (up with f32 x; up with f16
    x on I = 1056) is f32's 22 bits: the layer is within 2^-20 of f64 (norm over
    norm; each product's parts are good to 2^-22, its f32 sums to about 2^-21).
    A pair whose hi is not the one its lo completes is off by 2^-11 of a value."""
    print(f"prefill pairs {cfg}", flush=True)
    assert expert_tiles("layer", cfg.T, cfg.d, cfg.I, cfg.E, cfg.k, cfg.x_dtype) == (128, 128)
    inp = make_inputs(cfg, seed=21, keep_q=True, bias_rand=True)
    inp.residual.zero_()
    out = rt.moe_layer(inp.x, inp.router_w, inp.router_b, inp.glu, inp.lin, inp.down, inp.residual,
                       cfg.k)
    t = np.arange(0, cfg.T, 7)
    got = out.cpu().numpy().astype(np.float64)[t]
    _, want = _oracle(inp, cfg, t)
    assert np.linalg.norm(got - want) <= 2.0 ** -20 * np.linalg.norm(want)
