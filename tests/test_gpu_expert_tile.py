"""k_expert_tile (expert_tile.hip): row tiles of 16, 32 and 64 rows, each A
form (f16, f32 as f16 hi + lo, f32 as three bf16 planes under int4 weights),
plain and group scales, against the oracle's f64 products; f32's whole range
under int4 weights; infinities and NaN stay in their rows."""
import numpy as np
import pytest
import torch

import runntime_amd as rt
from oracle import ref

from runntime_amd.synth import MoeConfig, make_inputs
from tests.helpers import assert_close, expert_tiles, random_quant_weight

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (T, K, N, E, g, k), rows per tile: rows per expert from 1 to many 16-row tiles
# (a launch of fewer than 512 blocks takes no larger ones), then row tiles of 32
# and 64; K one 32-wide step past a piece or a ring turn or a part of a step, N
# with a partial unit group, a partial column block and a wavefront without
# columns.
SHAPES = [(1, 32, 8, 3, 32, 2), (5, 96, 72, 4, 32, 2), (40, 160, 136, 8, 32, 2),
          (60, 288, 264, 6, 96, 2), (129, 640, 200, 4, 640, 2), (70, 352, 64, 2, 352, 1),
          (260, 416, 520, 4, 416, 1), (33, 1408, 68, 1, 64, 1), (90, 64, 640, 128, 64, 4)]
LARGE = [((160, 104, 1416, 32, 104, 4), 32), ((160, 160, 1416, 32, 32, 4), 32),
         ((160, 288, 1352, 32, 96, 4), 32), ((320, 104, 1416, 32, 104, 4), 64),
         ((320, 160, 1416, 32, 32, 4), 64), ((320, 288, 1352, 32, 288, 4), 64)]
TILES = [(c, 0 if c[0] == 1 else 16) for c in SHAPES] + LARGE


def _route(T, E, k, seed):
    """Distinct random experts per token; slot 0 of every seventh token names none."""
    rng = np.random.default_rng(seed)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.float32)
    ids[3::7, 0] = -1.0
    gates = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    return np.concatenate([ids, gates], 1)


def _weight(E, K, N, g, bits, seed):
    q, sc = random_quant_weight(E, K, N, bits, g, seed)
    bias = ref.lcg_f32(E * N, seed + 2).reshape(E, N)
    words = rt.pack_expert_weights(q, bits)
    dev = rt.QuantExpertWeight(
        rt.QuantW(torch.from_numpy(words.view(np.int32)).to(DEV), (E * K, N)),
        torch.from_numpy(sc).to(DEV), torch.from_numpy(bias).to(DEV))
    w = q.astype(np.float64) * np.repeat(sc.reshape(E, K // g, N), g, 1).astype(np.float64)
    return dev, w, bias.astype(np.float64)


def _project(x, ids, w, b):
    """[A, N] rows x[a]·w[e] + b[e] and the sums of magnitudes (the error scale)."""
    y = np.zeros((len(ids), w.shape[2]))
    mag = np.zeros_like(y)
    for e in np.unique(ids[ids >= 0]).astype(int):
        r = ids == e
        y[r] = x[r] @ w[e] + b[e]
        mag[r] = np.abs(x[r]) @ np.abs(w[e]) + np.abs(b[e])
    return y, mag


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("xdtype", ["f32", "f16"])
@pytest.mark.parametrize("shape,rows", TILES)
def test_tile_products(bits, xdtype, shape, rows):
    T, K, N, E, g, k = shape
    if bits == 4:  # int4 runs here from one row on
        rows = max(rows, 16)
    assert expert_tiles("up", T, K, N, E, k, xdtype, bits, g, g)[0] == rows
    assert expert_tiles("down", T, N, K, E, k, "f32", bits, g, g)[1] == rows
    print(f"expert tile int{bits} {xdtype} {shape}", flush=True)
    route = _route(T, E, k, T + K)
    ids = route[:, :k].reshape(-1)
    glu, wg, bg = _weight(E, K, N, g, bits, 11)
    lin, wl, bl = _weight(E, K, N, g, bits, 23)
    x = (ref.lcg_f32(T * K, 5) * 2).reshape(T, K)
    if xdtype == "f16":
        x = x.astype(np.float16)
    rd = torch.from_numpy(route).to(DEV)
    opts = {"bits": bits, "groupSize": g}
    act = rt.moeUp(torch.from_numpy(x).to(DEV), rd, glu, lin, opts).cpu().numpy()
    xr = np.repeat(x.astype(np.float64), k, 0)
    yg, mg = _project(xr, ids, wg, bg)
    yl, ml = _project(xr, ids, wl, bl)
    gc, lc = np.minimum(yg, 7.0), np.clip(yl, -7.0, 7.0)
    want = np.where(ids[:, None] >= 0, gc / (1 + np.exp(-1.702 * gc)) * (lc + 1), 0.0)
    # Each product's f32 sums are off by at most ~(K/32 + 8)·2^-23 of the sum of
    # magnitudes, f32 x's two f16 parts by 2^-21 of it; SwiGLU's slopes are below
    # 1.2·8 (glu) and 7 (lin), its own arithmetic within 2^-20.
    eps = (K / 32 + 8) * 2.0 ** -23 + 2.0 ** -21
    np.testing.assert_array_less(np.abs(act - want), 9.6 * eps * mg + 7 * eps * ml
                                 + 2.0 ** -20 * (1 + np.abs(want)) + 1e-30)
    # down on plain f32 rows
    a = (ref.lcg_f32(T * k * K, 9)).reshape(T * k, K)
    res = ref.lcg_f32(T * N, 4).reshape(T, N)
    out = rt.moeDown(torch.from_numpy(a).to(DEV), rd, glu, torch.from_numpy(res).to(DEV),
                     opts).cpu().numpy()
    y, m = _project(a.astype(np.float64), ids, wg, bg)
    gates = route[:, k:].astype(np.float64)
    want = res + (y.reshape(T, k, N) * gates[..., None]).sum(1)
    mag = np.abs(res) + (m.reshape(T, k, N) * gates[..., None]).sum(1)
    np.testing.assert_array_less(np.abs(out - want), (eps + (k + 2) * 2.0 ** -23) * mag + 1e-30)


def test_int4_f32_range():
    """int4 weights take f32 x whole: rows near f32's largest and of 1e-20 keep
    f32's relative error, an infinity or a NaN stays in its row."""
    T, K, N, E = 40, 128, 64, 2
    print("expert tile int4 f32 range", flush=True)
    w, wd, _ = _weight(E, K, N, 32, 4, 3)
    w.bias = None
    a = ref.lcg_f32(T * K, 7).reshape(T, K)
    a[1] *= 1e35
    a[2] *= 1e-20
    a[3, 5] = np.inf
    a[4, 6] = np.nan
    route = np.zeros((T, 2), np.float32)
    route[:, 0] = np.arange(T) % E
    route[:, 1] = 1.0
    out = rt.moeDown(torch.from_numpy(a).to(DEV), torch.from_numpy(route).to(DEV), w, None,
                     {"bits": 4, "groupSize": 32}).cpu().numpy()
    fin = [t for t in range(T) if t not in (3, 4)]
    for t in fin:
        want = a[t].astype(np.float64) @ wd[t % E]
        mag = np.abs(a[t].astype(np.float64)) @ np.abs(wd[t % E])
        assert np.all(np.abs(out[t] - want) <= 16 * 2.0 ** -23 * mag), t
    with np.errstate(invalid="ignore"):
        want = a[3].astype(np.float64) @ wd[1]  # inf · 0 is NaN, else ±inf
    np.testing.assert_array_equal(np.isnan(out[3]), np.isnan(want))
    np.testing.assert_array_equal(out[3][~np.isnan(want)], want[~np.isnan(want)])
    assert np.isnan(out[4]).all()


def _unit_columns(words, e, u, K, N, bits):
    """Expert e's columns 4u .. 4u + 3 as f64 [K, 4], from quantW words."""
    n = K // 4 * bits // 2
    w = words[(e * (N // 4) + u) * n:][:n].view(torch.int8).to(torch.int32)
    v = w if bits == 8 else torch.stack([(w << 28) >> 28, w >> 4], -1)
    return v.reshape(K // 4, 4, 4).transpose(1, 2).reshape(K, 4).double()


# Experts of 2^29 bytes of weights, where K·N·bits is 2^32: one row an expert
# and several (int8: k_expert_skinny, then k_expert_tile).
@pytest.mark.parametrize("bits,K,N,T", [(4, 32768, 32768, 4), (8, 4096, 131072, 2),
                                        (8, 4096, 131072, 6)])
def test_experts_of_half_a_gib(bits, K, N, T):
    print(f"large experts int{bits} {K} x {N} T={T}", flush=True)
    E = 2
    g = torch.Generator(device=DEV).manual_seed(bits + T)
    words = torch.randint(-(1 << 31), 1 << 31, (E * K * N * bits // 32,), generator=g, device=DEV,
                          dtype=torch.int64).to(torch.int32)
    sc = torch.rand((E, N), generator=g, device=DEV) + 0.5
    a = torch.randn((T, K), generator=g, device=DEV)
    route = torch.ones((T, 2), device=DEV)
    route[:, 0] = torch.arange(T, device=DEV) % E
    w = rt.QuantExpertWeight(rt.QuantW(words, (E * K, N)), sc, None)
    out = rt.moeDown(a, route, w, None, {"bits": bits, "groupSize": K})
    for u in (0, 1, N // 8 + 3, N // 4 - 1):
        for e in range(E):
            q = _unit_columns(words, e, u, K, N, bits)
            s = sc[e, 4 * u:4 * u + 4].double()
            rows = a[e::E].double()
            got, want = out[e::E, 4 * u:4 * u + 4].double(), rows @ q * s
            bound = ((K / 32 + 8) * 2.0 ** -23 + 2.0 ** -21) * (rows.abs() @ q.abs()) * s
            assert torch.all((got - want).abs() <= bound), (u, e)


# Layers on each side of the rules, and the rows per tile of both products: few
# rows per expert on wide weights (decode kernels), row tiles of 16, 32 and 64
# (from 32 on the dispatch counts in them), K not a multiple of 32 (I = 1000), and
# the grouped GEMM's forms (f16 x: int8 limbs, an odd number of step pairs; f16
# pairs when I is not a multiple of 64; f32 x).
LAYERS = [(MoeConfig("t_wide3", 3, 1024, 16, 4, 2816, "f16"), 0),
          (MoeConfig("t_rows5", 40, 640, 32, 4, 640, "f32"), 16),
          (MoeConfig("t_rows20_i1000", 160, 768, 32, 4, 1000, "f16"), 16),
          (MoeConfig("t_rows40", 320, 640, 32, 4, 640, "f32"), 16),
          (MoeConfig("t_skew", 512, 640, 16, 2, 384, "f16", zipf=1.2, hot_share=0.5, empty=2), 16),
          (MoeConfig("t_limbs_odd", 300, 1024, 6, 2, 1088, "f16"), 16),
          (MoeConfig("t_rows20", 160, 256, 32, 4, 1408, "f16"), 32),
          (MoeConfig("t_rows20_f32", 160, 256, 32, 4, 1416, "f32"), 32),
          (MoeConfig("t_rows40_wide", 320, 256, 32, 4, 1408, "f16"), 64),
          (MoeConfig("t_rows40_f32", 320, 256, 32, 4, 1416, "f32"), 64),
          (MoeConfig("t_skew64", 320, 256, 32, 4, 1408, "f16", zipf=1.2, hot_share=0.5, empty=2), 64),
          (MoeConfig("g_limbs_odd", 1000, 1024, 20, 2, 1088, "f16"), 128),
          (MoeConfig("g_pairs_i1056", 1024, 1024, 8, 2, 1056, "f16"), 128),
          (MoeConfig("g_f32x", 1536, 1024, 8, 2, 1024, "f32"), 128)]
CHECKED = 150  # tokens checked against the oracle, spread over the call


@pytest.mark.parametrize("cfg,rows", LAYERS, ids=[c.name for c, _ in LAYERS])
def test_layer_paths(cfg, rows):
    print(f"layer path {cfg}", flush=True)
    assert expert_tiles("layer", cfg.T, cfg.d, cfg.I, cfg.E, cfg.k, cfg.x_dtype) == (rows, rows)
    inp = make_inputs(cfg, seed=12, keep_q=True, bias_rand=True)
    inp.residual.copy_(torch.randn(tuple(inp.residual.shape), generator=torch.Generator().manual_seed(6)))
    out, route = rt.moe_layer(inp.x, inp.router_w, inp.router_b, inp.glu, inp.lin, inp.down,
                              inp.residual, cfg.k, return_route=True)
    t = np.unique(np.linspace(0, cfg.T - 1, CHECKED).astype(int)) if cfg.T > 512 else np.arange(cfg.T)
    x = inp.x[t].float().cpu().numpy()
    want_route = ref.topk(ref.router_logits(x, inp.router_w.cpu().numpy(),
                                            inp.router_b.cpu().numpy()), cfg.k)
    w = {n: (ref.pack_ekn(inp.q[n].numpy(), 8), getattr(inp, n).scales.cpu().numpy(),
             getattr(inp, n).bias.cpu().numpy()) for n in ("glu", "lin", "down")}
    act = ref.moe_up(x, want_route, w["glu"], w["lin"], 8, cfg.d, cfg.E)
    want = ref.moe_down(act, want_route, w["down"], inp.residual[t].cpu().numpy(), 8, cfg.I, cfg.E)
    assert np.array_equal(route.cpu().numpy()[t, :cfg.k], want_route[:, :cfg.k])
    assert_close(out.cpu().numpy()[t], want, what=cfg.name)


# Dispatch over the routes of each sort kernel: one block (1, 2, 4 and 8
# chunks a wavefront, runs that end inside a chunk), three kernels above 8192
# assignments or 512 experts; ids that name no expert leave -1 at the end.
@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (63, 1, 5), (77, 4, 128), (257, 4, 130), (683, 3, 64),
                                   (1025, 4, 512), (1365, 6, 33), (2048, 4, 128), (2049, 4, 128),
                                   (40, 2, 700)])
def test_dispatch_one_block(T, k, E):
    print(f"dispatch T={T} k={k} E={E}", flush=True)
    rng = np.random.default_rng(T)
    route = np.ones((T, 2 * k), np.float32)
    route[:, :k] = rng.integers(0, E, (T, k))
    route[::5, 0] = rng.choice([-1.0, E, 0.5, np.nan], len(route[::5]))
    perm, off = rt.dispatch(torch.from_numpy(route).to(DEV), E)
    want_perm, _, want_off = ref.dispatch(route, E)
    np.testing.assert_array_equal(off.cpu().numpy(), want_off)
    np.testing.assert_array_equal(perm.cpu().numpy(), want_perm)


@pytest.mark.parametrize("T,hot", [(8192, 64), (8192, 1), (5000, 3), (1100, 2)])
def test_dispatch_experts_across_chunks(T, hot):
    """One block, up to eight chunks a wavefront, and an expert with rows in all
    of them: a chunk's places follow on those the chunk before it counted."""
    print(f"dispatch chunks T={T} hot={hot}", flush=True)
    E = 128
    route = np.ones((T, 2), np.float32)
    t = np.arange(T)
    route[:, 0] = np.where(t % 64 < hot, 7, t * 31 % E)
    perm, off = rt.dispatch(torch.from_numpy(route).to(DEV), E)
    want_perm, _, want_off = ref.dispatch(route, E)
    np.testing.assert_array_equal(off.cpu().numpy(), want_off)
    np.testing.assert_array_equal(perm.cpu().numpy(), want_perm)


@pytest.mark.parametrize("E,k", [(7, 3), (64, 8), (130, 4), (513, 16)])
def test_topk_special_logits(E, k):
    """Infinities, NaN, both zeros (equal, the lower id first), values at and
    below the −3.4e38 start, and rows with fewer candidates than k."""
    print(f"topk special E={E} k={k}", flush=True)
    rng = np.random.default_rng(E)
    x = rng.choice(np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, -3.4e38, -3.3e38, 1.5, -1.5,
                             1e-40, -1e-40], np.float32), (40, E))
    x[5] = -np.inf
    x[6] = np.nan
    x[7, 1:] = -np.inf
    x[8] = np.where(np.arange(E) % 2, 0.0, -0.0)
    with np.errstate(invalid="ignore", over="ignore"):
        want = ref.topk(x, k)
    got = rt.topk(torch.from_numpy(x).to(DEV), k).cpu().numpy()
    np.testing.assert_array_equal(got[:, :k], want[:, :k])
    np.testing.assert_allclose(got[:, k:], want[:, k:], atol=1e-7, rtol=1e-5, equal_nan=True)
