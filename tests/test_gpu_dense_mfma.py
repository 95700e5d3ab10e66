"""The f32 matrix-core kernels at the edges of their tiles, against f64:
k_linear (row tiles of 16 and 32, column tiles of 16, 32 and 64, K in whole
steps, quads or any), k_sdpa_mfma (row tiles, key steps, key parts) and
k_float_tile (row tiles of 16 and 32, K forms)."""
import numpy as np
import pytest
import torch

import runntime_amd as rt
from oracle import ref
from runntime_amd.linear import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# (T, K, N): 16 x 16 tiles up to 32 x 64 ones, the last of each partly empty;
# K of one step, past a step by 4 and by 1, fewer steps than wavefronts.
@pytest.mark.parametrize("T,K,N", [(1, 16, 1), (17, 20, 33), (16, 640, 64), (65, 640, 1152),
                                   (31, 132, 70), (321, 896, 644), (1000, 24, 260), (700, 647, 66),
                                   (160, 33, 1600), (65, 132, 1150)])
def test_linear_tiles(T, K, N):
    print(f"linear T={T} K={K} N={N}", flush=True)
    rng = np.random.default_rng(T + N)
    x, w = rng.standard_normal((T, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    b, a = rng.standard_normal(N).astype(np.float32), rng.standard_normal((T, N)).astype(np.float32)
    got = Linear(K, N, _dev(w), _dev(b)).forward(_dev(x), _dev(a)).cpu().numpy()
    xd, wd = x.astype(np.float64), w.astype(np.float64)
    want = xd @ wd + b + a
    mag = np.abs(xd) @ np.abs(wd) + np.abs(b) + np.abs(a)
    # chains of at most 32 products, then K / 32 sums, 8 parts, bias and addend
    np.testing.assert_array_less(np.abs(got - want), (32 + K / 32 + 12) * 2.0 ** -24 * mag + 1e-30)


# Rows of W so wide that 16 of them pass 32-bit offsets; K past a step, T past a
# row tile, an infinity in W's first row (K past K reads must not meet it).
@pytest.mark.parametrize("T,K,N", [(1, 3, (1 << 24) + 1), (17, 18, (1 << 24) + 35)])
def test_linear_more_than_2p24_columns(T, K, N):
    print(f"linear T={T} K={K} N={N}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randn((T, K), generator=g, device=DEV)
    w = torch.randn((K, N), generator=g, device=DEV)
    w[0, 5] = float("inf")
    b = torch.randn(N, generator=g, device=DEV)
    a = torch.randn((T, N), generator=g, device=DEV)
    got = Linear(K, N, w, b).forward(x, a)
    for c in (slice(0, 40), slice(N // 2 - 9, N // 2 + 50), slice(N - 60, N)):
        wc, bc, ac = w[:, c].double(), b[c].double(), a[:, c].double()
        want = torch.stack([(x[:, k:k + 1].double() * wc[k]) for k in range(K)]).sum(0) + bc + ac
        mag = (x.double().abs() @ wc.abs()) + bc.abs() + ac.abs()
        fin = torch.isfinite(want)
        assert torch.equal(got[:, c].double()[~fin], want[~fin])
        err = (got[:, c].double() - want)[fin].abs()
        assert torch.all(err <= (32 + 12) * 2.0 ** -24 * mag[fin] + 1e-30)


# Row tiles past a grid's second dimension, and outputs of more blocks than one
# grid holds threads for (16 x 16 tiles of 2^31 outputs and more).
@pytest.mark.parametrize("T,K,N", [(65535 * 32 + 33, 16, 64), (65535 * 32 + 33, 3, 1),
                                   (1050001, 1, 2047)])
def test_linear_many_rows(T, K, N):
    print(f"linear T={T} K={K} N={N}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randn((T, K), generator=g, device=DEV)
    w = torch.randn((K, N), generator=g, device=DEV)
    got = Linear(K, N, w).forward(x)
    for r in (slice(0, 40), slice(65535 * 16 - 20, 65535 * 16 + 20), slice(T - 40, T)):
        xr = x[r].double()
        err = (got[r].double() - xr @ w.double()).abs()
        assert torch.all(err <= (32 + 12) * 2.0 ** -24 * (xr.abs() @ w.double().abs()) + 1e-30)


@pytest.mark.parametrize("over", ["x", "addend", "w", "x shifted"])
def test_linear_into_its_inputs(over):
    """out over x (K = N), the addend, the weight (T = K), or rows below x's own:
    the result of a separate out."""
    print(f"linear into {over}", flush=True)
    from runntime_amd import _lib
    from runntime_amd.core import _ctx
    T = K = N = 640
    g = torch.Generator(device=DEV).manual_seed(9)
    buf = torch.randn((T + 8, K), generator=g, device=DEV)
    x = buf[:T]
    w = torch.randn((K, N), generator=g, device=DEV)
    a = torch.randn((T, N), generator=g, device=DEV)
    want = Linear(K, N, w.clone()).forward(x, a)
    out = {"x": x, "addend": a, "w": w, "x shifted": buf[8:]}[over]
    torch.cuda.synchronize()
    _lib.check(_lib.load().moe_linear(_ctx(x.device), x.data_ptr(), w.data_ptr(), None, a.data_ptr(),
                                      T, K, N, out.data_ptr()))
    torch.cuda.synchronize()
    assert torch.equal(out, want)


def test_linear_keeps_infinities_in_their_rows():
    print("linear infinities", flush=True)
    x = np.ones((40, 20), np.float32)
    x[7, 3], x[39, 19] = np.inf, np.nan
    w = np.ones((20, 33), np.float32)
    w[0, 5] = np.inf
    got = Linear(20, 33, _dev(w)).forward(_dev(x)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64)
    np.testing.assert_array_equal(got, want.astype(np.float32))


ATTN = [  # q_len, kv_len, q_heads, kv_heads, head_dim, left, right, offset, extra
    (1, 1, 2, 2, 64, -1, -1, 0, ""), (1, 300, 14, 2, 64, -1, -1, 299, ""),
    (15, 15, 14, 2, 64, 128, 128, 0, "sinks"), (17, 33, 3, 1, 128, 5, 0, 16, "sinks"),
    (33, 64, 8, 1, 64, 0, 0, 31, ""), (64, 64, 4, 2, 128, 40, 40, 0, "segments"),
    (97, 97, 9, 1, 64, 31, 7, 0, "segments sinks"), (50, 200, 2, 1, 64, -1, -1, 0, "bias"),
    (300, 300, 16, 2, 64, 128, 128, 0, "sinks"), (700, 700, 18, 2, 64, 30, 30, 0, "sinks"),
    # eight heads a block, the second block of a kv head with one of nine
    (500, 500, 72, 8, 64, 9, 3, 0, "segments sinks")]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("c", ATTN, ids=[f"q{c[0]}kv{c[1]}h{c[2]}-{c[3]}d{c[4]}" for c in ATTN])
def test_sdpa_tiles(dtype, c):
    qn, kn, qh, kh, hd, left, right, off, extra = c
    print(f"sdpa tiles {dtype} {c}", flush=True)
    rng = np.random.default_rng(qn + kn)
    npd = np.float16 if dtype == "f16" else np.float32
    q = (rng.standard_normal((qn, qh * hd)) * hd ** -0.25).astype(npd)
    k = (rng.standard_normal((kn, kh * hd)) * hd ** -0.25).astype(npd)
    v = rng.standard_normal((kn, kh * hd)).astype(npd)
    inf = float("inf")
    opts = {"qHeads": qh, "kvHeads": kh, "headDim": hd, "windowLeft": inf if left < 0 else left,
            "windowRight": inf if right < 0 else right, "qPosOffset": off}
    sinks = rng.standard_normal(qh).astype(np.float32) if "sinks" in extra else None
    segs = None
    if "segments" in extra:  # rows 10 to 19 see nothing
        cut = np.array([0, kn // 3, kn // 2, kn])
        seg = np.searchsorted(cut, np.arange(qn), side="right") - 1
        segs = np.stack([cut[seg], cut[seg + 1]], 1).astype(np.float32)
        segs[10:20] = (4, 4)
    score = np.zeros((qh, qn, kn))
    out = np.zeros((qn, qh * hd))
    pos = off + np.arange(qn)[:, None]
    key = np.arange(kn)[None, :]
    seen = np.ones((qn, kn), bool)
    if left >= 0:
        seen &= key >= pos - left
    if right >= 0:
        seen &= key <= pos + right
    if segs is not None:
        seen &= (key >= segs[:, :1]) & (key < segs[:, 1:])
    kb = {"start": 3, "end": kn // 2, "value": -1.5} if "bias" in extra else None
    for h in range(qh):
        g = h // (qh // kh)
        s = q[:, h * hd:(h + 1) * hd].astype(np.float64) @ k[:, g * hd:(g + 1) * hd].astype(np.float64).T
        if kb:
            s[:, kb["start"]:kb["end"]] += kb["value"]
        e = np.where(seen, np.exp(s - s.max(1, keepdims=True)), 0.0)
        den = e.sum(1, keepdims=True)
        if sinks is not None:
            den = den + np.exp(float(sinks[h]) * np.log(2.0) - s.max(1, keepdims=True))
        out[:, h * hd:(h + 1) * hd] = np.divide(e, den, out=np.zeros_like(e), where=den > 0) \
            @ v[:, g * hd:(g + 1) * hd].astype(np.float64)
    if sinks is not None:
        opts["sinks"] = _dev(sinks)
    if segs is not None:
        opts["segments"] = _dev(segs)
    if kb:
        opts["keyBias"] = kb
    got = rt.sdpa(_dev(q), _dev(k), _dev(v), opts).float().cpu().numpy()
    # f32 sums of head_dim and of the probabilities; f16 outputs round to 11 bits
    np.testing.assert_allclose(got, out, atol=(2e-5 if dtype == "f32" else 1e-3 * np.abs(v).max()),
                               rtol=(1e-4 if dtype == "f32" else 1e-3))


# An infinity or a NaN in V reaches the rows that see its key, and no other row
# of its 16-row tile: one step of keys, several, keys split over wavefronts,
# several heads a block; the last key, which pads a tile's last step.
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n,qh,kh,hd,left,right", [(70, 4, 2, 64, 9, 4), (70, 3, 1, 128, 40, 3),
                                                   (300, 14, 2, 64, 60, 60), (500, 72, 8, 64, 5, 0)])
def test_sdpa_keeps_infinities_from_rows_that_do_not_see_them(dtype, n, qh, kh, hd, left, right):
    print(f"sdpa infinities {dtype} {n} {qh}/{kh} {hd} {left} {right}", flush=True)
    rng = np.random.default_rng(n + hd)
    npd = np.float16 if dtype == "f16" else np.float32
    q = (rng.standard_normal((n, qh * hd)) * hd ** -0.25).astype(npd)
    k = (rng.standard_normal((n, kh * hd)) * hd ** -0.25).astype(npd)
    v = rng.standard_normal((n, kh * hd)).astype(npd)
    v[20], v[33, 3::5], v[n - 1, ::2] = np.inf, np.nan, -np.inf
    cut = np.array([0, 21, n // 2, n])
    seg = np.searchsorted(cut, np.arange(n), side="right") - 1
    segs = np.stack([cut[seg], cut[seg + 1]], 1).astype(np.float32)
    segs[10] = (4, 4)
    want = np.zeros((n, qh * hd))
    for r in range(n):
        lo, hi = int(max(r - left, segs[r, 0])), int(min(r + right + 1, segs[r, 1]))
        for h in range(qh if hi > lo else 0):
            c, g = slice(h * hd, (h + 1) * hd), h // (qh // kh)
            cg = slice(g * hd, (g + 1) * hd)
            s = k[lo:hi, cg].astype(np.float64) @ q[r, c].astype(np.float64)
            e = np.exp(s - s.max())
            with np.errstate(invalid="ignore"):
                want[r, c] = (e / e.sum()) @ v[lo:hi, cg].astype(np.float64)
    got = rt.sdpa(_dev(q), _dev(k), _dev(v),
                  {"qHeads": qh, "kvHeads": kh, "headDim": hd, "windowLeft": left, "windowRight": right,
                   "segments": _dev(segs)}).float().cpu().numpy()
    np.testing.assert_allclose(got, want, atol=2e-5 if dtype == "f32" else 4e-3,
                               rtol=1e-4 if dtype == "f32" else 1e-3)


@pytest.mark.parametrize("hd", [64, 32])  # k_sdpa_mfma, k_sdpa
def test_sdpa_windows_of_any_size(hd):
    """The C entry takes 64-bit windows: one past every key is unbounded, up to
    the largest, where a position plus the window would pass 64 bits."""
    print(f"sdpa windows {hd}", flush=True)
    from runntime_amd.core import _sdpa_launch
    n = 40
    g = torch.Generator(device=DEV).manual_seed(hd)
    q, k, v = (torch.randn((n, hd), generator=g, device=DEV) for _ in range(3))

    def run(left, right):
        return _sdpa_launch(q.device, q.data_ptr(), hd, k.data_ptr(), hd, v.data_ptr(), hd, n, n, 1, 1,
                            hd, left, right, 0, None, None, None, torch.float32)
    every, behind = run(-1, -1), run(-1, 2)
    want = torch.softmax(q.double() @ k.double().T, -1) @ v.double()
    torch.testing.assert_close(every.double(), want, atol=2e-5, rtol=1e-4)
    for big in (n, (1 << 31) - 1, 1 << 31, (1 << 32) - 1, 1 << 32, (1 << 63) - 1):
        # a bounded side may split the keys over wavefronts otherwise
        torch.testing.assert_close(run(big, big), every, atol=4e-5, rtol=1e-4)
        torch.testing.assert_close(run(big, 2), behind, atol=4e-5, rtol=1e-4)


# Rows per expert from one to a second 32-row tile; K whole steps, past one by
# 4, and odd; N a partial column block; few blocks, and 16-row tiles of 512 and
# more (no step ahead).
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("M,K,N,E", [(1, 16, 4, 1), (33, 36, 68, 2), (200, 640, 132, 40),
                                     (130, 19, 64, 3), (90, 48, 260, 90), (700, 260, 72, 16),
                                     (120, 640, 260, 120), (120, 260, 260, 120), (120, 19, 260, 120)])
def test_float_tiles(dtype, M, K, N, E):
    print(f"float tiles {dtype} M={M} K={K} N={N} E={E}", flush=True)
    rng = np.random.default_rng(M + K)
    npd = np.float16 if dtype == "f16" else np.float32
    a = rng.standard_normal((M, K)).astype(npd)
    w = rng.standard_normal((E * K, N)).astype(npd)
    b = rng.standard_normal((E, N)).astype(npd)
    idx = rng.integers(0, E, M).astype(np.float32)
    idx[::9] = -1.0
    got = rt.matmulGather(_dev(a), _dev(w), _dev(idx), {"bias": _dev(b)}).float().cpu().numpy()
    want, mag = np.zeros((M, N)), np.zeros((M, N))
    for e in range(E):
        r, we = idx == e, w[e * K:(e + 1) * K].astype(np.float64)
        want[r] = a[r].astype(np.float64) @ we + b[e]
        mag[r] = np.abs(a[r].astype(np.float64)) @ np.abs(we) + np.abs(b[e].astype(np.float64))
    eps = (16 + K / 16 + 10) * 2.0 ** -24
    bound = eps * mag + (2.0 ** -11 * np.abs(want) + 1e-7 if dtype == "f16" else 0.0) + 1e-30
    np.testing.assert_array_less(np.abs(got - want), bound)


# K past what a block's rows would fill in LDS (none are kept there): up and down,
# one row an expert and many, at d and I of 4100.
@pytest.mark.parametrize("T", [2, 40])
def test_float_block_of_long_rows(T):
    print(f"float block long rows T={T}", flush=True)
    from tests.helpers import assert_close
    d, I, E, k = 4100, 4100, 4, 2
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, d)).astype(np.float32)
    norm = np.ones(d, np.float32)
    rw = (0.02 * rng.standard_normal((d, E))).astype(np.float32)
    rb = np.zeros(E, np.float32)
    mk = lambda n, m, s: (s * rng.standard_normal((E * n, m))).astype(np.float32)
    glu, lin, down = mk(d, I, d ** -0.5), mk(d, I, d ** -0.5), mk(I, d, I ** -0.5)
    zi, zd = np.zeros((E, I), np.float32), np.zeros((E, d), np.float32)
    out, route = rt.moe_block_float(_dev(x), _dev(norm), 1e-5, _dev(rw), _dev(rb), _dev(glu), _dev(zi),
                                    _dev(lin), _dev(zi), _dev(down), _dev(zd), k=k, return_route=True)
    xn = ref.rmsnorm(x, norm, 1e-5)
    want_route = ref.topk(ref.router_logits(xn, rw, rb), k)
    assert np.array_equal(route.cpu().numpy()[:, :k], want_route[:, :k])
    want = ref.moe_block_float_f64(x, xn, want_route, (glu, zi), (lin, zi), (down, zd), k)
    assert_close(out.cpu().numpy(), want, atol=1e-4, rtol=1e-4, what="long rows")


# Weight rows so wide that 16 of them pass 32-bit offsets: 16- and 32-row tiles,
# K past a step, an infinity in an expert's first row.
@pytest.mark.parametrize("dtype,M,K", [("f32", 3, 5), ("f16", 40, 3), ("f32", 15, 18)])
def test_float_more_than_2p24_columns(dtype, M, K):
    print(f"float columns {dtype} M={M} K={K}", flush=True)
    E, N = 2, (1 << 24) + 36
    td = torch.float16 if dtype == "f16" else torch.float32
    g = torch.Generator(device=DEV).manual_seed(M)
    a = torch.randn((M, K), generator=g, device=DEV).to(td)
    w = torch.randn((E * K, N), generator=g, device=DEV).to(td)
    w[K, 4] = float("inf")
    idx = (torch.arange(M, device=DEV) % E).float()
    got = rt.matmulGather(a, w, idx, {"bias": torch.zeros((E, N), device=DEV, dtype=td)})
    for c in (slice(0, 70), slice(N // 2, N // 2 + 64), slice(N - 68, N)):
        for e in range(E):
            r, we = a[e::E].double(), w[e * K:(e + 1) * K, c].double()
            want = torch.stack([r[:, k:k + 1] * we[k] for k in range(K)]).sum(0)
            have, fin = got[e::E, c].double(), torch.isfinite(want)
            assert torch.equal(have[~fin], want[~fin])
            bound = (16 + 10) * 2.0 ** -24 * (r.abs() @ we.abs())[fin]
            if dtype == "f16":
                bound = bound + 2.0 ** -11 * want[fin].abs() + 1e-7
            assert torch.all((have - want)[fin].abs() <= bound + 1e-30)


def test_float_more_outputs_than_a_grid():
    """Past 2^34 outputs, 32-row tiles of 64 columns and eight wavefronts are more
    threads than one grid holds."""
    M, N = (1 << 22) + 40, 4096
    print(f"float outputs {M} x {N}", flush=True)
    a = ((torch.arange(M, device=DEV) % 1021) - 510).to(torch.float16).reshape(M, 1)
    w = ((torch.arange(N, device=DEV) % 7) - 3).to(torch.float16).reshape(1, N)
    got = rt.matmulGather(a, w, torch.zeros(M, device=DEV),
                          {"bias": torch.zeros((1, N), device=DEV, dtype=torch.float16)})
    for r in range(0, M, 1 << 20):
        assert torch.equal(got[r:r + (1 << 20)], a[r:r + (1 << 20)] * w), r
