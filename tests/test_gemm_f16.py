"""The fp16 tile product (rh_gemm_f16 and its split, SiLU and merge forms) against float64.

Products of fp16 values are exact in fp32, so an output is off by its fp32 sum over K terms:
|y - y_exact| <= 4 K 2^-24 sum_k |w x| (+ 2^-23 |beta y| for the added term). SiLU * mul adds
one fp16 rounding (2^-11 of the value) and, through g and u, the sums' own bound.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS32 = 2.0 ** -24
# One token and one quad of rows, a token or row past a tile, N not a multiple of 4, one 64-k step
# to many, on the three smallest tiles; the edges of all six are below (test_every_tile).
SHAPES = [(1, 4, 64), (17, 100, 128), (64, 64, 576), (65, 129, 192), (129, 1000, 1536), (200, 577, 320),
          (300, 2500, 256), (513, 3000, 448), (520, 6146, 128)]


def make(T, N, K, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((N, K)) * 0.05).astype(np.float16), rng.standard_normal((T, K)).astype(np.float16)


def up(torch, dev, a):
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.float16 else a).to(dev)


def exact(w, x):
    wd, xd = w.astype(np.float64), x.astype(np.float64)
    return xd @ wd.T, 4 * w.shape[1] * EPS32 * (np.abs(xd) @ np.abs(wd).T) + 1e-30


def padded(w, ldw):
    out = np.full((w.shape[0], ldw), 99, np.float16)
    out[:, :w.shape[1]] = w
    return out


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("T,N,K", SHAPES)
def test_product_matches_float64(torch_mod, dev, T, N, K, beta):
    from relay_amd import _lib

    w, x = make(T, N, K, T + N + K)
    ldw = K + 8
    y0 = np.random.default_rng(1).standard_normal((T, N)).astype(np.float32)
    W, X, Y = up(torch_mod, dev, padded(w, ldw)), up(torch_mod, dev, x), up(torch_mod, dev, y0)
    print(f"gemm_f16 case: T={T} N={N} K={K} beta={beta}", flush=True)
    _lib.check(_lib.lib().rh_gemm_f16(W.data_ptr(), ldw, X.data_ptr(), Y.data_ptr(), T, K, N, beta, None), "rh_gemm_f16")
    torch_mod.cuda.synchronize()
    want, bound = exact(w, x)
    want = want + beta * y0.astype(np.float64)
    err = np.abs(Y.cpu().numpy() - want)
    assert (err <= bound + 2 * EPS32 * (np.abs(want) + np.abs(beta * y0))).all()


@pytest.mark.parametrize("ks", [2, 3, 8])
@pytest.mark.parametrize("T,N,K", [(17, 100, 576), (65, 576, 1536), (300, 1000, 512), (520, 6144, 1024)])
def test_partials_add_up(torch_mod, dev, T, N, K, ks):
    """Every range of the split is written whole (the workspace starts as NaN), with an uneven
    deal of the 64-k steps where ks does not divide them."""
    from relay_amd import _lib

    w, x = make(T, N, K, T + N + K + ks)
    W, X = up(torch_mod, dev, w), up(torch_mod, dev, x)
    ws = torch_mod.full((ks, T, N), float("nan"), device=dev)
    print(f"gemm_f16_partials case: T={T} N={N} K={K} ks={ks}", flush=True)
    _lib.check(_lib.lib().rh_gemm_f16_partials(W.data_ptr(), K, X.data_ptr(), T, K, N, ks, ws.data_ptr(), None),
               "rh_gemm_f16_partials")
    torch_mod.cuda.synchronize()
    p = ws.cpu().numpy().astype(np.float64)
    cuts = [z * (K // 64) // ks * 64 for z in range(ks + 1)]
    for z in range(ks):
        want, bound = exact(w[:, cuts[z]:cuts[z + 1]], x[:, cuts[z]:cuts[z + 1]])
        assert (np.abs(p[z] - want) <= bound).all(), f"range {z}"


def silu_bound(w, x, I):
    y, b = exact(w, x)
    g, u, bg, bu = y[:, :I], y[:, I:], b[:, :I], b[:, I:]
    s = g / (1 + np.exp(-g))
    want = s * u
    # |d silu| <= 1.1 |dg|; expf and the fp32 division and products: a few ulp of fp32
    return want, 1.1 * bg * np.abs(u) + np.abs(s) * bu + 1.1 * bg * bu + np.abs(want) * (2.0 ** -11 + 16 * EPS32) + 2.0 ** -25


@pytest.mark.parametrize("T,I,K", [(1, 8, 64), (17, 104, 128), (65, 577, 192), (200, 1536, 576), (520, 2500, 256)])
def test_gate_up_silu(torch_mod, dev, T, I, K):
    """SiLU * mul in the product's epilogue, and behind partials (I a multiple of 8)."""
    from relay_amd import _lib

    L = _lib.lib()
    w, x = make(T, 2 * I, K, T + I + K)
    want, bound = silu_bound(w, x, I)
    W, X = up(torch_mod, dev, w), up(torch_mod, dev, x)
    act = torch_mod.full((T, I), float("nan"), device=dev, dtype=torch_mod.float16)
    print(f"gemm_f16_gate_up_silu case: T={T} I={I} K={K}", flush=True)
    _lib.check(L.rh_gemm_f16_gate_up_silu(W.data_ptr(), K, X.data_ptr(), act.data_ptr(), T, K, I, None), "gate_up_silu")
    torch_mod.cuda.synchronize()
    assert (np.abs(act.cpu().numpy().astype(np.float64) - want) <= bound).all()
    if I % 8 == 0 and K >= 128:
        ws = torch_mod.full((2, T, 2 * I), float("nan"), device=dev)
        act.fill_(float("nan"))
        _lib.check(L.rh_gemm_f16_partials(W.data_ptr(), K, X.data_ptr(), T, K, 2 * I, 2, ws.data_ptr(), None), "partials")
        _lib.check(L.rh_f16_merge_silu(ws.data_ptr(), 2, T, I, act.data_ptr(), None), "merge_silu")
        torch_mod.cuda.synchronize()
        assert (np.abs(act.cpu().numpy().astype(np.float64) - want) <= bound).all()


# (rows of W, tokens) of the tiles and the stages of their LDS rings.
STAGES = {(64, 64): 4, (128, 64): 3, (128, 128): 4, (192, 128): 3, (256, 128): 3, (128, 256): 3}


def shape_on(L, rows, toks, steps, form):
    """The smallest T and N whose product of `steps` 64-k steps (a range of two for "ranges") runs this
    tile with one token past a tile and the fewest rows past one."""
    ks = 2 if form == "ranges" else 1
    past = {"plain": 1, "silu": 2, "ranges": 4}[form]
    best = None
    for a in range(40):
        for b in range(24):
            T, N = a * toks + 1, b * rows + past
            if (best is None or T * N < best[0] * best[1]) and L.rh_gemm_f16_tile(T, 64 * steps * ks, N, ks) == 1000 * rows + toks:
                best = (T, N)
    return best


@pytest.mark.parametrize("form", ["plain", "silu", "ranges"])
@pytest.mark.parametrize("rows,toks,steps", [(r, t, n) for (r, t), s in STAGES.items()
                                             for n in (1, s - 1, s, s + 1, 2 * s + 1, 3 * s + 2)
                                             if (r, t, n) != (192, 128, 1)])  # which the plan never runs
def test_every_tile(torch_mod, dev, rows, toks, steps, form):
    """Every tile and form at its row and token tails, with a ring that is not filled, just filled and
    refilled to its last buffer and past it; nothing is written past the outputs."""
    from relay_amd import _lib

    L, torch = _lib.lib(), torch_mod
    shape = shape_on(L, rows, toks, steps, form)
    assert shape is not None
    T, N = shape
    ks = 2 if form == "ranges" else 1
    K, ldw, beta = 64 * steps * ks, 64 * steps * ks + 8, float(steps % 2)
    print(f"gemm_f16 tile case: {rows} x {toks} {form} T={T} N={N} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(1000 * rows + toks + steps)
    w = (torch.randn(N, ldw, generator=g, device=dev) * 0.05).half()
    x = torch.randn(T, K, generator=g, device=dev).half()
    wd, xd = w[:, :K].double(), x.double()
    tail = 4096

    def product(k0, k1):
        a, b = xd[:, k0:k1].contiguous(), wd[:, k0:k1].contiguous()
        return a @ b.T, 4 * (k1 - k0) * EPS32 * (a.abs() @ b.abs().T) + 1e-30

    if form == "plain":
        out = torch.randn(T * N + tail, generator=g, device=dev)
        y0 = out.clone()
        _lib.check(L.rh_gemm_f16(w.data_ptr(), ldw, x.data_ptr(), out.data_ptr(), T, K, N, beta, None), "rh_gemm_f16")
        want, bound = product(0, K)
        added = beta * y0[:T * N].view(T, N).double()
        want = want + added
        bound = bound + 2 * EPS32 * (want.abs() + added.abs())
        assert bool(((out[:T * N].view(T, N).double() - want).abs() <= bound).all())
        assert torch.equal(out[T * N:], y0[T * N:])
    elif form == "ranges":
        out = torch.full((ks * T * N + tail,), float("nan"), device=dev)
        _lib.check(L.rh_gemm_f16_partials(w.data_ptr(), ldw, x.data_ptr(), T, K, N, ks, out.data_ptr(), None), "partials")
        for z in range(ks):
            want, bound = product(64 * steps * z, 64 * steps * (z + 1))
            assert bool(((out[z * T * N:(z + 1) * T * N].view(T, N).double() - want).abs() <= bound).all()), z
        assert bool(out[ks * T * N:].isnan().all())
    else:
        I = N // 2
        out = torch.full((T * I + tail,), float("nan"), device=dev, dtype=torch.float16)
        _lib.check(L.rh_gemm_f16_gate_up_silu(w.data_ptr(), ldw, x.data_ptr(), out.data_ptr(), T, K, I, None), "silu")
        y, b = product(0, K)
        gate, u, bg, bu = y[:, :I], y[:, I:], b[:, :I], b[:, I:]
        s = gate * torch.sigmoid(gate)
        want = s * u  # the bound as in silu_bound
        bound = 1.1 * bg * u.abs() + s.abs() * bu + 1.1 * bg * bu + want.abs() * (2.0 ** -11 + 16 * EPS32) + 2.0 ** -25
        assert bool(((out[:T * I].view(T, I).double() - want).abs() <= bound).all())
        assert bool(out[T * I:].isnan().all())


@pytest.mark.parametrize("ks,scaled", [(1, False), (3, False), (2, True)])
@pytest.mark.parametrize("heads,kvh,D", [(9, 3, 64), (4, 2, 128), (2, 1, 8)])
def test_qkv_post_merge_matches_the_chain(torch_mod, dev, heads, kvh, D, ks, scaled):
    """The ranges added in order (and scaled), then rh_qkv_post_to_cache: the same bytes."""
    from relay_amd import _lib

    L = _lib.lib()
    T, bs, N = 37, 16, (heads + 2 * kvh) * D
    rng = np.random.default_rng(D + ks)
    ws = rng.standard_normal((ks, T, N)).astype(np.float32)
    total = ws[0].copy()
    for z in range(1, ks):
        total += ws[z]
    scale = rng.uniform(0.5, 2.0, N).astype(np.float32)
    if scaled:
        total *= scale
    seq = (np.arange(T) >= 20).astype(np.int32)
    pos = np.where(seq == 0, np.arange(T), np.arange(T) + 41).astype(np.int32)
    toff = np.array([0, 2], np.int32)
    tables = rng.permutation(8).astype(np.int32)
    inv = (10000.0 ** (-np.arange(0, D, 2) / D)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    d = {k: up(torch_mod, dev, v) for k, v in dict(ws=ws, total=total, scale=scale, seq=seq, pos=pos, toff=toff,
                                                   tables=tables, inv=inv, bias=bias).items()}
    outs = []
    for merged in (False, True):
        k = torch_mod.zeros(8 * kvh * bs * D, device=dev, dtype=torch_mod.float16)
        v, q = torch_mod.zeros_like(k), torch_mod.zeros(T * heads * D, device=dev, dtype=torch_mod.float16)
        rest = (d["bias"].data_ptr(), d["inv"].data_ptr(), d["pos"].data_ptr(), d["seq"].data_ptr(), d["toff"].data_ptr(),
                d["tables"].data_ptr(), k.data_ptr(), v.data_ptr(), q.data_ptr(), 0.125, heads, kvh, D, bs, None)
        if merged:
            rc = L.rh_qkv_post_merge(d["ws"].data_ptr(), ks, d["scale"].data_ptr() if scaled else None, T, *rest)
        else:
            rc = L.rh_qkv_post_to_cache(d["total"].data_ptr(), T, *rest)
        _lib.check(rc, "qkv_post")
        torch_mod.cuda.synchronize()
        outs.append([a.cpu().numpy().view(np.int16) for a in (q, k, v)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_merge_rmsnorm_without_scale(torch_mod, dev):
    """x += the ranges, out = rh_rmsnorm of the sum: the same bytes as the unmerged chain."""
    from relay_amd import _lib

    L = _lib.lib()
    ks, T, H = 3, 19, 1028
    rng = np.random.default_rng(4)
    ws, x = rng.standard_normal((ks, T, H)).astype(np.float32), rng.standard_normal((T, H)).astype(np.float32)
    w = rng.standard_normal(H).astype(np.float32)
    m = ws[0].copy()
    for z in range(1, ks):
        m += ws[z]
    want = m + x
    dws, dx, dw, dwant = (up(torch_mod, dev, a) for a in (ws, x, w, want))
    out, ref = (torch_mod.zeros(T, H, device=dev, dtype=torch_mod.float16) for _ in range(2))
    _lib.check(L.rh_f16_merge_rmsnorm(dws.data_ptr(), ks, T, H, dx.data_ptr(), dw.data_ptr(), 1e-5, out.data_ptr(), None), "merge")
    _lib.check(L.rh_rmsnorm(dwant.data_ptr(), None, T, dw.data_ptr(), H, 1e-5, ref.data_ptr(), None), "rmsnorm")
    torch_mod.cuda.synchronize()
    assert np.array_equal(dx.cpu().numpy(), want)
    assert torch_mod.equal(out, ref)


def test_refusals(torch_mod, dev):
    from relay_amd import _lib

    L = _lib.lib()
    b = torch_mod.zeros(4096, device=dev)
    p = b.data_ptr()
    assert L.rh_gemm_f16(p, 96, p, p, 4, 96, 4, 0.0, None) != 0          # K not a multiple of 64
    assert L.rh_gemm_f16(p, 60, p, p, 4, 64, 4, 0.0, None) != 0          # ldw < K
    assert L.rh_gemm_f16(None, 64, p, p, 4, 64, 4, 0.0, None) != 0
    assert L.rh_gemm_f16(p, 64, p, p + 4, 4, 64, 4, 0.0, None) != 0      # y not 16-byte aligned
    assert L.rh_gemm_f16_partials(p, 128, p, 4, 128, 4, 3, p, None) != 0  # more ranges than steps
    assert L.rh_gemm_f16_partials(p, 128, p, 4, 128, 5, 2, p, None) != 0  # N not a multiple of 4
    assert L.rh_gemm_f16(p, 64, p, p, 0, 64, 4, 0.0, None) == 0
    assert L.rh_gemm_f16_fits(4, 96, 4) == 0 and L.rh_gemm_f16_fits(4, 64, 4) == 1
    assert L.rh_w8_merge_silu(p, 1, 4, 8, None, p, None) != 0
    assert L.rh_w8_merge_rmsnorm(p, 1, 4, 8, None, p, p, 1e-5, p, None) != 0
