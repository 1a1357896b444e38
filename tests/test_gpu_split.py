"""The input and weight grads on split bf16 terms (split_gemm, wgrad_gemm),
against float64 on the CPU, where their tiles and chunks end: channels about
multiples of 16 and 32, output rows about 128, positions about 128 and 32,
windows that take all taps in one chunk and those that don't, and operands a
bf16 term cannot hold."""
import numpy as np
import pytest
import torch

from brosoundml_amd import native

pytestmark = pytest.mark.gpu
F = torch.nn.functional
P = native.ptr


@pytest.fixture(scope="module")
def K():
    return native.Context(0)


def rel(a, r):
    return float((a.double().cpu() - r).norm() / r.norm())


# A float dot product of n terms of one sign pattern errs by at most n 2^-24 of
# its terms' sum; the split one does no worse (24-bit operands, products to
# 2^-24 at worst and 2^-27.5 rms), so sqrt(n) 2^-24 of the result's norm bounds random terms: 2.2e-6 at
# the most terms here (1408), stated for all.
TOL = 2.5e-6


@pytest.mark.parametrize("N,ci,co,L,k,d", [
    (1, 1, 1, 1, 1, 1), (2, 127, 15, 127, 3, 1), (1, 128, 16, 128, 7, 3), (3, 129, 17, 129, 11, 5),
    (1, 128, 22, 401, 7, 1), (2, 128, 128, 1001, 11, 1), (1, 130, 40, 300, 11, 13), (1, 20, 20, 1500, 5, 200),
    (2, 22, 128, 257, 1, 1), (1, 1090, 64, 31, 3, 1), (1, 64, 128, 40000, 2, 9),
    (1, 35, 3, 200, 33, 1), (1, 5, 18, 300, 70, 1),  # weights packed in more than one group of taps
])
def test_dgrad_edges(K, N, ci, co, L, k, d):
    g = torch.Generator().manual_seed(ci * 1000 + L)
    rn = lambda *s: torch.randn(*s, generator=g)
    p = d * (k - 1) // 2
    Lo = L + 2 * p - d * (k - 1)
    w, dy = rn(co, ci * k), rn(N, co, Lo)
    dx = torch.full((N, ci, L), 7.0, device="cuda")
    wg, dyg = w.cuda(), dy.cuda()
    K.call("kdec_conv1d_dgrad", P(wg), P(dyg), co * Lo, P(dx), ci * L, N, ci, L, co, k, 1, p, d, 1.0, 0.0)
    w3 = w.double().reshape(co, ci, k)
    assert rel(dx, F.conv_transpose1d(dy.double(), w3, padding=p, dilation=d)) <= TOL


@pytest.mark.parametrize("value,where", [(v, w) for v in (np.inf, -np.inf, np.nan, 3.4e38) for w in "xw"] + [(1e-37, "x")])
def test_operands_past_bf16(K, value, where):
    # one such operand among ordinary ones: infinities and NaN where the float
    # product has them and nowhere else, large and tiny floats as themselves
    N, ci, co, L, k, p = 1, 130, 20, 300, 3, 1
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(N, co, L, generator=g), torch.rand(co, ci * k, generator=g) + 0.5
    if abs(value) < 1:
        x *= value
    elif where == "x":
        w *= 0.25
        x[0, 3, 150] = value
    else:
        x *= 0.1
        w[7, 4] = value
    y = torch.empty(N, ci, L, device="cuda")
    xg, wg = x.cuda(), w.cuda()
    K.call("kdec_conv1d_dgrad", P(wg), P(xg), co * L, P(y), ci * L, N, ci, L, co, k, 1, p, 1, 1.0, 0.0)
    ref = F.conv_transpose1d(x.double(), w.double().reshape(co, ci, k), padding=p)
    if np.isfinite(value):
        ref = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * np.inf, ref)
    got = y.double().cpu()
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
    f = ref.isfinite()
    assert (got[f] - ref[f]).norm() <= TOL * ref[f].norm()


@pytest.mark.parametrize("N,ci,co,L,k,s,d", [
    (1, 1, 1, 1, 1, 1, 1), (2, 31, 3, 33, 3, 1, 1), (1, 33, 127, 32, 3, 1, 5), (3, 32, 130, 31, 7, 1, 3),
    (1, 50, 128, 700, 11, 1, 5), (2, 20, 22, 257, 7, 1, 1), (1, 130, 64, 95, 1, 1, 1), (1, 9, 9, 900, 5, 1, 90),
    (2, 22, 40, 601, 12, 6, 1), (1, 1, 1, 131, 3, 2, 1), (1, 18, 20, 300, 4, 3, 5), (1, 40, 12, 500, 2, 1, 33),
    (1, 64, 128, 50001, 3, 1, 1),
    # few channels, all taps as channels; one channel more or one tap less, by taps
    (2, 1, 130, 333, 11, 1, 3), (1, 8, 20, 97, 31, 1, 1), (2, 16, 40, 260, 7, 1, 40), (1, 17, 9, 260, 7, 1, 1),
    (1, 1, 5, 401, 12, 2, 1), (1, 2, 3, 64, 2, 1, 1), (1, 40, 33, 130, 1, 3, 1), (1, 5, 7, 130, 2, 5, 1),
])
def test_wgrad_edges(K, N, ci, co, L, k, s, d):
    # column blocks of 32 channels by a tap (shared and separate windows), row
    # quads past C_out, chunks of 32 positions that end inside one, the
    # strided forms (a stride's phases as channels), and the bias sums
    g = torch.Generator().manual_seed(ci * 1000 + L)
    p = d * (k - 1) // 2
    Lo = (L + 2 * p - d * (k - 1) - 1) // s + 1
    x, dy = torch.randn(N, ci, L, generator=g), torch.randn(N, co, Lo, generator=g)
    dw, db = torch.ones(co, ci, k, device="cuda"), torch.ones(co, device="cuda")
    xg, dyg = x.cuda(), dy.cuda()
    K.call("kdec_conv1d_wgrad", P(xg), ci * L, P(dyg), co * Lo, P(dw), P(db), N, ci, L, co, k, s, p, d)
    xp = F.pad(x.double(), (p, p + s))
    cols = torch.stack([xp[:, :, t * d:t * d + (Lo - 1) * s + 1:s] for t in range(k)], 2)
    ref = 1.0 + torch.einsum("nml,nctl->mct", dy.double(), cols)
    assert rel(dw, ref) <= TOL
    assert rel(db, 1.0 + dy.double().sum((0, 2))) <= TOL


@pytest.mark.parametrize("k,s,L", [(20, 10, 33), (12, 6, 130), (3, 4, 9)])
def test_convt_wgrad_edges(K, k, s, L):
    N, ci, co, p = 2, 130, 24, max(0, (k - s) // 2)
    g = torch.Generator().manual_seed(k)
    Lo = (L - 1) * s - 2 * p + k
    x, dy = torch.randn(N, ci, L, generator=g), torch.randn(N, co, Lo, generator=g)
    dw = torch.zeros(ci, co, k, device="cuda")
    xg, dyg = x.cuda(), dy.cuda()
    K.call("kdec_convt1d_wgrad", P(xg), ci * L, P(dyg), co * Lo, P(dw), None, N, ci, L, co, k, s, p, 0)
    dp = F.pad(dy.double(), (p, p + s))
    cols = torch.stack([dp[:, :, t:t + (L - 1) * s + 1:s] for t in range(k)], 2)
    assert rel(dw, torch.einsum("nml,nctl->mct", x.double(), cols)) <= TOL


@pytest.mark.parametrize("value,where", [(v, w) for v in (np.inf, np.nan, 3.4e38) for w in ("x", "dy")])
def test_wgrad_operands_past_bf16(K, value, where):
    N, ci, co, L, k, p = 1, 40, 130, 300, 3, 1
    g = torch.Generator().manual_seed(6)
    x, dy = torch.randn(N, ci, L, generator=g) * 0.1, torch.randn(N, co, L, generator=g) * 0.1
    (x if where == "x" else dy)[0, 5, 150] = value
    dw = torch.zeros(co, ci, k, device="cuda")
    xg, dyg = x.cuda(), dy.cuda()
    K.call("kdec_conv1d_wgrad", P(xg), ci * L, P(dyg), co * L, P(dw), None, N, ci, L, co, k, 1, p, 1)
    xp = F.pad(x.double(), (p, p))
    ref = torch.stack([sum(torch.matmul(dy[n].double(), xp[n, :, t:t + L].t()) for n in range(N)) for t in range(k)], 2)
    got = dw.double().cpu()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    f = ref.isfinite()
    assert (got[f] - ref[f]).norm() <= TOL * ref[f].norm()


@pytest.mark.parametrize("N,ci,co,k,s,L", [
    (2, 130, 24, 20, 10, 33), (1, 127, 17, 12, 6, 130), (1, 9, 1, 3, 4, 9), (2, 20, 40, 5, 1, 140), (1, 64, 3, 7, 3, 257),
    (1, 30, 33, 1, 8, 260), (2, 9, 5, 3, 10, 40), (1, 130, 16, 7, 8, 31),
    (1, 40, 20, 32, 1, 90), (1, 33, 20, 32, 16, 9),
])
def test_convt_dgrad_edges(K, N, ci, co, k, s, L):
    # a stride's phases as channels: k a multiple of the stride and not, fewer
    # taps than phases, taps past k, channels that end inside a chunk
    g = torch.Generator().manual_seed(k)
    p = max(0, (k - s) // 2)
    Lo = (L - 1) * s - 2 * p + k
    w, dy = torch.randn(ci, co * k, generator=g), torch.randn(N, co, Lo, generator=g)
    dx = torch.full((N, ci, L), 7.0, device="cuda")
    wg, dyg = w.cuda(), dy.cuda()
    K.call("kdec_convt1d_dgrad", P(wg), P(dyg), co * Lo, P(dx), ci * L, N, ci, L, co, k, s, p, 0)
    assert rel(dx, F.conv1d(dy.double(), w.double().reshape(ci, co, k), stride=s, padding=p)[..., :L]) <= TOL


@pytest.mark.parametrize("value", [np.inf, np.nan, 3.4e38])
def test_convt_dgrad_operands_past_bf16(K, value):
    N, ci, co, k, s, p, L = 1, 40, 12, 12, 6, 3, 150
    g = torch.Generator().manual_seed(7)
    Lo = L * s
    w, dy = torch.rand(ci, co * k, generator=g) * 0.2, torch.randn(N, co, Lo, generator=g)
    dy[0, 3, 401] = value
    dx = torch.empty(N, ci, L, device="cuda")
    wg, dyg = w.cuda(), dy.cuda()
    K.call("kdec_convt1d_dgrad", P(wg), P(dyg), co * Lo, P(dx), ci * L, N, ci, L, co, k, s, p, 0)
    ref = F.conv1d(dy.double(), w.double().reshape(ci, co, k), stride=s, padding=p)
    got = dx.double().cpu()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    f = ref.isfinite()
    assert (got[f] - ref[f]).norm() <= TOL * ref[f].norm()


def bounded(got, ref, mag, n):
    # element by element: n terms of 24-bit operands err by at most n 2^-24 of
    # the sum of their magnitudes, and a result under 2^-126 by float's last step
    e = (got.double().cpu() - ref).abs()
    return bool((e <= n * 2.0 ** -24 * mag + 2.0 ** -148).all())


@pytest.mark.parametrize("e", [-104, -112, -118, -130])
@pytest.mark.parametrize("where", ["positions", "row", "all"])
@pytest.mark.parametrize("kind", ["dgrad", "convt_dgrad", "wgrad"])
def test_tiny_operands(K, kind, where, e):
    # operands about 2^e (subnormal ones too) in a few positions of the
    # gradient, in one row of the weights (of the gradient for a weight grad,
    # in one channel for "positions") or everywhere, beside ordinary ones: every
    # result to float precision by itself
    g = torch.Generator().manual_seed(-e)
    t = 2.0 ** e
    if kind == "wgrad":
        N, ci, co, L, k = 2, 40, 130, 70, 3
        x, dy = torch.randn(N, ci, L, generator=g), torch.randn(N, co, L, generator=g)
        if where == "positions":
            x[:, 5] *= t
        elif where == "row":
            dy[:, 70] *= t
        else:
            dy *= t
            x *= 1e3
        dw = torch.zeros(co, ci, k, device="cuda")
        xg, dyg = x.cuda(), dy.cuda()
        K.call("kdec_conv1d_wgrad", P(xg), ci * L, P(dyg), co * L, P(dw), None, N, ci, L, co, k, 1, 1, 1)
        f = lambda x, dy: torch.stack([sum(dy[n] @ F.pad(x[n], (1, 1))[:, j:j + L].t() for n in range(N)) for j in range(k)], 2)
        assert bounded(dw, f(x.double(), dy.double()), f(x.double().abs(), dy.double().abs()), N * L)
        return
    N, ci, co, L, k, s, p = (1, 130, 20, 300, 3, 1, 1) if kind == "dgrad" else (1, 130, 12, 150, 12, 6, 3)
    Lo = L * s
    dy = torch.randn(N, co, Lo, generator=g)
    w = torch.randn(*((co, ci, k) if kind == "dgrad" else (ci, co, k)), generator=g)
    if where == "positions":
        dy[:, :, 140 * s:160 * s] *= t
    elif where == "row":
        (w[:, 70] if kind == "dgrad" else w[70]).mul_(t)
    else:
        dy *= t
        w *= 1e3
    dx = torch.empty(N, ci, L, device="cuda")
    wg, dyg = w.cuda(), dy.cuda()
    if kind == "dgrad":
        K.call("kdec_conv1d_dgrad", P(wg), P(dyg), co * L, P(dx), ci * L, N, ci, L, co, k, 1, p, 1, 1.0, 0.0)
        f = lambda w, dy: F.conv_transpose1d(dy, w, padding=p)
    else:
        K.call("kdec_convt1d_dgrad", P(wg), P(dyg), co * Lo, P(dx), ci * L, N, ci, L, co, k, s, p, 0)
        f = lambda w, dy: F.conv1d(dy, w, stride=s, padding=p)
    assert bounded(dx, f(w.double(), dy.double()), f(w.double().abs(), dy.double().abs()), co * k)


def test_dgrad_refusals(K):
    # the forward's: more than 32 taps on a grid of a round of blocks or more,
    # a window past LDS; on a small grid the taps are taken
    def calls(N, c, L, k, d):
        p = d * (k - 1) // 2
        w, y = torch.ones(c, c * k, device="cuda"), torch.empty(N, c, L, device="cuda")
        x = torch.ones_like(y)
        yield lambda: K.call("kdec_conv1d_fwd", P(x), c * L, P(w), None, P(y), c * L, N, c, L, c, k, 1, p, d, None, 0, 1.0, 0.0)
        yield lambda: K.call("kdec_conv1d_dgrad", P(w), P(x), c * L, P(y), c * L, N, c, L, c, k, 1, p, d, 1.0, 0.0)

    for f in calls(1, 2, 128 * 4000, 33, 1):
        with pytest.raises(native.KdecError, match="bad chunk geometry"):
            f()
    for f in calls(1, 2, 128 * 4000, 31, 800):
        with pytest.raises(native.KdecError, match="does not fit LDS"):
            f()
    for f in calls(1, 2, 1000, 33, 1):
        f()


@pytest.mark.parametrize("kind", ["dgrad", "convt_dgrad"])
def test_large_weights(K, kind):
    # 1.6e9 weights: within 2^31 as floats, past it as split panels
    ci, co, k, s = (32768, 50000, 1, 1) if kind == "dgrad" else (32768, 25000, 2, 2)
    g = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randn(*((co, ci) if kind == "dgrad" else (ci, co * k)), generator=g, device="cuda")
    dy = torch.randn(1, co, k, generator=g, device="cuda")
    dx = torch.empty(1, ci, 1, device="cuda")
    if kind == "dgrad":
        K.call("kdec_conv1d_dgrad", P(w), P(dy), co, P(dx), ci, 1, ci, 1, co, 1, 1, 0, 1, 1.0, 0.0)
        ref = sum(w[c:c + 2000].double().t() @ dy[0, c:c + 2000, 0].double() for c in range(0, co, 2000))
    else:
        K.call("kdec_convt1d_dgrad", P(w), P(dy), co * k, P(dx), ci, 1, ci, 1, co, k, s, 0, 0)
        ref = torch.cat([w[m:m + 2048].double() @ dy.double().reshape(-1) for m in range(0, ci, 2048)])
    # 50 000 terms: sqrt(n) 2^-24
    assert rel(dx.reshape(-1), ref.cpu()) <= 1.4e-5


def test_dgrad_rows_past_2_27_bytes(K):
    # one channel of 2^28 positions: the chunk's other fifteen lie past the
    # input and read zero, so an infinity reaches three results and makes no NaN
    L, q = 1 << 28, 123_456_789
    w, dy = torch.full((1, 3), 0.5, device="cuda"), torch.zeros(1, 1, L, device="cuda")
    dy[0, 0, q] = float("inf")
    dy[0, 0, 5] = 2.0
    dx = torch.empty(1, 1, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(w), P(dy), L, P(dx), L, 1, 1, L, 1, 3, 1, 1, 1, 1.0, 0.0)
    assert torch.equal(dx[0, 0, q - 1:q + 2].cpu(), torch.full((3,), float("inf")))
    assert torch.equal(dx[0, 0, 4:7].cpu(), torch.ones(3))
    assert int(dx.count_nonzero()) == 6 and not bool(dx.isnan().any())


def families(K, f):
    """The profile's kernel families of one call."""
    K.profile(True)
    K.profile_reset()
    f()
    torch.cuda.synchronize()
    names = set(K.profile_read())
    K.profile(False)
    return names


@pytest.mark.parametrize("N,ci,co,L,k,d", [
    (1, 128, 128, 128 * 520 - 5, 3, 1),  # a round of whole tiles, eight in parts
    (259, 130, 96, 20, 31, 1),           # 518 tiles, 31 taps in parts that end between them
    (8, 1024, 1024, 100, 3, 1),          # less than a round, all in parts
    (1, 300, 260, 31, 11, 13),           # two tap groups per chunk
])
def test_dgrad_parts(K, N, ci, co, L, k, d):
    # tiles in parts (the profile shows their reduction), with whole ones and
    # without; dX = scale * sums + beta * dX
    g = torch.Generator().manual_seed(L)
    p = d * (k - 1) // 2
    w, dy, dx0 = (torch.randn(*s, generator=g) for s in ((co, ci * k), (N, co, L), (N, ci, L)))
    wg, dyg, dx = w.cuda(), dy.cuda(), dx0.cuda()
    f = lambda: K.call("kdec_conv1d_dgrad", P(wg), P(dyg), co * L, P(dx), ci * L, N, ci, L, co, k, 1, p, d, 0.5, 2.0)
    assert "tile_reduce" in families(K, f)
    ref = F.conv_transpose1d(dy.double(), w.double().reshape(co, ci, k), padding=p, dilation=d)
    # up to 3072 terms: sqrt(n) 2^-24
    assert rel(dx, 0.5 * ref + 2.0 * dx0.double()) <= 3.4e-6


@pytest.mark.parametrize("N,C,Co,L,k,d,act,with_r,parts", [
    (515, 256, 128, 20, 5, 1, 1, True, True),    # 1030 tiles, six in parts; taps at run time
    (515, 200, 128, 20, 3, 1, 2, True, True),    # a partial row tile, Snake
    (129, 128, 48, 1001, 11, 5, 2, False, True),  # 1032 tiles over row ends
    (515, 256, 96, 20, 5, 40, 0, False, True),   # tap groups
    (600, 256, 64, 20, 5, 1, 1, True, False),    # 1200 tiles, all whole
    (1024, 40, 20, 9, 1, 1, 2, True, False), (8, 128, 32, 128 * 128, 7, 1, 1, False, False),
])
def test_dgrad_adain_bwd_parts(K, N, C, Co, L, k, d, act, with_r, parts):
    # the AdaIN backward in the GEMM's epilogue and in the parts' reduction,
    # against the two calls the one replaces
    g = torch.Generator(device="cuda").manual_seed(C + L)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = d * (k - 1) // 2
    x, w, dy, r = rn(N, C, L) + 0.2, rn(Co, C * k) / (C * k) ** 0.5, rn(N, Co, L), rn(N, C, L)
    gm, bt, al = rn(N, C) * 0.4, rn(N, C) * 0.3, torch.rand(C, generator=g, device="cuda") + 0.5
    st, da0 = torch.empty(N * C, 2, device="cuda"), rn(C)
    K.call("kdec_instnorm_stats", P(x), C * L, N, C, L, 1e-5, P(st))
    R = P(r) if with_r else None
    got, ref = ([torch.empty(N, C, L, device="cuda"), torch.empty(N, C, device="cuda"), torch.empty(N, C, device="cuda"),
                 da0.clone()] for _ in range(2))
    out = lambda o: (P(o[0]), C * L, P(o[1]), P(o[2]), C, P(o[3]))
    fam = families(K, lambda: K.call(
        "kdec_conv1d_dgrad_adain_bwd", P(w), P(dy), Co * L, N, C, L, Co, k, 1, p, d, P(x), C * L, P(st), P(gm), P(bt), C,
        act, 0.2, P(al), R, C * L, *out(got)))
    assert ("tile_reduce" in fam) == parts
    t = torch.empty(N, C, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(w), P(dy), Co * L, P(t), C * L, N, C, L, Co, k, 1, p, d, 1.0, 0.0)
    K.call("kdec_adain_act_bwd", P(x), C * L, P(st), P(gm), P(bt), C, act, 0.2, P(al), P(t), C * L, R, C * L, *out(ref),
           N, C, L)
    # the same sums in another order: the row sums (L terms) and dalpha (N L terms) in double
    for a, b in zip(got, ref):
        assert rel(a, b.double().cpu()) <= 2e-6
