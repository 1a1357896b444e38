"""GPU parity of every kdec kernel family against the CPU oracle.

Each test draws seeded inputs, runs the HIP kernel through the C ABI (torch
only provides device memory and the stream) and the oracle's restatement of
the reference op on the same inputs, utterance by utterance, and checks the
relative L2 error. Tolerances: 1e-5 for forward values, 1e-4 for gradients
(the bars the reference path's parity is stated at); the max abs error is
reported on failure.
"""
import ctypes

import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FWD_TOL = 1e-5
GRAD_TOL = 1e-4


def rel_l2(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def assert_close(got, ref, tol, what):
    e = rel_l2(got, ref)
    mx = float(np.max(np.abs(np.asarray(got, np.float64).ravel() - np.asarray(ref, np.float64).ravel())))
    assert e <= tol, f"{what}: rel-L2 {e:.3e} > {tol:.0e} (max-abs {mx:.3e})"


@pytest.fixture(scope="module")
def K():
    from brosoundml_amd import native
    return native.Context(0)


_keep = []  # device inputs stay referenced until the test ends


@pytest.fixture(autouse=True)
def _release_inputs():
    yield
    torch.cuda.synchronize()
    _keep.clear()


def g(x):
    t = torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda()
    _keep.append(t)
    return t


def h(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def P(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


rng = np.random.default_rng(20251201)


def rnd(*shape, scale=1.0):
    return (rng.standard_normal(shape) * scale).astype(np.float32)


CONV = [
    # N, C_in, C_out, L, k, s, p, d
    (2, 3, 5, 37, 3, 1, 1, 1),
    (2, 64, 64, 300, 11, 1, 25, 5),
    (2, 128, 128, 777, 7, 1, 9, 3),
    (1, 130, 200, 64, 3, 1, 1, 1),       # channel tails on both sides
    (2, 22, 96, 241, 12, 6, 3, 1),       # noise_convs stage-0 geometry
    (2, 40, 22, 150, 7, 1, 3, 1),        # conv_post geometry
    (2, 90, 70, 50, 1, 1, 0, 1),         # 1x1 shortcut
    (1, 1, 1, 16, 3, 2, 1, 1),           # F0_conv
]


@pytest.mark.parametrize("N,C_in,C_out,L,k,s,p,d", CONV)
def test_conv1d_fwd_dgrad_wgrad(K, N, C_in, C_out, L, k, s, p, d):
    Lo = O.conv1d_out_len(L, k, s, p, d)
    x, W, b = rnd(N, C_in, L), rnd(C_out, C_in * k, scale=0.2), rnd(C_out)
    R = rnd(N, C_out, Lo)
    Y = torch.empty(N, C_out, Lo, device="cuda")
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y), C_out * Lo, N, C_in, L, C_out, k, s,
           p, d, P(g(R)), C_out * Lo, 0.5, 0.0)
    ref = np.stack([0.5 * (O.conv1d(x[n], W, b, C_in, L, C_out, k, s, p, d).reshape(C_out, Lo) + R[n])
                    for n in range(N)])
    assert_close(h(Y), ref, FWD_TOL, "conv1d forward")
    dY = rnd(N, C_out, Lo)
    if s == 1:
        dX = torch.empty(N, C_in, L, device="cuda")
        K.call("kdec_conv1d_dgrad", P(g(W)), P(g(dY)), C_out * Lo, P(dX), C_in * L, N, C_in, L, C_out, k, s, p,
               d, 1.0, 0.0)
        ref = np.stack([O.conv1d_dgrad(W, dY[n], C_in, L, C_out, k, s, p, d) for n in range(N)])
        assert_close(h(dX), ref, GRAD_TOL, "conv1d backward_input")
    dW = torch.zeros(C_out, C_in * k, device="cuda")
    db = torch.zeros(C_out, device="cuda")
    K.call("kdec_conv1d_wgrad", P(g(x)), C_in * L, P(g(dY)), C_out * Lo, P(dW), P(db), N, C_in, L, C_out, k, s,
           p, d)
    rW = np.zeros(C_out * C_in * k)
    rb = np.zeros(C_out)
    for n in range(N):
        a, bb = O.conv1d_wgrad(x[n], dY[n], C_in, L, C_out, k, s, p, d)
        rW += a
        rb += bb
    assert_close(h(dW), rW, GRAD_TOL, "conv1d backward_weight")
    assert_close(h(db), rb, GRAD_TOL, "conv1d backward_bias")


@pytest.mark.parametrize("C_out,L", [
    (128, 4000),    # ~31 splits: partials in row quads, four split groups per column
    (22, 30000),    # C_out not a multiple of 4: row-major partials, 16-byte reduce, eight groups
    (128, 61441),   # hundreds of splits: row quads, eight groups
])
def test_conv1d_wgrad_split_plans(K, C_out, L):
    # The weight grad's split-K partial layouts and reduce plans against
    # torch's float64 weight grad, with the bias grad.
    N, C_in, k, d = 2, 128, 7, 3
    p = d * (k - 1) // 2
    x, dY = rnd(N, C_in, L, scale=0.5), rnd(N, C_out, L, scale=0.5)
    dW = torch.zeros(C_out, C_in * k, device="cuda")
    db = torch.zeros(C_out, device="cuda")
    K.call("kdec_conv1d_wgrad", P(g(x)), C_in * L, P(g(dY)), C_out * L, P(dW), P(db), N, C_in, L, C_out, k, 1, p,
           d)
    ref = torch.nn.grad.conv1d_weight(torch.from_numpy(x).double(), (C_out, C_in, k),
                                      torch.from_numpy(dY).double(), padding=p, dilation=d)
    assert_close(h(dW), ref.reshape(C_out, C_in * k).numpy(), GRAD_TOL, "conv1d backward_weight, split plans")
    assert_close(h(db), dY.astype(np.float64).sum(axis=(0, 2)), GRAD_TOL, "conv1d backward_bias, split plans")


@pytest.mark.parametrize("k,d", [(7, 3), (3, 1)])
def test_conv1d_grid_beyond_one_round(K, k, d):
    # 1301 output tiles: more than one round of resident blocks, so the
    # forward's last tiles run as channel-chunk parts reduced by tile_reduce
    # while the others run whole (the input grad's all run whole: its parts are
    # test_gpu_split.py's test_dgrad_parts). Reference: torch's float64 conv1d
    # on the CPU (the C oracle covers the same kernel at the small sizes above).
    N, C_in, C_out, L = 1, 32, 128, 128 * 1300 + 1
    p = d * (k - 1) // 2
    x, W, b = rnd(N, C_in, L), rnd(C_out, C_in * k, scale=0.2), rnd(C_out)
    R = rnd(N, C_out, L)
    Y = torch.empty(N, C_out, L, device="cuda")
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y), C_out * L, N, C_in, L, C_out, k, 1,
           p, d, P(g(R)), C_out * L, 0.5, 0.0)
    F = torch.nn.functional
    xt = torch.from_numpy(x).double()
    Wt = torch.from_numpy(W).double().reshape(C_out, C_in, k)
    ref = 0.5 * (F.conv1d(xt, Wt, torch.from_numpy(b).double(), padding=p, dilation=d) + torch.from_numpy(R).double())
    assert_close(h(Y), ref.numpy(), FWD_TOL, "conv1d forward, split tail tiles")
    dY = rnd(N, C_out, L)
    dX = torch.empty(N, C_in, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(g(W)), P(g(dY)), C_out * L, P(dX), C_in * L, N, C_in, L, C_out, k, 1, p, d,
           1.0, 0.0)
    ref = F.conv_transpose1d(torch.from_numpy(dY).double(), Wt, padding=p, dilation=d)
    assert_close(h(dX), ref.numpy(), GRAD_TOL, "conv1d backward_input, split tail tiles")


@pytest.mark.parametrize("k,d", [(11, 5), (3, 3)])
def test_conv1d_quad_panel_multi_tile(K, k, d):
    # Grids past one round of resident blocks at k = 3 / 7 / 11 run the
    # quad-packed weight kernel. Two output-channel tiles (C_out = 200) and
    # 40 input channels exercise the m-tile-major panel, the zero rows past
    # C_out and the zero channels past C_in, in the forward and (with the
    # roles swapped: 200 GEMM input channels, 40 output rows) the input grad.
    N, C_in, C_out, L = 2, 40, 200, 128 * 650 + 5
    p = d * (k - 1) // 2
    x, W, b = rnd(N, C_in, L), rnd(C_out, C_in * k, scale=0.1), rnd(C_out)
    Y = torch.empty(N, C_out, L, device="cuda")
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y), C_out * L, N, C_in, L, C_out, k, 1,
           p, d, None, 0, 1.0, 0.0)
    F = torch.nn.functional
    xt = torch.from_numpy(x).double()
    Wt = torch.from_numpy(W).double().reshape(C_out, C_in, k)
    ref = F.conv1d(xt, Wt, torch.from_numpy(b).double(), padding=p, dilation=d)
    assert_close(h(Y), ref.numpy(), FWD_TOL, "conv1d forward, quad panel")
    dY = rnd(N, C_out, L)
    dX = torch.empty(N, C_in, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(g(W)), P(g(dY)), C_out * L, P(dX), C_in * L, N, C_in, L, C_out, k, 1, p, d,
           1.0, 0.0)
    ref = F.conv_transpose1d(torch.from_numpy(dY).double(), Wt, padding=p, dilation=d)
    assert_close(h(dX), ref.numpy(), GRAD_TOL, "conv1d backward_input, quad panel")


@pytest.mark.parametrize("case", ["quad_residual", "split_tiles", "small_grid"])
def test_conv1d_fwd_stats(K, case):
    # kdec_conv1d_fwd_stats against kdec_conv1d_fwd + kdec_instnorm_stats:
    # Y bit for bit (the epilogue stores what the plain conv stores) and the
    # per-row (mean, rstd) within 1e-6, on the quad GEMM's whole tiles (C =
    # 128, 1400 tiles, residual and scale, rows with a large common offset),
    # with split tail tiles reduced by tile_reduce_stats (C = 256), and on a
    # small grid (the two calls). kdec_conv1d_fwd_stats_fused reports which.
    N, C_in, C_out, L, k, d, with_r, fused = {
        "quad_residual": (2, 128, 128, 128 * 700, 11, 5, True, 1),
        "split_tiles": (2, 256, 256, 128 * 330 - 9, 7, 3, False, 1),
        "small_grid": (1, 64, 96, 1000, 3, 1, True, 0),
    }[case]
    p = d * (k - 1) // 2
    x = rnd(N, C_in, L)
    W = rnd(C_out, C_in * k, scale=1.0 / np.sqrt(C_in * k))
    b = rnd(C_out) + 4.0  # an offset much larger than the rows' spread
    R = rnd(N, C_out, L) if with_r else None
    assert K.L.kdec_conv1d_fwd_stats_fused(K.h, N, C_in, L, C_out, k, 1, p, d) == fused
    Y0 = torch.empty(N, C_out, L, device="cuda")
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y0), C_out * L, N, C_in, L, C_out, k, 1, p, d,
           P(g(R) if with_r else None), C_out * L, 0.75, 0.0)
    st0 = torch.empty(N * C_out, 2, device="cuda")
    K.call("kdec_instnorm_stats", P(Y0), C_out * L, N, C_out, L, 1e-5, P(st0))
    Y1 = torch.empty(N, C_out, L, device="cuda")
    st1 = torch.empty(N * C_out, 2, device="cuda")
    K.call("kdec_conv1d_fwd_stats", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y1), C_out * L, N, C_in, L, C_out, k, 1,
           p, d, P(g(R) if with_r else None), C_out * L, 0.75, 1e-5, P(st1))
    np.testing.assert_array_equal(h(Y1), h(Y0))
    a, r = h(st1), h(st0)
    assert_close(a[:, 0], r[:, 0], 1e-6, f"fused statistics ({case}) mean")
    assert_close(a[:, 1], r[:, 1], 1e-6, f"fused statistics ({case}) rstd")


@pytest.mark.parametrize("case", ["quad_snake_residual", "split_tiles_leaky", "small_grid_none"])
def test_conv1d_dgrad_adain_bwd_fused(K, case):
    # kdec_conv1d_dgrad_adain_bwd against the two calls it replaces
    # (kdec_conv1d_dgrad, then kdec_adain_act_bwd, each checked against the
    # oracle elsewhere): the GEMM with the AdaIN epilogue on whole tiles (C =
    # 128, 1400 tiles, Snake, residual grad R; C = 256, 1320 tiles in two
    # output-channel tiles, leaky), and the two calls on a small grid (tiles in
    # parts are test_gpu_split.py's test_dgrad_adain_bwd_parts). dX, dgamma,
    # dbeta and dalpha (accumulated onto a nonzero start) agree to summation
    # order.
    N, C, Co, L, k, d, act, with_r = {
        "quad_snake_residual": (2, 128, 128, 128 * 700, 11, 5, "snake", True),
        "split_tiles_leaky": (2, 256, 256, 128 * 330 - 9, 7, 3, "leaky", False),
        "small_grid_none": (1, 64, 96, 1000, 3, 1, "none", True),
    }[case]
    p = d * (k - 1) // 2
    x = rnd(N, C, L, scale=1.3) + 0.2
    W = rnd(Co, C * k, scale=1.0 / np.sqrt(C * k))
    dYc = rnd(N, Co, L)
    gm, bt = rnd(N, C, scale=0.4), rnd(N, C, scale=0.3)
    alpha = rng.uniform(0.5, 2.0, C).astype(np.float32)
    R = rnd(N, C, L) if with_r else None
    st = torch.empty(N * C, 2, device="cuda")
    K.call("kdec_instnorm_stats", P(g(x)), C * L, N, C, L, 1e-5, P(st))
    a0 = rng.standard_normal(C).astype(np.float32)
    outs = []
    for fused in (False, True):
        dX = torch.empty(N, C, L, device="cuda")
        dg = torch.empty(N, C, device="cuda")
        db = torch.empty(N, C, device="cuda")
        da = g(a0).clone()
        if fused:
            K.call("kdec_conv1d_dgrad_adain_bwd", P(g(W)), P(g(dYc)), Co * L, N, C, L, Co, k, 1, p, d, P(g(x)),
                   C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2, P(g(alpha)), P(g(R) if with_r else None),
                   C * L, P(dX), C * L, P(dg), P(db), C, P(da))
        else:
            t = torch.empty(N, C, L, device="cuda")
            K.call("kdec_conv1d_dgrad", P(g(W)), P(g(dYc)), Co * L, P(t), C * L, N, C, L, Co, k, 1, p, d, 1.0, 0.0)
            K.call("kdec_adain_act_bwd", P(g(x)), C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2, P(g(alpha)),
                   P(t), C * L, P(g(R) if with_r else None), C * L, P(dX), C * L, P(dg), P(db), C, P(da), N, C, L)
        outs.append([h(dX), h(dg), h(db), h(da)])
    ref, got = outs
    for i, what in enumerate(("dX", "dgamma", "dbeta", "dalpha")):
        if what == "dalpha" and act != "snake":
            assert np.array_equal(got[i], a0), "dalpha changed for a non-Snake activation"
            continue
        assert_close(got[i], ref[i], 2e-6, f"fused dgrad + adain backward ({case}) {what}")


@pytest.mark.parametrize("k,d", [(3, 5), (11, 1)])
def test_conv1d_small_grid_split_parts(K, k, d):
    # 200 (forward) and 400 (input-grad) output tiles: fewer than one round of
    # resident blocks. The forward's tiles run their channel-chunk parts one
    # after the other in a block, the input grad's run whole (parts in blocks of
    # their own: test_gpu_small_grids.py's test_conv_fwd_parts, test_dgrad_parts).
    # Reference: torch float64.
    N, C_in, C_out, L = 2, 256, 128, 128 * 100 - 7
    p = d * (k - 1) // 2
    x, W, b = rnd(N, C_in, L), rnd(C_out, C_in * k, scale=0.1), rnd(C_out)
    Y = torch.empty(N, C_out, L, device="cuda")
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y), C_out * L, N, C_in, L, C_out, k, 1,
           p, d, None, 0, 1.0, 0.0)
    F = torch.nn.functional
    xt = torch.from_numpy(x).double()
    Wt = torch.from_numpy(W).double().reshape(C_out, C_in, k)
    ref = F.conv1d(xt, Wt, torch.from_numpy(b).double(), padding=p, dilation=d)
    assert_close(h(Y), ref.numpy(), FWD_TOL, "conv1d forward, split parts")
    dY = rnd(N, C_out, L)
    dX = torch.empty(N, C_in, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(g(W)), P(g(dY)), C_out * L, P(dX), C_in * L, N, C_in, L, C_out, k, 1, p, d,
           1.0, 0.0)
    ref = F.conv_transpose1d(torch.from_numpy(dY).double(), Wt, padding=p, dilation=d)
    assert_close(h(dX), ref.numpy(), GRAD_TOL, "conv1d backward_input, split parts")


def test_conv1d_batch_stride_and_accumulate(K):
    # outputs written into a channel slice of a wider tensor, beta accumulate
    N, C_in, C_out, L, k = 2, 16, 8, 40, 3
    x, W = rnd(N, C_in, L), rnd(C_out, C_in * k, scale=0.3)
    Ywide = g(rnd(N, C_out + 5, L))
    before = h(Ywide).copy()
    Yv = Ywide[:, 2:2 + C_out]
    K.call("kdec_conv1d_fwd", P(g(x)), C_in * L, P(g(W)), None, P(Yv), (C_out + 5) * L, N, C_in, L, C_out, k, 1,
           1, 1, None, 0, 1.0, 1.0)
    got = h(Ywide)
    ref = before.copy()
    for n in range(N):
        ref[n, 2:2 + C_out] += O.conv1d(x[n], W, None, C_in, L, C_out, k, 1, 1, 1).reshape(C_out, L)
    assert_close(got, ref, FWD_TOL, "strided accumulate")
    assert np.array_equal(got[:, :2], before[:, :2]) and np.array_equal(got[:, 2 + C_out:], before[:, 2 + C_out:])


CONVT = [
    # N, C_in, C_out, L, k, s, p
    (2, 64, 32, 40, 20, 10, 5),    # ups0 geometry
    (2, 32, 16, 50, 12, 6, 3),     # ups1 geometry
    (1, 5, 7, 13, 5, 3, 1),        # k not a multiple of s
    (2, 6, 4, 9, 4, 2, 1),
    (1, 3, 3, 11, 3, 1, 1),        # stride 1
]


@pytest.mark.parametrize("N,C_in,C_out,L,k,s,p", CONVT)
def test_convt1d(K, N, C_in, C_out, L, k, s, p):
    Lo = O.convt1d_out_len(L, k, s, p, 0, 1)
    x, W, b = rnd(N, C_in, L), rnd(C_in, C_out * k, scale=0.2), rnd(C_out)
    Y = torch.empty(N, C_out, Lo, device="cuda")
    K.call("kdec_convt1d_fwd", P(g(x)), C_in * L, P(g(W)), P(g(b)), P(Y), C_out * Lo, N, C_in, L, C_out, k, s, p, 0)
    ref = np.stack([O.convt1d(x[n], W, b, C_in, L, C_out, k, s, p) for n in range(N)])
    assert_close(h(Y), ref, FWD_TOL, "conv_transpose1d forward")
    dY = rnd(N, C_out, Lo)
    dX = torch.empty(N, C_in, L, device="cuda")
    K.call("kdec_convt1d_dgrad", P(g(W)), P(g(dY)), C_out * Lo, P(dX), C_in * L, N, C_in, L, C_out, k, s, p, 0)
    ref = np.stack([O.convt1d_dgrad(W, dY[n], C_in, L, C_out, k, s, p) for n in range(N)])
    assert_close(h(dX), ref, GRAD_TOL, "conv_transpose1d backward_input")
    dW = torch.zeros(C_in, C_out * k, device="cuda")
    db = torch.zeros(C_out, device="cuda")
    K.call("kdec_convt1d_wgrad", P(g(x)), C_in * L, P(g(dY)), C_out * Lo, P(dW), P(db), N, C_in, L, C_out, k, s,
           p, 0)
    rW, rb = np.zeros(C_in * C_out * k), np.zeros(C_out)
    for n in range(N):
        a, bb = O.convt1d_wgrad(x[n], dY[n], C_in, L, C_out, k, s, p)
        rW += a
        rb += bb
    assert_close(h(dW), rW, GRAD_TOL, "conv_transpose1d backward_weight")
    assert_close(h(db), rb, GRAD_TOL, "conv_transpose1d backward_bias")


@pytest.mark.parametrize("N,C_out,L,k,s,p", [
    (4, 256, 512, 20, 10, 5),    # one block per row, float4 reads (the ups0 backward case, 5120 outputs)
    (3, 130, 167, 12, 6, 3),     # one block per row, scalar reads (1002 outputs)
    (2, 128, 11667, 12, 6, 3),   # rows past 128 K positions (2 x 70002): slice partials, then their sum
])
def test_convt1d_bias_grad(K, N, C_out, L, k, s, p):
    """The transposed conv's bias grad alone (dW null): db += sum over (n, l)
    of dY[n, c, l], against a float64 sum, for both of its reduction plans."""
    C_in = 8
    Lo = O.convt1d_out_len(L, k, s, p, 0, 1)
    dY = rnd(N, C_out, Lo)
    db0 = rnd(C_out)
    db = g(db0)
    K.call("kdec_convt1d_wgrad", P(g(rnd(N, C_in, L))), C_in * L, P(g(dY)), C_out * Lo, None, P(db), N, C_in, L,
           C_out, k, s, p, 0)
    ref = db0.astype(np.float64) + dY.astype(np.float64).sum(axis=(0, 2))
    assert_close(h(db), ref, GRAD_TOL, "conv_transpose1d backward_bias")


def test_pool(K):
    N, C, L = 2, 9, 33
    x, W, b = rnd(N, C, L), rnd(C, 3), rnd(C)
    Y = torch.empty(N, C, 2 * L, device="cuda")
    K.call("kdec_pool_fwd", P(g(x)), C * L, P(g(W)), P(g(b)), P(Y), 2 * C * L, N, C, L)
    ref = np.stack([O.convt1d(x[n], W, b, C, L, C, 3, 2, 1, 1, 1, C) for n in range(N)])
    assert_close(h(Y), ref, FWD_TOL, "pool forward")
    dY = rnd(N, C, 2 * L)
    dX = torch.empty(N, C, L, device="cuda")
    K.call("kdec_pool_dgrad", P(g(W)), P(g(dY)), 2 * C * L, P(dX), C * L, N, C, L)
    ref = np.stack([O.convt1d_dgrad(W, dY[n], C, L, C, 3, 2, 1, 1, 1, C) for n in range(N)])
    assert_close(h(dX), ref, GRAD_TOL, "pool backward_input")
    dW = torch.zeros(C, 3, device="cuda")
    db = torch.zeros(C, device="cuda")
    K.call("kdec_pool_wgrad", P(g(x)), C * L, P(g(dY)), 2 * C * L, P(dW), P(db), N, C, L)
    rW, rb = np.zeros(C * 3), np.zeros(C)
    for n in range(N):
        a, bb = O.convt1d_wgrad(x[n], dY[n], C, L, C, 3, 2, 1, 1, 1, C)
        rW += a
        rb += bb
    assert_close(h(dW), rW, GRAD_TOL, "pool backward_weight")
    assert_close(h(db), rb, GRAD_TOL, "pool backward_bias")


ACTS = {"none": 0, "leaky": 1, "snake": 2}


@pytest.mark.parametrize("act", ["none", "leaky", "snake"])
# lengths cover every row-kernel shape (256x4, 256x16, 1024x16, 1024x48),
# with 4-byte accesses (L not a multiple of 4) and 16-byte ones, and the
# chunked path for longer rows
# rows held by one block up to 49152; rows of 49155..62464 with 16-B aligned
# bases and batch strides (C a multiple of 4 here) add a per-row head and
# rest, at every head offset c*L mod 4 (4 x 61441, the shortest such row
# 8 x 49155, the longest 4 x 62464); other long rows take the chunked passes
# (C = 2, 49153, and 70000)
@pytest.mark.parametrize("C,L", [(5, 31), (3, 1500), (16, 4099), (3, 8192), (2, 48000), (2, 61441), (2, 70000),
                                 (4, 61441), (8, 49155), (4, 49153), (4, 62464)])
def test_adain_act(K, act, C, L):
    N = 2
    x = rnd(N, C, L, scale=1.7) + 0.3
    gm, bt = rnd(N, C, scale=0.4), rnd(N, C, scale=0.3)
    alpha = rng.uniform(0.5, 2.0, C).astype(np.float32)
    st = torch.empty(N * C, 2, device="cuda")
    K.call("kdec_instnorm_stats", P(g(x)), C * L, N, C, L, 1e-5, P(st))
    Y = torch.empty(N, C, L, device="cuda")
    K.call("kdec_adain_act_fwd", P(g(x)), C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2, P(g(alpha)), P(Y),
           C * L, None, 0, N, C, L)
    refs = []
    for n in range(N):
        y = O.adain_affine(x[n], gm[n], bt[n], C, L)
        if act == "leaky":
            y = O.leaky(y, 0.2)
        elif act == "snake":
            y = O.snake(y, alpha, C, L)
        refs.append(y)
    assert_close(h(Y), np.stack(refs), FWD_TOL, f"adain+{act} forward")
    # statistics and affine + activation in one pass
    st2 = torch.empty(N * C, 2, device="cuda")
    Y2 = torch.empty(N, C, L, device="cuda")
    K.call("kdec_adain_act_fwd_stats", P(g(x)), C * L, 1e-5, P(st2), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2,
           P(g(alpha)), P(Y2), C * L, None, 0, N, C, L)
    assert_close(h(st2), h(st), 1e-6, f"adain+{act} fused statistics")
    assert_close(h(Y2), np.stack(refs), FWD_TOL, f"adain+{act} fused forward")

    dY = rnd(N, C, L)
    R = rnd(N, C, L)
    dX = torch.empty(N, C, L, device="cuda")
    dg = torch.empty(N, C, device="cuda")
    db = torch.empty(N, C, device="cuda")
    da = torch.zeros(C, device="cuda")
    K.call("kdec_adain_act_bwd", P(g(x)), C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2, P(g(alpha)),
           P(g(dY)), C * L, P(g(R)), C * L, P(dX), C * L, P(dg), P(db), C, P(da), N, C, L)
    rdx, rdg, rdb, rda = [], [], [], np.zeros(C)
    for n in range(N):
        s = O.adain_affine(x[n], gm[n], bt[n], C, L)
        ds = dY[n].ravel()
        if act == "leaky":
            ds = O.leaky_bwd(s, ds, 0.2)
        elif act == "snake":
            ds, a_ = O.snake_bwd(s, alpha, ds, C, L)
            rda += a_
        dx, dgg, dbb = O.adain_affine_bwd(x[n], gm[n], ds, C, L)
        rdx.append(dx + R[n].ravel())
        rdg.append(dgg)
        rdb.append(dbb)
    assert_close(h(dX), np.stack(rdx), GRAD_TOL, f"adain+{act} dX")
    assert_close(h(dg), np.stack(rdg), GRAD_TOL, f"adain+{act} dGamma")
    assert_close(h(db), np.stack(rdb), GRAD_TOL, f"adain+{act} dBeta")
    if act == "snake":
        assert_close(h(da), rda, GRAD_TOL, "snake dAlpha")


@pytest.mark.parametrize("C,L", [(3, 1500), (2, 70000)])
def test_adain_snake_large_arguments(K, C, L):
    # alpha in [6, 10] and (1 + gamma) ~ 9: |alpha * s| reaches several hundred,
    # where the Snake's sin^2 and the backward's (sin^2, sin 2th) come from a
    # multi-turn argument reduction; row kernel (1500) and chunked passes.
    # Inputs from a generator of the test's own, whatever ran before it.
    N = 2
    r = np.random.default_rng(1000 + L)
    x = (r.standard_normal((N, C, L)) * 1.1).astype(np.float32)
    gm = (8.0 + r.standard_normal((N, C)) * 0.5).astype(np.float32)
    bt = (r.standard_normal((N, C)) * 2.0).astype(np.float32)
    alpha = r.uniform(6.0, 10.0, C).astype(np.float32)
    st = torch.empty(N * C, 2, device="cuda")
    K.call("kdec_instnorm_stats", P(g(x)), C * L, N, C, L, 1e-5, P(st))
    Y = torch.empty(N, C, L, device="cuda")
    K.call("kdec_adain_act_fwd", P(g(x)), C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS["snake"], 0.0, P(g(alpha)),
           P(Y), C * L, None, 0, N, C, L)
    pre = [O.adain_affine(x[n], gm[n], bt[n], C, L) for n in range(N)]
    assert max(float(np.abs(p.reshape(C, L) * alpha[:, None]).max()) for p in pre) > 150.0
    assert_close(h(Y), np.stack([O.snake(pre[n], alpha, C, L) for n in range(N)]), FWD_TOL, "snake forward")
    dY = r.standard_normal((N, C, L)).astype(np.float32)
    dX = torch.empty(N, C, L, device="cuda")
    dg, db = torch.empty(N, C, device="cuda"), torch.empty(N, C, device="cuda")
    da = torch.zeros(C, device="cuda")
    K.call("kdec_adain_act_bwd", P(g(x)), C * L, P(st), P(g(gm)), P(g(bt)), C, ACTS["snake"], 0.0, P(g(alpha)),
           P(g(dY)), C * L, None, 0, P(dX), C * L, P(dg), P(db), C, P(da), N, C, L)
    rdx, rdg, rdb, rda = [], [], [], np.zeros(C)
    for n in range(N):
        ds, a_ = O.snake_bwd(pre[n], alpha, dY[n].ravel(), C, L)
        rda += a_
        dx, dgg, dbb = O.adain_affine_bwd(x[n], gm[n], ds, C, L)
        rdx.append(dx)
        rdg.append(dgg)
        rdb.append(dbb)
    assert_close(h(dX), np.stack(rdx), GRAD_TOL, "snake dX")
    assert_close(h(dg), np.stack(rdg), GRAD_TOL, "snake dGamma")
    assert_close(h(db), np.stack(rdb), GRAD_TOL, "snake dBeta")
    # d(alpha) = sum dY (th sin 2th - sin^2 th) / a^2 moves by about 2 th^2
    # times the rounding of s: at these arguments one ulp of s on half the
    # elements shifts it by 1e-5 to 4e-5 rel-L2 (measured with the oracle), and
    # the kernel's statistics differ from the oracle's by a few ulp in step
    # across a row. Against the oracle's own s it is therefore held to 4e-4,
    # and to the 1e-4 bar against s formed from the kernel's statistics
    # (float32, the kernel's order of operations), which leaves only the
    # kernel's own arithmetic.
    assert_close(h(da), rda, 4 * GRAD_TOL, "snake dAlpha (oracle statistics)")
    sk = h(st).reshape(N, C, 2)
    rda_k = np.zeros(C)
    for n in range(N):
        xh = (x[n] - sk[n, :, 0:1]) * sk[n, :, 1:2]
        s_k = ((np.float32(1.0) + gm[n])[:, None] * xh + bt[n][:, None]).astype(np.float32)
        rda_k += O.snake_bwd(s_k.ravel(), alpha, dY[n].ravel(), C, L)[1]
    assert_close(h(da), rda_k, GRAD_TOL, "snake dAlpha (kernel statistics)")


@pytest.mark.parametrize("act", ["leaky", "snake"])
# 4-byte row kernel (1500), 16-byte row kernel (8192), chunked passes (70000),
# long row with a head and rest (4 x 61441)
@pytest.mark.parametrize("C,L", [(3, 1500), (4, 8192), (2, 70000), (4, 61441)])
def test_adain_act_pre_activation_output(K, act, C, L):
    # Ypre, the AdaIN output before the activation, written beside Y
    N = 2
    x = rnd(N, C, L, scale=1.3) - 0.2
    gm, bt = rnd(N, C, scale=0.4), rnd(N, C, scale=0.3)
    alpha = rng.uniform(0.5, 2.0, C).astype(np.float32)
    st = torch.empty(N * C, 2, device="cuda")
    Y = torch.empty(N, C, L, device="cuda")
    Yp = torch.empty(N, C, L, device="cuda")
    K.call("kdec_adain_act_fwd_stats", P(g(x)), C * L, 1e-5, P(st), P(g(gm)), P(g(bt)), C, ACTS[act], 0.2,
           P(g(alpha)), P(Y), C * L, P(Yp), C * L, N, C, L)
    pre = np.stack([O.adain_affine(x[n], gm[n], bt[n], C, L) for n in range(N)])
    assert_close(h(Yp).reshape(N, -1), pre, FWD_TOL, f"adain+{act} pre-activation output")
    post = np.stack([O.leaky(pre[n], 0.2) if act == "leaky" else O.snake(pre[n], alpha, C, L) for n in range(N)])
    assert_close(h(Y).reshape(N, -1), post, FWD_TOL, f"adain+{act} output beside Ypre")


def test_elementwise(K):
    N, C, L = 2, 3, 17
    x = rnd(N, C, L)
    Y = torch.empty(N, C, L + 1, device="cuda")
    K.call("kdec_pad_reflect_left1_fwd", P(g(x)), C * L, P(Y), C * (L + 1), N, C, L)
    assert np.array_equal(h(Y), np.stack([O.pad_reflect_left1(x[n], C, L).reshape(C, L + 1) for n in range(N)]))
    dY = rnd(N, C, L + 1)
    dX = torch.empty(N, C, L, device="cuda")
    K.call("kdec_pad_reflect_left1_bwd", P(g(dY)), C * (L + 1), P(dX), C * L, N, C, L)
    assert_close(h(dX), np.stack([O.pad_reflect_left1_bwd(dY[n], C, L) for n in range(N)]), 1e-7, "pad bwd")
    Y2 = torch.empty(N, C, 2 * L, device="cuda")
    K.call("kdec_nearest2x_fwd", P(g(x)), C * L, P(Y2), 2 * C * L, N, C, L)
    assert np.array_equal(h(Y2), np.repeat(x, 2, axis=2))
    d2 = rnd(N, C, 2 * L)
    dx2 = torch.empty(N, C, L, device="cuda")
    K.call("kdec_nearest2x_bwd", P(g(d2)), 2 * C * L, P(dx2), C * L, N, C, L, 1.0, 0.0)
    assert_close(h(dx2), d2[..., 0::2] + d2[..., 1::2], 1e-7, "nearest2x bwd")
    Yl = torch.empty(N, C * L, device="cuda")
    K.call("kdec_leaky_fwd", P(g(x)), C * L, P(Yl), C * L, N, C * L, 0.1)
    assert np.array_equal(h(Yl).ravel(), O.leaky(x.ravel(), 0.1))
    F = torch.empty(1000, device="cuda")
    K.call("kdec_fill", P(F), 1000, 3.5)
    assert np.all(h(F) == 3.5)


@pytest.mark.parametrize("cols,bs,off", [(4096, 4096, 0), (4099, 4100, 0), (1024, 1028, 1)])
def test_add3_in_order(K, cols, bs, off):
    # (A + B) + C in float32, bit for bit: whole float4s on aligned rows of a
    # multiple of 4, the scalar path on a ragged row and on an offset base;
    # the output aliases A, as the generator's resblock sum uses it
    N = 3
    a, b, c = (rnd(N, bs + off) for _ in range(3))
    ref = (a[:, off:off + cols] + b[:, off:off + cols]) + c[:, off:off + cols]
    ta, tb, tc = g(a), g(b), g(c)
    pa, pb, pc = (ctypes.c_void_p(t.data_ptr() + 4 * off) for t in (ta, tb, tc))
    K.call("kdec_add3", pa, bs + off, pb, bs + off, pc, bs + off, pa, bs + off, N, cols)
    out = h(ta)
    assert np.array_equal(out[:, off:off + cols], ref.astype(np.float32))
    assert np.array_equal(out[:, :off], a[:, :off]) and np.array_equal(out[:, off + cols:], a[:, off + cols:])


@pytest.mark.parametrize("cols,bs", [(4096, 4096), (4099, 4100), (128 * 10241, 128 * 10241)])
def test_fused_elementwise_passes(K, cols, bs):
    # kdec_leaky_bwd_scaled against kdec_leaky_bwd and a scaling pass, and
    # kdec_add3_leaky against kdec_add3 and kdec_leaky_fwd, bit for bit (the
    # fused passes the generator runs in place of the pairs); aligned rows of
    # a multiple of 4 (the float4 path) and a ragged one; zeros and negative
    # zeros in the inputs
    N = 2
    x = rnd(N, bs)
    x[:, ::97] = 0.0
    x[:, 5::101] = -0.0
    dy = rnd(N, bs)
    tx, tdy = g(x), g(dy)
    got = torch.empty(N, bs, device="cuda")
    K.call("kdec_leaky_bwd_scaled", P(tx), bs, P(tdy), bs, P(got), bs, N, cols, 0.1, 1.0 / 3.0)
    t = torch.empty(N, bs, device="cuda")
    ref = torch.empty(N, bs, device="cuda")
    K.call("kdec_leaky_bwd", P(tx), bs, P(tdy), bs, P(t), bs, N, cols, 0.1)
    K.call("kdec_axpby", 1.0 / 3.0, P(t), bs, 0.0, None, 0, P(ref), bs, N, cols)
    assert torch.equal(got[:, :cols], ref[:, :cols])
    # the leaky backward against numpy's float32 arithmetic (exact), and
    # axpby with both operands
    xs, dys = x[:, :cols], dy[:, :cols]
    assert np.array_equal(h(t)[:, :cols], np.where(xs > 0, dys, np.float32(0.1) * dys))
    K.call("kdec_axpby", 0.5, P(tx), bs, -2.0, P(tdy), bs, P(ref), bs, N, cols)
    assert_close(h(ref)[:, :cols], 0.5 * xs.astype(np.float64) - 2.0 * dys.astype(np.float64), 1e-7, "axpby")
    a, b, c = g(rnd(N, bs)), g(rnd(N, bs)), g(rnd(N, bs))
    y, z = torch.empty(N, bs, device="cuda"), torch.empty(N, bs, device="cuda")
    K.call("kdec_add3_leaky", P(a), bs, P(b), bs, P(c), bs, P(y), bs, P(z), bs, N, cols, 0.01)
    y2, z2 = torch.empty(N, bs, device="cuda"), torch.empty(N, bs, device="cuda")
    K.call("kdec_add3", P(a), bs, P(b), bs, P(c), bs, P(y2), bs, N, cols)
    K.call("kdec_leaky_fwd", P(y2), bs, P(z2), bs, N, cols, 0.01)
    assert torch.equal(y[:, :cols], y2[:, :cols]) and torch.equal(z[:, :cols], z2[:, :cols])
    # Y aliasing A, as the generator calls it
    K.call("kdec_add3_leaky", P(a), bs, P(b), bs, P(c), bs, P(a), bs, P(z), bs, N, cols, 0.1)
    K.call("kdec_leaky_fwd", P(y2), bs, P(z2), bs, N, cols, 0.1)
    assert torch.equal(a[:, :cols], y2[:, :cols]) and torch.equal(z[:, :cols], z2[:, :cols])


@pytest.mark.parametrize("N,C,L", [(2, 3, 17), (1, 2, 2), (2, 5, 1023), (3, 4, 1024), (2, 128, 10240)])
def test_add3_unpad_left1(K, N, C, L):
    # the fused resblock-grad sum and reflect-pad adjoint against the two
    # passes it replaces, bit for bit, with Y aliasing A as the generator's
    # last stage calls it; row lengths either side of the 1024-sample blocks
    a, b, c = (rnd(N, C * (L + 1)) for _ in range(3))
    y_ref = ((a + b) + c).astype(np.float32).reshape(N, C, L + 1)
    z_ref = y_ref[..., 1:].copy()
    z_ref[..., 1] = z_ref[..., 1] + y_ref[..., 0]
    ta, tb, tc = g(a), g(b), g(c)
    Z = torch.empty(N, C * L, device="cuda")
    K.call("kdec_add3_unpad_left1", P(ta), C * (L + 1), P(tb), C * (L + 1), P(tc), C * (L + 1), P(ta), C * (L + 1),
           P(Z), C * L, N, C, L)
    assert np.array_equal(h(ta).reshape(N, C, L + 1), y_ref)
    assert np.array_equal(h(Z).reshape(N, C, L), z_ref)
    a2 = g(a)
    Z2 = torch.empty(N, C * L, device="cuda")
    K.call("kdec_add3", P(a2), C * (L + 1), P(tb), C * (L + 1), P(tc), C * (L + 1), P(a2), C * (L + 1), N, C * (L + 1))
    K.call("kdec_pad_reflect_left1_bwd", P(a2), C * (L + 1), P(Z2), C * L, N, C, L)
    assert torch.equal(Z, Z2) and torch.equal(ta, a2)


@pytest.mark.parametrize("n_fft,hop,L,C", [(20, 5, 301, 24), (8, 2, 65, 6)])
def test_spectral_head(K, n_fft, hop, L, C):
    N = 2
    k = 7
    x = rnd(N, C, L, scale=0.8)
    W = rnd(n_fft + 2, C * k, scale=0.3 / np.sqrt(C * k))
    b = rnd(n_fft + 2, scale=0.1)
    xl = torch.empty(N, C * L, device="cuda")
    K.call("kdec_leaky_fwd", P(g(x)), C * L, P(xl), C * L, N, C * L, 0.01)
    post = torch.empty(N, n_fft + 2, L, device="cuda")
    K.call("kdec_conv1d_fwd", P(xl), C * L, P(g(W)), P(g(b)), P(post), (n_fft + 2) * L, N, C, L, n_fft + 2, k, 1,
           3, 1, None, 0, 1.0, 0.0)
    S = (L - 1) * hop
    audio = torch.empty(N, S, device="cuda")
    K.call("kdec_spectral_fwd", P(post), (n_fft + 2) * L, None, P(audio), S, N, L, n_fft, hop)
    ref = [O.spectral_head(x[n], C, L, W, b, k, n_fft, hop) for n in range(N)]
    assert_close(h(audio), np.stack([r[0] for r in ref]), FWD_TOL, "spectral head forward")
    dA = rnd(N, S)
    dpost = torch.empty(N, n_fft + 2, L, device="cuda")
    K.call("kdec_spectral_bwd", P(post), (n_fft + 2) * L, None, P(g(dA)), S, P(dpost), (n_fft + 2) * L, N, L, n_fft,
           hop)
    dxl = torch.empty(N, C, L, device="cuda")
    K.call("kdec_conv1d_dgrad", P(g(W)), P(dpost), (n_fft + 2) * L, P(dxl), C * L, N, C, L, n_fft + 2, k, 1, 3, 1,
           1.0, 0.0)
    dx = torch.empty(N, C, L, device="cuda")
    K.call("kdec_leaky_bwd", P(g(x)), C * L, P(dxl), C * L, P(dx), C * L, N, C * L, 0.01)
    rdx = np.stack([O.spectral_head_bwd(x[n], C, L, W, b, k, n_fft, hop, dA[n])[0] for n in range(N)])
    assert_close(h(dx), rdx, GRAD_TOL, "spectral head backward")


def test_harmonic_source(K):
    # F0 with unvoiced (zero) frames; magnitudes compare tightly, phases only
    # where the bin holds energy (atan2 of a ~1e-8 bin is noise in any float
    # evaluation, CPU or GPU).
    N, fc, us, n_fft, hop = 2, 16, 60, 20, 5
    F0 = rng.uniform(80, 300, (N, fc)).astype(np.float32)
    F0[0, 3:6] = 0.0
    F0[1, 10] = 0.0
    lW = rnd(9, scale=0.3)
    lb = rnd(1, scale=0.1)
    frames = fc * us // hop + 1
    har = torch.empty(N, n_fft + 2, frames, device="cuda")
    K.call("kdec_harmonic_source", P(g(F0)), fc, P(har), (n_fft + 2) * frames, N, fc, P(g(lW)), P(g(lb)), 8, 24000,
           us, n_fft, hop)
    got = h(har)
    F = n_fft // 2 + 1
    for n in range(N):
        ref, fr = O.harmonic_source(F0[n], lW, lb, 8, 24000, us, n_fft, hop)
        assert fr == frames
        ref = ref.reshape(2 * F, frames)
        mag_ref, mag = ref[:F], got[n, :F]
        assert_close(mag, mag_ref, 1e-5, "harmonic source magnitude")
        strong = mag_ref > 1e-3 * mag_ref.max()
        dphi = np.angle(np.exp(1j * (got[n, F:][strong].astype(np.float64) - ref[F:][strong])))
        assert np.max(np.abs(dphi)) < 1e-3, f"phase error {np.max(np.abs(dphi))}"


@pytest.mark.parametrize("N,rows,S", [(3, 700, 128), (8, 37396, 128), (11, 1001, 128), (2, 95, 64), (4, 300, 256),
                                      (3, 77, 40), (2, 50, 16)])
def test_style_projection(K, N, rows, S):
    # the decoder's 37 396 fc rows at B = 8, ragged row blocks, more than one
    # pass of utterances, and style widths for both kernel families
    W, b = rnd(rows, S, scale=0.1), rnd(rows)
    st = rnd(N, S, scale=0.3)
    out = torch.empty(N, rows, device="cuda")
    K.call("kdec_style_proj_fwd", P(g(W)), P(g(b)), P(g(st)), S, P(out), rows, N, rows, S)
    ref = st.astype(np.float64) @ W.T.astype(np.float64) + b
    assert_close(h(out), ref, FWD_TOL, "style projection")
    dout = rnd(N, rows)
    dst = torch.empty(N, S, device="cuda")
    dW = torch.zeros(rows, S, device="cuda")
    db = torch.zeros(rows, device="cuda")
    K.call("kdec_style_proj_bwd", P(g(W)), P(g(st)), S, P(g(dout)), rows, P(dst), S, 0.0, P(dW), P(db), N, rows, S)
    assert_close(h(dst), dout.astype(np.float64) @ W.astype(np.float64), GRAD_TOL, "d(style)")
    assert_close(h(dW), dout.T.astype(np.float64) @ st.astype(np.float64), GRAD_TOL, "d(fc.weight)")
    assert_close(h(db), dout.sum(0), GRAD_TOL, "d(fc.bias)")


def test_error_paths(K):
    from brosoundml_amd import native
    # shape errors are reported, not launched
    with pytest.raises(native.KdecError, match="stride 1"):
        K.call("kdec_conv1d_dgrad", P(g(rnd(4, 6))), P(g(rnd(1, 4, 8))), 32, P(g(rnd(1, 2, 16))), 32, 1, 2, 16, 4,
               3, 2, 1, 1, 1.0, 0.0)
    with pytest.raises(native.KdecError):
        K.call("kdec_conv1d_fwd", None, 0, None, None, None, 0, 1, 1, 1, 1, 1, 1, 0, 1, None, 0, 1.0, 0.0)


@pytest.mark.parametrize("shared_gate", [False, True])
def test_lora_projection(K, shared_gate):
    # three AdaIN units (2C = 6, 10, 4 rows) stacked, N = 3 utterances, rank 5
    N, S, rank, scale = 3, 16, 5, 0.9
    sizes = [6, 10, 4]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    R, U = int(off[-1]), len(sizes)
    W, b = rnd(R, S, scale=0.3), rnd(R, scale=0.2)
    A, B = rnd(U * rank, S, scale=0.3), rnd(R, rank, scale=0.3)
    style = rnd(N, S)
    gate = rnd(1 if shared_gate else N, rank)
    g_bs = 0 if shared_gate else rank
    offd = torch.from_numpy(off).cuda()
    H = torch.empty(N, U * rank, device="cuda")
    out = torch.empty(N, R, device="cuda")
    K.call("kdec_lora_proj_fwd", P(g(W)), P(g(b)), P(g(A)), P(g(B)), P(g(gate)), g_bs, scale, P(offd), U, rank,
           P(g(style)), S, P(H), P(out), R, N, R, S)
    ref_y = np.zeros((N, R))
    ref_h = np.zeros((N, U * rank))
    for n in range(N):
        gn = gate[0 if shared_gate else n]
        for u in range(U):
            r0, r1 = off[u], off[u + 1]
            y, hh = O.lora_fwd(W[r0:r1], b[r0:r1], A[u * rank:(u + 1) * rank], B[r0:r1], gn, scale, style[n])
            ref_y[n, r0:r1] = y
            ref_h[n, u * rank:(u + 1) * rank] = hh
    assert_close(h(out), ref_y, FWD_TOL, "lora projection forward")
    dout = rnd(N, R)
    dstyle = torch.empty(N, S, device="cuda")
    dW = torch.zeros(R, S, device="cuda")
    db = torch.zeros(R, device="cuda")
    dA = torch.zeros(U * rank, S, device="cuda")
    dB = torch.zeros(R, rank, device="cuda")
    dG = torch.zeros(gate.shape[0], rank, device="cuda")
    K.call("kdec_lora_proj_bwd", P(g(W)), P(g(A)), P(g(B)), P(g(gate)), g_bs, scale, P(offd), U, rank,
           P(g(style)), S, P(H), P(g(dout)), R, P(dstyle), S, 0.0, P(dW), P(db), P(dA), P(dB), P(dG), N, R, S)
    rs = np.zeros((N, S)); rW = np.zeros((R, S)); rb = np.zeros(R)
    rA = np.zeros((U * rank, S)); rB = np.zeros((R, rank)); rG = np.zeros(gate.shape)
    for n in range(N):
        gi = 0 if shared_gate else n
        for u in range(U):
            r0, r1 = off[u], off[u + 1]
            gr = O.lora_bwd(W[r0:r1], A[u * rank:(u + 1) * rank], B[r0:r1], gate[gi], scale, style[n],
                            ref_h[n, u * rank:(u + 1) * rank].astype(np.float32), dout[n, r0:r1])
            rs[n] += gr["dstyle"]; rW[r0:r1] += gr["dW"]; rb[r0:r1] += gr["db"]
            rA[u * rank:(u + 1) * rank] += gr["dA"]; rB[r0:r1] += gr["dB"]; rG[gi] += gr["dG"]
    for name, got, ref in (("dstyle", dstyle, rs), ("dW", dW, rW), ("db", db, rb), ("dA", dA, rA), ("dB", dB, rB),
                           ("dG", dG, rG)):
        assert_close(h(got), ref, GRAD_TOL, f"lora projection {name}")


def test_length_regulate(K):
    # the reference's host loop is a per-phoneme repeat: np.repeat pins it;
    # two utterances of different totals in one padded batch, zero and
    # negative durations, frames past a total zero
    from brosoundml_amd import native
    r = np.random.default_rng(21)
    N, C, L, T = 2, 40, 37, 150
    te = r.normal(size=(N, C, L)).astype(np.float32)
    dur = r.integers(0, 5, size=(N, L)).astype(np.int32)
    dur[0, 3] = -2
    dur[1, :5] = 0
    out = torch.full((N, C, T), 7.0, device="cuda")
    totals = torch.zeros(N, dtype=torch.int32, device="cuda")
    t_dur = torch.from_numpy(dur).cuda()
    K.call("kdec_length_regulate", P(g(te)), C * L, P(t_dur), L, N, C, L, P(out), C * T, T, P(totals))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for n in range(N):
        d = np.maximum(dur[n], 0)
        ref = np.repeat(te[n], d, axis=1)[:, :T]
        assert totals[n].item() == d.sum()
        np.testing.assert_array_equal(got[n, :, :ref.shape[1]], ref)
        assert np.all(got[n, :, ref.shape[1]:] == 0.0)
    with pytest.raises(native.KdecError):
        K.call("kdec_length_regulate", P(g(te)), C * L - 1, P(t_dur), L, N, C, L, P(out), C * T, T, P(totals))
