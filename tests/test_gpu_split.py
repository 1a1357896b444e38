"""The input grads on split bf16 terms (split_gemm), against float64 on the
CPU, where their tiles and chunks end: channels about multiples of 16, output
rows about 128, positions about 128, windows that take all taps in one chunk and
those that don't, and operands a bf16 term cannot hold."""
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
# 2^-26), so sqrt(n) 2^-24 of the result's norm bounds random terms: 2.2e-6 at
# the most terms here (1408), stated for all.
TOL = 2.5e-6


@pytest.mark.parametrize("N,ci,co,L,k,d", [
    (1, 1, 1, 1, 1, 1), (2, 127, 15, 127, 3, 1), (1, 128, 16, 128, 7, 3), (3, 129, 17, 129, 11, 5),
    (1, 128, 22, 401, 7, 1), (2, 128, 128, 1001, 11, 1), (1, 130, 40, 300, 11, 13), (1, 20, 20, 1500, 5, 200),
    (2, 22, 128, 257, 1, 1), (1, 1090, 64, 31, 3, 1), (1, 64, 128, 40000, 2, 9),
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
