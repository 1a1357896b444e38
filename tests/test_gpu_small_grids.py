"""The stride-1 forwards on grids of less than a round of blocks (corr_gemm),
and the style projection's weight grad, against float64 on the CPU where their
tiles, chunks, parts and staging forms end."""
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


# Float sums of up to 3270 random terms err by about sqrt(n) 2^-24 of the
# result's norm (3.4e-6 at most here); half of that is seen.
TOL = 3.5e-6


@pytest.mark.parametrize("N,ci,co,L,k,d", [
    (1, 1, 1, 1, 1, 1),            # less than one of everything
    (1, 1090, 1024, 21, 3, 1),     # parts, one 32-column block per tile
    (1, 1090, 200, 33, 3, 1),      # parts, the second block of a tile with one column
    (2, 40, 130, 500, 3, 3),       # an odd octet at the end, a partial row tile
    (1, 128, 128, 7681, 7, 5),     # all parts in one block, plan chunks of 4 and 3 taps
    (1, 128, 128, 24121, 11, 5),   # parts that end inside an octet
    (2, 120, 128, 20001, 3, 1),    # all parts in one block, an odd count of octets
    (1, 128, 22, 24121, 7, 1),
    (1, 64, 40, 3000, 2, 1), (1, 24, 40, 3000, 5, 1), (1, 200, 512, 400, 1, 1),
    (1, 32, 64, 2000, 5, 60),      # a window past the staging items: taps in groups
    (1, 32, 64, 2000, 3, 300),     # taps further apart than the block's columns
    (1, 40, 64, 2000, 5, 200), (4, 32, 64, 20000, 5, 200),  # those in blocks of 32 and of 64 columns, all at once
    (1, 40, 64, 2000, 7, 100), (1, 24, 130, 400, 11, 33), (4, 24, 64, 20000, 7, 33),  # an octet's at once
    (4, 24, 64, 20000, 9, 70), (1, 72, 40, 1500, 20, 40),   # and in groups
    (1, 32, 64, 2000, 3, 32), (1, 32, 64, 2000, 3, 33), (4, 24, 64, 20000, 3, 64), (4, 24, 64, 20000, 3, 65),
    (1, 9, 17, 1500, 2, 500), (1, 16, 130, 33, 3, 90),
])
def test_conv_fwd_edges(K, N, ci, co, L, k, d):
    g = torch.Generator().manual_seed(ci + L)
    p = d * (k - 1) // 2
    Lo = L + 2 * p - d * (k - 1)
    x, w = torch.randn(N, ci, L, generator=g), torch.randn(co, ci * k, generator=g)
    b, r, y0 = torch.randn(co, generator=g), torch.randn(N, co, Lo, generator=g), torch.randn(N, co, Lo, generator=g)
    xg, wg, bg, rg, y = x.cuda(), w.cuda(), b.cuda(), r.cuda(), y0.cuda()
    K.call("kdec_conv1d_fwd", P(xg), ci * L, P(wg), P(bg), P(y), co * Lo, N, ci, L, co, k, 1, p, d, P(rg), co * Lo, 0.5, 2.0)
    ref = F.conv1d(x.double(), w.double().reshape(co, ci, k), b.double(), padding=p, dilation=d)
    assert rel(y, 0.5 * (ref + r.double()) + 2.0 * y0.double()) <= TOL


def test_conv_fwd_parts(K):
    # 64 tiles of 384 steps: in parts, a block each, summed by tile_reduce
    N, ci, co, L, k, p = 8, 1024, 1000, 100, 3, 1
    g = torch.Generator().manual_seed(1)
    x, w, b, r, y0 = (torch.randn(*s, generator=g) for s in ((N, ci, L), (co, ci * k), (co,), (N, co, L), (N, co, L)))
    xg, wg, bg, rg, y = x.cuda(), w.cuda(), b.cuda(), r.cuda(), y0.cuda()
    K.profile(True)
    K.profile_reset()
    K.call("kdec_conv1d_fwd", P(xg), ci * L, P(wg), P(bg), P(y), co * L, N, ci, L, co, k, 1, p, 1, P(rg), co * L, 0.5, 2.0)
    torch.cuda.synchronize()
    assert "tile_reduce" in K.profile_read()
    K.profile(False)
    ref = F.conv1d(x.double(), w.double().reshape(co, ci, k), b.double(), padding=p)
    assert rel(y, 0.5 * (ref + r.double()) + 2.0 * y0.double()) <= TOL


@pytest.mark.parametrize("N,ci,co,L,k,s", [(2, 33, 130, 2600, 20, 10), (1, 5, 7, 5200, 32, 16)])
def test_conv_fwd_long_strides(K, N, ci, co, L, k, s):
    # strided windows of which two stages leave two blocks per CU: staged once
    g = torch.Generator().manual_seed(k)
    p = (k - s) // 2
    Lo = (L + 2 * p - k) // s + 1
    x, w, b = torch.randn(N, ci, L, generator=g), torch.randn(co, ci * k, generator=g), torch.randn(co, generator=g)
    xg, wg, bg, y = x.cuda(), w.cuda(), b.cuda(), torch.full((N, co, Lo), 7.0, device="cuda")
    K.call("kdec_conv1d_fwd", P(xg), ci * L, P(wg), P(bg), P(y), co * Lo, N, ci, L, co, k, s, p, 1, None, 0, 1.0, 0.0)
    assert rel(y, F.conv1d(x.double(), w.double().reshape(co, ci, k), b.double(), stride=s, padding=p)) <= TOL


@pytest.mark.parametrize("k,s,L", [(20, 10, 42), (20, 10, 400), (12, 6, 4000), (3, 4, 9), (5, 1, 140)])
def test_convt_fwd_edges(K, k, s, L):
    N, ci, co, p = 1, 72, 136, max(0, (k - s) // 2)
    g = torch.Generator().manual_seed(k + L)
    x, w = torch.randn(N, ci, L, generator=g), torch.randn(ci, co * k, generator=g)
    Lo = (L - 1) * s - 2 * p + k
    y = torch.full((N, co, Lo), 7.0, device="cuda")
    xg, wg = x.cuda(), w.cuda()
    K.call("kdec_convt1d_fwd", P(xg), ci * L, P(wg), None, P(y), co * Lo, N, ci, L, co, k, s, p, 0)
    assert rel(y, F.conv_transpose1d(x.double(), w.double().reshape(ci, co, k), stride=s, padding=p)) <= TOL


@pytest.mark.parametrize("N,rows,S", [(1, 1, 128), (8, 33, 128), (9, 100, 64), (40, 17, 256), (3, 31, 4), (80, 20, 128),
                                      # above, an element per thread; from 208 blocks of 32 rows on (N = 8,
                                      # S = 128) by rows: whole blocks, a part of the last, one block less
                                      (8, 6656, 128), (8, 6655, 128), (8, 6624, 128), (9, 17471, 64), (1, 8900, 64),
                                      (3, 3195, 256), (1, 197700, 4), (1, 803, 1024), (1, 803, 1022)])
def test_style_weight_grad(K, N, rows, S):
    g = torch.Generator().manual_seed(N)
    st, do = torch.randn(N, S, generator=g), torch.randn(N, rows, generator=g)
    dw0, db0 = torch.randn(rows, S, generator=g), torch.randn(rows, generator=g)
    w, stg, dog, dw, db = torch.zeros(rows, S).cuda(), st.cuda(), do.cuda(), dw0.cuda(), db0.cuda()
    K.call("kdec_style_proj_bwd", P(w), P(stg), S, P(dog), rows, None, 0, 0.0, P(dw), P(db), N, rows, S)
    # double sums, rounded once and added in float: half an ulp of each
    assert rel(dw, dw0.double() + do.double().t() @ st.double()) <= 2 ** -23
    assert rel(db, db0.double() + do.double().sum(0)) <= 2 ** -23
