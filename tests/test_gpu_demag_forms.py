"""Which form of the convolution a plan takes at the edges of its rules, seen from
outside: HS_DEMAG_FORCE="-1,-1,-1" keeps a plan's FP32 field in the five passes
with the variants it would have, so the fields agree bit for bit where the plan
takes the five passes by itself, and differ in rounding where it takes three
kernels."""
import numpy as np
import pytest

from hotspin_amd.api import Demag
from hotspin_amd._lib import check
from tests.gpu_util import P, dev, empty, host, relerr, require_gpu, torch

pytestmark = pytest.mark.gpu

CELL = (2e-9, 3e-9, 2.5e-9)


@pytest.fixture(autouse=True)
def _gpu():
    require_gpu()
    yield
    check("demag forms")


def _f32(N, m):
    d, B = Demag(N, CELL), empty(m.shape, torch.float32)
    d.field_f32(P(m), None, 8e5, P(B))
    out = host(B)
    d.close()
    return out


# more than 16 planes on compiled lengths that would have to fold axis 1; a fold that
# takes blocks of more than 256 threads (26 planes in items of six, 64 points: 320)
FIVE = [(20, 64, 16), (24, 64, 64), (24, 48, 32), (32, 64, 16), (32, 128, 8), (26, 256, 16)]
# at the other side: 16 planes, 24 and 32 unfolded, padded plane counts, 20 planes unfolded
THREE = [(16, 64, 16), (24, 32, 16), (32, 32, 16), (20, 32, 16), (17, 64, 16), (30, 64, 16), (26, 128, 16),
         (10, 320, 16), (16, 256, 16)]


@pytest.mark.parametrize("N,five", [(N, True) for N in FIVE] + [(N, False) for N in THREE])
def test_form_of_the_fp32_convolution(monkeypatch, N, five):
    n = N[0] * N[1] * N[2]
    m = np.random.default_rng(n).standard_normal((3, n))
    m32 = dev(m, np.float32)
    own = _f32(N, m32)
    monkeypatch.setenv("HS_DEMAG_FORCE", "-1,-1,-1")
    forced = _f32(N, m32)
    monkeypatch.delenv("HS_DEMAG_FORCE")
    assert np.array_equal(own, forced) == five
    d, dm, B = Demag(N, CELL), dev(m), empty((3, n))
    d.field_f64(P(dm), None, 8e5, P(B))
    want = host(B)
    d.close()
    # FP32 round-off of transforms of up to 2048 points and sums of up to 96 products
    assert relerr(own, want) <= 2e-6 and relerr(forced, want) <= 2e-6


def _compiled(d):
    """Which of the plan's row, column and axis-0 passes run compiled kernels."""
    import ctypes as C
    from hotspin_amd._lib import lib
    cnt = (C.c_int * 3)()
    assert lib().hs_demag_variant_count(d._h, cnt) == 0
    return tuple(c > 0 for c in cnt)


# an open axis without a compiled length (more than 128 planes, more than 1024 rows,
# more than 2048 cells along x) beside others that have one at 2 N, could be padded to
# one, or gain by it: (rows, columns, axis 0) compiled
BESIDE_RUN_TIME = [((140, 64, 100), (False, True, False)), ((130, 49, 49), (False, False, False)),
                   ((140, 16, 37), (True, True, False)), ((200, 20, 33), (True, True, False)),
                   ((7, 1100, 49), (False, False, True)), ((3, 1300, 10), (True, False, True)),
                   ((3, 37, 2100), (False, True, True)), ((129, 3, 4), (True, True, False))]


@pytest.mark.parametrize("N,compiled", BESIDE_RUN_TIME)
def test_padding_beside_a_run_time_length(N, compiled):
    from oracle import pyoracle as po
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(n)
    m, msk = rng.standard_normal((3, n)), rng.random(n)
    d, o = Demag(N, CELL), po.Demag(N, CELL)
    assert d.P == o.P and d.K == o.K
    assert _compiled(d) == compiled
    assert relerr(d.kernel(), o.kernel()) <= 1e-12
    want = o.B(m, msk, 8e5).reshape(3, n)
    dm, dw, B = dev(m), dev(msk), empty((3, n))
    d.field_f64(P(dm), P(dw), 8e5, P(B))
    assert relerr(host(B), want) <= 1e-12
    dm, dw, B = dev(m, np.float32), dev(msk, np.float32), empty((3, n), torch.float32)
    d.field_f32(P(dm), P(dw), 8e5, P(B))
    assert relerr(host(B), want) <= 2e-6
    d.close()


# three-kernel meshes beyond the size whose FP64 table is kept for hs_demag_field_f64_noalloc
@pytest.mark.parametrize("N", [(8, 256, 256), (1, 1024, 1024), (2, 640, 640), (16, 512, 512)])
def test_three_kernel_plan_holds_no_five_pass_kernel(monkeypatch, N):
    """The footprint by which requests are admitted is no larger than with the five
    passes, whose FP32 kernel octant (16 to 114 MB here) nothing reads."""
    from hotspin_amd.api import SlotBatch
    kw = dict(msat0T0Mul=1e6, demag=1, gammaLL=2.211e5, torque=1)
    own = SlotBatch(N, CELL, 1, **kw)
    monkeypatch.setenv("HS_DEMAG_FORCE", "-1,-1,-1")
    five = SlotBatch(N, CELL, 1, **kw)
    assert own.footprint() <= five.footprint()
    own.close()
    five.close()


# padded plans in five passes: the tiles (pencils a block, threads) of two-level rows,
# two-level columns and the axis-0 pass with four lanes a pencil, one lane below 16 points
@pytest.mark.parametrize("N,pbc,tiles", [((36, 100, 100), (0, 0, 0), [8, 128, 8, 128, 8, 192]),
                                         ((33, 33, 31), (0, 0, 0), [8, 64, 8, 80, 8, 192]),
                                         ((40, 129, 129), (0, 0, 0), [8, 128, 8, 160, 8, 192]),
                                         ((33, 300, 70), (0, 0, 0), [8, 80, 8, 256, 8, 192]),
                                         ((8, 190, 100), (1, 0, 0), [8, 128, 8, 192, 32, 192])])
def test_fixed_variants_of_padded_five_pass_plans(N, pbc, tiles):
    import ctypes as C
    from hotspin_amd._lib import lib
    n = N[0] * N[1] * N[2]
    d, t = Demag(N, CELL, pbc), (C.c_int * 6)()
    assert lib().hs_demag_tiles(d._h, t) == 0
    assert list(t) == tiles
    m = np.random.default_rng(n).standard_normal((3, n))
    dm, B = dev(m), empty((3, n))
    d.field_f64(P(dm), None, 8e5, P(B))
    m32, Bf = dev(m, np.float32), empty((3, n), torch.float32)
    d.field_f32(P(m32), None, 8e5, P(Bf))
    assert relerr(host(Bf), host(B)) <= 2e-6  # FP32 round-off of transforms of up to 1280 points
    d.close()


# meshes whose FP64 spectra fit the static array of hs_demag_field_f64_noalloc at 2 N but
# not padded: three kernels, folded; five passes
@pytest.mark.parametrize("N", [(24, 140, 110), (40, 129, 65)])
def test_fp32_is_padded_where_fp64_stays_at_the_logic_size(N):
    """The FP32 field runs compiled passes; both FP64 entries take the mesh and agree
    bit for bit; the octant is that of 2 N."""
    from oracle import pyoracle as po
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(n)
    m, msk = rng.standard_normal((3, n)), rng.random(n)
    d, o = Demag(N, CELL), po.Demag(N, CELL)
    assert d.P == o.P and d.K == o.K
    assert _compiled(d) == (True, True, True)
    assert relerr(d.kernel(), o.kernel()) <= 1e-12
    want = o.B(m, msk, 8e5).reshape(3, n)
    dm, dw = dev(m), dev(msk)
    out = []
    for field in (d.field_f64_noalloc, d.field_f64):
        B = empty((3, n))
        field(P(dm), P(dw), 8e5, P(B))
        out.append(host(B))
    assert np.array_equal(out[0], out[1])
    assert relerr(out[0], want) <= 1e-12
    m32, w32, Bf = dev(m, np.float32), dev(msk, np.float32), empty((3, n), torch.float32)
    d.field_f32(P(m32), P(w32), 8e5, P(Bf))
    assert relerr(host(Bf), want) <= 2e-6
    d.close()


@pytest.mark.parametrize("N,pbc,form", [((16, 512, 512), (0, 0, 0), [8, 0]), ((8, 256, 256), (0, 0, 0), [4, 4]),
                                        ((4, 8, 16), (0, 0, 0), [1, 1]), ((4, 8, 16), (1, 0, 0), [0, 0]),
                                        ((33, 8, 16), (0, 0, 0), [0, 0]), ((24, 140, 110), (0, 0, 0), [4, 0])])
def test_form_that_a_plan_reports(N, pbc, form):
    import ctypes as C
    from hotspin_amd._lib import lib
    d, out = Demag(N, CELL, pbc), (C.c_int * 2)()
    assert lib().hs_demag_form(d._h, out) == 0 and list(out) == form
    d.close()
