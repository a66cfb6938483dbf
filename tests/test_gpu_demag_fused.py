"""The three-kernel demag convolution (column tiles in LDS, axis 0 convolved
directly) against the FP64 oracle, at the sizes where its tiling can go wrong:
plane counts below, at and beyond one axis-0 item (1..8 planes, then blocks of
6 and 8 with a remainder), column counts that leave a partial tile, row counts
that leave a partial row block, each length family, masks and batches.
(Batches and slots: test_gpu_demag_folded.py.)

Bars: FP64 1e-12 of max|B| (as the five-pass convolution); FP32 2e-6, the
round-off of FP32 transforms of up to 2048 points and sums of up to 3 N0
products (eps (log2 P1 P2 + N0) ~ 6e-8 (20 + 33) = 3e-6 at worst, rms 1/10)."""
import numpy as np
import pytest

from hotspin_amd.api import Demag
from hotspin_amd._lib import check
from oracle import pyoracle as po
from tests.gpu_util import P, dev, empty, host, relerr, require_gpu, torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    require_gpu()
    yield
    check("demag fused")


# folded axis 1 (FP32 beyond 2048 points of N0 P1, FP64 beyond 1024): 2, 4, 8 and 16 ways
# (the folds compiled are 2, 4 and 8, in FP64 2 and 4; more than 16 planes on compiled
# lengths do not fold in FP32)
SHAPES = ([(16, 128, 8), (64, 64, 16), (8, 256, 16), (20, 96, 12), (33, 80, 10), (3, 512, 8), (16, 512, 16)] +
          [(n0, 8, 16) for n0 in range(1, 10)] +           # planes per item, first of the blocked form
          [(10, 8, 16), (12, 4, 8), (13, 8, 8), (16, 16, 8), (17, 4, 16), (33, 8, 8)] +
          [(2, 5, 10), (3, 6, 12), (2, 10, 20), (1, 12, 24), (3, 24, 48), (2, 20, 40), (4, 80, 10)] +
          [(1, 32, 128), (8, 256, 8), (2, 512, 8), (1, 384, 16), (5, 64, 512)])


@pytest.mark.parametrize("N", SHAPES)
def test_fields_match_oracle(N):
    cell = (2e-9, 3e-9, 2.5e-9)
    rng = np.random.default_rng(sum(N))
    n = N[0] * N[1] * N[2]
    m = rng.standard_normal((3, n))
    msk = rng.random(n)
    d, o = Demag(N, cell), po.Demag(N, cell)
    for w in (None, msk):
        want = o.B(m, w, 8e5).reshape(3, n)
        dm, dw = dev(m), None if w is None else dev(w)
        B = empty((3, n))
        d.field_f64(P(dm), P(dw), 8e5, P(B))
        assert relerr(host(B), want) <= 1e-12
        dm, dw = dev(m, np.float32), None if w is None else dev(w, np.float32)
        B = empty((3, n), torch.float32)
        d.field_f32(P(dm), P(dw), 8e5, P(B))
        assert relerr(host(B), want) <= 2e-6
    d.close()


@pytest.mark.parametrize("N", [(2, 8, 16), (9, 6, 24)])
def test_periodic_x_and_the_other_axes(N):
    """A periodic x axis keeps the three kernels (rows without padding); a
    periodic axis 0 or 1 takes the five passes.  Both match the oracle."""
    cell = (2e-9, 3e-9, 2.5e-9)
    n = N[0] * N[1] * N[2]
    m = np.random.default_rng(3).standard_normal((3, n))
    for pbc in ((0, 0, 1), (0, 1, 0), (1, 0, 0), (1, 1, 1)):
        d = Demag(N, cell, pbc)
        want = po.Demag(N, cell, pbc).B(m, None, 8e5).reshape(3, n)
        dm, B = dev(m), empty((3, n))
        d.field_f64(P(dm), None, 8e5, P(B))
        assert relerr(host(B), want) <= 1e-12
        dm, B = dev(m, np.float32), empty((3, n), torch.float32)
        d.field_f32(P(dm), None, 8e5, P(B))
        assert relerr(host(B), want) <= 2e-6
        d.close()


# open axes whose 2 N has no compiled transform run at the next compiled length: one
# ragged axis at a time, all three, odd x lengths, a folded axis 1 with rows missing
# in its upper half (300 -> 640 points, FP32 folded 8 ways), more than 32 planes
# (the five passes), one plane, and ragged axes next to periodic ones
RAGGED = [((2, 8, 9), 0), ((2, 7, 16), 0), ((7, 8, 16), 0), ((7, 75, 100), 0), ((6, 45, 150), 0), ((1, 11, 13), 0),
          ((16, 300, 18), 0), ((3, 23, 31), 0), ((8, 113, 37), 0), ((35, 9, 14), 0), ((49, 27, 22), 0),
          ((3, 9, 26), (0, 0, 1)), ((3, 14, 18), (0, 1, 0)), ((7, 16, 18), (1, 0, 0)), ((5, 1, 22), 0), ((5, 22, 1), 0)]


@pytest.mark.parametrize("N,pbc", RAGGED)
def test_ragged_lengths(N, pbc):
    cell, pbc = (2e-9, 3e-9, 2.5e-9), pbc or (0, 0, 0)
    rng = np.random.default_rng(sum(N))
    n = N[0] * N[1] * N[2]
    m, msk = rng.standard_normal((3, n)), rng.random(n)
    d, o = Demag(N, cell, pbc), po.Demag(N, cell, pbc)
    assert d.P == tuple(2 * a if a > 1 and not p else a for a, p in zip(N, pbc))  # the logic size is reported
    assert relerr(d.kernel(), o.kernel()) <= 1e-12
    for w in (None, msk):
        want = o.B(m, w, 8e5).reshape(3, n)
        dm, dw = dev(m), None if w is None else dev(w)
        for field in (d.field_f64, d.field_f64_noalloc):
            B = empty((3, n))
            field(P(dm), P(dw), 8e5, P(B))
            assert relerr(host(B), want) <= 1e-12
        dm, dw = dev(m, np.float32), None if w is None else dev(w, np.float32)
        B = empty((3, n), torch.float32)
        d.field_f32(P(dm), P(dw), 8e5, P(B))
        assert relerr(host(B), want) <= 2e-6
    d.close()


# folded FP32 rows that go through LDS in halves, 32 or 16 to a block, against the FP64 field
@pytest.mark.parametrize("N", [(3, 384, 1024), (8, 320, 384), (16, 512, 512), (9, 200, 768), (4, 512, 640), (16, 500, 333)])
def test_folded_long_rows(N):
    n = N[0] * N[1] * N[2]
    m = np.random.default_rng(n).standard_normal((3, n))
    d = Demag(N, (2e-9, 3e-9, 2.5e-9))
    dm, df = dev(m), dev(m, np.float32)
    B, Bf = empty((3, n)), empty((3, n), torch.float32)
    d.field_f64(P(dm), None, 8e5, P(B))
    d.field_f32(P(df), None, 8e5, P(Bf))
    assert relerr(host(Bf), host(B)) <= 2e-6
    d.close()
