"""The three-kernel demag convolution with a folded axis 1, for many solves at once:
the rows of a pencil, the columns of a solve and the kernels' early exit on an
idle solve depend on the solve's index there.  Meshes folded 4 and 8 ways, whose
row kernels pass through LDS whole or in halves (rows of 384 points and more),
with rows missing in the folded half, and one unfolded.  Every solve gives the
same bits alone and in the mix.  And single fields at the plane counts where the
form of the convolution changes."""
import numpy as np
import pytest

from hotspin_amd import workloads as W
from hotspin_amd.api import Batch, Demag, SlotBatch, Solver
from hotspin_amd._lib import check
from oracle import pyoracle as po
from tests.gpu_util import P, dev, empty, host, relerr, require_gpu, torch

pytestmark = pytest.mark.gpu

CELL = (2e-9, 3e-9, 2.5e-9)
MAT = W.MATERIAL_WIDE_T


@pytest.fixture(autouse=True)
def _gpu():
    require_gpu()
    yield
    check("demag folded")


def _states(N, k):
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(n + k)
    T = rng.uniform(200, 900, k)
    return T, np.stack([W.random_state(n, W.equilibrium_m(t, MAT["Tc"], MAT["J"]), rng) for t in T])


# rows of 8 and of 64 points folded 4 ways; 384 points in halves, 4 and 8 ways; 150 of 160
# rows, and an odd number of cells along x; not folded
FOLDED = [(16, 128, 8), (4, 256, 64), (3, 384, 384), (10, 320, 384), (7, 150, 101), (5, 20, 33)]


@pytest.mark.parametrize("N", FOLDED)
def test_batch_equals_solves_alone(N):
    kw = W.llbr_params(T=300.0, seed=5, material=MAT)
    T, m = _states(N, 3)
    seeds = np.arange(3, dtype=np.uint64) + 11
    b = Batch(N, CELL, 3, TMuls=T, seeds=seeds, **kw)
    b.set_m(m)
    b.run("rk4", 2, 2e-15)
    mb = b.get_m()
    b.close()
    assert np.isfinite(mb).all() and not np.array_equal(mb[0], mb[2])
    for q in range(3):
        s = Solver(N, CELL, **dict(kw, TMul=float(T[q]), seed=int(seeds[q])))
        s.set_m(m[q])
        s.run("rk4", 2, 2e-15)
        assert np.array_equal(s.get_m(), mb[q]), q
        s.close()


@pytest.mark.parametrize("N", [(16, 128, 8), (3, 384, 384), (7, 150, 101), (5, 20, 33)])
def test_slots_beside_an_idle_one_equal_slots_alone(N):
    kw = W.llbr_params(T=300.0, seed=5, material=MAT)
    T, m = _states(N, 2)

    def run(which):
        g = SlotBatch(N, CELL, 3, **kw)
        for i, slot in which:  # slot 1 is idle; slot 2 ends earlier and is idle from then on
            g.admit(slot, m[i], float(T[i]), 40 + i, 6 - 2 * i, 1e-15, maxErr=1e-4, maxdt=1e-13)
        g.run_to_end(chunk=2)
        out = [g.get_m(slot) for _, slot in which]
        g.close()
        return out

    both = run([(0, 0), (1, 2)])
    assert np.isfinite(both[0]).all() and np.isfinite(both[1]).all()
    assert np.array_equal(both[0], run([(0, 0)])[0])
    assert np.array_equal(both[1], run([(1, 2)])[0])


# up to 32 planes in three kernels, 16 where axis 1 folds on compiled lengths; items of
# eight and of six planes, with and without a remainder
PLANES = [(16, 64, 24), (17, 64, 24), (20, 16, 16), (20, 64, 24), (24, 8, 16), (24, 64, 16), (30, 64, 16), (31, 8, 16),
          (31, 64, 16), (32, 8, 16), (32, 32, 16), (32, 64, 16), (33, 32, 16)]


@pytest.mark.parametrize("N", PLANES)
def test_plane_counts_match_oracle(N):
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(n)
    m, msk = rng.standard_normal((3, n)), rng.random(n)
    d = Demag(N, CELL)
    want = po.Demag(N, CELL).B(m, msk, 8e5).reshape(3, n)
    dm, dw, B = dev(m), dev(msk), empty((3, n))
    d.field_f64(P(dm), P(dw), 8e5, P(B))
    assert relerr(host(B), want) <= 1e-12
    dm, dw, B = dev(m, np.float32), dev(msk, np.float32), empty((3, n), torch.float32)
    d.field_f32(P(dm), P(dw), 8e5, P(B))
    # FP32 transforms of up to 256 points and sums of up to 96 products
    assert relerr(host(B), want) <= 2e-6
    d.close()


# unfolded, more than eight planes: items of four planes in a launch of fewer than 1024 waves
# (the solve alone), of six or eight beyond (the batch); plane counts that fill items of each
# size and that do not
@pytest.mark.parametrize("N,k", [((32, 32, 32), 9), ((24, 32, 16), 24), ((9, 16, 16), 64), ((13, 12, 10), 96),
                                 ((20, 8, 16), 64), ((31, 10, 12), 96)])
def test_small_and_large_launches_give_the_same_bits(N, k):
    kw = W.llbr_params(T=300.0, seed=5, material=MAT)
    T, m = _states(N, k)
    seeds = np.arange(k, dtype=np.uint64) + 11
    b = Batch(N, CELL, k, TMuls=T, seeds=seeds, **kw)
    b.set_m(m)
    _, h = b.rhs()
    b.run("rk4", 1, 2e-15)
    mb = b.get_m()
    b.close()
    for q in (0, k // 2, k - 1):
        s = Solver(N, CELL, **dict(kw, TMul=float(T[q]), seed=int(seeds[q])))
        s.set_m(m[q])
        assert np.array_equal(s.rhs()[1], h[q]), q
        s.run("rk4", 1, 2e-15)
        assert np.array_equal(s.get_m(), mb[q]), q
        s.close()
