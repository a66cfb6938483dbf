"""Demag passes that take the length at run time.  Open axes are padded to compiled
lengths, so they are reached by periodic axes (7, 9, 11, 13, 25, 100 cells; an
odd x length), by one-cell axes and by open axes beyond the compiled lengths.
Rows, columns and axis 0 (which holds the spectrum of all P0 rows), each alone
and together, in a batch, in slots with an idle one, and through the
no-allocation entry."""
import ctypes as C

import numpy as np
import pytest

from hotspin_amd import workloads as W
from hotspin_amd.api import Batch, Demag, SlotBatch, Solver
from hotspin_amd._lib import check, lib
from oracle import pyoracle as po
from tests.gpu_util import P, dev, empty, host, relerr, require_gpu, torch

pytestmark = pytest.mark.gpu

CELL = (2e-9, 3e-9, 2.5e-9)


@pytest.fixture(autouse=True)
def _gpu():
    require_gpu()
    yield
    check("demag run-time lengths")


# mesh, periodic images, run-time (rows, columns, axis 0)
CASES = [((11, 8, 8), (1, 0, 0), (False, False, True)), ((7, 9, 14), (1, 1, 0), (False, True, True)),
         ((13, 4, 6), (2, 0, 0), (False, False, True)), ((2, 100, 16), (0, 1, 0), (False, True, False)),
         ((3, 25, 14), (0, 1, 1), (True, True, False)), ((4, 8, 9), (0, 0, 1), (True, False, False)),
         ((7, 13, 11), (1, 1, 1), (True, True, True)), ((5, 6, 1), (0, 0, 0), (True, False, False)),
         ((130, 3, 4), (0, 0, 0), (False, False, True)), ((2, 3, 2050), (0, 0, 0), (True, False, False))]


@pytest.mark.parametrize("N,pbc,runtime", CASES)
def test_fields_match_oracle(N, pbc, runtime):
    d, o = Demag(N, CELL, pbc), po.Demag(N, CELL, pbc)
    cnt = (C.c_int * 3)()
    assert lib().hs_demag_variant_count(d._h, cnt) == 0
    assert tuple(c == 0 for c in cnt) == runtime
    assert d.P == o.P and d.K == o.K
    assert relerr(d.kernel(), o.kernel()) <= 1e-12
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(n)
    m, msk = rng.standard_normal((3, n)), rng.random(n)
    want = o.B(m, msk, 8e5).reshape(3, n)
    dm, dw = dev(m), dev(msk)
    out = []
    for field in (d.field_f64_noalloc, d.field_f64):  # the first before the plan has FP64 spectra
        B = empty((3, n))
        B.fill_(np.nan)
        field(P(dm), P(dw), 8e5, P(B))
        out.append(host(B))
    assert np.array_equal(out[0], out[1])
    assert relerr(out[0], want) <= 1e-12
    dm, dw, B = dev(m, np.float32), dev(msk, np.float32), empty((3, n), torch.float32)
    d.field_f32(P(dm), P(dw), 8e5, P(B))
    assert relerr(host(B), want) <= 2e-6
    d.close()


MAT = W.MATERIAL_WIDE_T


def _states(N, k, seed):
    n = N[0] * N[1] * N[2]
    rng = np.random.default_rng(seed)
    T = rng.uniform(200, 900, k)
    return T, np.stack([W.random_state(n, W.equilibrium_m(t, MAT["Tc"], MAT["J"]), rng) for t in T])


@pytest.mark.parametrize("N,pbc", [((7, 8, 10), (1, 0, 0)), ((11, 9, 6), (1, 1, 0))])
def test_batch_equals_solves_alone_and_oracle(N, pbc):
    """The spectrum of all P0 rows is held per solve."""
    kw = W.llbr_params(T=300.0, seed=5, material=MAT, Bext=(0.01, -0.02, 0.03))
    T, m = _states(N, 3, 2)
    seeds = np.arange(3, dtype=np.uint64) + 11
    b = Batch(N, CELL, 3, pbc=pbc, TMuls=T, seeds=seeds, **kw)
    b.set_m(m)
    b.run("rk4", 4, 2e-15)
    mb = b.get_m()
    for q in range(3):
        kq = dict(kw, TMul=float(T[q]), seed=int(seeds[q]))
        s = Solver(N, CELL, pbc=pbc, **kq)
        s.set_m(m[q])
        s.run("rk4", 4, 2e-15)
        assert np.array_equal(s.get_m(), mb[q])
    o = po.LLB(N, CELL, pbc=pbc, **kq)
    mo = m[2].copy()
    for i in range(4):
        o.step("rk4", mo, 2e-15, i)
    assert np.abs(mb[2] - mo).max() <= 1e-5


def test_slots_with_an_idle_one_equal_slots_alone():
    N, pbc = (7, 8, 10), (1, 0, 0)
    kw = W.llbr_params(T=300.0, seed=5, material=MAT)
    T, m = _states(N, 2, 3)

    def run(which):
        g = SlotBatch(N, CELL, 3, pbc=pbc, **kw)
        for i, slot in which:
            g.admit(slot, m[i], float(T[i]), 40 + i, 6, 1e-15, maxErr=1e-4, maxdt=1e-13)
        g.run_to_end(chunk=2)
        return [g.get_m(slot) for _, slot in which]

    both = run([(0, 0), (1, 2)])
    assert np.isfinite(both).all()
    assert np.array_equal(both[0], run([(0, 0)])[0])
    assert np.array_equal(both[1], run([(1, 2)])[0])
