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
