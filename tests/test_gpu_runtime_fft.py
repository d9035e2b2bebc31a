"""The FFT passes of lengths without a compile-time plan (csrc/fft_gen.inl)
against numpy's transforms: every group of prime radices, lengths whose widest
stage has more butterflies than a workgroup has threads, odd ones, the longest,
and line counts that leave a workgroup's last lines empty."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from openspacecharge_amd import _capi as K

pytestmark = pytest.mark.gpu

# one length per group of radices, then several stages, then the edges
LENGTHS = [1, 2, 3, 5, 7, 4, 6, 9, 10, 8, 11, 13, 17, 19, 23, 15, 14, 21, 22, 26, 12, 45, 20,
           25, 40, 50, 70, 100, 105, 150, 200, 230, 242, 294, 500, 529, 1058, 1000, 1331, 1750,
           1920]


def primes(n):
    out, p = [], 2
    while n > 1:
        while n % p == 0:
            out.append(p)
            n //= p
        p += 1
    return out


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_line_transform(L, axis):
    assert K.load().osc_fft_length_supported(L)
    shape = [3, 5, 2]
    shape[axis] = L
    rng = np.random.default_rng(L)
    a = np.asfortranarray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    b = np.zeros_like(a, order="F")
    ctx = osc.Context(0)
    osc.ccfft3d(a, b, (1, -1, 1), ctx=ctx)
    ctx.close()
    e = np.fft.ifft(a, axis=0, norm="forward")
    e = np.fft.fft(e, axis=1)
    e = np.fft.ifft(e, axis=2, norm="forward")
    # relative 2-norm: each prime stage adds up r rounded products
    tol = np.finfo(float).eps * sum(sum(p + 3 for p in primes(m)) + 1 for m in shape)
    assert np.linalg.norm(b - e) <= tol * np.linalg.norm(e)
