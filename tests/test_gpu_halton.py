"""The device's Halton values take their digits by multiplying with a
reciprocal of the digit base; the oracle divides.  Every dimension at the
indexes where such a division can go wrong: each side of a multiple of the
base and of its powers, and the ends of the 32-bit range."""
import numpy as np
import pytest
import torch

from psychopath_cpp_amd import gpu

pytestmark = pytest.mark.gpu


def _bases():
    primes = [p for p in range(2, 1700) if all(p % k for k in range(2, int(p**0.5) + 1))][:256]
    for d, p in enumerate(primes):
        b = p
        while b * p <= 500:
            b *= p
        yield d, b


@pytest.mark.parametrize("part", range(4))
def test_gpu_halton_digits_are_exact(gpu_ctx, oracle, part):
    rng = np.random.default_rng(part)
    for d, b in _bases():
        if d % 4 != part:
            continue
        top = 2**32 - 1
        idx = {0, 1, top, top - 1, 2**31, 2**31 - 1, (top // b) * b, (top // b) * b - 1}
        power = b
        while power <= top:
            idx |= {power - 1, power, power + 1, (top // power) * power, (top // power) * power - 1}
            power *= b
        idx = np.array(sorted(i for i in idx if 0 <= i <= top) + list(rng.integers(0, 2**32, 40)), np.uint32)
        t = torch.from_numpy(idx.view(np.int32)).cuda()
        got = gpu.halton(gpu_ctx, d, t).cpu().numpy()
        want = np.array([oracle.lib().ora_halton(d, int(i)) for i in idx], np.float32)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), d

