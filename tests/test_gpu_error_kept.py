"""Rounding errors of single kernels against longer arithmetic, at bounds that
an extra rounding per term, per output or per bin pair exceeds.  u is the unit
roundoff; C u = 0.42 u is the rms of one rounding to nearest (uniform error,
logarithmic mantissas)."""
import numpy as np
import pytest
import torch

from wgpufft_amd import FftConfig, FftPlan, FftPrecision

pytestmark = pytest.mark.gpu

U32, U64, C = 2.0 ** -24, 2.0 ** -53, 0.42


def uniform(count, seed, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(count, generator=g, device="cuda", dtype=dtype) * 2 - 1


def rel_l2(y, ref):
    return (torch.linalg.norm(y.to(ref.dtype) - ref) / torch.linalg.norm(ref)).item()


@pytest.mark.parametrize("n0,n1,volumes", [(17, 17, 256), (59, 47, 32)])
def test_small_volume_direct_sums_round_once_per_term(n0, n1, volumes):
    """A direct sum of n terms whose accumulator rounds once per term errs by C u
    sqrt(n / 2), a term by C u sqrt(2.5) (product, its difference, the factor);
    twice per term would be C u sqrt(n) (measured 1.31 and 1.36 times as much)."""
    x = torch.view_as_complex(uniform(2 * n0 * n1 * volumes, n0).view(volumes, n1, n0, 2))
    y = torch.empty_like(x)
    plan = FftPlan.c2c(FftConfig.new_nd([n0, n1]).with_batch(volumes))
    assert plan.describe().startswith("small-volume"), plan.describe()
    plan.execute(x, y)
    torch.cuda.synchronize()
    e = rel_l2(y, torch.fft.fft2(x.to(torch.complex128)))
    assert e <= 1.1 * C * U32 * np.sqrt((n0 + n1) / 2 + 5), e
