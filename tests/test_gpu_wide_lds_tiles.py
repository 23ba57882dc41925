"""512-thread tiles of the kernels that still run from LDS to LDS: lines and
convolutions of one stage, at tiles that take more than half of a CU's LDS
(2-point f32 lines, 2048 to a tile; f64 and df64 Rader of 5 and 7 and Bluestein
of 2 and 3 points forced on their axis), against torch.fft in complex128.  Longer
convolutions and lines, whose tiles were such ones, run the register stages.
Bounds as everywhere in this suite: f32 relative L2 <= 1e-6, f64 <= 1e-13, df64
<= 1e-11."""
import pytest
import torch

from wgpufft_amd import FftConfig, FftPlan, FftPrecision, FftTuning

pytestmark = pytest.mark.gpu

PREC = {"f32": FftPrecision.F32, "f64": FftPrecision.F64, "df64": FftPrecision.Df64}
TOL = {"f32": 1e-6, "f64": 1e-13, "df64": 1e-11}


# (precision, points, lines, forced kind, route, lines of a tile); the last tile
# of each is not full
@pytest.mark.parametrize("prec,n,lines,forced,route,lpw", [
    ("f32", 2, 5001, None, "lds N=2", 2048),
    ("f64", 5, 262147, "rader", "rader p=5 M=4", 512), ("df64", 5, 262147, "rader", "rader p=5 M=4", 512),
    ("f64", 7, 174800, "rader", "rader p=7 M=6", 341),
    ("f64", 3, 209500, "bluestein", "bluestein N=3 M=5", 409), ("df64", 2, 349500, "bluestein", "bluestein N=2 M=3", 682)])
@pytest.mark.parametrize("inverse", [False, True])
def test_wide_tiles(torch_cuda, prec, n, lines, forced, route, lpw, inverse):
    tuning = FftTuning()
    if forced:
        tuning = getattr(tuning, f"with_force_{forced}_axes")([0])
    cfg = (FftConfig.inverse(n) if inverse else FftConfig.new(n)).with_batch(lines).with_precision(PREC[prec])
    plan = FftPlan.c2c(cfg.with_tuning(tuning))
    assert plan.describe().startswith(route) and f"lpw={lpw}" in plan.describe() and " nt=" not in plan.describe(), \
        plan.describe()
    g = torch.Generator(device="cuda").manual_seed(n)
    v = torch.rand(lines * n * 2, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    if prec == "df64":
        hi = v.float()
        x = torch.stack([hi, (v - hi.double()).float()], -1).view(lines, n, 4)
        v = hi.double() + x.view(-1, 2)[:, 1].double()
    else:
        v = v.float().double() if prec == "f32" else v
        x = torch.view_as_complex((v.float() if prec == "f32" else v).view(lines, n, 2))
    y = torch.empty_like(x)
    plan.execute(x, y)
    torch.cuda.synchronize()
    got = torch.view_as_complex(y.double().view(lines, n, 2, 2).sum(-1)) if prec == "df64" else y.to(torch.complex128)
    want = (torch.fft.ifft if inverse else torch.fft.fft)(torch.view_as_complex(v.view(lines, n, 2)))
    e = (torch.linalg.norm(got - want) / torch.linalg.norm(want)).item()
    assert e <= TOL[prec], (e, plan.describe())
