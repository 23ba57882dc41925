"""The autotuner times what an untuned plan runs: the runtime schedule's own tile
(any line and thread count) is the candidate lds:auto."""
import re

import pytest

import wgpufft_amd as W
from wgpufft_amd import FftConfig, FftPlan, FftTransformKind

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _clean():
    W.clear_tuning()
    yield
    W.clear_tuning()


@pytest.mark.parametrize("kind,n,lines", [("r2c", 400, 48000), ("c2c", 270, 20000), ("c2c", 540, 8000), ("c2r", 286, 9000)])
def test_untuned_shape_is_timed(torch_cuda, kind, n, lines):
    cfg = (FftConfig.inverse(n) if kind == "c2r" else FftConfig.new(n)).with_batch(lines)
    build = getattr(FftPlan, kind)
    untuned = build(cfg).describe()
    count, report = W.autotune(cfg, {"c2c": FftTransformKind.C2c, "r2c": FftTransformKind.R2c,
                                     "c2r": FftTransformKind.C2r}[kind], reps=5)
    assert count == 1, report
    times = {name: float(us) for name, us in re.findall(r"(lds:\S+?)=([\d.]+)us", report)}
    assert "lds:auto" in times and len(times) > 2, report
    assert report.split("->")[1].strip() in times and min(times, key=times.get) == report.split("->")[1].strip(), report
    key = report.split(":", 1)[0]
    W.clear_tuning()
    W.parse_tuning(key + " = lds:auto\n")
    assert build(cfg).describe() == untuned
