"""Choices that saved tuning tables may hold: each stays a valid one (a table
with an unknown choice is refused as a whole)."""
import pytest

import wgpufft_amd as W


@pytest.fixture(autouse=True)
def _clean():
    W.clear_tuning()
    yield
    W.clear_tuning()


# the runtime schedule's own tile, and kernels that no default picks
@pytest.mark.parametrize("choice", [
    "lds:auto", "lds:lpw=3",
    "reg:f32:n1024:t128:l2:lf00:m0/0:p0:v1:8x8x4x4:pipe2",
    "reg:f32:n1024:t64:l2:lf00:m0/0:p0:v1:16x16x4:pipe2",
    "reg:f32:n4096:t512:l1:lf00:m0/0:p0:v1:8x8x8x8:pipe1",
    "reg:f32:n4096:t256:l2:lf00:m0/0:p0:v2:8x8x8x8:fold:adj",
    "reg:f32:n2048:t128:l2:lf00:m0/0:p0:v2:16x16x8:fold",
    "reg:f32:n1024:t64:l2:lf00:m0/0:p0:v2:16x16x4:fold",
    "reg:f32:n2048:t128:l2:lf00:m1/1:p0:v1:16x16x8:pipe2"])
def test_choice_is_accepted(choice):
    n = choice.split(":n")[1].split(":")[0] if ":n" in choice else "1000"
    assert W.parse_tuning(f"f32|n{n}|lf00|m0/0|p0|pair0|lines2^12 = {choice}\n") == 1


@pytest.mark.parametrize("choice", ["lds:", "lds:automatic", "lds:auto=1"])
def test_choice_is_refused(choice):
    with pytest.raises(W.FftError):
        W.parse_tuning(f"f32|n1000|lf00|m0/0|p0|pair0|lines2^12 = {choice}\n")
