"""Which registered shape a pass of power-of-two lines takes, on both sides of
the lines that the rules draw."""
import pytest

import wgpufft_amd as W
from wgpufft_amd import FftConfig, FftPlan, FftPrecision
from wgpufft_amd.tune import DEFAULT_TABLE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,points,pipelined", [
    ("r2c", 512, 4 << 20, False), ("r2c", 1024, 4 << 20, False), ("r2c", 2048, 4 << 20, False),
    ("c2r", 1024, 4 << 20, False), ("c2r", 2048, 4 << 20, False),
    ("r2c", 512, 6 << 20, True), ("r2c", 1024, 6 << 20, True), ("r2c", 2048, 6 << 20, True),
    ("c2r", 1024, 6 << 20, True), ("c2r", 2048, 6 << 20, True),
    ("r2c", 256, 4 << 20, False), ("r2c", 256, 8 << 20, True), ("r2c", 256, 32 << 20, False),
    ("r2c", 4096, 32 << 20, True)])
def test_real_lines_are_pipelined_where_it_pays(torch_cuda, kind, n, points, pipelined):
    cfg = (FftConfig.new(n) if kind == "r2c" else FftConfig.inverse(n)).with_batch(points // n)
    plan = getattr(FftPlan, kind)(cfg)
    assert ("pipe" in plan.describe()) == pipelined, plan.describe()


@pytest.mark.parametrize("n,columns,shape", [
    (4096, 512, "vec=1 lpw=4"), (4096, 1024, "vec=1 lpw=4"), (4096, 2048, "vec=2 lpw=8"), (4096, 1025, "vec=1 lpw=4"),
    (2048, 2048, "vec=2 lpw=8"), (2048, 1025, "vec=1 lpw=8"), (2048, 2049, "vec=1 lpw=4"), (2048, 3880 + 1, "vec=1 lpw=8"),
    (1024, 1024, "vec=2 lpw=8"), (1024, 2049, "vec=1 lpw=8")])
def test_column_tiles(torch_cuda, n, columns, shape):
    """Tiles that have a CU to themselves: 8 lines of 4096 points, or of 2048 one
    by one (columns of an odd count)."""
    plan = FftPlan.c2c(FftConfig.new_nd([columns, n]).with_axes([1]))
    assert shape in plan.describe(), plan.describe()


@pytest.mark.parametrize("n,batch,shape", [
    (65536, 64, "N=256 16x16 lines=16384 tpl=16 vec=1 lpw=16"), (65536, 4, "N=256 16x16 lines=1024 tpl=16 vec=1 lpw=8"),
    (131072, 4, "lpw=8"), (262144, 16, "lpw=16"), (16384, 256, "N=128 16x8 lines=32768 tpl=8 vec=1 lpw=32"),
    (16384, 128, "N=128 16x8 lines=16384 tpl=8 vec=1 lpw=8")])
def test_twiddled_columns_tile(torch_cuda, n, batch, shape):
    """The columns of a two-pass split: 16 lines of 256 and 512 points where that
    fills every CU, 32 of 128 from four tiles per CU on."""
    first = FftPlan.c2c(FftConfig.new(n).with_batch(batch)).describe().split(";")[0]
    assert " post" in first and shape in first, first


def test_twiddled_columns_of_one_line(torch_cuda):
    """4096 columns of 128 points, the middle pass of 2^19: eight lines per tile."""
    middle = FftPlan.c2c(FftConfig.new(1 << 19)).describe().split(";")[1]
    assert " post" in middle and "N=128 16x8 lines=4096 tpl=8 vec=1 lpw=8" in middle, middle


@pytest.mark.parametrize("shape,axes,pipelined", [
    ([256, 256, 64], None, False), ([256, 256, 128], None, False), ([512, 128, 64], None, False),
    ([512, 256, 64], None, True), ([1024, 64, 64], None, True), ([256, 256, 64], [0], True), ([512, 128, 64], [0], True)])
def test_complex_lines_of_several_axes(torch_cuda, shape, axes, pipelined):
    cfg = FftConfig.new_nd(shape)
    desc = FftPlan.c2c(cfg.with_axes(axes) if axes else cfg).describe()
    assert ("pipe" in desc) == pipelined, desc


@pytest.mark.parametrize("n,lines,f64,tile", [(41, 64, False, 8), (41, 300, False, 8), (29, 300, False, 9), (71, 64, False, 4),
                                              (211, 64, False, 4), (74, 64, True, 1)])
def test_few_convolution_lines_spread(torch_cuda, n, lines, f64, tile):
    """Short of two workgroups per CU a tile takes no more lines than a wave has
    threads for their butterflies."""
    cfg = FftConfig.new(n).with_batch(lines).with_precision(FftPrecision.F64 if f64 else FftPrecision.F32)
    desc = FftPlan.c2c(cfg).describe()
    assert " nt=" in desc and int(desc.split("lpw=")[1].split()[0]) <= tile, desc


@pytest.mark.parametrize("shape,axes,batch,kind", [([1024], None, 3072, "c2c"), ([256], None, 32768, "c2c"),
                                                   ([24576, 256], [1], 1, "c2c"), ([3072, 2048], [1], 1, "c2c"),
                                                   ([2048], None, 2048, "r2c")])
def test_committed_table_leaves_better_rules_alone(torch_cuda, shape, axes, batch, kind):
    """Passes where the built-in rule runs the faster shape (or the same): the
    committed table holds no choice for them."""
    cfg = FftConfig.new_nd(shape).with_batch(batch)
    if axes:
        cfg = cfg.with_axes(axes)
    W.clear_tuning()
    built_in = getattr(FftPlan, kind)(cfg).describe()
    W.load_tuning(DEFAULT_TABLE)
    try:
        assert getattr(FftPlan, kind)(cfg).describe() == built_in
    finally:
        W.clear_tuning()
