"""The kernel shape of power-of-two lines is chosen by their number: every
shape of a length runs the same radix schedule, so a line's result is the same
bits whichever one runs (and the one of a few lines is checked against numpy).

The bound of the comparison with numpy: f32 Stockham stages err by about
eps * sqrt(log2 n) <= 6e-8 * 3.5 in the L2 norm; 6e-7 leaves a factor three.
"""
import numpy as np
import pytest
import torch

from wgpufft_amd import FftConfig, FftPlan

pytestmark = pytest.mark.gpu


def run(shape, batch, x):
    y = torch.empty_like(x)
    plan = FftPlan.c2c(FftConfig.new_nd(shape).with_axes([len(shape) - 1]).with_batch(batch))
    plan.execute(x, y)
    torch.cuda.synchronize()
    return y, plan


def uniform(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(2 * n, device="cuda", generator=g) * 2 - 1


# lines below, at and above the persistent form's eight tiles per CU, with a last
# tile that is not full
@pytest.mark.parametrize("n,counts", [
    (256, (16376, 16391)), (512, (8188, 8195)), (1024, (4091, 4099)), (2048, (2047, 2049, 4099)),
    (4096, (2047, 2049))])
def test_contiguous_counts_agree(n, counts):
    x = uniform(n * max(counts), n)
    few, _ = run([n], 3, x[:2 * n * 3])
    ref = np.fft.fft(x[:2 * n * 3].cpu().numpy().astype(np.float64).view(np.complex128).reshape(3, n))
    got = few.cpu().numpy().view(np.complex64).reshape(3, n)
    assert np.linalg.norm(got - ref) <= 6e-7 * np.linalg.norm(ref)
    outs = [run([n], c, x[:2 * n * c]) for c in counts]
    assert ("pipe" in outs[-1][1].describe()) and "pipe" not in run([n], 3, x[:6 * n])[1].describe()
    assert torch.equal(outs[-1][0][:few.numel()], few)
    for y, _ in outs[:-1]:
        m = min(y.numel(), outs[-1][0].numel())
        assert torch.equal(y[:m], outs[-1][0][:m])
    # the tail of the longest batch, by itself
    tail, _ = run([n], 5, x[:2 * n * counts[-1]][-10 * n:])
    assert torch.equal(outs[-1][0][-10 * n:], tail)


# columns: few (the tile halves), odd and even numbers of them, arrays below
# and above the cache lines of the rule
@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024, 2048, 4096])
def test_column_counts_agree(n):
    widths = [2, 37, 96, 1056]
    if n in (256, 1024):
        widths.append((13 << 20) // n // 2 * 2)
    base = None
    for w in widths:
        x = uniform(n * w, 7).view(n, w, 2)
        if base is not None:
            x[:, :2] = base[0]
        y = run([w, n], 1, x.contiguous())[0].view(n, w, 2)
        if base is None:
            base = (x[:, :2].clone(), y[:, :2].clone())
            ref = np.fft.fft(x.cpu().numpy().astype(np.float64)[..., 0] + 1j * x.cpu().numpy()[..., 1], axis=0)
            got = y.cpu().numpy()[..., 0] + 1j * y.cpu().numpy()[..., 1]
            assert np.linalg.norm(got - ref) <= 6e-7 * np.linalg.norm(ref)
        else:
            assert torch.equal(y[:, :2], base[1]), (n, w)


# real lines below and above the persistent form's eight tiles per CU
@pytest.mark.parametrize("kind,n,counts", [
    ("r2c", 256, (8189, 8195)), ("r2c", 512, (8189, 8195)),
    ("r2c", 1024, (4093, 4099)), ("r2c", 2048, (2047, 2049)), ("r2c", 4096, (2047, 2049)),
    ("c2r", 1024, (4093, 4099)), ("c2r", 2048, (2047, 2049)), ("c2r", 4096, (2047, 2049)),
    ("c2r", 64, (5, 4099)), ("c2r", 512, (3, 2049))])
def test_real_counts_agree(kind, n, counts):
    pin, pout = (n, n + 2) if kind == "r2c" else (n + 2, n)  # floats per line
    x = uniform(pin * max(counts) // 2 + 1, n)[:pin * max(counts)].view(-1, pin)
    if kind == "c2r":  # Hermitian: real first and last bins
        x[:, 1] = 0
        x[:, n + 1] = 0
    outs = []
    for c in counts:
        cfg = (FftConfig.new(n) if kind == "r2c" else FftConfig.inverse(n)).with_batch(c)
        plan = getattr(FftPlan, kind)(cfg)
        y = torch.empty(c * pout, device="cuda")
        plan.execute(x[:c].contiguous(), y)
        torch.cuda.synchronize()
        outs.append(y.view(c, pout))
    m = min(counts)
    assert torch.equal(outs[0][:m], outs[1][:m])
    xs = x[:3].cpu().numpy().astype(np.float64)
    if kind == "r2c":
        ref = np.fft.rfft(xs).view(np.float64).reshape(3, pout)
    else:
        ref = np.fft.irfft(xs.view(np.complex128), n)
    got = outs[0][:3].cpu().numpy()
    assert np.linalg.norm(got - ref) <= 6e-7 * np.linalg.norm(ref)
