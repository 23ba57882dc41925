"""Batched transforms at every 16-byte offset of a 128-byte line: the passes
over adjacent lines start their tiles at 128-byte lines, which must not change
a bit of the results nor touch a point outside of them."""
import pytest
import torch

from wgpufft_amd import FftBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lines", [(65536, 3), (16384, 2), (32768, 1), (4096, 3)])
@pytest.mark.parametrize("off_in,off_out", [(0, 0), (2, 0), (0, 2), (6, 10), (14, 8), (8, 14)])
def test_offsets(n, lines, off_in, off_out):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.view_as_complex(torch.rand(n * lines, 2, device="cuda", generator=g) * 2 - 1)
    want = torch.empty_like(x)
    FftBatch([dict(n=n, batch=lines, input=x, output=want)]).execute()
    src = torch.full((n * lines + 32,), complex(float("nan"), 0), dtype=torch.complex64, device="cuda")
    dst = torch.full_like(src, 7)
    src[off_in:off_in + n * lines] = x
    FftBatch([dict(n=n, batch=lines, input=src[off_in:off_in + n * lines],
                   output=dst[off_out:off_out + n * lines])]).execute()
    torch.cuda.synchronize()
    assert torch.equal(dst[off_out:off_out + n * lines], want)
    assert torch.all(dst[:off_out] == 7) and torch.all(dst[off_out + n * lines:] == 7)
