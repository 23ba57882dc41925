"""Index maps of the runtime-schedule register lines (mix_kernels.hpp) against
numpy's FFT: LDS slot of a stage's outputs, the slots the next stage reads, and
its twiddle index, for schedules of two to five stages in any order."""
import numpy as np
import pytest


def simulate(x, radices):
    n = len(x)
    L, buf, w = 1, None, None
    for s, R in enumerate(radices):
        nr = n // R
        if s == 0:
            w = x.reshape(R, nr).T.copy()  # butterfly j holds points j + m n / R
        else:
            Rp, Lp = radices[s - 1], L // radices[s - 1]
            nrp_prev, rstep = (n // Rp) | 1, n // (L * R) * Lp
            w = np.empty((nr, R), complex)
            for j in range(nr):
                kq, k = divmod(j, L)
                m, kk = divmod(k, Lp)
                at = m * nrp_prev + kq * Lp + kk
                for i in range(R):
                    w[j, i] = buf[at + i * rstep] * np.exp(-2j * np.pi * k * i / (L * R))
        w = np.fft.fft(w, axis=1)
        if s + 1 == len(radices):
            out = np.empty(n, complex)
            for i in range(R):
                out[np.arange(nr) + i * nr] = w[:, i]
            return out
        nrp = nr | 1
        buf = np.full(R * nrp, np.nan, complex)
        for i in range(R):
            buf[i * nrp + np.arange(nr)] = w[:, i]
        L *= R


@pytest.mark.parametrize("radices", [(9, 2), (12, 9), (16, 16), (15, 6, 12), (2, 13, 3), (3, 3, 3, 3), (7, 5, 8, 5),
                                     (2, 3, 5, 7, 11)])
def test_mix_exchange_layout(radices):
    n = int(np.prod(radices))
    x = np.random.default_rng(n).standard_normal((n, 2)) @ [1, 1j]
    assert np.max(np.abs(simulate(x, radices) - np.fft.fft(x))) < 1e-10 * n


@pytest.mark.parametrize("r1,r2", [(2, 3), (2, 5), (4, 3), (2, 7), (3, 5)])
def test_coprime_butterfly(r1, r2):
    """DftCoprime: input and output index maps without a twiddle between the factors."""
    r = r1 * r2
    v = np.random.default_rng(r).standard_normal((r, 2)) @ [1, 1j]
    y = np.array([[v[(r2 * n1 + r1 * n2) % r] for n1 in range(r1)] for n2 in range(r2)])
    y = np.fft.fft(np.fft.fft(y, axis=1), axis=0)
    out = np.empty(r, complex)
    for k1 in range(r1):
        for k2 in range(r2):
            out[next(k for k in range(k1, r, r1) if k % r2 == k2)] = y[k2, k1]
    assert np.allclose(out, np.fft.fft(v))
