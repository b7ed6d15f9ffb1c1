"""Workgroup LDS FFT vs numpy (FP64), on the GPU; lengths whose transform
exceeds one workgroup's LDS (complex 36000 and 37044, real 72000, 72576 and
74088: the dt 0.05 s lengths) run the four-step transform over HBM."""
import numpy as np
import pytest

from oracle.xc import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 98, 2001, 18000, 18144, 18522, 36000, 37044])
def test_c2c_forward_inverse(gpu, n):
    import torch
    from fastxc_amd import ops

    rng = np.random.default_rng(n)
    x = (rng.standard_normal((3, n)) + 1j * rng.standard_normal((3, n))).astype(np.complex64)
    xd = torch.from_numpy(x).to(gpu)
    f = ops.fft_c2c(xd).cpu().numpy()
    assert rel_l2(f, np.fft.fft(x.astype(np.complex128))) < 1e-6
    b = ops.fft_c2c(xd, inverse=True).cpu().numpy()
    assert rel_l2(b, np.fft.ifft(x.astype(np.complex128)) * n) < 1e-6


@pytest.mark.parametrize("n,in_len", [(36000, 36000), (36288, 36000), (37044, 36000), (24, 20),
                                      (72000, 72000), (72576, 72000), (74088, 72000)])
def test_r2c_c2r(gpu, n, in_len):
    import torch
    from fastxc_amd import ops

    rng = np.random.default_rng(n)
    x = rng.standard_normal((4, in_len)).astype(np.float32)
    X = ops.fft_r2c(torch.from_numpy(x).to(gpu), n=n).cpu().numpy()
    want = np.fft.rfft(x.astype(np.float64), n=n)
    assert rel_l2(X, want) < 1e-6
    assert np.all(X[:, 0].imag == 0) and np.all(X[:, -1].imag == 0)
    y = ops.fft_c2r(torch.from_numpy(want.astype(np.complex64)).to(gpu), n).cpu().numpy()
    assert rel_l2(y, np.fft.irfft(want, n=n) * n) < 1e-6


@pytest.mark.parametrize("n,in_len,rows", [(40960, 40959, 3), (40000, 1, 2), (72900, 72900, 300),
                                           (75000, 70001, 2), (79380, 79380, 2)])
def test_real_halves(gpu, n, in_len, rows):
    """Real transforms of two half-length LDS transforms: about the shortest and the longest
    length that takes them, odd and even halves, zero padding that ends inside a sample group,
    more rows than workgroups."""
    import torch
    from fastxc_amd import ops

    rng = np.random.default_rng(n)
    x = rng.standard_normal((rows, in_len)).astype(np.float32)
    X = ops.fft_r2c(torch.from_numpy(x).to(gpu), n=n).cpu().numpy()
    want = np.fft.rfft(x.astype(np.float64), n=n)
    assert rel_l2(X, want) < 1e-6
    assert np.all(X[:, 0].imag == 0) and np.all(X[:, -1].imag == 0)
    z = (rng.standard_normal((rows, n // 2 + 1)) + 1j * rng.standard_normal((rows, n // 2 + 1)))
    z = z.astype(np.complex64)
    ref = np.fft.irfft(z.astype(np.complex128), n=n) * n
    for out_len in (n, in_len, n // 2 + 1):
        y = ops.fft_c2r(torch.from_numpy(z).to(gpu), n, out_len=out_len).cpu().numpy()
        assert rel_l2(y, ref[:, :out_len]) < 1e-6
