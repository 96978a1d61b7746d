"""The conjugate-transposed GEMV at the edges of its tiles, against float64 /
complex128 numpy."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float64, torch.float32, torch.complex128, torch.complex64]
EPS = {torch.float64: 2.0**-53, torch.float32: 2.0**-24, torch.complex128: 2.0**-53, torch.complex64: 2.0**-24}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,M,N,K", [(1, 1, 1, 1), (3, 17, 2, 63), (2, 64, 1, 64), (2, 65, 2, 257), (1, 300, 1, 5),
                                         (5, 33, 1, 1000)])
def test_conjt_gemv(gpu, dtype, batch, M, N, K):
    """A^H B + C for one and two columns: remainders of the column tiles and of
    the rows each slice walks; K eps |A|^T |B| bounds the sum's rounding."""
    from jaxhps_amd.adjoint import _gemm_conjt

    print(f"conjt gemv {dtype} {(batch, M, N, K)}", flush=True)
    rng = np.random.default_rng(M + K)

    def rand(*s):
        x = rng.standard_normal(s) + (1j * rng.standard_normal(s) if dtype.is_complex else 0)
        return torch.as_tensor(x).to(dtype)

    A, B, C = rand(batch, K, M), rand(batch, K, N), rand(batch, M, N)
    out = _gemm_conjt(A.to(gpu), M, K * M, M, K, B.to(gpu), N, K * N, N, batch, C=C.to(gpu), beta=1.0)
    a, b, c = (t.numpy().astype(complex) for t in (A, B, C))
    ref = a.conj().transpose(0, 2, 1) @ b + c
    bound = 4 * (K + 2) * EPS[dtype] * (np.abs(a).transpose(0, 2, 1) @ np.abs(b) + np.abs(c))
    assert (np.abs(out.cpu().numpy() - ref) <= bound).all()
