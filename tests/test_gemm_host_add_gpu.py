"""The host-pointer GEMM adds A.B to C on the host as it comes back: int32 wrap-around, the first and last
elements of every thread's part and chunk (sizes at and around 4 MiB chunks and the 1 MiB threading limit,
more chunks than staging slots out and in), C at a 4-byte aligned address."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
import x100hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,off", [(1, 1, 1, 0), (3, 5, 7, 1), (512, 512, 16, 0), (511, 513, 33, 3), (1024, 1024, 16, 1),
                                       (1024, 1025, 8, 0), (1031, 4093, 17, 2), (2500, 2100, 32, 0),
                                       # more than four chunks in: a slot is used again (B; A and then B)
                                       (64, 1500, 16000, 0), (1400, 33, 16000, 1)])
def test_host_gemm_adds(dev, M, N, K, off):
    A, B = synth.gemm_inputs(M, N, K, seed=M + N)
    rng = np.random.default_rng(K)
    buf = np.full(M * N + off + 8, 12345, np.int32)
    C = buf[off:off + M * N].reshape(M, N)
    C[:] = rng.integers(-2**31, 2**31, (M, N), dtype=np.int64).astype(np.int32)   # sums wrap
    ref = C.copy()
    ol.gemm_ref_i8(A, B, ref, threads=16)
    x100hip.gemm_host(A, B, C)
    assert np.array_equal(C, ref)
    assert (buf[:off] == 12345).all() and (buf[off + M * N:] == 12345).all()
