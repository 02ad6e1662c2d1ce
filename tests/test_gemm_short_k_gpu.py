"""int8 products of a short K with many outputs (k_gemm_mfma) at the edges of its tiles, stages and dispatch,
bit for bit against the oracle, in both forms."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
import x100hip

pytestmark = pytest.mark.gpu

# 128x128 tiles: whole, ragged rows / columns / last stage, one to seven stages; 64x64 tiles the same, by size and
# for up to 64 rows or columns; sizes on both sides of the line to k_gemm_tile
SHAPES = [(2048, 2176, 64), (2050, 2064, 16), (2049, 2128, 80), (4096, 1152, 192), (8000, 4112, 176), (6400, 6416, 448),
          (6400, 6416, 464), (1024, 1024, 64), (1601, 1040, 48), (1500, 1200, 112), (64, 65536, 64), (33, 131088, 80),
          (70001, 32, 64), (17, 65552, 16), (1024, 1024, 256)]


@pytest.mark.parametrize("acc", [True, False])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_short_k(dev, M, N, K, acc):
    import torch
    A, B = synth.gemm_inputs(M, N, K, seed=M + N + K)
    C0 = synth.rand_int8(3, (M, N)).astype(np.int32) * 4099
    dA, dB = torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev)
    dC = torch.full((M * N + 64,), 77, dtype=torch.int32, device=dev)
    dC[:M * N] = torch.from_numpy(C0).to(dev).reshape(-1)
    f = x100hip.gemm_dev if acc else x100hip.gemm_dev_set
    f(M, N, K, dA.data_ptr(), dB.data_ptr(), dC.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = dC.cpu().numpy()
    assert (got[M * N:] == 77).all()
    ref = C0.copy() if acc else np.zeros((M, N), np.int32)
    ol.gemm_ref_i8(A, B, ref, threads=16)
    assert np.array_equal(got[:M * N].reshape(M, N), ref)
