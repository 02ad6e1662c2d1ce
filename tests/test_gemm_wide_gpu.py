"""int8 GEMM on operands too large to multiply on the host, checked on sampled columns against exact 64-bit
products: rows of C beyond the 32-bit offsets of the 256x256 tiles."""
import numpy as np
import pytest

import x100hip

pytestmark = pytest.mark.gpu


def check(dev, M, N, K, acc, variant=x100hip.GEMM_AUTO):
    import torch
    print("M %d N %d K %d acc %d variant %d" % (M, N, K, acc, variant), flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    A = torch.randint(-128, 128, (M, K), generator=g, device=dev, dtype=torch.int8)
    B = torch.randint(-128, 128, (K, N), generator=g, device=dev, dtype=torch.int8)
    C = torch.randint(-(1 << 20), 1 << 20, (M, N), generator=g, device=dev, dtype=torch.int32)
    rng = np.random.default_rng(N)
    cols = np.unique(np.concatenate([np.arange(min(N, 64)), np.arange(max(N - 64, 0), N), rng.integers(0, N, 512)]))
    rows = np.unique(np.concatenate([np.arange(min(M, 64)), np.arange(max(M - 64, 0), M), rng.integers(0, M, 512)]))
    at = (torch.from_numpy(rows).to(dev)[:, None], torch.from_numpy(cols).to(dev)[None, :])
    old = C[at].cpu().numpy().astype(np.int64)
    f = x100hip.gemm_dev if acc else x100hip.gemm_dev_set
    f(M, N, K, A.data_ptr(), B.data_ptr(), C.data_ptr(), torch.cuda.current_stream().cuda_stream, variant)
    torch.cuda.synchronize()
    got = C[at].cpu().numpy()
    # float64 products are exact: |sum| <= 2^14 K < 2^53
    a, b = A[at[0][:, 0]].cpu().numpy().astype(np.float64), B[:, at[1][0]].cpu().numpy().astype(np.float64)
    want = (a @ b).astype(np.int64) + (old if acc else 0)
    del A, B, C
    torch.cuda.empty_cache()
    assert np.array_equal(got, ((want + 2**31) % 2**32 - 2**31).astype(np.int32))


# the last and the first N on each side of k_gemm_big's limit where C is added; past the first wrap of a signed
# offset; the overwrite form beyond it
@pytest.mark.parametrize("M,N,K,acc", [(256, 6029312, 512, True), (256, 7508480, 512, True), (256, 7508736, 512, True),
                                       (512, 7508736, 576, True), (256, 1 << 23, 512, False)])
def test_wide_256_tiles(dev, M, N, K, acc):
    check(dev, M, N, K, acc, x100hip.GEMM_TILE256)
    check(dev, M, N, K, acc)
