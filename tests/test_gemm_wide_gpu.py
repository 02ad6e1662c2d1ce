"""int8 GEMM on operands too large to multiply on the host, checked on sampled columns against exact 64-bit
products: rows of C beyond the 32-bit offsets of the 256x256 tiles, and N or K from 2^24 on k_gemm_mfma."""
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
    e, r = (64, 512) if K < 1 << 20 else (8, 16)   # the ends of the range and some between
    rows, cols = (np.unique(np.concatenate([np.arange(min(n, e)), np.arange(max(n - e, 0), n), rng.integers(0, n, r)]))
                  for n in (M, N))
    at = (torch.from_numpy(rows).to(dev)[:, None], torch.from_numpy(cols).to(dev)[None, :])
    old = C[at].cpu().numpy().astype(np.int64)
    f = x100hip.gemm_dev if acc else x100hip.gemm_dev_set
    f(M, N, K, A.data_ptr(), B.data_ptr(), C.data_ptr(), torch.cuda.current_stream().cuda_stream, variant)
    torch.cuda.synchronize()
    got = C[at].cpu().numpy()
    # float64 products are exact: |sum| <= 2^14 K < 2^53
    want = old if acc else np.zeros_like(old)
    for k in range(0, K, 1 << 20):
        a = A[:, k:k + (1 << 20)][at[0][:, 0]].cpu().numpy().astype(np.float64)
        b = B[k:k + (1 << 20)][:, at[1][0]].cpu().numpy().astype(np.float64)
        want = want + (a @ b).astype(np.int64)
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


# N and K just past 2^24 and where 127 rows pass 2^32 bytes; ragged rows, columns and last K stages; sums that wrap
@pytest.mark.parametrize("M,N,K,variants", [
    (48, 1 << 24, 64, (0, 6, 7)), (33, (1 << 24) + 16, 400, (0, 6)), (20, (1 << 26) + 48, 32, (0,)), (130, (1 << 24) + 80, 1168, (0, 6)),
    (64, 128, 1 << 24, (0, 2)), (70, 112, (1 << 25) + 48, (0, 6))])
def test_rows_of_2_24(dev, M, N, K, variants):
    for variant in variants:   # AUTO, TILE128, TILE64, TILE32
        for acc in (True, False):
            check(dev, M, N, K, acc, variant)


# more rows than one launch of k_gemm_tile holds (2^32 - 1 threads)
def test_2_30_rows(dev):
    check(dev, (1 << 30) + 33, 16, 16, True)
