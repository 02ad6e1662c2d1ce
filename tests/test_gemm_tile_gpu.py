"""k_gemm_tile at the edges of its tiles, K stages and operands, bit-exact against the oracle.

M and N around the 32 / 64 / 128 tiles; K around the 128-k stage, the 4-slot ring's turn and the loop
that unrolls it, with remainders that 16-byte chunks divide (global->LDS DMA) and that they do not
(unaligned loads, the matrix's last chunk shifted); odd base addresses; operands of one chunk."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
import x100hip

pytestmark = pytest.mark.gpu

TILES = [x100hip.GEMM_TILE128, x100hip.GEMM_TILE64, x100hip.GEMM_TILE32]


def run(dev, M, N, K, acc, variant=None, off=(0, 0, 0)):
    import torch
    A, B = synth.gemm_inputs(M, N, K, seed=M + 3 * N + 7 * K)
    C0 = synth.rand_int8(9, (M, N)).astype(np.int32) * 4099

    def at(x, o):   # a device copy whose first byte is o elements past an aligned address, nothing after it
        buf = torch.empty(x.size + o, dtype=torch.int8 if x.dtype == np.int8 else torch.int32, device=dev)
        buf[o:].copy_(torch.from_numpy(np.ascontiguousarray(x)).reshape(-1))
        return buf, buf.data_ptr() + o * x.itemsize

    (_a, pa), (_b, pb), (c, pc) = at(A, off[0]), at(B, off[1]), at(C0, off[2])
    f = x100hip.gemm_dev if acc else x100hip.gemm_dev_set
    f(M, N, K, pa, pb, pc, torch.cuda.current_stream().cuda_stream, *([] if variant is None else [variant]))
    torch.cuda.synchronize()
    ref = C0.copy() if acc else np.zeros((M, N), np.int32)
    ol.gemm_ref_i8(A, B, ref, threads=16)
    assert np.array_equal(c[off[2]:].cpu().numpy().reshape(M, N), ref)


@pytest.mark.parametrize("variant", TILES)
@pytest.mark.parametrize("M,N,K", [(17, 16, 16), (127, 112, 112), (128, 128, 128), (129, 144, 144), (65, 80, 256),
                                   (33, 272, 384), (96, 48, 528), (160, 64, 896), (31, 144, 1008), (64, 128, 1040),
                                   (130, 32, 1152), (40, 48, 1664), (257, 240, 2064)])
def test_tile_aligned(dev, variant, M, N, K):
    run(dev, M, N, K, True, variant)
    run(dev, M, N, K, False, variant)


@pytest.mark.parametrize("M,N,K", [(1, 16, 17), (1, 17, 16), (16, 1, 1), (3, 5, 6), (33, 31, 127), (64, 65, 129),
                                   (63, 17, 255), (31, 3, 257), (5, 70, 385), (100, 33, 514), (129, 67, 643),
                                   (700, 513, 131), (1030, 777, 1), (2, 1300, 1000), (1300, 2, 999), (1025, 1600, 270)])
def test_tile_unaligned(dev, M, N, K):
    run(dev, M, N, K, True)
    run(dev, M, N, K, False)


@pytest.mark.parametrize("off", [(1, 0, 0), (0, 3, 0), (7, 13, 1), (0, 0, 3)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 128), (8, 256, 512), (300, 256, 400), (1024, 1024, 272)])
def test_tile_base_address(dev, M, N, K, off):
    run(dev, M, N, K, True, off=off)
    run(dev, M, N, K, False, off=off)


@pytest.mark.parametrize("M,N,K", [(17, 4096, 1024), (200, 2048, 640), (333, 2048, 512), (1024, 512, 256),
                                   (2000, 1008, 320), (16, 1280, 1280), (2048, 2048, 512)])
def test_tile_auto(dev, M, N, K):
    run(dev, M, N, K, True)
    run(dev, M, N, K, False)


# Every form of the automatic choice over its pipeline: (tile, aligned, M, N, K).  The aligned 32x64 tile, which no
# variant selects, over the ring's unrolled turn (8 stages and more) and K tails; the unaligned tiles over two to
# twenty stages.  test_gemm_plan.py checks that the sizes take these tiles.
FORMS = [("32x64", 1, 97, 3088, 272), ("32x64", 1, 130, 2064, 1040), ("32x64", 1, 97, 2064, 1168), ("32x64", 1, 180, 1040, 2096),
         ("128", 0, 1001, 1503, 999), ("128", 0, 1300, 1503, 514), ("128", 0, 700, 2049, 1155), ("128", 0, 2047, 1601, 385),
         ("64", 0, 1100, 1300, 257), ("64", 0, 2049, 1153, 515), ("64", 0, 1025, 1600, 270),
         ("32x64", 0, 700, 777, 131), ("32x64", 0, 700, 777, 387), ("32x64", 0, 700, 777, 514), ("32x64", 0, 513, 771, 1023),
         ("32", 0, 37, 41, 2500), ("32", 0, 300, 300, 1201)]


@pytest.mark.parametrize("tile,aligned,M,N,K", FORMS)
def test_tile_forms(dev, tile, aligned, M, N, K):
    run(dev, M, N, K, True)
    run(dev, M, N, K, False)
