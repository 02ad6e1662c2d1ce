"""The matrix-core forms of the block-quantized GEMV (k_q_mm) and of the tile GEMV (k_gemv_tile_mm) at the
edges of their plans, against the oracle: bit for bit (k_q_mm keeps the dot-product kernels' summation
order), exact integers (tiles)."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
import x100hip

pytestmark = pytest.mark.gpu

# K on both sides of each plan's limit (512, 1024, 2048, 4096, 8192), whole and with blocks missing;
# N below, at and past the 16- and 32-row tiles and the 4096 / 8192 / 16384-row plan changes
I8 = [(16, 512, 2), (17, 480, 8), (33, 32, 3), (100, 544, 3), (31, 1024, 5), (48, 992, 8), (512, 2048, 5), (8200, 2048, 8),
      (15, 1056, 6), (777, 2016, 8), (2048, 4096, 5), (130, 2080, 8), (65, 3968, 7), (129, 8192, 7), (40, 4128, 8),
      (1, 2048, 8),
      # K <= 1024 and few rows of x: both sides of the lines by N
      (8191, 96, 2), (8192, 512, 2), (12287, 32, 3), (12288, 480, 3), (114689, 64, 3), (24575, 128, 4), (24576, 256, 4),
      (57345, 32, 4), (2047, 1024, 3), (2048, 992, 4), (81921, 544, 4)]
Q4 = [(16, 512, 5), (512, 2048, 8), (4099, 2048, 5), (8193, 1024, 2), (31, 1984, 7), (1, 32, 8), (129, 4096, 8),
      (8200, 2080, 3), (16390, 4096, 2), (33, 3968, 6), (17, 8192, 2), (130, 4128, 4), (48, 8160, 8)]


def check(dev, qtype, N, K, M):
    import torch
    s = torch.cuda.current_stream().cuda_stream
    W = synth.quant_weight(qtype, N, K, N + K)
    x = synth.normal_f32(N + M, (M, K))
    x[0, :32] = 0.0                    # an all-zero block
    raw = torch.from_numpy(np.ascontiguousarray(W).view(np.uint8).reshape(-1)).to(dev)
    packed = torch.empty(x100hip.packed_bytes(qtype, N, K), dtype=torch.uint8, device=dev)
    x100hip.pack(qtype, N, K, raw.data_ptr(), packed.data_ptr(), s)
    dx = torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev)
    dy = torch.full((M * N + 64,), float("nan"), dtype=torch.float32, device=dev)
    x100hip.qgemv(qtype, M, N, K, packed.data_ptr(), dx.data_ptr(), dy.data_ptr(), s)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert np.isnan(got[M * N:]).all(), "wrote past y"
    got, ref = got[:M * N].reshape(M, N), ol.qgemv(qtype, W, x)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("N,K,M", I8)
def test_i8_path(dev, N, K, M):
    check(dev, synth.Q8_0, N, K, M)


@pytest.mark.parametrize("N,K,M", Q4)
def test_q4_0(dev, N, K, M):
    check(dev, synth.Q4_0, N, K, M)


def test_q4_0_past_2_27_blocks(dev):
    # 2^20 + 3 rows of 128 blocks: the dot-product kernel's 64-bit offsets; sampled rows against the oracle
    import torch
    M, N, K = 5, (1 << 20) + 3, 4096
    s = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(1)
    raw = torch.randint(0, 256, (N, K // 32, 18), generator=g, device=dev, dtype=torch.uint8)
    raw[..., 1] = 0x18                 # fp16 scales of about 0.002
    packed = torch.empty(x100hip.packed_bytes(synth.Q4_0, N, K), dtype=torch.uint8, device=dev)
    x100hip.pack(synth.Q4_0, N, K, raw.data_ptr(), packed.data_ptr(), s)
    x = synth.normal_f32(2, (M, K))
    dx, dy = torch.from_numpy(x).to(dev), torch.empty((M, N), dtype=torch.float32, device=dev)
    x100hip.qgemv(synth.Q4_0, M, N, K, packed.data_ptr(), dx.data_ptr(), dy.data_ptr(), s)
    torch.cuda.synchronize()
    rows = np.concatenate([np.arange(8), np.random.default_rng(3).integers(0, N, 100), np.arange(N - 8, N)])
    at = torch.from_numpy(rows).to(dev)
    W, got = raw[at].cpu().numpy(), dy[:, at].cpu().numpy()
    del raw, packed, dy
    torch.cuda.empty_cache()
    ref = ol.qgemv(synth.Q4_0, np.ascontiguousarray(W), x)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("int4", [True, False])
@pytest.mark.parametrize("N,K,M", [(8, 32, 2), (24, 160, 3), (16, 992, 5), (1000, 1056, 8), (1024, 2080, 2), (264, 4864, 8),
                                   (16384, 1024, 4), (65536, 1024, 1), (40, 6528, 7), (2056, 96, 6),
                                   # fewer waves per 16 rows: 16384 and 65536 rows, K to 8 steps, last block part full
                                   (16384, 32, 2), (16392, 480, 5), (65528, 512, 8), (65536, 64, 3), (65544, 544, 2),
                                   (65544, 992, 8), (80008, 160, 7),
                                   # two rows: both sides of the lines to the dot products
                                   (4088, 160, 2), (4096, 512, 2), (65528, 480, 2), (65536, 480, 2), (4088, 2080, 2), (4096, 2080, 2)])
def test_tile(dev, int4, N, K, M):
    import torch
    W = synth.rand_int8(N + K, (N, K))
    if int4:
        W = (W >> 4).astype(np.int8)
    x = synth.rand_int8(N + K + 1, (M, K))
    dw = torch.from_numpy(x100hip.pack_w(int4, W).view(np.uint8)).to(dev)
    dx = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    dy = torch.full((M * N + 64,), -7, dtype=torch.int32, device=dev)
    x100hip.gemv_tile(int4, M, N, K, dw.data_ptr(), dx.data_ptr(), dy.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    assert (got[M * N:] == -7).all()
    assert np.array_equal(got[:M * N].reshape(M, N), ol.gemv_int(W, x))


@pytest.mark.parametrize("int4,K", [(False, 16), (False, 32), (True, 32)])
def test_tile_2_28_rows(dev, int4, K):
    # one launch of four waves per 16 rows would pass 2^32 - 1 threads; the first, last and some other rows
    import torch
    M, N = 2, 1 << 28
    g = torch.Generator(device=dev).manual_seed(K)
    nb = N * K // (2 if int4 else 1)
    W = torch.randint(0, 256, (nb,), generator=g, device=dev, dtype=torch.uint8)
    x = synth.rand_int8(K, (M, K))
    dx = torch.from_numpy(x).to(dev)
    dy = torch.full((M * N + 64,), -7, dtype=torch.int32, device=dev)
    x100hip.gemv_tile(int4, M, N, K, W.data_ptr(), dx.data_ptr(), dy.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (dy[M * N:] == -7).all()
    blocks = np.unique(np.concatenate([np.arange(16), N // 8 - 16 + np.arange(16), np.random.default_rng(K).integers(0, N // 8, 500)]))
    tiles = W.reshape(N // 8, -1, 8, 16)[torch.from_numpy(blocks).to(dev)].cpu().numpy()   # [block][tile][row][16 bytes]
    got = dy[:M * N].reshape(M, N // 8, 8)[:, torch.from_numpy(blocks).to(dev)].cpu().numpy()
    del W, dy
    torch.cuda.empty_cache()
    if int4:
        lo, hi = (tiles << 4).view(np.int8) >> 4, tiles.view(np.int8) >> 4
        rows = np.concatenate([lo, hi], axis=3)
    else:
        rows = tiles.view(np.int8)
    rows = rows.transpose(0, 2, 1, 3).reshape(len(blocks), 8, K).astype(np.int64)
    assert np.array_equal(got, np.einsum("mk,bnk->mbn", x.astype(np.int64), rows))
