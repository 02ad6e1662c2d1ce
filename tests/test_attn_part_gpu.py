"""Decode attention at the edges of k_attn_part's passes against the oracle, bit for bit: chunks of 16 to
200 positions (passes of 64, part passes), 1 to 16 query heads per KV head, pos alone in its chunk, and
cache rows at and after pos holding NaN (the kernel reads the row of pos before it is written)."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
from test_decode_gpu import GpuLayer, close
from test_decode_oracle import caches, make_cfg

pytestmark = pytest.mark.gpu
T = (synth.Q4_K,) * 4


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# (query heads, KV heads, positions pos): with 256 / KV heads chunks, 8 KV heads give CH = pos / 32
# rounded up to 8.  pos = 4 CH k leaves pos alone in the last chunk.
@pytest.mark.parametrize("nh,nkv,positions", [
    (8, 8, (511, 520, 767, 768, 2047, 2048, 2304)),   # 1 head per KV head: CH 16, 24, 24, 32, 64, 72, 80
    (24, 8, (2000, 4160, 6399)),                       # 3: CH 64, 136, 200
    (40, 8, (1000, 2112)),                             # 5
    (64, 8, (900, 2048, 4095)),                        # 8
    (32, 2, (1500, 3080, 8192)),                       # 16: CH 16, 32, 72
])
def test_attn_part(dev, nh, nkv, positions):
    ctx = max(positions) + 9
    cfg = make_cfg(T, n_head=nh, n_head_kv=nkv, ctx=ctx)
    L = synth.decode_layer_weights(512, nh, nkv, 128, 256, 8, T, seed=nh + nkv)
    gl = GpuLayer(cfg, L, T, dev)
    for pos in positions:
        kc, vc = caches(cfg, pos, 77 + pos)
        rk, rv = kc.copy(), vc.copy()
        kc[:, pos:] = np.nan
        vc[:, pos:] = np.nan
        gl.set_cache(kc, vc)
        h = synth.normal_f32(pos, (cfg.d,))
        got, _, _ = gl.run(pos, h)
        rh = h.copy()
        ol.attn_decode(cfg, L, rk, rv, pos, rh)
        close(got, rh, "h pos %d" % pos)
        gk, gv = gl.kc.cpu().numpy(), gl.vc.cpu().numpy()
        close(gk[:, pos], rk[:, pos], "k row")
        close(gv[:, pos], rv[:, pos], "v row")
        for g, r in ((gk, kc), (gv, vc)):
            assert np.array_equal(bits(np.delete(g, pos, 1)), bits(np.delete(r, pos, 1)))
