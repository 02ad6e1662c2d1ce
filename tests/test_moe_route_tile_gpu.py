"""Many-row MoE at the edges of the LDS router (k_moe_route_tile: 48 rows and more, d <= 2048; 16 rows and 1, 2
or 4 experts per block, the last ones part full) and of the expert chunks' XCD order, against the oracle, bit
for bit."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
import x100hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,d,ff,n_exp,n_act", [(47, 512, 256, 8, 2), (48, 256, 256, 60, 8), (49, 2048, 256, 6, 3),
                                                (65, 768, 256, 33, 4), (130, 2048, 256, 130, 2), (300, 512, 512, 61, 3),
                                                (512, 256, 256, 1, 1), (511, 1792, 256, 19, 2), (64, 2304, 256, 9, 2)])
def test_moe_many_rows(dev, M, d, ff, n_exp, n_act):
    import torch
    s = torch.cuda.current_stream().cuda_stream
    Wg, Wu, Wd = synth.moe_weights(n_exp, d, ff, seed=M + d)
    R = synth.moe_router(n_exp, d, seed=M + 1)
    hn = synth.normal_f32(M + 2, (M, d))
    dW = [torch.from_numpy(np.ascontiguousarray(w).view(np.uint8).reshape(-1)).to(dev) for w in (Wg, Wu, Wd)]
    dR, dh = torch.from_numpy(R).to(dev), torch.from_numpy(hn).to(dev)
    out = torch.empty((M, d), dtype=torch.float32, device=dev)
    sel = torch.empty((M, n_act), dtype=torch.int32, device=dev)
    sw = torch.empty((M, n_act), dtype=torch.float32, device=dev)
    x100hip.moe_layer(M, d, ff, n_exp, n_act, dh.data_ptr(), dR.data_ptr(), dW[0].data_ptr(), dW[1].data_ptr(),
                      dW[2].data_ptr(), out.data_ptr(), False, sel.data_ptr(), sw.data_ptr(), s)
    torch.cuda.synchronize()
    ref, rsel, rsw = ol.moe_layer(hn, R, Wg, Wu, Wd, n_act)
    assert np.array_equal(sel.cpu().numpy(), rsel)
    assert np.array_equal(sw.cpu().numpy().view(np.uint32), rsw.view(np.uint32))
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
