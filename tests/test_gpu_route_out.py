"""The routing that a device-pointer forward hands its caller: the same ids and weights as
the host form's, for decode, batched and multi-chunk calls, and only where it is asked for;
a layer's and an FFN block's."""
import numpy as np
import pytest
import torch

import zzref as Z
import zunzuncito_amd as zz
from test_gpu_gemma import close_all, gpu_block
from test_gpu_parity import gpu_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["gemma", "lfm", "maple", "ling"])
def test_device_routing_outputs(kind):
    zz.init()
    L = Z.make_layer(kind, seed=37, E=16, K=4, D=512, MI=256)
    if kind == "ling":
        L.n_group, L.topk_group = 4, 2
    m = gpu_layer(L)
    try:
        for S in (1, 2, 5, 17, 64, 2100):         # 2048 tokens a chunk at K = 4
            print("case", kind, S, flush=True)
            x = Z.make_input(L, S, 3)
            _, ids, wts = m.forward(x)
            xd = torch.from_numpy(x).cuda()
            out = torch.empty_like(xd)
            for want_i, want_w in ((True, True), (True, False), (False, True)):
                ei = torch.full((S + 1, L.K), -7, dtype=torch.int32, device="cuda")
                ew = torch.full((S + 1, L.K), -7.0, device="cuda")
                m.forward_dev(xd.data_ptr(), out.data_ptr(), S, ei.data_ptr() if want_i else 0,
                              ew.data_ptr() if want_w else 0, torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                assert np.array_equal(ei[:S].cpu().numpy().ravel(), ids) if want_i else bool((ei == -7).all())
                assert np.array_equal(ew[:S].cpu().numpy().ravel(), wts) if want_w else bool((ew == -7).all())
                assert bool((ei[S] == -7).all()) and bool((ew[S] == -7).all())
    finally:
        m.close()


def test_block_routing_outputs():
    """The block's routing is its MoE layer's, by the fused decode launches (up to 4 rows)
    and by the batched path, either output alone too."""
    zz.init()
    L = Z.make_layer("gemma", seed=39, E=16, K=4, D=512, MI=256)
    b, m, d = gpu_block(L, Z.make_dense(L.D, 512, 40))
    try:
        for S in (1, 3, 4, 5, 33):
            print("case block", S, flush=True)
            x = Z.make_input(L, S, 5)
            _, ids, wts = m.forward(x)
            for want_i, want_w in ((True, True), (True, False), (False, True)):
                H = torch.from_numpy(x).cuda()
                ei = torch.full((S + 1, L.K), -7, dtype=torch.int32, device="cuda")
                ew = torch.full((S + 1, L.K), -7.0, device="cuda")
                b.forward_dev(H.data_ptr(), S, ei.data_ptr() if want_i else 0, ew.data_ptr() if want_w else 0,
                              torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                assert np.array_equal(ei[:S].cpu().numpy().ravel(), ids) if want_i else bool((ei == -7).all())
                assert np.array_equal(ew[:S].cpu().numpy().ravel(), wts) if want_w else bool((ew == -7).all())
                assert bool((ei[S] == -7).all()) and bool((ew[S] == -7).all())
    finally:
        close_all(b, m, d)
