"""Routing and permutation of many tokens: every token count per workgroup that the one-launch
routing chooses between, and the permutation on either side of where it takes more workgroups
and where the waves' runs end.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from berth_amd import kernels as K
from berth_amd import synth
from oracle import oracle as O
from tests.gpu_util import DEV
from tests.test_gpu_moe import _route

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,k,per_workgroup", [(256, 256, 128, 4, 1), (257, 256, 66, 4, 2), (700, 128, 128, 8, 3),
                                                   (1021, 64, 60, 5, 4), (1501, 2048, 128, 8, 6), (200, 128, 1024, 10, 4)])
def test_routing_of_many_tokens(T, H, E, k, per_workgroup):
    x, wr = synth.activations(T, T, H), synth.router_weight(E, H, E)
    idx, w, logits = _route(x, wr, k)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert f"moe_route_slab_kernel<{per_workgroup}>" in K.moe.last_launch(), K.moe.last_launch()
    oi, ow, ol = O.moe_route(x, wr, k, want_logits=True)
    assert np.array_equal(logits.view(np.uint32), ol.view(np.uint32))
    assert np.array_equal(idx, oi)
    assert np.allclose(w, ow, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("T,k,E,hot", [(70, 1, 1, False), (127, 8, 128, False), (128, 8, 128, True), (129, 8, 60, False),
                                       (1500, 8, 128, True), (1024, 16, 512, False), (4097, 16, 1024, True)])
def test_permutation_of_many_pairs(T, k, E, hot):
    rng = np.random.default_rng(T + E)
    score = rng.random((T, E)) - (np.log(np.arange(E) + 1.0) if hot else 0.0)
    idx = np.argsort(-score, axis=1)[:, :k].astype(np.int32)
    d_idx = torch.from_numpy(idx).to(DEV)
    off = torch.zeros(E + 1, dtype=torch.int32, device=DEV)
    perm, inv = (torch.zeros(T * k, dtype=torch.int32, device=DEV) for _ in range(2))
    scratch = torch.zeros(K.moe.permute_scratch_bytes(T, k, E), dtype=torch.uint8, device=DEV)
    K.moe.permute(d_idx.data_ptr(), off.data_ptr(), perm.data_ptr(), inv.data_ptr(), scratch.data_ptr(), T, k, E)
    torch.cuda.synchronize()
    ooff, operm = O.moe_permute(idx, E)
    assert np.array_equal(off.cpu().numpy(), ooff)
    assert np.array_equal(perm.cpu().numpy(), operm)
    assert np.array_equal(inv.cpu().numpy()[operm], np.arange(T * k))
