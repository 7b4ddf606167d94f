"""How dense launches of 128-row tiles are cut up, as the cost rule decides it: whole tiles for a short K, in
less than a round of the compute units, in several, and for bundles whose slices differ in width; dealt out
for a longer one.  Bar: rtol 2e-3 / atol 1e-3 of the oracle's fp32 sums; a second call gives the same bits."""
import numpy as np
import pytest
import torch

from berth_amd import kernels as K
from berth_amd import synth
from berth_amd.kernels import Codebook, OutDtype
from oracle import oracle as O
from tests.gpu_util import DEV, close, dev, host_f16
from tests.test_gpu_linear import _run_linear

pytestmark = pytest.mark.gpu

WHOLE, DEALT = "exl3_gemm_kernel<{},{},128x256>", "exl3_gemm_balanced_kernel<{},{},128x256>"


@pytest.mark.parametrize("rows,Kk,N,bits,cb,fp32,kernel", [
    (449, 128, 4096, 4, 2, True, WHOLE),        # one k-block, 64 tiles, the last of one row
    (512, 384, 8192, 3, 1, False, WHOLE),       # half a round
    (600, 256, 16640, 4, 2, True, WHOLE),       # a round and a quarter, half of the last column tile empty
    (1400, 128, 16384, 5, 0, False, WHOLE),     # nearly three rounds
    (460, 2048, 4096, 4, 2, False, DEALT),
])
def test_kernel_by_cost_matches_the_oracle_and_repeats(rows, Kk, N, bits, cb, fp32, kernel):
    got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, cb, fp32, 40 + rows, prefill=True)
    assert kernel.format(bits, cb) in launch, launch
    if kernel == WHOLE:
        assert "split_k=1 " in launch, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)
    again = _run_linear(rows, Kk, N, bits, cb, fp32, 40 + rows, prefill=True)[0]
    assert np.array_equal(got.view(np.uint8), again.view(np.uint8)), launch


def test_bundle_of_narrower_slices_as_whole_tiles():
    rows, Kk, width, widths, bits = 460, 256, 4096, (4096, 1024, 384), 4
    lins = [synth.linear(340 + i, Kk, n, bits) for i, n in enumerate(widths)]
    d = [[dev(t.view(np.uint16)) for t in lin] for lin in lins]
    x = synth.activations(350, rows, Kk)
    outs = [torch.full((rows, n), 5.0, dtype=torch.float16, device=DEV) for n in widths]
    i64 = lambda v: torch.tensor(v, dtype=torch.int64, device=DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    lists = [i64([dd[j].data_ptr() for dd in d]) for j in range(3)]
    c_ptrs, n_list, src = i64([o.data_ptr() for o in outs]), i32(list(widths)), i32([0, 1, 2])
    a_had = torch.zeros((3, rows, Kk), dtype=torch.float16, device=DEV)
    d_x = dev(x.view(np.uint16))
    K.ops.exl3_mgemm(d_x.data_ptr(), lists[0].data_ptr(), outs[0].data_ptr(), lists[1].data_ptr(), a_had.data_ptr(),
                     lists[2].data_ptr(), rows, Kk, width, bits, Codebook.MUL1, OutDtype.F16, 1, 3, n_list.data_ptr(),
                     c_ptrs.data_ptr(), n_list.data_ptr(), src.data_ptr(), 3)
    torch.cuda.synchronize()
    assert WHOLE.format(4, 2) in K.ops.last_launch(), K.ops.last_launch()
    for i, (tr, suh, svh) in enumerate(lins):
        want, _ = O.linear(x, tr, suh, svh, Kk, widths[i], bits, 2, out_fp32=False)
        assert close(host_f16(outs[i]), want)[0] == 0, i
