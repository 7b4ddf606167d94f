"""The row-block MFMA kernel (more than 32 rows; blocks of up to 128 rows x 128 columns, steps of
256 rows of K dealt out evenly) at the sizes where it can go wrong, against the oracle: blocks
that are full, of one row more than a tile of sixteen, of every height class; K that leaves
k groups of the last step empty; tiles inside one workgroup and shared by many; bundles with
narrower slices.  Bar: rtol 2e-3 / atol 1e-3 of the oracle's fp32 sums; a second call gives the
same bits."""
import numpy as np
import pytest
import torch

from berth_amd import kernels as K
from berth_amd import synth
from berth_amd.kernels import Codebook, OutDtype
from oracle import oracle as O
from tests.gpu_util import DEV, close, dev, host_f16, host_u16, knobs
from tests.test_gpu_linear import _run_linear

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _every_size():
    with knobs(BERTH_GEMM_BLOCK_ROWS=1 << 30, BERTH_GEMM_BLOCK_STEPS=0):
        yield


@pytest.mark.parametrize("rows,Kk,N,bits,cb,fp32", [
    (33, 128, 128, 4, 2, True),         # one step with two of four k groups, one workgroup
    (48, 256, 256, 3, 1, False),        # one full step
    (49, 384, 1280, 5, 0, True),        # two steps, the second half empty
    (64, 4096, 384, 2, 2, False),       # three tiles cut into many parts
    (65, 1408, 640, 6, 2, True),        # 80-row blocks
    (97, 2176, 256, 8, 2, False),       # 112-row blocks
    (128, 1024, 1024, 4, 2, True),
    (129, 1024, 1152, 7, 1, True),      # two blocks of 80 rows, the second short
    (300, 640, 4352, 1, 2, False),      # three blocks; more tiles than fit the parts: ranges across tiles
    (520, 256, 8192, 4, 2, True),       # five blocks, several whole tiles per workgroup
])
def test_row_blocks_match_the_oracle_and_repeat(rows, Kk, N, bits, cb, fp32):
    got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, cb, fp32, 60 + rows, prefill=True)
    assert "exl3_gemm_block_kernel" in launch, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)
    again = _run_linear(rows, Kk, N, bits, cb, fp32, 60 + rows, prefill=True)[0]
    assert np.array_equal(got.view(np.uint8), again.view(np.uint8)), launch


@pytest.mark.parametrize("rows", [34, 48, 50, 66, 80, 81, 96, 99, 112, 113, 210])
def test_every_height_with_whole_and_shared_tiles(rows):
    """Blocks of 48 to 128 rows, full and not: the last row tiles of the exchange between the k groups, operand loads that do not
    divide evenly.  136 tiles (or 272) of two steps for 256 workgroups: some inside one, some shared."""
    Kk, N, bits = 512, 17408, 4
    got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, 2, True, 160 + rows, prefill=True)
    height = (rows if rows <= 128 else rows // 2) + 15 & ~15
    assert f"exl3_gemm_block_kernel<4,2,{height}x128>" in launch and "exl3_gemm_finish_kernel" in launch, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)


@pytest.mark.parametrize("rows,Kk,N,cb,blocks", [
    (200, 2048, 8192, 2, True),         # two blocks of 112 rows, four steps a compute unit
    (300, 1024, 8192, 2, False),        # three steps a compute unit
    (200, 2048, 8192, 1, True),         # MCG: beside up to half a chip of tiles
    (300, 2048, 8192, 2, True),         # three blocks: up to half a chip
    (300, 2048, 12288, 2, False),
    (400, 2048, 8192, 2, True),         # four blocks: up to a whole chip, 32 steps a compute unit
    (400, 8448, 8192, 2, False),
    (450, 2048, 8192, 2, True),         # blocks of 128: one tile a workgroup
    (450, 3072, 6144, 2, False),        # ranges across tiles
    (513, 2048, 8192, 2, False),        # above the limit of rows
])
def test_the_rule_beside_wide_tiles(rows, Kk, N, cb, blocks):
    """Both sides of the rule that sends several row blocks of wide outputs to this kernel, each against the oracle."""
    with knobs(BERTH_GEMM_BLOCK_ROWS=511, BERTH_GEMM_BLOCK_STEPS=-1):        # the rule as it is, on a card of 256 compute units
        got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, 3, cb, False, 260 + rows, prefill=True)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert ("exl3_gemm_block_kernel" in launch) == blocks, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)


@pytest.mark.parametrize("rows,Kk,N,cb,blocks", [
    (36, 3072, 512, 2, True),           # 48 steps
    (36, 3072, 384, 2, False),
    (35, 4096, 1024, 2, False),
    (96, 2944, 1024, 2, False),         # not deep enough
    (97, 4096, 1024, 2, False),         # blocks of more than 96 rows
    (160, 3584, 512, 1, True),          # two blocks of 80
    (160, 3456, 512, 0, False),
    (288, 4096, 512, 2, False),         # three
])
def test_the_rule_of_deep_weights(rows, Kk, N, cb, blocks):
    """Both sides of the rule that sends deep and narrow weights to this kernel, each against the oracle."""
    with knobs(BERTH_GEMM_BLOCK_ROWS=511, BERTH_GEMM_BLOCK_STEPS=-1):
        got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, 4, cb, True, 280 + rows, prefill=True)
    assert ("exl3_gemm_block_kernel" in launch) == blocks, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)


@pytest.mark.parametrize("rows,Kk,N,blocks", [
    (385, 640, 12288, False),           # three steps a tile, in ranges across tiles
    (450, 2304, 8064, False),           # ranges across tiles, in as many row blocks as 8192 columns in whole tiles have
    (511, 3072, 2048, False),           # beside one round of 32-row tiles
    (450, 3072, 2048, True),            # beside one and a half
    (505, 2304, (1536, 256, 256), False),
    (174, 5120, (384, 128, 128), False),        # 200 steps of deep weights, three inputs
    (155, 4096, (1536, 256, 256), True),        # 512
])
def test_several_row_blocks_only_where_they_cost_less(rows, Kk, N, blocks):
    """Launches of several row blocks that tiles are quicker for, and their neighbours, each against the oracle."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rule goes by the compute units")
    with knobs(BERTH_GEMM_BLOCK_ROWS=511, BERTH_GEMM_BLOCK_STEPS=-1):
        if isinstance(N, int):
            got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, 2, 2, True, 270 + rows, prefill=True)
            assert np.array_equal(ah, want_ah) and close(got, want)[0] == 0, launch
        else:
            from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
            gpu, lins = Gpu(0), [synth.linear(660 + i, Kk, n, 2) for i, n in enumerate(N)]
            x, outs = synth.activations(670 + rows, rows, Kk), [torch.zeros((rows, n), dtype=torch.float16, device=DEV) for n in N]
            Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *lin) for i, lin in enumerate(lins)]).forward(
                gpu, dev(x.view(np.uint16)), outs, OutDtype.F16, rows)
            torch.cuda.synchronize()
            launch = K.ops.last_launch()
            for out, lin, n in zip(outs, lins, N):
                assert close(host_f16(out), O.linear(x, *lin, Kk, n, 2, 2, out_fp32=False)[0])[0] == 0, launch
    assert ("exl3_gemm_block_kernel" in launch) == blocks, launch


@pytest.mark.parametrize("rows,unit", [(40, 128), (150, 128), (70, 0)])
def test_bundle_with_narrower_slices(rows, unit):
    """Sliced lists whose widths differ: blocks past a slice's end are empty and touch nothing.  unit 0: four slices of one
    column block each."""
    Kk, width, widths, bits = 640, 640, (640, 256, 128, 640), 4
    if not unit:
        width, widths = 128, (128, 128, 128, 128)
    lins = [synth.linear(640 + i, Kk, n, bits) for i, n in enumerate(widths)]
    d = [[dev(t.view(np.uint16)) for t in lin] for lin in lins]
    x = synth.activations(650 + rows, rows, Kk)
    outs = [torch.full((rows, n), 5.0, dtype=torch.float16, device=DEV) for n in widths]
    i64 = lambda v: torch.tensor(v, dtype=torch.int64, device=DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    lists = [i64([dd[j].data_ptr() for dd in d]) for j in range(3)]
    c_ptrs, n_list, src = i64([o.data_ptr() for o in outs]), i32(list(widths)), i32([0, 1, 2, 3])
    a_had = torch.zeros((4, rows, Kk), dtype=torch.float16, device=DEV)
    d_x = dev(x.view(np.uint16))
    K.ops.exl3_mgemm(d_x.data_ptr(), lists[0].data_ptr(), outs[0].data_ptr(), lists[1].data_ptr(), a_had.data_ptr(),
                     lists[2].data_ptr(), rows, Kk, width, bits, Codebook.MUL1, OutDtype.F16, 1, 4, n_list.data_ptr(),
                     c_ptrs.data_ptr(), n_list.data_ptr(), src.data_ptr(), 4)
    torch.cuda.synchronize()
    assert "exl3_gemm_block_kernel" in K.ops.last_launch(), K.ops.last_launch()
    for i, (tr, suh, svh) in enumerate(lins):
        want, want_had = O.linear(x, tr, suh, svh, Kk, widths[i], bits, 2, out_fp32=False)
        assert close(host_f16(outs[i]), want)[0] == 0, i
        assert np.array_equal(host_u16(a_had).reshape(4, -1)[i], want_had.view(np.uint16).reshape(-1)), i


@pytest.mark.parametrize("rows,H,I,bits,steps", [
    (33, 1024, 4096, 4, -1),            # by the rule of sizes the down projection takes 32-row tiles: no operand-ordered rows
    (100, 2048, 5632, 3, 0),            # tiles inside one workgroup and shared ones
    (145, 1152, 4224, 5, 0),            # two row blocks, the second with 65 rows; a ragged last step of K
    (48, 1280, 3072, 2, 0),             # parts of its own for every tile
    (64, 128, 17408, 4, 0),             # every tile inside one workgroup
])
def test_gate_up_finished_with_the_next_rotation(rows, H, I, bits, steps):
    """Gate, activation, rotated activation and output of an MLP call, and the rotated activation and output of the block
    call, whose launch that finishes gate and up forms them."""
    from berth_amd.device import Gpu
    from tests.test_gpu_mlp import _block_inputs, _layer, run_mlp_block
    with knobs(BERTH_GEMM_BLOCK_STEPS=steps):
        launch = run_mlp_block(rows, H, I, bits)
    assert "exl3_gemm_silu_mul_finish_kernel" in launch and "silu_mul_had_r_128_kernel" not in launch, launch
    assert ("exl3_gemm_block_kernel" in launch.split(" ; ")[1]) == (steps == 0), launch
    gpu = Gpu(0)
    lins, mlp = _layer(gpu, H, I, bits, 9900 + rows, rows)
    x, res, w = _block_inputs(gpu, H, rows, 9950 + rows)
    res_out, y = torch.zeros_like(res), torch.zeros((rows, H), dtype=torch.float32, device=DEV)
    mlp.forward_block(gpu, x, res, res_out, w, y, rows=rows)
    torch.cuda.synchronize()
    act = host_f16(mlp.u)[:rows * I].reshape(rows, I)
    assert np.array_equal(host_u16(mlp.act_had)[:rows * I], O.had_rows_f16(act, lins[2][1], True).view(np.uint16).ravel())
    # the output from that activation: the down projection as a call of its own, the residual added behind it
    d = [dev(t.view(np.uint16)) for t in lins[2]]
    c, had = torch.zeros_like(y), torch.zeros((rows, I), dtype=torch.float16, device=DEV)
    with knobs(BERTH_GEMM_BLOCK_STEPS=0):
        K.prefill_lin.exl3_linear(mlp.u.data_ptr(), d[0].data_ptr(), c.data_ptr(), d[1].data_ptr(), had.data_ptr(), d[2].data_ptr(),
                                  torch.zeros(I * H, dtype=torch.float16, device=DEV).data_ptr() if rows > 144 else None, rows, I, H,
                                  bits, Codebook.MUL1, OutDtype.F32)
    torch.cuda.synchronize()
    assert torch.equal(y, c + res_out)
