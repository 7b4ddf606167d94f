"""The few-row MFMA kernel (2..32 rows, units of 64 x 128 weights dealt out evenly) at the sizes
where its split can go wrong, against the oracle: one and two tiles of 16 rows with and without
a remainder, the smallest launch there is, ranges that start or end on a column block, ranges
that touch many column blocks (shallow weights, several rounds of workgroups), odd numbers of
k-blocks, narrower slices of a bundle.  Bar: rtol 2e-3 / atol 1e-3 of the oracle's fp32 sums;
a second call gives the same bits."""
import numpy as np
import pytest
import torch

from berth_amd import kernels as K
from berth_amd import synth
from berth_amd.kernels import Codebook, OutDtype
from oracle import oracle as O
from tests.gpu_util import DEV, close, dev, host_f16, host_u16, knobs
from tests.test_gpu_linear import _run_linear
from tests.test_gpu_mlp import run_mlp_block

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _every_size():
    """The kernel at every size it can serve, not only where it is the faster one."""
    with knobs(BERTH_GEMM_ROWS_UNITS=1):
        yield


@pytest.mark.parametrize("rows,Kk,N,bits,cb", [
    (2, 128, 256, 4, 2),            # four units: one workgroup, one unit per wave group
    (3, 1408, 640, 4, 2),           # 110 units
    (5, 5120, 1024, 3, 1),          # ranges shared by many workgroups
    (8, 1152, 4864, 5, 0),          # nine k-blocks
    (16, 4096, 2048, 2, 2),         # a full tile; every range starts and ends on a unit of its own block
    (17, 2176, 3200, 6, 2),         # second tile with one row
    (32, 2048, 4096, 8, 2),
    (31, 128, 128 * 2600, 1, 2),    # shallow: ranges of many column blocks, two rounds of workgroups
    (9, 16384, 512, 7, 1),          # deep and narrow: one column block over most of the launch
])
def test_few_rows_match_the_oracle_and_repeat(rows, Kk, N, bits, cb):
    got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, cb, True, 40 + rows, prefill=True)
    assert "exl3_gemm_rows_kernel" in launch, launch
    assert np.array_equal(ah, want_ah), launch
    bad, worst = close(got, want)
    assert bad == 0, (bad, worst, launch)
    again = _run_linear(rows, Kk, N, bits, cb, True, 40 + rows, prefill=True)[0]
    assert np.array_equal(got.view(np.uint8), again.view(np.uint8)), launch


@pytest.mark.parametrize("rows,unit", [(3, 128), (20, 128), (5, 0)])
def test_bundle_with_narrower_slices(rows, unit):
    """Sliced lists whose widths differ (the last one a single column block): blocks past a
    slice's end are empty and touch nothing.  unit 0: four slices of one
    column block each."""
    Kk, width, widths, bits = 1024, 1664, (1664, 640, 128, 1664), 4
    if not unit:
        width, widths = 128, (128, 128, 128, 128)
    lins = [synth.linear(600 + i, Kk, n, bits) for i, n in enumerate(widths)]
    d = [[dev(t.view(np.uint16)) for t in lin] for lin in lins]
    x = synth.activations(610 + rows, rows, Kk)
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
    assert "exl3_gemm_rows_kernel" in K.ops.last_launch(), K.ops.last_launch()
    for i, (tr, suh, svh) in enumerate(lins):
        want, want_had = O.linear(x, tr, suh, svh, Kk, widths[i], bits, 2, out_fp32=False)
        assert close(host_f16(outs[i]), want)[0] == 0, i
        assert np.array_equal(host_u16(a_had).reshape(4, -1)[i], want_had.view(np.uint16).reshape(-1)), i


@pytest.mark.parametrize("rows", [4, 12])
def test_mlp_of_few_rows_stage_by_stage(rows):
    launch = run_mlp_block(rows, 1536, 4096, 4)
    assert launch.count("exl3_gemm_rows_kernel") == 2 and "silu_mul_had_r_128_kernel" in launch, launch


@pytest.mark.parametrize("rows,H,I,bits", [
    (2, 2048, 16384, 2),        # one column block a workgroup, each pair shared by two
    (5, 2048, 5632, 4),         # column blocks in two parts
    (8, 1152, 8448, 3),         # ranges across pairs; up stays in its buffer
    (9, 1152, 8448, 5),         # the activation in its place
    (16, 384, 8704, 4),         # pairs shared by four workgroups
    (17, 640, 17408, 6),        # two rows a wave, the second of one wave only
    (24, 128, 40960, 4),        # whole pairs inside a workgroup
    (32, 640, 17408, 1),
    (12, 256, 5120, 4),         # the down projection reads the row-major copy
])
def test_mlp_whose_gate_and_up_leave_the_next_input(rows, H, I, bits):
    """Gate, up or activation, rotated activation and output, stage by stage; a second call gives the same bits."""
    from berth_amd.device import Gpu
    from tests.test_gpu_mlp import _layer
    with knobs(BERTH_GEMM_ROWS_UNITS=192 if I == 5120 else 1):
        launch = run_mlp_block(rows, H, I, bits)
    assert ",silu,rotate>" in launch and "silu_mul_had_r_128_kernel" not in launch, launch
    assert ("exl3_gemm_rows_kernel" in launch.split(" ; ")[1]) == (I != 5120), launch
    gpu = Gpu(0)
    _, mlp = _layer(gpu, H, I, bits, 9700 + rows, rows)
    x = gpu.upload((synth.activations(9800 + rows, rows, H) / np.sqrt(H)).astype(np.float16).view(np.uint16))
    got = []
    for _ in range(2):
        y = torch.zeros((rows, H), dtype=torch.float32, device=DEV)
        mlp.forward(gpu, x, y, rows=rows)
        got.append([y] + [getattr(mlp, n).clone() for n in ("g", "u", "act_had")])
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("rows,H,I,bits,cb", [(5, 2048, 5632, 3, 1), (24, 640, 17408, 4, 1),       # one tile of sixteen rows and two
                                              (8, 1152, 8448, 2, 0), (17, 1152, 8448, 5, 0)])
def test_gate_and_up_leave_the_next_input_with_the_other_codebooks(rows, H, I, bits, cb):
    launch = run_mlp_block(rows, H, I, bits, cb)
    assert f"exl3_gemm_rows_kernel<{bits},{cb},{16 if rows <= 16 else 32}x128,silu,rotate>" in launch, launch


@pytest.mark.parametrize("rows,H,I,bits", [(2, 128, 256, 4),        # one block a row: a quarter of a wave
                                           (9, 1152, 1280, 3),      # a workgroup with a half-empty wave
                                           (33, 8320, 8320, 2),     # two chunks a thread, one row block with one row past its first 32
                                           (3, 17408, 17408, 1)])   # three chunks
def test_block_with_fused_norm_equals_the_separate_calls(rows, H, I, bits):
    """Residual add, norm and both rotations in one launch, the residual added by the down launch:
    the residual stream, rotated inputs, gate / up results and the output bit for bit as
    berth_ops_rms_norm_res_in -> berth_exl3_mlp -> berth_ops_add_f32 give them."""
    from berth_amd.device import Gpu, ptr
    from tests.test_gpu_mlp import _block_inputs, _layer
    gpu = Gpu(0)
    _, mlp = _layer(gpu, H, I, bits, 9900 + rows, rows)
    x, res, w = _block_inputs(gpu, H, rows, 9950 + rows)
    res_ref, h = res.clone(), torch.zeros((rows, H), dtype=torch.float16, device=DEV)
    K.ops.rms_norm_res_in(ptr(x), ptr(w), ptr(h), ptr(res_ref), rows, H, 1e-6, 1.0, 1.0, True, gpu.raw_stream())
    y_ref = torch.zeros((rows, H), dtype=torch.float32, device=DEV)
    mlp.forward(gpu, h, y_ref, rows=rows)
    K.ops.add_f32(ptr(y_ref), ptr(res_ref), ptr(y_ref), rows * H, gpu.raw_stream())
    names = ("x_had", "g", "u", "act_had")
    want = {n: getattr(mlp, n).clone() for n in names}
    for n in names:
        getattr(mlp, n).zero_()
    res_out, y = torch.zeros_like(res), torch.zeros_like(y_ref)
    mlp.forward_block(gpu, x, res, res_out, w, y, rows=rows)
    torch.cuda.synchronize()
    launch = K.last_launch()
    assert "add_rms_norm_had_r_128_kernel" in launch and "+add" in launch, launch
    bits_of = lambda t: t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)
    assert torch.equal(bits_of(res_out), bits_of(res_ref)) and torch.equal(bits_of(y), bits_of(y_ref)), launch
    for n in names:
        assert torch.equal(bits_of(getattr(mlp, n)), bits_of(want[n])), (n, launch)


@pytest.mark.parametrize("rows,Kk,N,bits,cb", [
    (2, 2048, 2048, 4, 2),          # parts of 4 units: two 128 blocks
    (5, 4224, 2048, 3, 1),          # 66 units in 16 parts: 4 and 5 units, odd starts
    (16, 4096, 3968, 5, 0),         # 31 blocks
    (17, 2176, 3200, 6, 2),         # a second tile with one row
    (24, 6144, 5120, 4, 2),         # 192 items: three a lane group
    (32, 6144, 5120, 3, 2),         # 256: four
    (17, 10240, 5120, 2, 2),        # 238: some lane groups with three
    (32, 1024, 2048, 2, 2),
    (8, 17408, 1024, 8, 2),
])
@pytest.mark.parametrize("fp32", [False, True])
def test_rotation_inside_the_launch(rows, Kk, N, bits, cb, fp32):
    """Every column block is cut into parts of its own and a workgroup rotates the part of the input that it needs: the
    rotated rows as the oracle has them, and the bits of the form with a launch for the rotation (whose input
    lies in the buffer of the rotated rows, which keeps the two launches)."""
    tr, suh, svh = synth.linear(rows + Kk, Kk, N, bits)
    x = synth.activations(rows + N, rows, Kk)
    d_tr, d_suh, d_svh, d_x = (dev(a.view(np.uint16)) for a in (tr, suh, svh, x))
    res = []
    for in_place in (False, True):
        c = torch.zeros((rows, N), dtype=torch.float32 if fp32 else torch.float16, device=DEV)
        a_had = d_x.clone() if in_place else torch.zeros_like(d_x)
        K.prefill_lin.exl3_linear((a_had if in_place else d_x).data_ptr(), d_tr.data_ptr(), c.data_ptr(), d_suh.data_ptr(),
                                  a_had.data_ptr(), d_svh.data_ptr(), None, rows, Kk, N, bits, Codebook(cb),
                                  OutDtype.F32 if fp32 else OutDtype.F16)
        torch.cuda.synchronize()
        launch = K.prefill_lin.last_launch()
        assert (",rotate>" in launch) != in_place and ("had_r_128_slabs_kernel" in launch) == in_place, launch
        res.append((c, a_had))
    want, want_had = O.linear(x, tr, suh, svh, Kk, N, bits, cb, out_fp32=fp32)
    assert np.array_equal(host_u16(res[0][1]).reshape(-1), want_had.view(np.uint16).reshape(-1))
    assert torch.equal(res[0][1], res[1][1]) and torch.equal(res[0][0], res[1][0])
    assert close(res[0][0].cpu().numpy() if fp32 else host_f16(res[0][0]), want)[0] == 0


@pytest.mark.parametrize("rows,by_value,Kk", [(3, False, 2304), (8, False, 2304), (9, True, 2304), (20, True, 2304), (20, False, 2304),
                                              (9, True, 512), (16, True, 1024), (31, True, 768)])
def test_bundle_that_rotates_its_input(rows, by_value, Kk):
    """Three sources of one input, two slices of the first: every source's rotated rows are left once.  With the lists in
    device memory, which no check of the host sees, a launch of its own rotates."""
    from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
    gpu = Gpu(0)
    widths, bits = (1024, 512, 512), 3
    lins = [synth.linear(700 + i, Kk, n, bits) for i, n in enumerate(widths)]
    multi = Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *l) for i, l in enumerate(lins)])
    x = synth.activations(710 + rows, rows, Kk)
    outs = [torch.zeros((rows, n), dtype=torch.float16, device=DEV) for n in widths]
    multi.forward(gpu, dev(x.view(np.uint16)), outs, OutDtype.F16, rows, by_value=by_value)
    torch.cuda.synchronize()
    launch = K.ops.last_launch()
    assert (",rotate>" in launch) == by_value and ("had_r_128_slabs_kernel" in launch) != by_value, launch
    for i, (tr, suh, svh) in enumerate(lins):
        want, want_had = O.linear(x, tr, suh, svh, Kk, widths[i], bits, 2, out_fp32=False)
        assert close(host_f16(outs[i]), want)[0] == 0, i
        slab = host_u16(multi.a_had)[i * rows * Kk:(i + 1) * rows * Kk]
        assert np.array_equal(slab, want_had.view(np.uint16).reshape(-1)), i


def test_outputs_over_the_input_or_its_rotated_rows():
    """Two launches where the output lies over a buffer that the launch would rotate from or into: the bits of
    buffers of their own (the first launch has read the input and left its copy before anything is stored)."""
    rows, Kk, N, bits = 6, 2304, 1024, 4
    lins = [[dev(t.view(np.uint16)) for t in synth.linear(720 + i, Kk, N, bits)] for i in range(2)]
    d_x = dev(synth.activations(725, rows, Kk).view(np.uint16))
    tr, suh, svh = lins[0]
    a_had = torch.zeros_like(d_x)
    c = torch.zeros((rows, N), dtype=torch.float16, device=DEV)
    res = []
    for out in (c, a_had):
        K.prefill_lin.exl3_linear(d_x.data_ptr(), tr.data_ptr(), out.data_ptr(), suh.data_ptr(), a_had.data_ptr(),
                                  svh.data_ptr(), None, rows, Kk, N, bits, Codebook.MUL1, OutDtype.F16)
        torch.cuda.synchronize()
        assert (",rotate>" in K.prefill_lin.last_launch()) == (out is c), K.prefill_lin.last_launch()
        res.append(host_u16(out).reshape(-1)[:rows * N].copy())
    assert np.array_equal(*res)

    # a uniform bundle: its outputs follow from one pointer also where the lists are in device memory
    lists = [torch.tensor([lin[j].data_ptr() for lin in lins], dtype=torch.int64, device=DEV) for j in range(3)]
    slabs = torch.zeros((2, rows, Kk), dtype=torch.float16, device=DEV)
    res = []
    for over in (False, True):
        x = d_x.clone()
        out = x if over else torch.zeros((2, rows, N), dtype=torch.float16, device=DEV)
        K.ops.exl3_mgemm(x.data_ptr(), lists[0].data_ptr(), out.data_ptr(), lists[1].data_ptr(), slabs.data_ptr(),
                         lists[2].data_ptr(), rows, Kk, N, bits, Codebook.MUL1, OutDtype.F16, 1, 2)
        torch.cuda.synchronize()
        assert (",rotate>" in K.ops.last_launch()) == (not over), K.ops.last_launch()
        res.append(host_u16(out).reshape(-1)[:2 * rows * N].copy())
    assert np.array_equal(*res)


def _bundle_lists(sources, slices, outs):
    """The seven lists of a sliced bundle in device memory: slices of (source, first column, width)."""
    t64, t32 = (lambda v: torch.tensor(v, dtype=torch.int64, device=DEV)), (lambda v: torch.tensor(v, dtype=torch.int32, device=DEV))
    bits, sizes = sources[0]["bits"], [s["n"] for s in sources]
    b = t64([sources[s]["d"][0].data_ptr() + n0 // 16 * 16 * bits * 2 for s, n0, _ in slices])
    svh = t64([sources[s]["d"][2].data_ptr() + 2 * n0 for s, n0, _ in slices])
    suh = t64([s["d"][1].data_ptr() for s in sources])
    c = t64([outs[s].data_ptr() + 2 * n0 for s, n0, _ in slices])
    return b, suh, svh, t32([w for _, _, w in slices]), c, t32([sizes[s] for s, _, _ in slices]), t32([s for s, _, _ in slices])


def _sources(seed, Kk, widths, bits):
    return [{"bits": bits, "n": n, "np": lin, "d": [dev(t.view(np.uint16)) for t in lin]}
            for n, lin in ((n, synth.linear(seed + i, Kk, n, bits)) for i, n in enumerate(widths))]


def _device_bundle(x, a_had, lists, rows, Kk, width, bits, outs, sources):
    b, suh, svh, n, c, stride, src = lists
    K.ops.exl3_mgemm(x.data_ptr(), b.data_ptr(), outs[0].data_ptr(), suh.data_ptr(), a_had.data_ptr(), svh.data_ptr(), rows, Kk,
                     width, bits, Codebook.MUL1, OutDtype.F16, 1, len(src), n.data_ptr(), c.data_ptr(), stride.data_ptr(),
                     src.data_ptr(), sources)
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows", [3, 8, 9, 20, 32])
@pytest.mark.parametrize("over", ["input", "rotated rows"])
def test_outputs_of_device_lists_over_the_input(rows, over):
    """Slices whose lists are in device memory may store over the input or over the rotated rows: both have been read when the
    first output is stored, so the bits are those of buffers of their own."""
    Kk, widths, bits = 2304, (1024, 512, 512), 4
    sources = _sources(730, Kk, widths, bits)
    slices = [(0, 0, 512), (0, 512, 512), (1, 0, 512), (2, 0, 512)]
    d_x = dev(synth.activations(735 + rows, rows, Kk).view(np.uint16))
    res = []
    for own in (True, False):
        x, a_had = d_x.clone(), torch.zeros((3, rows, Kk), dtype=torch.float16, device=DEV)
        outs = [torch.zeros((rows, n), dtype=torch.float16, device=DEV) for n in widths]
        if not own:         # outputs one behind the other in the input (their columns fit) or in the rotated rows
            at, flat = 0, (x if over == "input" else a_had).view(torch.float16).reshape(-1)
            for i, n in enumerate(widths):
                outs[i] = flat[at:at + rows * n].view(rows, n)
                at += rows * n
        _device_bundle(x, a_had, _bundle_lists(sources, slices, outs), rows, Kk, 512, bits, outs, 3)
        assert ",rotate>" not in K.ops.last_launch(), K.ops.last_launch()
        res.append([host_u16(o).copy() for o in outs])
    for i in range(3):
        assert np.array_equal(res[0][i], res[1][i]), i


@pytest.mark.parametrize("rows", [4, 17])
def test_rotated_rows_of_a_source_without_slices(rows):
    """A source that no slice of a bundle in device memory uses: its rotated rows are left all the same."""
    Kk, widths, bits = 2304, (1024, 512, 1024), 3
    sources = _sources(740, Kk, widths, bits)
    x = synth.activations(745 + rows, rows, Kk)
    a_had = torch.zeros((3, rows, Kk), dtype=torch.float16, device=DEV)
    outs = [torch.zeros((rows, n), dtype=torch.float16, device=DEV) for n in widths]
    lists = _bundle_lists(sources, [(0, 0, 512), (0, 512, 512), (2, 0, 512), (2, 512, 512)], outs)
    _device_bundle(dev(x.view(np.uint16)), a_had, lists, rows, Kk, 512, bits, outs, 3)
    for i, s in enumerate(sources):
        want, want_had = O.linear(x, *s["np"], Kk, widths[i], bits, 2, out_fp32=False)
        assert np.array_equal(host_u16(a_had)[i].reshape(-1), want_had.view(np.uint16).reshape(-1)), i
        assert i == 1 or close(host_f16(outs[i]), want)[0] == 0, i


def _bundle(rows, Kk, widths, bits):
    """Sources of different widths, lists in device memory."""
    from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
    gpu = Gpu(0)
    lins = [synth.linear(640 + i, Kk, n, bits) for i, n in enumerate(widths)]
    bundle = Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *lin) for i, lin in enumerate(lins)])
    x = synth.activations(650 + rows, rows, Kk)
    outs = [torch.full((rows, n), 5.0, dtype=torch.float16, device=DEV) for n in widths]
    bundle.forward(gpu, gpu.upload(x.view(np.uint16)), outs, OutDtype.F16, rows, by_value=False)
    torch.cuda.synchronize()
    for out, lin, n in zip(outs, lins, widths):
        assert close(host_f16(out), O.linear(x, *lin, Kk, n, bits, 2, out_fp32=False)[0])[0] == 0, K.ops.last_launch()


@pytest.mark.parametrize("rows,Kk,widths,bits,fp32,rotates", [
    (2, 1024, (1024, 512, 512), 4, False, True),
    (4, 512, (512, 256), 3, True, True),            # four k-blocks, the fewest rows
    (3, 512, (512, 256), 3, False, False),          # the dot-product kernel, from the device lists
    (8, 2304, (1024, 512, 512), 2, True, True),
    (5, 384, (512, 256), 4, False, False),          # three k-blocks
    (8, 1152, (128 * 17, 128), 4, False, False),    # eighteen slices stay in device memory
    (7, 640, (256, 256, 128), 6, False, True),      # five k-blocks
])
def test_few_rows_of_a_bundle_by_value(rows, Kk, widths, bits, fp32, rotates):
    """Lists on both sides: every source and its rotated rows, which the launch that rotates leaves once; twice the same bits."""
    from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
    gpu = Gpu(0)
    lins = [synth.linear(760 + i, Kk, n, bits) for i, n in enumerate(widths)]
    multi = Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *l) for i, l in enumerate(lins)])
    x = synth.activations(770 + rows, rows, Kk)
    res = []
    for _ in range(2):
        outs = [torch.zeros((rows, n), dtype=torch.float32 if fp32 else torch.float16, device=DEV) for n in widths]
        with knobs(BERTH_GEMM_ROWS_UNITS=-1):
            multi.forward(gpu, dev(x.view(np.uint16)), outs, OutDtype.F32 if fp32 else OutDtype.F16, rows)
            launch = K.ops.last_launch()
        torch.cuda.synchronize()
        assert (",rotate>" in launch) == rotates == ("by value" in launch), launch
        res.append([o.cpu().numpy() for o in outs])
    for i, lin in enumerate(lins):
        want, want_had = O.linear(x, *lin, Kk, widths[i], bits, 2, out_fp32=fp32)
        assert close(res[0][i], want)[0] == 0 and np.array_equal(res[0][i], res[1][i]), i
        slab = host_u16(multi.a_had)[i * rows * Kk:(i + 1) * rows * Kk]
        assert np.array_equal(slab, want_had.view(np.uint16).reshape(-1)), i


@pytest.mark.parametrize("rows,bits,cb", [(2, 4, 0), (5, 3, 1), (8, 6, 1)])
def test_few_rows_of_a_bundle_by_value_with_the_other_codebooks(rows, bits, cb):
    from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
    gpu, Kk, widths = Gpu(0), 2304, (1024, 512, 512)
    lins = [synth.linear(790 + i, Kk, n, bits) for i, n in enumerate(widths)]
    multi = Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *lin, Codebook(cb)) for i, lin in enumerate(lins)])
    x, outs = synth.activations(795 + rows, rows, Kk), [torch.zeros((rows, n), dtype=torch.float16, device=DEV) for n in widths]
    with knobs(BERTH_GEMM_ROWS_UNITS=-1):
        multi.forward(gpu, dev(x.view(np.uint16)), outs, OutDtype.F16, rows)
    torch.cuda.synchronize()
    launch = K.ops.last_launch()
    assert "by value" in launch and f"exl3_gemm_rows_kernel<{bits},{cb},16x128,rotate>" in launch, launch
    for out, lin, n in zip(outs, lins, widths):
        assert close(host_f16(out), O.linear(x, *lin, Kk, n, bits, cb, out_fp32=False)[0])[0] == 0, launch


def test_few_rows_by_value_with_outputs_over_the_input():
    """The host sees that an output lies over the input: a launch of its own rotates, and the bits are those of other buffers."""
    from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu
    gpu, rows, Kk, widths = Gpu(0), 6, 2304, (1024, 512)
    multi = Exl3MultiLinear(gpu, [Exl3Linear(gpu, f"l{i}", *synth.linear(780 + i, Kk, n, 4)) for i, n in enumerate(widths)])
    d_x = dev(synth.activations(785, rows, Kk).view(np.uint16))
    res = []
    for over in (False, True):
        a, flat = d_x.clone(), torch.zeros(rows * Kk, dtype=torch.float16, device=DEV)
        flat = a.view(torch.float16).reshape(-1) if over else flat
        outs, at = [], 0
        for n in widths:
            outs.append(flat[at:at + rows * n].view(rows, n))
            at += rows * n
        multi.forward(gpu, a, outs, OutDtype.F16, rows)
        torch.cuda.synchronize()
        assert (",rotate>" in K.ops.last_launch()) == (not over), K.ops.last_launch()
        res.append([host_u16(o).copy() for o in outs])
    assert all(np.array_equal(u, v) for u, v in zip(*res))


@pytest.mark.parametrize("kind,rows,Kk,N,bits,cb,matrix", [
    ("linear", 2, 768, 768, 4, 2, True),        # six k-blocks
    ("linear", 2, 512, 1024, 4, 2, False),
    ("linear", 4, 512, 512, 3, 1, True),        # 32 units, four k-blocks
    ("linear", 8, 512, 384, 4, 2, False),       # 24
    ("linear", 8, 384, 4096, 2, 0, False),      # three k-blocks
    ("linear", 3, 3072, 256, 5, 0, True),
    ("bundle", 4, 1024, 512, 4, 2, False), ("bundle", 5, 1024, 512, 4, 2, True), ("bundle", 8, 896, 512, 4, 2, False),
    ("mlp", 4, 1152, 1280, 4, 2, False), ("mlp", 5, 1152, 1280, 4, 2, True), ("mlp", 8, 1024, 1152, 3, 2, False),
])
def test_small_weights_beside_the_dot_product_kernel(kind, rows, Kk, N, bits, cb, matrix):
    """Which kernel two to eight rows of small weights take, on both sides of every line, and its results."""
    with knobs(BERTH_GEMM_ROWS_UNITS=-1):
        if kind == "linear":
            got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, cb, True, 70 + rows, prefill=True)
            assert np.array_equal(ah, want_ah) and close(got, want)[0] == 0, launch
        elif kind == "bundle":
            _bundle(rows, Kk, (N, N // 4), bits)
            launch = K.ops.last_launch()
        else:
            launch = run_mlp_block(rows, Kk, N, bits)
    assert ("exl3_gemm_rows_kernel" in launch) == matrix and ("exl3_gemv_kernel" in launch) != matrix, launch


@pytest.mark.parametrize("rows,Kk,N,kernel", [
    (2, 1024, 1024, "exl3_gemm_rows_kernel"),       # up to the knob's rows: whichever is the quicker
    (3, 3072, 2048, "exl3_gemm_kernel"),            # above: 768 units of three rows want 3072
    (8, 1024, 1024, "exl3_gemm_kernel"),            # 128 of eight 1024
    (8, 2048, 4096, "exl3_gemm_rows_kernel"),
])
def test_rows_above_the_knob_of_the_dot_product_kernel(rows, Kk, N, kernel):
    """BERTH_GEMV_MAX_ROWS: above it small weights take the MFMA tiles of 32 rows, large ones the few-row kernel."""
    with knobs(BERTH_GEMM_ROWS_UNITS=-1, BERTH_GEMV_MAX_ROWS=2):
        got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, 3, 2, True, 75 + rows, prefill=True)
    assert kernel + "<" in launch and np.array_equal(ah, want_ah) and close(got, want)[0] == 0, launch


@pytest.mark.parametrize("rows,H,I,bits", [(2, 512, 512, 4), (8, 640, 768, 3), (4, 384, 512, 4)])
def test_small_block_with_fused_norm(rows, H, I, bits):
    """From 512 of `hidden` on a block's MLP takes the kernel at any of these row counts: gate and up, the rotated
    activation and the output, each from the device's own results of the stage before."""
    from berth_amd.device import Gpu, ptr
    from tests.test_gpu_mlp import _block_inputs, _layer
    gpu = Gpu(0)
    (gate, up, down), mlp = _layer(gpu, H, I, bits, 9300 + rows, rows)
    x, res, w = _block_inputs(gpu, H, rows, 9350 + rows)
    res_ref, h = res.clone(), torch.zeros((rows, H), dtype=torch.float16, device=DEV)
    res_out, y = torch.zeros_like(res), torch.zeros_like(res)
    K.ops.rms_norm_res_in(ptr(x), ptr(w), ptr(h), ptr(res_ref), rows, H, 1e-6, 1.0, 1.0, True, gpu.raw_stream())
    with knobs(BERTH_GEMM_ROWS_UNITS=-1):
        mlp.forward_block(gpu, x, res, res_out, w, y, rows=rows)
        launch = K.last_launch()
    torch.cuda.synchronize()
    assert ("add_rms_norm_had_r_128_kernel" in launch and "+add" in launch) == (H >= 512), launch
    assert torch.equal(res_out, res_ref)
    normed = host_f16(h)
    g, u = (host_f16(t)[:rows * I].reshape(rows, I) for t in (mlp.g, mlp.u))
    for got, lin in ((g, gate), (u, up)):
        assert close(got, O.linear(normed, *lin, H, I, bits, 2)[0].reshape(rows, I))[0] == 0, launch
    act = O.silu_mul(g, u).reshape(rows, I)
    want, act_had = O.linear(act, *down, I, H, bits, 2, out_fp32=True)
    assert np.array_equal(host_u16(mlp.act_had)[:rows * I], act_had.view(np.uint16).ravel())
    # rows of a norm reach 5e4 here, and where they cancel what is left is the rounding of the sums: a wave adds eight
    # products at a time, I / 8 roundings of half an ulp of partial sums as large as the row's largest output
    want = want.reshape(rows, H)
    atol = np.maximum(1e-3, I / 8 * 2.0 ** -24 * np.abs(want).max(axis=1, keepdims=True))
    assert close(y.cpu().numpy(), want + res_ref.cpu().numpy(), atol=atol)[0] == 0, launch


@pytest.mark.parametrize("rows,H,I,bits,same", [
    (2, 512, 512, 4, False), (8, 640, 768, 3, False),   # the block takes the few-row kernel, the call the dot-product kernel
    (4, 384, 512, 4, True),                             # both the dot-product kernel
    (5, 1280, 3072, 2, True), (9, 1152, 1280, 3, True), # both the few-row kernel
])
def test_block_beside_the_separate_calls_at_default_knobs(rows, H, I, bits, same):
    """berth_exl3_mlp_block against norm -> berth_exl3_mlp -> add: the same bits where both take the same kernels.  Elsewhere
    gate, up and the output are fp32 sums of the same products in another order: four fp16 roundings (gate, up, activation,
    rotated activation) of half a unit, 2^-11, may fall either way, and rotations and random weights keep a row's
    relative 2-norm."""
    from berth_amd.device import Gpu, ptr
    from tests.test_gpu_mlp import _block_inputs, _layer
    gpu = Gpu(0)
    _, mlp = _layer(gpu, H, I, bits, 9400 + rows, rows)
    x, res, w = _block_inputs(gpu, H, rows, 9450 + rows)
    stream, h, add = res.clone(), torch.zeros((rows, H), dtype=torch.float16, device=DEV), torch.zeros_like(res)
    res_out, y = torch.zeros_like(res), torch.zeros_like(res)
    with knobs(BERTH_GEMM_ROWS_UNITS=-1):
        K.ops.rms_norm_res_in(ptr(x), ptr(w), ptr(h), ptr(stream), rows, H, 1e-6, 1.0, 1.0, True, gpu.raw_stream())
        mlp.forward(gpu, h, add, rows=rows)
        separate = K.last_launch()
        sums, x_had = add.clone(), mlp.x_had.clone()
        K.ops.add_f32(ptr(add), ptr(stream), ptr(add), rows * H, gpu.raw_stream())
        mlp.forward_block(gpu, x, res, res_out, w, y, rows=rows)
        launch = K.last_launch()
    torch.cuda.synchronize()
    assert torch.equal(res_out, stream) and torch.equal(x_had, mlp.x_had), launch
    assert (("exl3_gemv_kernel" in separate) == ("exl3_gemv_kernel" in launch)) == same, (separate, launch)
    if same:
        assert torch.equal(y, add), launch
    else:
        off = (y.double() - add.double()).norm(dim=1) / sums.double().norm(dim=1)
        assert float(off.max()) <= 4 * 2 * 2.0 ** -11, (off, launch)


@pytest.mark.parametrize("rows,H,I,matrix,dots", [
    (4, 1024, 3072, 0, 2),      # 768 units of gate and up: two launches of the dot-product kernel
    (4, 1024, 4096, 1, 1),      # 1024, from which gate and up take the few-row kernel whatever hidden is
    (4, 512, 8192, 1, 1),
    (3, 1024, 4096, 0, 2),      # 3072 at two and three rows
    (8, 1024, 2048, 0, 2), (4, 1152, 2048, 0, 2),
    (5, 1152, 2048, 2, 0),      # above 1024 of hidden five rows and more
])
def test_launches_of_small_mlps(rows, H, I, matrix, dots):
    with knobs(BERTH_GEMM_ROWS_UNITS=-1):
        launch = run_mlp_block(rows, H, I, 2)
    assert (launch.count("exl3_gemm_rows_kernel"), launch.count("exl3_gemv_kernel")) == (matrix, dots), launch


@pytest.mark.parametrize("rows,Kk,N,bits,own", [
    (2, 2944, 256, 5, True),            # parts of four and five units beside an even share of four
    (9, 1152, 512, 4, True),            # 18 units in four parts
    (16, 4096, 3072, 3, True),          # ten parts of six and seven, in a grid of fewer than the compute units
    (23, 2816, 11264, 2, True),         # two of 22 beside a share of 16
    (16, 3072, 11264, 2, False),        # two of 24 beside 17
])
def test_parts_longer_than_the_even_share(rows, Kk, N, bits, own):
    """Column blocks cut into parts of their own, whose launch rotates its input, up to six units above the even share."""
    got, want, ah, want_ah, launch = _run_linear(rows, Kk, N, bits, 2, True, 90 + rows, prefill=True)
    assert "exl3_gemm_rows_kernel" in launch and ("had_r_128" not in launch) == own, launch
    assert np.array_equal(ah, want_ah) and close(got, want)[0] == 0, launch
