"""MoE launches by token count.  Routing and permutation of many tokens: every token count per
workgroup that the one-launch routing chooses between, and the permutation on either side of where
it takes more workgroups and where the waves' runs end, bit-exact against the oracle.  Layers of up
to 16 tokens: the grouped few-row kernel, stage by stage."""
import numpy as np
import pytest
import torch

from berth_amd import kernels as K
from berth_amd import synth
from berth_amd.device import Gpu
from berth_amd.moe import MoeLayer
from oracle import oracle as O
from tests.gpu_util import DEV, dev, knobs
import tests.test_gpu_moe as stages
from tests.test_gpu_moe import _check_stages, _make_layer, _route

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,k,per_workgroup", [(256, 256, 128, 4, 1), (257, 256, 66, 4, 2), (700, 128, 128, 8, 3), (1, 2048, 512, 10, 1), (1, 64, 130, 3, 1),
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


@pytest.mark.parametrize("T,H,E,k,I,bits,shared_I", [
    (16, 256, 2, 1, 256, 4, 256),       # sixteen rows in one problem, four units a column block, the shared expert among them
    (9, 1024, 20, 8, 128, 3, 0),        # down projection of one k-block: the 32-row kernel on 16-row problems
    (16, 2048, 128, 8, 768, 4, 0),
    (5, 512, 300, 7, 384, 6, 0),        # three column blocks, ranges of one and a bit of them
    (3, 256, 4, 3, 256, 2, 128),        # fewer units than four for every compute unit
    (12, 640, 40, 8, 512, 5, 512),
])
def test_few_token_layers_on_the_grouped_few_row_kernel(T, H, E, k, I, bits, shared_I):
    gpu = Gpu(0)
    wr, experts_np, experts, shared_np, shared = _make_layer(gpu, 9100 + T + H, H, E, I, bits, shared_I, 10.0)
    layer = MoeLayer(gpu, wr, experts, k, shared=shared)
    x = (synth.activations(T + H, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    out, again = (torch.zeros((T, H), dtype=torch.float32, device=DEV) for _ in range(2))
    idx = torch.zeros((T, k), dtype=torch.int32, device=DEV)
    w = torch.zeros((T, k), dtype=torch.float32, device=DEV)
    d_x = dev(x.view(np.uint16))
    layer.forward(gpu, d_x, out, T, idx, w)
    torch.cuda.synchronize()
    assert "exl3_gemm_rows_kernel" in K.moe.last_launch(), K.moe.last_launch()
    want, oi, _ = O.moe_layer(x, wr, experts_np, k, I, bits, 2, shared=shared_np, shared_I=shared_I)
    assert np.array_equal(idx.cpu().numpy(), oi)
    _check_stages(layer, x, experts_np, shared_np, oi, w.cpu().numpy(), out.cpu().numpy(), T, H, E, k, I, bits, shared_I)
    for _ in range(3):
        layer.forward(gpu, d_x, again, T)
        torch.cuda.synchronize()
        assert torch.equal(again, out)


def test_one_token_of_many_experts():
    """More experts than the one-token kernels take: the one-launch routing sorts the choices too."""
    gpu = Gpu(0)
    T, H, E, k, I, bits, shared_I = 1, 256, 300, 7, 128, 4, 128
    wr, experts_np, experts, shared_np, shared = _make_layer(gpu, 9300, H, E, I, bits, shared_I, 10.0)
    layer = MoeLayer(gpu, wr, experts, k, shared=shared)
    x = (synth.activations(9301, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    out = torch.zeros((T, H), dtype=torch.float32, device=DEV)
    idx = torch.zeros((T, k), dtype=torch.int32, device=DEV)
    w = torch.zeros((T, k), dtype=torch.float32, device=DEV)
    layer.forward(gpu, dev(x.view(np.uint16)), out, T, idx, w)
    torch.cuda.synchronize()
    assert "moe_route_slab_kernel<1>" in K.moe.last_launch() and "sort" in K.moe.last_launch(), K.moe.last_launch()
    want, oi, _ = O.moe_layer(x, wr, experts_np, k, I, bits, 2, shared=shared_np, shared_I=shared_I)
    assert np.array_equal(idx.cpu().numpy(), oi)
    _check_stages(layer, x, experts_np, shared_np, oi, w.cpu().numpy(), out.cpu().numpy(), T, H, E, k, I, bits, shared_I)


@pytest.mark.parametrize("T,bits", [(150, 4), (150, 3), (240, 4), (240, 6), (330, 4), (330, 2)])
def test_problems_of_two_three_and_four_row_blocks(T, bits):
    """About 50, 80 and 110 rows an expert: the 128-row problems run as many 32-row blocks as they
    have rows for, with the bits of 32-row problems."""
    gpu = Gpu(0)
    H, E, k, I = 256, 6, 2, 384
    wr, _, experts, _, _ = _make_layer(gpu, 9400 + T + bits, H, E, I, bits, 0, 1.0)
    x = (synth.activations(9401 + T, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    d_x, res = dev(x.view(np.uint16)), []
    for big_min in (0, 33):
        with knobs(BERTH_MOE_BIG_MIN=big_min):
            layer = MoeLayer(gpu, wr, experts, k)
            out = torch.zeros((T, H), dtype=torch.float32, device=DEV)
            layer.forward(gpu, d_x, out, T)
            torch.cuda.synchronize()
            assert ("exl3_gemm_mixed_kernel" in K.moe.last_launch()) == (big_min > 0), K.moe.last_launch()
            res.append(out)
    assert torch.equal(res[0], res[1])


def _tiles_in_halves(rows, tiles):
    """Which problems of a mixed launch run as halves, from the rows of each expert (the kernel's rule for 256 compute units)."""
    big = small = 0
    for m in rows:
        left = m % 128
        big += m // 128 + (left >= 33)
        small += 0 < left < 33
    return "both" if 2 * (big + small) * tiles <= 512 else "first" if (2 * big + small) * tiles <= 512 else "none"


@pytest.mark.parametrize("T,H,E,k,I,bits,codebook,shared_I,gate_up,down", [
    (150, 384, 6, 2, 384, 4, 2, 0, "both", "both"),         # a column block and a half
    (330, 256, 6, 2, 384, 5, 0, 384, "both", "both"),       # problems of four row blocks and the shared expert's
    (240, 256, 6, 2, 128, 3, 1, 0, "both", "both"),
    (700, 128, 66, 4, 384, 4, 2, 0, "first", "both"),       # few problems in the second list
    (700, 128, 66, 4, 256, 2, 1, 128, "both", "both"),
    (600, 384, 200, 4, 256, 3, 2, 256, "first", "first"),   # nearly all experts of up to sixteen rows, whole
    (600, 128, 200, 4, 384, 4, 0, 384, "none", "both"),     # as halves in the down projection
    (360, 384, 60, 4, 384, 3, 0, 0, "both", "both"),        # nearly all of 17..32 rows, on either side of both rules
    (560, 256, 100, 4, 384, 3, 1, 384, "first", "both"),
    (900, 384, 150, 4, 384, 3, 2, 0, "none", "first"),
])
def test_launches_of_few_128_row_tiles_run_them_as_halves(T, H, E, k, I, bits, codebook, shared_I, gate_up, down):
    """Halves of both lists, of the first alone and of none, against the bits of a launch of 32-row problems only (whole
    tiles; K of up to 384 is not cut there either)."""
    gpu = Gpu(0)
    wr, _, experts, _, shared = _make_layer(gpu, 9600 + T + bits, H, E, I, bits, shared_I, 1.0)
    x = (synth.activations(9601 + T, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    d_x, res = dev(x.view(np.uint16)), []
    idx = torch.zeros((T, k), dtype=torch.int32, device=DEV)
    w = torch.zeros((T, k), dtype=torch.float32, device=DEV)
    for big_min in (0, 33):
        with knobs(BERTH_MOE_BIG_MIN=big_min):
            layer = MoeLayer(gpu, wr, experts, k, shared=shared, codebook=codebook)
            out = torch.zeros((T, H), dtype=torch.float32, device=DEV)
            layer.forward(gpu, d_x, out, T, idx, w)
            torch.cuda.synchronize()
            assert ("exl3_gemm_mixed_kernel" in K.moe.last_launch()) == (big_min > 0), K.moe.last_launch()
            assert torch.isfinite(out).all() and (out != 0).any()
            res.append(out)
    assert torch.equal(res[0], res[1])
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        return
    rows = [int(r) for r in torch.bincount(idx.flatten().long(), minlength=E).cpu()] + ([T] if shared_I == I else [])
    assert _tiles_in_halves(rows, 2 * -(-I // 256)) == gate_up
    assert _tiles_in_halves(rows, -(-H // 256)) == down


@pytest.mark.parametrize("T,H,E,k", [(3, 128, 128, 8), (2, 128, 300, 10), (5, 128, 512, 32), (2, 64, 1000, 9), (1, 64, 65, 3)])
@pytest.mark.parametrize("finite", [0, 2, None])
def test_choice_among_equal_and_minus_infinite_logits(T, H, E, k, finite):
    """Columns repeat, so that the same logit stands in many lanes and several times in one lane; with a bias
    of minus infinity fewer than k experts (or none at all) are left and the lowest of the others follow."""
    x = synth.activations(T + E, T, H)
    wr = synth.router_weight(E, H, E)[:, np.arange(E) * 7 % 11]
    bias = None
    if finite is not None:
        bias = np.full(E, -np.inf, np.float32)
        bias[E // 3:E // 3 + finite] = 0.25
    idx, w, logits = _route(x, wr, k, bias=bias)
    # the rule on the device's own logits: largest first, ties to the lowest index (a stable sort)
    want = np.argsort(-logits, axis=1, kind="stable")[:, :k]
    assert np.array_equal(idx, want)
    if finite != 0:
        oi, ow = O.moe_route(x, wr, k, bias=bias)
        assert np.array_equal(idx, oi) and np.allclose(w, ow, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("T,H,E,k,experts", [(2, 2048, 130, 3, 16), (17, 2048, 512, 10, 16), (33, 4032, 194, 6, 16), (31, 6144, 1000, 8, 16),
                                             (270, 2048, 512, 10, 32), (513, 2048, 142, 4, 32)])
def test_routing_tiles_of_sixteen_tokens(T, H, E, k, experts):
    """Ragged token groups and slabs, a last pass with one segment missing, three passes: the oracle's bits."""
    x, wr = synth.activations(T, T, H), synth.router_weight(E, H, E)
    bias = synth.zipf_bias(5, E) if E % 4 == 0 else None
    with knobs(BERTH_MOE_ROUTE_SLAB=2):         # also where the other form is the quicker one
        idx, w, logits = _route(x, wr, k, bias=bias)
    assert "moe_route_slab_kernel<16," in K.moe.last_launch(), K.moe.last_launch()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert f"moe_route_slab_kernel<16,{experts}>" in K.moe.last_launch(), K.moe.last_launch()
    oi, ow, ol = O.moe_route(x, wr, k, bias=bias, want_logits=True)
    assert np.array_equal(logits.view(np.uint32), ol.view(np.uint32))
    assert np.array_equal(idx, oi)
    assert np.allclose(w, ow, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("T,H,E,k,tiles", [
    (17, 2048, 2, 2, False), (256, 2048, 128, 8, False), (257, 2048, 128, 8, True), (512, 2048, 100, 4, True), (600, 1920, 34, 6, True),
    (1000, 2048, 128, 8, True), (1025, 2048, 128, 8, False), (1500, 2048, 64, 6, True), (1090, 4096, 16, 4, True), (1037, 2048, 62, 9, True),
    (700, 1024, 64, 4, False)])
def test_routing_tiles_of_up_to_128_experts(T, H, E, k, tiles):
    """One slab, several, ragged ones, on either side of the rule's lines: the oracle's bits, from tiles and from slabs of 128."""
    x, wr = synth.activations(T, T, H), synth.router_weight(E, H, E)
    bias = synth.zipf_bias(6, E) if E % 4 == 0 else None
    idx, w, logits = _route(x, wr, k, bias=bias)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert ("moe_route_slab_kernel<16," in K.moe.last_launch()) == tiles, K.moe.last_launch()
    with knobs(BERTH_MOE_ROUTE_SLAB=2):
        again = _route(x, wr, k, bias=bias)
    assert "moe_route_slab_kernel<16," in K.moe.last_launch(), K.moe.last_launch()
    assert all(np.array_equal(a, b) for a, b in zip((idx, w, logits), again))
    oi, ow, ol = O.moe_route(x, wr, k, bias=bias, want_logits=True)
    assert np.array_equal(logits.view(np.uint32), ol.view(np.uint32))
    assert np.array_equal(idx, oi)
    assert np.allclose(w, ow, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("T,H,E,tokens", [
    (8, 2048, 512, 16), (9, 2048, 512, 1), (64, 2048, 512, 1), (128, 2048, 512, 2), (256, 2048, 512, 16), (384, 2048, 512, 6),
    (512, 2048, 512, 16), (128, 2048, 256, 1), (129, 2048, 256, 16), (500, 1856, 160, 16), (500, 1792, 160, 4), (500, 2112, 160, 4)])
def test_routing_form_by_whole_rounds(T, H, E, tokens):
    """On either side of the rule's lines: tokens of a workgroup, and the same logits and choices from the other forms."""
    x, wr = synth.activations(T, T, H), synth.router_weight(E, H, E)
    res = []
    for form in (1, 2, 0):
        with knobs(BERTH_MOE_ROUTE_SLAB=form):
            res.append(_route(x, wr, 8))
        if form == 1 and torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert f"moe_route_slab_kernel<{tokens}" in K.moe.last_launch(), K.moe.last_launch()
        if form == 2:
            assert "moe_route_slab_kernel<16," in K.moe.last_launch(), K.moe.last_launch()
    for other in res[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(res[0], other))


@pytest.mark.parametrize("T,H,E,k,I,bits", [
    (12, 256, 5, 3, 384, 4),         # problems of sixteen rows
    (40, 384, 3, 2, 128, 5),         # of 32 rows, a last one of fewer
    (200, 256, 6, 2, 128, 3),        # of two to four row blocks, and the rest of 32
])
def test_rows_found_through_the_permutation(T, H, E, k, I, bits):
    """The layer leaves the rotated rows in the order of the pairs, the stages on their own in sorted order."""
    stages.test_stage_entry_points_compose_to_the_layer(T, H, E, k, I, bits)


@pytest.mark.parametrize("T,H,E,k,I,bits,shared_I", [
    (17, 128, 40, 3, 128, 4, 0),        # one k-block, one column block
    (70, 256, 2, 2, 384, 3, 384),       # experts with 32, 32 and 6 rows, the always-on one among them
    (128, 384, 9, 1, 640, 6, 128),      # an always-on expert of another width
    (33, 256, 64, 8, 256, 2, 0),
])
def test_gate_up_and_the_next_rotation_in_one_launch(T, H, E, k, I, bits, shared_I):
    """17..128 tokens: every workgroup holds gate and up of its columns and leaves the down projection's rotated input."""
    gpu = Gpu(0)
    wr, experts_np, experts, shared_np, shared = _make_layer(gpu, 9500 + T + H, H, E, I, bits, shared_I, 10.0)
    layer = MoeLayer(gpu, wr, experts, k, shared=shared)
    x = (synth.activations(T + H, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    out, again = (torch.zeros((T, H), dtype=torch.float32, device=DEV) for _ in range(2))
    idx = torch.zeros((T, k), dtype=torch.int32, device=DEV)
    w = torch.zeros((T, k), dtype=torch.float32, device=DEV)
    layer.forward(gpu, dev(x.view(np.uint16)), out, T, idx, w)
    torch.cuda.synchronize()
    assert "exl3_gemm_pair_kernel" in K.moe.last_launch() and "had_rows" not in K.moe.last_launch(), K.moe.last_launch()
    want, oi, _ = O.moe_layer(x, wr, experts_np, k, I, bits, 2, shared=shared_np, shared_I=shared_I)
    assert np.array_equal(idx.cpu().numpy(), oi)
    _check_stages(layer, x, experts_np, shared_np, oi, w.cpu().numpy(), out.cpu().numpy(), T, H, E, k, I, bits, shared_I)
    layer.forward(gpu, dev(x.view(np.uint16)), again, T)
    torch.cuda.synchronize()
    assert torch.equal(again, out)


@pytest.mark.parametrize("T,H,E,k,I,bits,shared_I", [
    (140, 256, 20, 2, 384, 4, 0),       # experts on either side of sixteen rows; 80 tiles of gate and up: halves
    (150, 128, 150, 3, 384, 3, 0),      # nearly all below; 150 x 4 tiles whole, 150 of the down projection as halves
    (150, 384, 60, 2, 384, 3, 0),       # both launches as halves, of a column block and a half
    (16, 384, 2, 1, 128, 5, 128),       # sixteen rows of the always-on expert
    (60, 384, 5, 1, 640, 2, 0),         # gate, up and the next rotation in one launch
])
@pytest.mark.parametrize("codebook", [0, 1, 2])
def test_experts_of_up_to_sixteen_rows(T, H, E, k, I, bits, shared_I, codebook):
    """They take the 16-row matrix instructions: against the oracle, stage by stage.  From 129 tokens on whichever list
    their problem is in (BERTH_MOE_BIG_MIN=9: most of them in that of the 128-row problems), with the same bits (K of
    up to 384 is not cut)."""
    gpu, res = Gpu(0), []
    wr, experts_np, experts, shared_np, shared = _make_layer(gpu, 9900 + T, H, E, I, bits, shared_I, 1.0)
    x = (synth.activations(9901 + T, T, H).astype(np.float32) / np.sqrt(H)).astype(np.float16)
    want, oi, _ = O.moe_layer(x, wr, experts_np, k, I, bits, codebook, shared=shared_np, shared_I=shared_I)
    rows = np.bincount(oi.reshape(-1), minlength=E)
    assert (rows[rows > 0] <= 16).any() or shared_I
    for big_min in (0, 9, 33) if T >= 129 and T * k >= 256 else (0,):
        with knobs(BERTH_MOE_BIG_MIN=big_min, BERTH_MOE_FEW_TOKENS=0):
            layer = MoeLayer(gpu, wr, experts, k, shared=shared, codebook=codebook)
            out = torch.zeros((T, H), dtype=torch.float32, device=DEV)
            idx = torch.zeros((T, k), dtype=torch.int32, device=DEV)
            w = torch.zeros((T, k), dtype=torch.float32, device=DEV)
            layer.forward(gpu, dev(x.view(np.uint16)), out, T, idx, w)
            torch.cuda.synchronize()
            assert ("exl3_gemm_mixed_kernel" in K.moe.last_launch()) == (big_min > 0), K.moe.last_launch()
            assert ("exl3_gemm_pair_kernel" in K.moe.last_launch()) == (big_min == 0), K.moe.last_launch()
            assert np.array_equal(idx.cpu().numpy(), oi)
            _check_stages(layer, x, experts_np, shared_np, oi, w.cpu().numpy(), out.cpu().numpy(), T, H, E, k, I, bits, shared_I,
                          codebook)
        res.append(out)
    assert all(torch.equal(res[0], other) for other in res[1:])


def test_rows_beyond_four_gigabytes_of_rotated_input():
    """16-row problems over 65535 rows of 32896 columns: the rotated rows span more than 32-bit offsets reach, and the last
    ones are read where they are."""
    T, Kk, N, E, bits = 65535, 32896, 128, 2, 4
    tr, suh, svh = synth.linear(9701, Kk, N, bits)
    x = synth.activations(9702, 8, Kk)
    d = [dev(t.view(np.uint16)) for t in (tr, suh, svh)]
    table = torch.tensor([[t.data_ptr() for t in d]] * E, dtype=torch.int64, device=DEV)
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32, device=DEV)
    idx, off, perm, inv = i32(T), i32(E + 1), i32(T), i32(T)
    idx[T // 2:] = 1
    gather = (torch.arange(T, device=DEV) % 8).int()
    d_x, out = dev(x.view(np.uint16)), torch.zeros((T, N), dtype=torch.float32, device=DEV)
    a_had = torch.zeros((T, Kk), dtype=torch.float16, device=DEV)
    with knobs(BERTH_MOE_FEW_TOKENS=T, BERTH_MOE_BIG_MIN=0):
        scratch = torch.zeros(K.moe.permute_scratch_bytes(T, 1, E), dtype=torch.uint8, device=DEV)
        K.moe.permute(idx.data_ptr(), off.data_ptr(), perm.data_ptr(), inv.data_ptr(), scratch.data_ptr(), T, 1, E)
        K.moe.grouped_exl3(d_x.data_ptr(), None, gather.data_ptr(), 1, table.data_ptr(), 1, 0, 1, out.data_ptr(), None,
                           scratch.data_ptr(), a_had.data_ptr(), T, 1, E, Kk, N, bits, 2, True)
        torch.cuda.synchronize()
    want, _ = O.linear(x, tr, suh, svh, Kk, N, bits, 2, out_fp32=True)
    for r in (0, T // 2, T - 250, T - 1):
        assert np.abs(out[r].cpu().numpy() - want[r % 8]).max() <= 2e-3 * np.abs(want).max(), r
    assert torch.equal(out[:8], out[T - 7 - 8:T - 7])


def test_sixteen_row_problems_beside_128_row_ones():
    """64 experts with 25 rows each as problems of 16 rows, in a call that may also have 128-row problems: two problems
    per expert, all of them in the list, and the bits of the 32-row problems."""
    T, k, E, Kk, N, bits = 200, 8, 64, 256, 384, 4
    lins = [synth.linear(9800 + e, Kk, N, bits) for e in range(E)]
    d = [[dev(t.view(np.uint16)) for t in lin] for lin in lins]
    table = torch.tensor([[t.data_ptr() for t in lin] for lin in d], dtype=torch.int64, device=DEV)
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32, device=DEV)
    idx = (torch.arange(T * k, device=DEV) % E).int()
    d_x, res = dev(synth.activations(9801, T, Kk).view(np.uint16)), []
    for few in (16, T):
        off, perm, inv = i32(E + 1), i32(T * k), i32(T * k)
        out = torch.zeros((T * k, N), dtype=torch.float32, device=DEV)
        a_had = torch.zeros((T * k, Kk), dtype=torch.float16, device=DEV)
        with knobs(BERTH_MOE_FEW_TOKENS=few):
            scratch = torch.zeros(K.moe.permute_scratch_bytes(T, k, E), dtype=torch.uint8, device=DEV)
            K.moe.permute(idx.data_ptr(), off.data_ptr(), perm.data_ptr(), inv.data_ptr(), scratch.data_ptr(), T, k, E)
            K.moe.grouped_exl3(d_x.data_ptr(), None, perm.data_ptr(), k, table.data_ptr(), 1, 0, 1, out.data_ptr(), None,
                               scratch.data_ptr(), a_had.data_ptr(), T, k, E, Kk, N, bits, 2, True)
            torch.cuda.synchronize()
        assert (out != 0).any(dim=1).all()
        res.append(out)
    assert torch.equal(res[0], res[1])
