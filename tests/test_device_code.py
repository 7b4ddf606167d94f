"""What the compiler cannot see around inline assembly, checked in the gfx950 assembly of the kernels themselves.

Loads that write LDS directly are issued as inline assembly, so the compiler inserts no wait for them: a
kernel has to wait itself before anything else uses the bytes they land in.  The decode of two codebooks
is inline assembly, so the compiler does not keep a matrix instruction away from its results.  The kernels
are compiled here (no GPU), and every path through their control flow is followed.
"""
import re
import subprocess

import pytest

from berth_amd import build as B

# the row-block kernel at every height and over the bit rates' load shapes
BLOCK_KERNELS = [f"exl3_gemm_block_kernel<{bits}, {cb}, {mt}>" for bits, cb, mt in
                 ((4, 2, 4), (4, 2, 6), (4, 2, 8), (1, 2, 4), (3, 1, 8), (8, 0, 6), (4, 2, 3), (4, 2, 5), (3, 1, 7))]

# every loop that multiplies freshly decoded weights, with the codebooks whose decode is inline assembly
DECODING_KERNELS = (["exl3_gemm_kernel<3, 1, 4>", "exl3_gemm_balanced_kernel<3, 1, 4>", "exl3_gemm_kernel<4, 0, 1>",
                     "exl3_gemm_wide_kernel<4, 1>"] +
                    [f"exl3_gemm_mixed_kernel<{bits}, {cb}>" for bits, cb in ((1, 1), (2, 1), (3, 1), (4, 0))] +
                    [f"exl3_gemm_rows_kernel<3, 1, {mt}, {grouped}>" for mt, grouped in ((1, "false"), (2, "false"), (1, "true"))] +
                    ["exl3_gemm_block_kernel<3, 1, 4>", "exl3_gemm_block_kernel<5, 0, 8>"])
STREAM_KERNELS = ["exl3_gemv_stream_kernel<4, 1, kInPlain, 0>", "exl3_gemv_stream_kernel<5, 0, kInPlain, 0>",
                  "exl3_gemv_stream_kernel<4, 1, kInPlainLong, 0>"]


def _operands(text):
    """Registers of one operand list, operand by operand: [('v', 3), ...] each."""
    out = []
    for op in re.split(r",(?![^\[]*\])", text):
        m = re.match(r"\s*[-|]*([vas])\[(\d+):(\d+)\]", op) or re.match(r"\s*[-|]*([vas])(\d+)\b", op)
        out.append([] if not m else [(m[1], i) for i in range(int(m[2]), int(m[m.lastindex]) + 1)])
    return out


class Function:
    """Instructions of one kernel as (opcode, operand text, inside inline assembly), with successors."""

    def __init__(self, name, lines):
        self.name, self.code, labels = name, [], {}
        in_asm = False
        for line in lines:
            if "#ASMSTART" in line or "#ASMEND" in line:
                in_asm = "#ASMSTART" in line
            text = line.split(";")[0].strip()
            if m := re.match(r"(\.LBB\w+):", text):
                labels[m[1]] = len(self.code)
            elif text and not text.startswith(".") and not text.endswith(":"):
                op, _, rest = text.partition(" ")
                self.code.append((op, rest.strip(), in_asm))
        self.next = []
        for i, (op, rest, _) in enumerate(self.code):
            after = [] if op in ("s_endpgm", "s_branch") else [i + 1]
            if op == "s_branch" or op.startswith("s_cbranch"):
                after.append(labels[rest])
            assert op not in ("s_setpc_b64", "s_swappc_b64"), "an indirect branch cannot be followed"
            self.next.append(after)

    def states(self, entry, step, join):
        """The state before every instruction, as the join over all paths that reach it."""
        before = {0: entry}
        work = [0]
        while work:
            i = work.pop()
            out = step(before[i], *self.code[i])
            for j in self.next[i]:
                new = out if j not in before else join(before[j], out)
                if j not in before or new != before[j]:
                    before[j] = new
                    work.append(j)
        return before


def _assembly(tmp_path, kernels, headers, params="GemmParams"):
    source = tmp_path / "kernels.hip"
    source.write_text("".join(f'#include "{h}"\n' for h in headers) + "namespace berth {\n" +
                      "".join(f"template __global__ void {k}({params});\n" for k in sorted(set(kernels))) + "}\n")
    out = tmp_path / "kernels.gfx950"
    r = subprocess.run([B.HIPCC, *B.FLAGS, "--offload-device-only", "-S", "-I" + B.CSRC, str(source), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out.read_text()


def _compile(tmp_path, kernels, headers, params="GemmParams"):
    functions, lines = [], None
    for line in _assembly(tmp_path, kernels, headers, params).splitlines():
        if m := re.match(r"(_Z\w+):", line):
            name, lines = m[1], []
        elif lines is not None and line.startswith(".Lfunc_end"):
            functions.append(Function(name, lines))
            lines = None
        elif lines is not None:
            lines.append(line)
    return functions


def _is_vector_load(op):
    return op.startswith(("global_load", "buffer_load", "scratch_load"))


def _lds_loads_step(younger, op, rest, in_asm):
    """State: None when every load to LDS has landed, else the fewest vector loads issued behind the
    youngest of them.  Loads come back in order, so vmcnt(n) covers it from n younger loads on."""
    if "load_lds" in op:
        return 0
    if younger is not None and _is_vector_load(op):
        return min(younger + 1, 64)
    if younger is not None and op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", rest)):
        return None if younger >= int(m[1]) else younger
    return younger


def _fewest(a, b):
    return b if a is None else a if b is None else min(a, b)


@pytest.fixture(scope="module")
def block_kernels(tmp_path_factory):
    found = _compile(tmp_path_factory.mktemp("block"), BLOCK_KERNELS, ["exl3_gemm_block_kernel.cuh"])
    found = [f for f in found if "exl3_gemm_block_kernel" in f.name]
    assert len(found) == len(BLOCK_KERNELS)
    return found


def test_loads_to_lds_have_landed_before_their_bytes_are_used_again(block_kernels):
    """The register dumps at the end of a tile lie over the operand buffers, some of them over what another
    wave loaded: no load to LDS may be outstanding at a barrier of the finish (the loop's own barriers are
    inline assembly), where LDS is written, or where the workgroup gives its LDS back."""
    for f in block_kernels:
        before = f.states(None, _lds_loads_step, _fewest)
        assert any("load_lds" in op for op, _, _ in f.code), f.name
        late = [(i, op) for i, (op, _, in_asm) in enumerate(f.code)
                if ((op == "s_barrier" and not in_asm) or op.startswith("ds_write") or op == "s_endpgm")
                and before.get(i) is not None]
        assert not late, f"{f.name}: loads to LDS outstanding at {late[:4]} ({len(late)} in all)"


def test_the_loops_wait_covers_the_loads_of_its_step(block_kernels):
    """`s_waitcnt vmcnt(n)` + `s_barrier` in the loop: on every path the loads to LDS are older than at
    least n other loads, so the operands that are read behind the barrier are there."""
    for f in block_kernels:
        before = f.states(None, _lds_loads_step, _fewest)
        waits = [i for i, (op, rest, in_asm) in enumerate(f.code) if in_asm and op == "s_waitcnt" and "vmcnt" in rest]
        assert waits, f.name
        for i in waits:
            assert _lds_loads_step(before[i], *f.code[i]) is None, (f.name, i, f.code[i])


VALU_TO_MFMA = 2        # wait states; what the compiler leaves between its own instructions


def _asm_results_step(ages, op, rest, in_asm):
    """State: wait states since inline assembly wrote a vector register, while fewer than VALU_TO_MFMA.
    (An exchange of two registers writes both of its operands.)"""
    passed = int(rest, 0) + 1 if op == "s_nop" else 1
    ages = {reg: age + passed for reg, age in ages if age + passed < VALU_TO_MFMA}
    if op.startswith(("v_", "ds_read", "global_load", "buffer_load", "scratch_load")):
        for operand in _operands(rest)[:2 if re.match(r"v_(permlane\d+_)?swap_b(16|32)", op) else 1]:
            for reg in operand:
                ages.pop(reg, None)
                if in_asm and op.startswith("v_"):
                    ages[reg] = 0
    return frozenset(ages.items())


def _youngest(a, b):
    joined = dict(a)
    for reg, age in b:
        joined[reg] = min(age, joined.get(reg, age))
    return frozenset(joined.items())


def _read_too_soon(f):
    """(matrix instruction, register) pairs of a kernel that stand too close to inline assembly."""
    before, found = f.states(frozenset(), _asm_results_step, _youngest), []
    for i, (op, rest, _) in enumerate(f.code):
        if op.startswith("v_mfma") and i in before:
            fresh = dict(before[i])
            found += [(f"{op} {rest}", reg) for operand in _operands(rest)[1:4] for reg in operand if reg in fresh]
    return found


@pytest.mark.parametrize("kernels,headers,params", [
    (DECODING_KERNELS, ("exl3_gemm_block_kernel.cuh", "exl3_gemm_wide_kernel.cuh"), "GemmParams"),
    (STREAM_KERNELS, ("exl3_gemv_stream_kernel.cuh",), "StreamParams")])
def test_matrix_instructions_keep_their_distance_from_inline_assembly(tmp_path, kernels, headers, params):
    functions = [f for f in _compile(tmp_path, kernels, headers, params) if "finish_kernel" not in f.name]
    assert len(functions) == len(set(kernels))
    for f in functions:
        assert any(op.startswith("v_mfma") for op, _, _ in f.code), f.name
        assert any(a and op.startswith("v_") for op, _, a in f.code), f"{f.name}: no inline assembly left to check"
        close = _read_too_soon(f)
        assert not close, f"{f.name}: too soon: {close[:4]} ({len(close)} in all)"


@pytest.mark.parametrize("write,regs", [
    ("v_permlane16_swap_b32 v4, v12", (4, 12)), ("v_permlane32_swap_b32_e32 v5, v13", (5, 13)), ("v_swap_b32 v6, v14", (6, 14)),
    ("v_add_u32_e32 v7, v15, v16", (7,))])
@pytest.mark.parametrize("waits,close", [("s_nop 0", True), ("s_nop 1", False)])
def test_every_register_that_inline_assembly_writes_counts(write, regs, waits, close):
    """A matrix instruction right behind inline assembly is found by each register that it writes, and only by those."""
    for reg in range(4, 17):
        f = Function("synthetic", [";#ASMSTART", write, waits, ";#ASMEND",
                                   f"v_mfma_f32_32x32x16_f16 v[32:47], v[20:23], v[{reg}:{reg}], v[32:47]", "s_endpgm"])
        assert bool(_read_too_soon(f)) == (close and reg in regs), (write, waits, reg)


@pytest.mark.parametrize("kernels,params", [
    (["exl3_gemm_pair_kernel<3, 1>", "exl3_gemm_pair_kernel<4, 0>", "exl3_gemm_kernel<4, 0, 1, false>"], "GemmParams"),
    (["exl3_gemm_rows_kernel<3, 1, 1, false, true>", "exl3_gemm_rows_kernel<4, 0, 2, false, true>"], "GemmRotateParams"),
    (["exl3_gemm_rows_kernel<3, 1, 1, false, false, true>", "exl3_gemm_rows_kernel<4, 0, 2, false, false, true>"], "RowsPairParams")])
def test_the_same_of_the_fused_launches(tmp_path, kernels, params):
    test_matrix_instructions_keep_their_distance_from_inline_assembly(tmp_path, kernels, ("exl3_gemm_rows_kernel.cuh",), params)


def _registers(tmp_path, kernels, headers, params="GemmParams"):
    """(vector registers, scratch bytes a lane) of each kernel"""
    found = {}
    for entry in _assembly(tmp_path, kernels, headers, params).split("  - .agpr_count:")[1:]:
        found[re.search(r"\.name:\s+(\S+)", entry)[1]] = tuple(int(re.search(rf"\.{key}:\s+(\d+)", entry)[1])
                                                                for key in ("vgpr_count", "private_segment_fixed_size"))
    assert len(found) == len(kernels)
    return found


def test_grouped_tiles_of_one_block_leave_room_for_four_workgroups(tmp_path):
    """Four workgroups of four waves on a compute unit: at most 128 of a SIMD's 512 registers a lane, and no scratch.
    (8 bits outside the pair kernel and MUL1 above 6 take three.)"""
    kernels = ([f"exl3_gemm_pair_kernel<{bits}, {cb}>" for bits, cb in ((3, 0), (4, 0), (4, 1), (4, 2), (8, 0))] +
               [f"exl3_gemm_kernel<{bits}, {cb}, 1, false>" for bits, cb in ((3, 0), (3, 1), (3, 2), (4, 0), (7, 1))])
    found = _registers(tmp_path, kernels, ("exl3_gemm_kernel.cuh",))
    assert {name: at for name, at in found.items() if at[0] > 128 or at[1]} == {}


def test_one_token_gate_and_up_leave_room_for_five_workgroups(tmp_path):
    """The one-token launch that works the routing out: at most 96 registers up to 5 bits, and no scratch."""
    kernels = [f"exl3_gemv_kernel<{bits}, {cb}, 1, false, {trs}, true>" for bits, cb, trs in ((2, 2, 8), (4, 0, 8), (4, 2, 4), (5, 1, 8))]
    found = _registers(tmp_path, kernels, ("exl3_gemv_kernel.cuh",), "GemvParams")
    assert {name: at for name, at in found.items() if at[0] > 96 or at[1]} == {}


def test_every_tile_of_a_mixed_launch_is_taken_once(tmp_path):
    """mixed_place over two lists of any length within their room: each problem whole, or both of its halves, once each
    and within the grid; all of the second list (few rows or many) as halves where twice its tiles have places."""
    source, program = tmp_path / "places.hip", tmp_path / "places"
    source.write_text("""#include "exl3_gemm_kernel.cuh"
#include <cstdio>
#include <map>
#include <tuple>
using namespace berth;
int main() {
    for (int tiles : {1, 2, 3, 4, 8, 14, 64}) for (int places : {32, 64, 512, 608})
    for (int big = 0; big <= 70; big += big < 4 ? 1 : 11) for (int small = 0; small <= 300; small += small < 4 ? 1 : 37) {
        const bool all = 2 * (big + small) * tiles <= places, first = (2 * big + small) * tiles <= places;
        std::map<std::tuple<bool, int, bool>, int> seen;
        const int grid = 8 * (int)group_grid(tiles, 1, big + small + mixed_extra(tiles, places)).y;     // full lists: the tightest
        for (int i = 0; i < grid; ++i) {
            const MixedPlace m = mixed_place(i, big, small, tiles, places);
            if (m.empty) continue;
            if (m.halves != (m.first_list ? first : all) || (m.second && !m.halves)) return 1;
            ++seen[{m.first_list, m.at, m.second}];
        }
        if ((int)seen.size() != big * (first ? 2 : 1) + small * (all ? 2 : 1)) return 2;
        for (auto& [place, times] : seen)
            if (times != 1 || std::get<1>(place) < 0 || std::get<1>(place) >= (std::get<0>(place) ? big : small)) return 3;
    }
    std::puts("ok");
}
""")
    subprocess.run([B.HIPCC, *B.FLAGS, "-I" + B.CSRC, str(source), "-o", str(program)], check=True, capture_output=True)
    assert subprocess.run([str(program)], capture_output=True, text=True).stdout == "ok\n"
