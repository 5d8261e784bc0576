"""What the build looks for in the compiled kernels."""
import os
import re
import subprocess

import pytest

from cobalt_amd import build as B

KERNEL = """
.amdgcn_target "amdgcn-amd-amdhsa--gfx950"
.text
.globl k
.p2align 8
.type k,@function
k:
  v_mov_b32_e32 v{amount}, 4
  {op} v[0:1], v{amount}, v[2:3]
  s_endpgm
.size k, .-k
.rodata
.p2align 6
.amdhsa_kernel k
  .amdhsa_next_free_vgpr {n}
  .amdhsa_next_free_sgpr 8
  .amdhsa_accum_offset {accum}
.end_amdhsa_kernel
.amdgpu_metadata
---
amdhsa.version: [1, 2]
amdhsa.target: amdgcn-amd-amdhsa--gfx950
amdhsa.kernels:
  - .name: k
    .symbol: k.kd
    .agpr_count: {agpr}
    .vgpr_count: {n}
    .sgpr_count: 8
    .kernarg_segment_size: 0
    .kernarg_segment_align: 8
    .group_segment_fixed_size: 0
    .private_segment_fixed_size: 0
    .wavefront_size: 64
    .max_flat_workgroup_size: 64
...
.end_amdgpu_metadata
"""


@pytest.mark.parametrize("op,amount,n,agpr,hit", [
    ("v_lshrrev_b64", 7, 8, 0, True), ("v_lshlrev_b64", 15, 16, 0, True), ("v_ashrrev_i64", 223, 224, 0, True),
    ("v_lshrrev_b64", 255, 256, 0, True), ("v_lshrrev_b64", 15, 24, 8, True),   # (the next one is an accumulation register)
    ("v_lshrrev_b64", 7, 16, 0, False), ("v_lshrrev_b64", 223, 232, 0, False), ("v_lshrrev_b64", 6, 8, 0, False),
    ("v_lshrrev_b64", 14, 15, 0, False)])
def test_shift_hazards_are_found(tmp_path, op, amount, n, agpr, hit):
    """Assembled here, never run: a 64-bit shift by the last register of the allocation, and shifts that are not."""
    src, obj = tmp_path / "k.s", str(tmp_path / "k.co")
    src.write_text(KERNEL.format(op=op, amount=amount, n=n, agpr=agpr, accum=(n - agpr + 3) // 4 * 4))
    subprocess.run([B._llvm("clang"), "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", str(src), "-o", obj], check=True)
    assert B.shift_hazards(obj) == ([("k", op, amount)] if hit else [])


def test_no_kernel_of_the_library_has_one():
    if not os.path.exists(B.LIB):
        pytest.skip("the library is not built")
    assert B.shift_hazards_of(B.LIB) == []


@pytest.mark.parametrize("name,lds,hit", [("_ZN3cbk18gemm_skinny_kernelILi4EEEvNS_6SkArgsE", 16, True),
                                          ("_ZN3cbk18gemm_skinny_kernelILi4EEEvNS_6SkArgsE", 0, False), ("other", 16, False)])
def test_static_lds_before_a_table_at_address_0_is_found(tmp_path, name, lds, hit):
    src, obj = tmp_path / "k.s", str(tmp_path / "k.co")
    text = KERNEL.format(op="v_lshrrev_b64", amount=6, n=8, agpr=0, accum=8)
    text = text.replace(".group_segment_fixed_size: 0", f".group_segment_fixed_size: {lds}").replace(" .name: k", f" .name: {name}")
    src.write_text(text.replace(".symbol: k.kd", f".symbol: {name}.kd"))
    subprocess.run([B._llvm("clang"), "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", str(src), "-o", obj], check=True)
    assert B.static_lds(obj) == ([(name, lds)] if hit else [])


def test_kernels_that_read_from_lds_address_0_have_no_static_lds():
    """And the library holds kernels of the names that are looked for."""
    if not os.path.exists(B.LIB):
        pytest.skip("the library is not built")
    assert B.static_lds_of(B.LIB) == []
    names = B._of_every_code_object(B._kernels, B.LIB)
    assert all(any(n in k for k in names) for n in B.LDS_FROM_ZERO)


def assembled(tmp_path, code):
    """A kernel of these instructions, assembled and never run."""
    src, obj = tmp_path / "k.s", str(tmp_path / "k.co")
    text = KERNEL.format(op="v_lshrrev_b64", amount=6, n=264, agpr=8, accum=256)
    begin, end = text.index("  v_mov_b32_e32"), text.index("  s_endpgm")
    src.write_text(text[:begin] + "".join(f"  {c}\n" for c in code) + text[end:])
    subprocess.run([B._llvm("clang"), "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", str(src), "-o", obj], check=True)
    return obj


LDS_COPY = "buffer_load_dwordx4 v2, s[4:7], s9 offen lds"


@pytest.mark.parametrize("code,hit", [
    (["v_readfirstlane_b32 s4, v0", "s_add_u32 m0, s8, 16", "s_nop 0", LDS_COPY], "s4"),
    (["v_readfirstlane_b32 s4, v0", "s_add_u32 m0, s8, 16", "s_nop 4", LDS_COPY], None),
    (["v_readlane_b32 s9, v0, 3", "s_nop 3", LDS_COPY], "s9"),           # the offset, one state short
    (["v_readlane_b32 s9, v0, 3", "s_nop 3", "s_nop 0", LDS_COPY], None),
    (["v_readfirstlane_b32 s10, v0", LDS_COPY], None),                 # another register
    (["v_cmp_lt_u32_e64 s[4:5], v0, v1", "v_mov_b32_e32 v3, 0", LDS_COPY], "s4"),
    (["v_readfirstlane_b32 s4, v0", "s_cbranch_scc1 2", "s_nop 7", "s_nop 7", LDS_COPY], "s4"),   # only on the path that jumps
    (["v_readfirstlane_b32 s4, v0", "s_branch 2", LDS_COPY, "s_endpgm", "s_nop 3", LDS_COPY], None),
    (["s_nop 7", LDS_COPY, "s_nop 7", "v_readfirstlane_b32 s4, v0", "s_cbranch_scc1 65531"], "s4")])   # around a loop (to the copy)
def test_scalar_registers_read_too_soon_are_found(tmp_path, code, hit):
    found = B.wait_hazards(assembled(tmp_path, code))
    assert [f[3] for f in found] == ([hit] if hit else [])


MFMA = "v_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[8:11], a[0:3]"
READ = "v_accvgpr_read_b32 v0, a3"


@pytest.mark.parametrize("code,hit", [
    ([MFMA, "s_nop 6", READ], "a3"), ([MFMA, "s_nop 7", READ], None),
    ([MFMA, "s_nop 6", "v_accvgpr_write_b32 a2, 0"], "a2"),
    ([MFMA, "s_nop 6", "v_accvgpr_read_b32 v0, a4"], None),
    ([MFMA, MFMA, "s_nop 7", READ], None),                              # the same sums again: chained
    ([MFMA, "s_nop 6", "v_mfma_f32_16x16x32_f16 a[4:7], v[4:7], v[8:11], a[0:3]"], "a0"),
    ([MFMA, "s_nop 6", "v_mfma_f32_16x16x32_f16 a[4:7], a[0:3], v[8:11], a[4:7]"], "a0"),
    ([MFMA, "s_nop 7", "v_mfma_f32_16x16x32_f16 a[4:7], a[0:3], v[8:11], a[4:7]"], None),
    ([MFMA, "s_cbranch_scc1 1", "s_nop 7", READ], "a3"),
    (["s_nop 0", READ, "s_nop 7", MFMA, "s_cbranch_scc0 65530"], "a3"),    # around a loop
    (["v_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]", "s_nop 10", "v_accvgpr_read_b32 v0, a15"], "a15"),
    (["v_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]", "s_nop 11", "v_accvgpr_read_b32 v0, a15"], None),
    (["v_mov_b32_e32 v5, 0", "s_nop 0", MFMA, "s_nop 7"], "v5"), (["v_mov_b32_e32 v5, 0", "s_nop 1", MFMA, "s_nop 7"], None),
    (["v_accvgpr_write_b32 a1, 0", MFMA, "s_nop 7"], "a1"), (["v_mov_b32_e32 v12, 0", MFMA, "s_nop 7"], None)])
def test_wait_states_around_matrix_instructions_are_looked_for(tmp_path, code, hit):
    found = B.wait_hazards(assembled(tmp_path, code))
    assert [f[3] for f in found] == ([hit] if hit else [])


def test_the_wait_states_are_the_compilers_own(tmp_path):
    """The figures of build.py against what the compiler leaves around its own instructions: a source that needs every one of them
    has no hazard, and would have with one state more."""
    src, obj = tmp_path / "k.hip", str(tmp_path / "k.o")
    src.write_text("""
#include <hip/hip_runtime.h>
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
__global__ void read4(const v8h* p, v4f* o) { const v4f c = __builtin_amdgcn_mfma_f32_16x16x32_f16(p[threadIdx.x], p[64], o[threadIdx.x], 0, 0, 0); o[64 + threadIdx.x] = c + 1.f; }
__global__ void read16(const v8h* p, v16f* o) { const v16f c = __builtin_amdgcn_mfma_f32_32x32x16_f16(p[threadIdx.x], p[64], o[threadIdx.x], 0, 0, 0); o[64 + threadIdx.x] = c + 1.f; }
__global__ void write(const v8h* p, v4f* o) { const v8h a = p[threadIdx.x]; o[64 + threadIdx.x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a + a, p[64], o[threadIdx.x], 0, 0, 0); }
__global__ void scalar(const int* q, int* o) {
  const int s = __builtin_amdgcn_readfirstlane(q[threadIdx.x]);
  o[threadIdx.x] = __builtin_amdgcn_raw_buffer_load_b32(__builtin_amdgcn_make_buffer_rsrc((void*)q, 0, -1, 0x27000), threadIdx.x * 4, s, 0);
}
""")
    subprocess.run(["/opt/rocm/bin/hipcc"] + [f for f in B.FLAGS if f != "-shared"] + ["-c", str(src), "-o", obj], check=True, capture_output=True)
    assert B._of_every_code_object(B.wait_hazards, obj) == []
    kept = B.MFMA_TO_READ, B.VALU_TO_MFMA, B.VALU_TO_VMEM
    try:
        B.MFMA_TO_READ = {k: v + 1 for k, v in kept[0].items()}
        assert {f[2] for f in B._of_every_code_object(B.wait_hazards, obj)} == set(kept[0])
        B.MFMA_TO_READ, B.VALU_TO_MFMA, B.VALU_TO_VMEM = kept[0], kept[1], kept[2] + 1
        assert {f[4] for f in B._of_every_code_object(B.wait_hazards, obj)} == {"buffer_load_dword"}
    finally:
        B.MFMA_TO_READ, B.VALU_TO_MFMA, B.VALU_TO_VMEM = kept


def test_no_kernel_of_the_library_reads_a_register_too_soon():
    if not os.path.exists(B.LIB):
        pytest.skip("the library is not built")
    assert B.wait_hazards_of(B.LIB) == []


def main_loop(body):
    """Of a function's instructions, those of the loop with most matrix instructions."""
    at = {b[0]: i for i, b in enumerate(body)}
    loops = [body[at[b[3]]:i + 1] for i, b in enumerate(body) if b[3] in at and at[b[3]] < i]
    return max(loops, key=lambda l: sum("mfma" in b[1] for b in l), default=[])


def tile_loops(code_object):
    return [(fn, [(b[1], b[2]) for b in main_loop(body)]) for fn, body in B._functions(code_object) if "gemm_big_kernel" in fn]


@pytest.fixture(scope="module")
def loops():
    if not os.path.exists(B.LIB):
        pytest.skip("the library is not built")
    return dict(B._in_processes(tile_loops, B.LIB))


def test_tile_kernels_keep_their_state_in_registers(loops):
    """Every function named after one is a kernel with its matrix instructions in a loop: none calls a closure, which has its
    variables in memory (as the generic reader did, a quarter of its time)."""
    assert len(loops) > 300
    assert [fn for fn, l in loops.items() if sum(op.startswith("v_mfma") for op, _ in l) not in (128, 256, 512)] == []
    assert [fn for fn, l in loops.items() if any(op.startswith("scratch_") for op, _ in l)] == []


def waits(loop):
    """(matrix instructions so far, loads since the barrier and whether one of those lies behind the last matrix instruction, the
    count that is waited for, whether a barrier follows) of every wait for loads in a loop."""
    mfma, loads, fresh, out = 0, 0, False, []
    for i, (op, args) in enumerate(loop):
        if op.startswith("v_mfma"):
            mfma, fresh = mfma + 1, False
        elif op == "s_barrier":
            loads = 0
        elif op.startswith("global_load"):
            loads, fresh = loads + 1, True
        elif op == "s_waitcnt" and "vmcnt" in args:
            count = int(args[args.index("vmcnt(") + 6:].partition(")")[0])
            out.append((mfma, loads, fresh, count, any(o == "s_barrier" for o, _ in loop[i:i + 4])))
    return out


def test_tile_kernels_do_not_wait_for_loads_where_they_issue_them(loops):
    """A chunk of weights is loaded two stages before its use: nothing beside its loads may need what they load."""
    assert [(fn, w) for fn, l in loops.items() for w in waits(l) if w[2] and w[3] < w[1]] == []


def test_tile_kernels_wait_for_loads_at_their_barriers_only(loops):
    """Four waits for everything in a trip of four stages, each before a barrier, and none that the compiler adds: such a one
    would wait for the direct copies of the next stage."""
    for fn, l in loops.items():
        if "gemm_big_kernelILi0E" not in fn:                              # (calls of the generic reader wait for what they load)
            assert [w[3:] for w in waits(l)] == [(0, True)] * 4, fn


def test_streams_of_three_dwords_are_shifted_on(loops):
    """23 of 32 codes of four bits (three widened) fill three dwords.  Shifted on from byte to byte they take at most 30 vector
    instructions a block (eight in a trip) more than the two dwords of 16 codes: reading, widening and shifting the third.  Windows at
    a running position took 36 and 42."""
    vector = {}
    for fn, l in loops.items():
        key = tuple(map(int, re.search(r"gemm_big_kernelILi(\d)ELi(\d+)ELi(\d+)ELi(\d)ELi(\d)E", fn).groups()))
        vector[key] = sum(op.startswith("v_") and "mfma" not in op for op, _ in l)
    for (bits, keep, group, vectors, tile), n in vector.items():
        if keep == 23 and bits > 2:
            assert n - vector[bits, 16, group, vectors, tile] <= 8 * 30, (bits, group, vectors, tile)


def decode_kernels(code_object):
    """[(kernel, bits, group, rows, wide table, instructions, of those the blocks that have matrix instructions)] of the decode kernels."""
    out = []
    for fn, body in B._functions(code_object):
        m = re.search(r"gemv_(mfma|split)_kernelILi(\d)ELi(\d+)ELi(\d+)ELi(\d)ELb(\d)", fn)
        if not m:
            continue
        ops, steps, block = [b[1] for b in body], [], []
        for op in ops:
            block.append(op)
            if op.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                if any(o.startswith("v_mfma") for o in block):
                    steps.append(block)
                block = []
        out.append((m.group(1), *map(int, m.groups()[1:]), ops, steps))
    return out


@pytest.fixture(scope="module")
def decoders():
    if not os.path.exists(B.LIB):
        pytest.skip("the library is not built")
    return B._in_processes(decode_kernels, B.LIB)


def test_decode_steps_keep_their_state_in_registers(decoders):
    """A value of the loop that lies in scratch memory is read back behind the weights on their way, and waits for them."""
    assert len(decoders) > 200
    scratch = lambda ops: any(op.startswith("scratch_") for op in ops)
    assert [d[:6] for d in decoders if any(map(scratch, d[7])) and (d[1] != 8 or d[0] == "split")] == []
    assert [d[:6] for d in decoders if scratch(d[6]) and d[0] == "mfma" and d[1] != 8 and d[3] == 128] == []


def test_small_launches_end_without_spilled_scalars(decoders):
    """One activation row, small table: a launch of a step or two per wavefront is as long as what stands before and after
    them.  With more scalars spilled than there are here, every store of the end reads its pointers back from vector lanes:
    130 reads and more in a kernel, 33 to 51 without."""
    small = [d for d in decoders if d[0] == "mfma" and d[4] == 1 and not d[5] and d[1] in (2, 4) and d[2] in (10, 16)]
    assert len(small) == 8 and max(d[6].count("v_readlane_b32") for d in small) <= 64


def test_small_launches_of_every_format_end_without_spilled_scalars(decoders):
    """The same of 3- and 6-bit codes, 23 of 32 kept and dense layouts: where an output goes is read from the arguments at the end."""
    small = [d for d in decoders if d[0] == "mfma" and d[4] == 1 and not d[5]]
    assert len(small) > 25 and [d[:6] for d in small if d[6].count("v_readlane_b32") > 64] == []
