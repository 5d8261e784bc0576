"""Builds libcbk_hip.so (the C-ABI HIP library, hipcc for gfx950) and _native.so (its operators for
Python) in-tree."""
import multiprocessing
import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ProcessPoolExecutor, ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libcbk_hip.so")
SOURCES = ["cbk_api.hip", "cbk_dequant.hip", "cbk_gemv_generic.hip", "cbk_gemv.hip", "cbk_gemm.hip", "cbk_gemm_big.hip",
           "cbk_gemm_big_b2.hip", "cbk_gemm_big_b3.hip", "cbk_gemm_big_b4.hip", "cbk_gemm_big_b6.hip"] + [
           f"cbk_gemm_big_b{b}_t{t}.hip" for b in (2, 3, 4) for t in (1, 2, 4)] + ["cbk_act.hip", "cbk_pack.hip", "cbk_gemm_skinny.hip", "cbk_gemm_skinny_b2.hip",
           "cbk_gemm_skinny_b3.hip", "cbk_gemm_skinny_b4.hip", "cbk_gemm_skinny_b68.hip"]
FLAGS = ["-O3", "--offload-arch=gfx950", "-fPIC", "-shared", "-std=c++17",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument", "-Wno-inline-asm"]


def _llvm(tool):
    return os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "llvm", "bin", tool)


_KD = re.compile(r"\.(agpr_count|group_segment_fixed_size|vgpr_count|symbol):\s+(\S+)")
_SHIFT64 = re.compile(r"\b(v_(?:lshl|lshr|ashr)rev_[bi]64)\S*\s+v\[\d+:\d+\], v(\d+),")


def _kernels(code_object):
    """{kernel: its architectural vector registers and bytes of static LDS}, from the notes of a code object."""
    notes = subprocess.run([_llvm("llvm-readelf"), "--notes", code_object], check=True, capture_output=True, text=True).stdout
    out, cur = {}, {}
    for key, val in _KD.findall(notes):                                # (the keys of a kernel come in alphabetical order)
        if key == "agpr_count":
            cur = {"agpr": int(val)}
        elif key == "group_segment_fixed_size":
            cur["lds"] = int(val)
        elif key == "symbol":
            cur["symbol"] = val[:-3] if val.endswith(".kd") else val
        elif key == "vgpr_count" and "symbol" in cur:
            out[cur["symbol"]] = (int(val) - cur.get("agpr", 0), cur.get("lds", 0))
    return out


def shift_hazards(code_object):
    """[(function, instruction, register)]: the 64-bit shifts of a gfx950 code object whose shift amount
    is in the last vector register its wavefronts are given.

    Measured on gfx950: such a shift can work with another amount (0 in every case seen), in some
    wavefronts and not in others.  The 64-token tile of 6-bit codes had its amount in v223 of 224
    registers and returned sums off by 1e-2 that changed from run to run; the same instructions with
    232 registers given are exact.  The compiler knows the case for gfx90a, where it moves the
    amount, but does not look for it on gfx950.  Registers are given in blocks of eight."""
    arch = {k: v[0] for k, v in _kernels(code_object).items()}
    out, fn = [], ""
    dis = subprocess.Popen([_llvm("llvm-objdump"), "-d", "--no-show-raw-insn", code_object], stdout=subprocess.PIPE, text=True)
    for line in dis.stdout:
        if line.endswith(">:\n"):
            fn = line[line.index("<") + 1:-3]
            continue
        m = _SHIFT64.search(line)
        if not m:
            continue
        r = int(m.group(2))
        if r % 8 != 7:
            continue
        # a function that is no kernel runs with the registers of any kernel that can hold it
        n = arch.get(fn, min((v for v in arch.values() if v > r), default=0))
        if r + 1 >= n or r == 255:
            out.append((fn, m.group(1), r))
    if dis.wait() != 0:
        raise RuntimeError(f"llvm-objdump failed on {code_object}")
    return out


# Wait states between two instructions that the hardware does not keep apart.  The compiler fills them in, but not around
# instructions written by hand (cbk_gemm_big.h): the values are those it leaves on gfx950 around its own.  An instruction
# is one wait state, s_nop n is n + 1.
MFMA_TO_READ = {"v_mfma_f32_16x16x32_f16": 8, "v_mfma_f32_32x32x16_f16": 12}   # until anything but the next product of the same sums touches them
VALU_TO_MFMA = 2                                                       # a vector register written -> a matrix instruction reads it
VALU_TO_VMEM = 5                                                       # a scalar register written by a vector instruction -> a memory instruction reads it
_REG = re.compile(r"(?<![\w])([vas])(?:(\d+)\b|\[(\d+):(\d+)\])")
_TARGET = re.compile(r"<(\S+?)(?:\+0x([0-9a-f]+))?>$")


def _registers(text):
    return {(k, r) for k, n, lo, hi in _REG.findall(text) for r in (range(int(lo), int(hi) + 1) if lo else (int(n),))}


def _functions(code_object):
    """(name, [(address, mnemonic, operands, branch target or None)]) of every function of a code object."""
    dis = subprocess.Popen([_llvm("llvm-objdump"), "-d", "--no-show-raw-insn", code_object], stdout=subprocess.PIPE, text=True)
    name, start, body = "", 0, []
    for line in dis.stdout:
        if line.endswith(">:\n"):
            if body:
                yield name, body
            name, start, body = line[line.index("<") + 1:-3], int(line[:line.index(" ")], 16), []
            continue
        text, _, note = line.partition("//")
        op, _, args = text.strip().partition(" ")
        if not op or not note:
            continue
        target = None
        if op.startswith(("s_cbranch", "s_branch")):
            m = _TARGET.search(note.strip())
            if m and m.group(1) == name:
                target = start + int(m.group(2) or "0", 16)
        body.append((int(note[:note.index(":")], 16), op, args.strip(), target))
    if body:
        yield name, body
    if dis.wait() != 0:
        raise RuntimeError(f"llvm-objdump failed on {code_object}")


def wait_hazards(code_object):
    """[(function, address, instruction, register, instruction that follows too soon)] of a gfx950 code object: the pairs
    above that lie closer together, along any path of branches inside a function."""
    out = []
    for fn, body in _functions(code_object):
        at = {b[0]: i for i, b in enumerate(body)}
        regs = [None] * len(body)

        def touched(i):
            if regs[i] is None:
                regs[i] = _registers(body[i][2])
            return regs[i]

        def followers(i, states):
            """Instructions that can begin fewer than `states` wait states after instruction i."""
            todo, seen = [(i, states)], {}
            while todo:
                j, left = todo.pop()
                _, op, args, target = body[j]
                if j != i:
                    left -= int(args, 0) + 1 if op == "s_nop" else 1
                nxt = [] if op in ("s_branch", "s_endpgm", "s_setpc_b64") else [j + 1]
                if target is not None and target in at:
                    nxt.append(at[target])
                for n in nxt:
                    if left > 0 and n < len(body) and seen.get(n, 0) < left:
                        if n not in seen:
                            yield n
                        seen[n] = left
                        todo.append((n, left))

        for i, (addr, op, args, _) in enumerate(body):
            if not op.startswith("v_"):
                continue
            if op in MFMA_TO_READ:
                sums = args.partition(", ")[0]
                dst = _registers(sums)
                for j in followers(i, MFMA_TO_READ[op]):
                    hit = dst & touched(j)
                    if hit and body[j][1] == op:
                        d, a, b, c = body[j][2].split(", ")[:4]
                        if c == d == sums:                             # the next product of the same sums: chained by the hardware
                            hit = dst & _registers(a + " " + b)
                    if hit:
                        out.append((fn, addr, op, "%s%d" % min(hit), body[j][1]))
            elif op.startswith("v_mfma") or op.startswith("v_smfma"):
                continue
            else:
                dst = args.split(", ", 2)
                first = _registers(dst[0])
                if len(dst) > 1 and any(o in op for o in ("_co_", "v_div_scale", "v_mad_u64", "v_mad_i64")):
                    first |= _registers(dst[1])
                if any(k == "s" for k, _ in first):
                    for j in followers(i, VALU_TO_VMEM):
                        if body[j][1].startswith(("buffer_", "global_", "scratch_", "flat_")):
                            hit = {r for r in first if r[0] == "s"} & touched(j)
                            if hit:
                                out.append((fn, addr, op, "%s%d" % min(hit), body[j][1]))
                if any(k != "s" for k, _ in first) and any(b[1] in MFMA_TO_READ for b in body[i + 1:i + 1 + VALU_TO_MFMA]):
                    for j in followers(i, VALU_TO_MFMA):
                        hit = first & _registers(body[j][2].partition(", ")[2]) if body[j][1] in MFMA_TO_READ else None
                        if hit:
                            out.append((fn, addr, op, "%s%d" % min(hit), body[j][1]))
    return out


# Kernels whose table reads take an entry's offset in dynamic LDS as its address: nothing else may lie before it.
LDS_FROM_ZERO = ("gemm_skinny_kernel", "gemv_mfma_kernel", "gemv_split_kernel")


def static_lds(code_object):
    """[(kernel, bytes)]: the kernels of LDS_FROM_ZERO that have static LDS, which would move their table off address 0
    and have them multiply with wrong weights."""
    return [(k, lds) for k, (_, lds) in _kernels(code_object).items() if lds and any(n in k for n in LDS_FROM_ZERO)]


def _of_every_code_object(check, path, executor=ThreadPoolExecutor):
    """What `check` finds in every gfx950 code object inside an object file or library."""
    with tempfile.TemporaryDirectory() as tmp:
        link = os.path.join(tmp, "o")
        os.symlink(os.path.abspath(path), link)
        subprocess.run([_llvm("llvm-objdump"), "--offloading", link], check=True, capture_output=True)
        objs = [os.path.join(tmp, f) for f in sorted(os.listdir(tmp)) if "gfx950" in f]
        with executor(8) as ex:
            return [h for hs in ex.map(check, objs) for h in hs]


def shift_hazards_of(path):
    return _of_every_code_object(shift_hazards, path)


def _in_processes(check, path):                                       # (for what takes python itself long)
    return _of_every_code_object(check, path, lambda n: ProcessPoolExecutor(n, multiprocessing.get_context("fork")))


def wait_hazards_of(path):
    return _in_processes(wait_hazards, path)


def static_lds_of(path):
    return _of_every_code_object(static_lds, path)


def build_lib(verbose=True, extra=()):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objs = []
    procs = []
    for s in SOURCES:
        o = os.path.join(CSRC, s.replace(".hip", ".o"))
        cmd = [hipcc] + [f for f in FLAGS if f != "-shared"] + list(extra) + ["-c", os.path.join(CSRC, s), "-o", o]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((s, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(o)
    for s, p in procs:
        out, _ = p.communicate()
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed on {s}:\n{out}")
        if verbose and out.strip():
            print(out)
    cmd = [hipcc, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIB] + objs
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    bad = static_lds_of(LIB)
    if bad:
        os.remove(LIB)
        raise RuntimeError("static LDS in kernels that read from LDS address 0 (see static_lds):\n" +
                           "\n".join(f"  {n} bytes in {fn}" for fn, n in bad))
    bad = shift_hazards_of(LIB)
    if bad:
        os.remove(LIB)
        raise RuntimeError("64-bit shifts with their amount in the last register (see shift_hazards):\n" +
                           "\n".join(f"  {op} amount v{r} in {fn}" for fn, op, r in bad))
    bad = wait_hazards_of(LIB)
    if bad:
        os.remove(LIB)
        raise RuntimeError("instructions that follow each other too soon (see wait_hazards):\n" +
                           "\n".join(f"  {op} of {r}, then {then}, at {at:#x} of {fn}" for fn, at, op, r, then in bad))
    return LIB


NATIVE = os.path.join(HERE, "_native.so")


def build_native(verbose=True):
    """_native.so: the operators of ops.py as a CPython extension on torch's C++ API (host code,
    linked to libcbk_hip.so beside it)."""
    import sysconfig
    from torch.utils import cpp_extension as X
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    inc = list(X.include_paths()) + [sysconfig.get_paths()["include"], os.path.join(rocm, "include")]
    libs = X.library_paths()
    cmd = (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]
           + [a for d in inc for a in ("-isystem", d)] + [os.path.join(CSRC, "cbk_torch.cpp"), "-o", NATIVE]
           + ["-L" + d for d in libs + [HERE]] + ["-Wl,-rpath," + d for d in libs] + ["-Wl,-rpath,$ORIGIN"]
           + ["-lcbk_hip", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-lamdhip64",
              "-L" + os.path.join(rocm, "lib")])
    if verbose:
        print(" ".join(cmd), flush=True)
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if out.returncode != 0:
        raise RuntimeError("g++ failed on cbk_torch.cpp:\n" + out.stdout)
    return NATIVE


BENCH_LIB = os.path.join(HERE, "libcbk_bench.so")


def build_bench_lib(verbose=True):
    """libcbk_bench.so: the measured-ceiling probes bench.py reports beside the published peaks."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc] + FLAGS + [os.path.join(CSRC, "cbk_bench.hip"), "-o", BENCH_LIB]
    if verbose:
        print(" ".join(cmd), flush=True)
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if out.returncode != 0:
        raise RuntimeError("hipcc failed on cbk_bench.hip:\n" + out.stdout)
    return BENCH_LIB


if __name__ == "__main__":
    build_lib()
    build_native()
    build_bench_lib()
    print("built", LIB, NATIVE, BENCH_LIB)
