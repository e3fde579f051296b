"""Static check of the compiled matrix-core kernels: no vector instruction may read the destination of a matrix
instruction within a few issue slots of it on ANY control-flow path.

One build of the backward kernel had a branch between the last matrix instruction of a score tile and the first read
of its result; the compiler's wait states covered the fall-through path only, and the taken path read half-finished
sums (wrong gradients for some shapes, no error).  The kernels avoid such branches; this test compiles them to
assembly (no GPU needed) and walks every path behind every matrix instruction.

And no memory instruction may take its address from a scalar register that a vector instruction wrote less than five wait states
before: the compiler sees to it, except in asm blocks, which it does not look into (load_to_lds16 of common.h).

And the bf16 backward reloads no spilled register between the end of a direction and the staging of the next: the counter a reload is
waited for with goes down in the order of issue, so that it waits for everything the wave has just stored (3 to 6 % of a call).  Its
workgroups of two tiles send no more through memory than LDS has no room for."""
import functools
import os
import re
import subprocess
import tempfile

import pytest

from vig_amd import build as B

SOURCES = ["gla_tiles.hip", "gla_mfma.hip", "gla_backward_mfma.hip", "gates.hip", "patch_conv.hip", "linear.hip", "gla_states.hip",
           "wgrad.hip"]
WINDOW = 8  # issue slots behind a 32x32x16 matrix instruction in which its destination must not be read


def _regs(text):
    out = set()
    for m in re.finditer(r"\bv\[(\d+):(\d+)\]", text):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1))
    for m in re.finditer(r"\bv(\d+)\b", text):
        out.add(int(m.group(1)))
    return out


def early_reads(asm: str, window: int = WINDOW):
    lines = asm.split("\n")
    labels = {m.group(1): i for i, l in enumerate(lines) if (m := re.match(r"^(\.LBB\w+):", l))}
    mfma = re.compile(r"v_mfma_\w+\s+v\[(\d+):(\d+)\]")
    found = []
    for i, l in enumerate(lines):
        m = mfma.search(l)
        if not m:
            continue
        dst = set(range(int(m.group(1)), int(m.group(2)) + 1))
        stack, seen = [(i + 1, 0)], set()
        while stack:
            k, slots = stack.pop()
            while k < len(lines) and slots < window and k not in seen:
                seen.add(k)
                t = lines[k].strip()
                k += 1
                if not t or t.startswith(";") or t.startswith(".") or t.endswith(":"):
                    continue
                op = t.split()[0]
                if op == "s_nop":
                    slots += int(t.split()[1]) + 1
                elif op.startswith("s_cbranch"):
                    if t.split()[1] in labels:
                        stack.append((labels[t.split()[1]], slots + 1))
                    slots += 1
                elif op == "s_branch":
                    k = labels.get(t.split()[1], len(lines))
                    slots += 1
                elif op == "s_endpgm":
                    break
                elif op.startswith("v_mfma"):
                    if _regs(t.split(",")[0]) & dst:
                        break  # accumulates into / overwrites the same registers: interlocked by hardware
                    slots += 8
                else:
                    stores = ("ds_write", "buffer_store", "global_store", "scratch_store")
                    srcs = t if op.startswith(stores) else (",".join(t.split(",")[1:]) if "," in t else "")
                    if _regs(srcs) & dst:
                        found.append((i + 1, l.strip(), k, slots, t))
                        break
                    slots += 1
    return found


SCALAR_WAIT = 5  # wait states between a vector instruction's write of a scalar register and a memory instruction's read of it
VMEM = ("buffer_", "global_", "scratch_", "flat_")


def _sregs(text):
    out = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]", text):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1))
    for m in re.finditer(r"\bs(\d+)\b", text):
        out.add(int(m.group(1)))
    return out


def stale_scalars(asm: str):
    lines = asm.split("\n")
    labels = {m.group(1): i for i, l in enumerate(lines) if (m := re.match(r"^(\.LBB\w+):", l))}
    found = []
    for i, l in enumerate(lines):
        t = l.strip()
        dst = _sregs(t.split(",")[0]) if t.startswith("v_") else set()
        if not dst:
            continue
        stack, seen = [(i + 1, 0, frozenset(dst))], set()
        while stack:
            k, waited, live = stack.pop()
            while k < len(lines) and waited < SCALAR_WAIT and live and (k, waited) not in seen:
                seen.add((k, waited))
                t = lines[k].split(";")[0].strip()
                k += 1
                if not t or t.startswith(".") or t.endswith(":"):
                    continue
                op = t.split()[0]
                if op.startswith(VMEM) and _sregs(t) & live:
                    found.append((i + 1, l.strip(), k, waited, t))
                    break
                if op == "s_endpgm":
                    break
                if op.startswith("s_cbranch") and t.split()[1] in labels:
                    stack.append((labels[t.split()[1]], waited + 1, live))
                if op == "s_branch":
                    k = labels.get(t.split()[1], len(lines))
                if "," in t and op.startswith("s_"):
                    live = live - _sregs(t.split(",")[0])  # (written anew)
                waited += int(t.split()[1]) + 1 if op == "s_nop" else 1
    return found


def test_walk_sees_stale_scalars():
    asm = """
\tv_readfirstlane_b32 s5, v1
\tv_readfirstlane_b32 s4, v0
\t;;#ASMSTART
\ts_mov_b32 m0, s8
\ts_nop %d
\tglobal_load_lds_dwordx4 v3, s[4:5]
\t;;#ASMEND
"""
    assert len(stale_scalars(asm % 0)) == 2 and len(stale_scalars(asm % 2)) == 1 and stale_scalars(asm % 3) == []
    assert stale_scalars((asm % 0).replace("v_readfirstlane_b32 s5, v1", "s_mov_b32 s5, 0").replace("v_readfirstlane_b32 s4, v0", "s_mov_b32 s4, 0")) == []


def test_checker_sees_the_pattern():
    asm = """
.LBB0_1:
\tv_mfma_f32_32x32x16_bf16 v[0:15], v[70:73], v[28:31], v[0:15]
\ts_cbranch_scc1 .LBB0_3
\ts_nop 10
\tv_cndmask_b32_e64 v0, v0, 0, s[44:45]
.LBB0_3:
\tv_cvt_pk_bf16_f32 v71, v2, v3
\ts_endpgm
"""
    hits = early_reads(asm)
    assert len(hits) == 1 and "v_cvt_pk_bf16_f32" in hits[0][4]
    assert early_reads(asm.replace("\ts_cbranch_scc1 .LBB0_3\n", "")) == []


def reloads_while_staging(asm: str, kernels: str):
    """(kernel, reload) for every reload between two barriers around a direction's factors, 32 exponentials and more."""
    found, seen = [], 0
    for name, body in re.findall(rf"^({kernels}\w*):[^\n]*\n(.*?)^\.Lfunc_end", asm, re.S | re.M):
        for part in re.split(r"^\ts_barrier", body, flags=re.M):
            if part.count("v_exp_f32") >= 32:
                seen += 1
                found += [(name, l.strip()) for l in part.split("\n") if "scratch_load" in l]
    return found, seen


@functools.lru_cache(maxsize=None)
def _assembly(src):
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, src + ".s")
        cmd = [B.HIPCC, *[f for f in B.FLAGS if f != "-fPIC"], "-S", "--cuda-device-only", "-I", B.CSRC,
               os.path.join(B.CSRC, src), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return open(out).read()


def _report(hits):
    return "\n".join(f"line {a}: {b}  ->  line {c} after {d} slots: {e}" for a, b, c, d, e in hits[:10])


@pytest.mark.parametrize("src", SOURCES)
def test_no_early_read_of_matrix_results(src):
    hits = early_reads(_assembly(src))
    assert hits == [], _report(hits)


LDS_LOADS = [f for f in B.SOURCES if "load_to_lds16(" in open(os.path.join(B.CSRC, f)).read()]


@pytest.mark.parametrize("src", LDS_LOADS)
def test_no_stale_scalar_address(src):
    hits = stale_scalars(_assembly(src))
    assert hits == [], _report(hits)


def test_no_reload_between_the_directions():
    # whole sequences, 64 key channels, both directions: two to eight waves
    found, seen = reloads_while_staging(_assembly("gla_backward_mfma.hip"), r"_ZN3vig24gla_backward_mfma_kernelILi4ELb1ELb0ELi[23478]E")
    assert seen == 10 and found == []


def test_two_tiles_park_one_unit_of_four_in_memory():
    # 64 key channels, both directions, two waves: dv, dk, dq and either gate's gradient in four stores each, and what is left of the
    # first direction's dq (all four units through memory: 600 slabs of 64 tokens 27.6 us instead of 26.9)
    name, = re.findall(r"^(_ZN3vig24gla_backward_mfma_kernelILi4ELb1ELb0ELi2E\w*):", _assembly("gla_backward_mfma.hip"), re.M)
    body = re.search(rf"^{name}:.*?^\.Lfunc_end", _assembly("gla_backward_mfma.hip"), re.S | re.M).group(0)
    assert body.count("buffer_store_dwordx4") == 5 * 4 + 1
