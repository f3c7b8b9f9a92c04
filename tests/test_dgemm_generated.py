"""Host-side checks of the machine code of the medium-row kernels (exl3_dgemm.kspec.hip, exl3_dgemm_wide.kspec.hip) as built -- no GPU.  Both count their outstanding loads by hand, and the wide
one writes its matrix instructions as asm statements, which the compiler's hazard logic does not see:

  * every request into LDS is waited for in front of the next barrier (the count of the wait is at most the number of loads issued behind the last request), and nothing is requested whose barrier
    is followed by the output tile in the same LDS;
  * wide kernel: accumulators stay in their registers from the first to the last matrix instruction, no vector instruction writes a matrix instruction's operand right in front of it, and the
    accumulators are read only behind the closing wait states, on every way out of the loop."""
import os
import re
import subprocess
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJ = os.path.join(ROOT, "build", "obj")
BIN = "/opt/rocm/llvm/bin"
TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"


def _kernels(unit, tmp):
    """{(codebook, row tiles): [(address, instruction, branch target or None)]} of one built unit."""
    obj = os.path.join(OBJ, unit + ".o")
    if not os.path.exists(obj) or not os.path.exists(f"{BIN}/llvm-objdump"):
        pytest.skip("the units are not built here")
    run = lambda *a: subprocess.run(a, check=True, capture_output=True, text=True).stdout
    # (dumping a section rewrites the object: the copy, so that the build keeps its own)
    fat, code, copy = str(tmp / "fat"), str(tmp / "code"), str(tmp / "copy.o")
    run(f"{BIN}/llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, obj, copy)
    run(f"{BIN}/clang-offload-bundler", "--unbundle", "--type=o", "--targets=" + TARGET, "--input=" + fat, "--output=" + code)
    out, cur, base = {}, None, 0
    for line in run(f"{BIN}/llvm-objdump", "-d", "--no-show-raw-insn", code).splitlines():
        m = re.match(r"^([0-9a-f]+) <(\S+)>:", line)
        if m:
            k = re.search(r"kernelILi\d+ELi(\d+)ELi(\d+)EE", m.group(2))
            cur, base = (out.setdefault((int(k.group(1)), int(k.group(2))), []) if k else None), int(m.group(1), 16)
        elif cur is not None and line.startswith("\t"):
            text, _, note = line.partition("//")
            if not note:
                continue                                      # (the fill behind a kernel)
            target = re.search(r"<\S+\+0x([0-9a-f]+)>", note)
            cur.append((int(note.split(":")[0], 16), " ".join(text.split()), base + int(target.group(1), 16) if target else None))
    assert len(out) in (12, 15)
    return out


def _is_dma(s):
    return s.startswith("buffer_load") and s.endswith(" lds")


def _is_load(s):
    return s.startswith(("global_load", "buffer_load", "flat_load", "scratch_load", "global_store", "buffer_store", "scratch_store"))


def _regs(operand):
    m = re.match(r"^([va])\[(\d+):(\d+)\]$", operand) or re.match(r"^([va])(\d+)()$", operand)
    return {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3) or m.group(2)) + 1)} if m else set()


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("unit", ["exl3_dgemm", "exl3_dgemm_wide"])
def test_requests_into_lds_are_waited_for(unit, K, tmp_path):
    for (cb, mt), code in _kernels(f"{unit}_k{K}", tmp_path).items():
        requests = behind = wait = total = 0
        for _, s, _ in code:
            if _is_dma(s):
                requests, behind, wait, total = requests + 1, 0, None, total + 1
            elif _is_load(s):
                behind += 1
            elif s.startswith("s_waitcnt") and "vmcnt" in s and requests:
                n = int(re.search(r"vmcnt\((\d+)\)", s).group(1))
                if n <= behind:
                    wait = n
            elif s == "s_barrier":
                assert not requests or wait is not None, (cb, mt)
                requests = behind = 0
        assert total == 3 * mt, (cb, mt, total)               # the first block and the two of the loop; the block behind the loop requests nothing


@pytest.mark.parametrize("K", range(1, 9))
def test_wide_kernel_keeps_its_accumulators_and_operands_in_place(K, tmp_path):
    for (cb, mt), code in _kernels(f"exl3_dgemm_wide_k{K}", tmp_path).items():
        where = [i for i, (_, s, _) in enumerate(code) if s.startswith("v_mfma")]
        assert len(where) == 3 * 8 * mt
        first, last = where[0], where[-1]
        loop_end = max(i for i, (a, s, t) in enumerate(code) if s.startswith("s_cbranch") and t is not None and t < a and first < i < last and any(i > j for j in where))
        recent = []
        for i, (_, s, _) in enumerate(code):
            op, _, rest = s.partition(" ")
            operands = [o.strip().split()[0] for o in rest.split(",") if o.strip()]
            if op.startswith("v_mfma"):
                dst, a, b, c = (_regs(o) for o in operands[:4])
                assert dst == c and all(r[0] == "a" for r in dst), s
                for written in recent[-4:]:
                    assert not written & (a | b | c), (cb, mt, s)
                recent.append(set())
                continue
            recent.append(_regs(operands[0]) if op.startswith("v_") and operands else set())
            if first < i < last and op.startswith("v_"):
                assert not any(r[0] == "a" for o in operands for r in _regs(o)), (cb, mt, s)
            if first < i < loop_end:
                assert not op.startswith("scratch_"), (cb, mt, s)
        nops = [i for i in range(last, len(code)) if code[i][1] == "s_nop 15"][:2]
        read = next(i for i in range(last + 1, len(code)) if re.search(r"\ba(\[|\d)", code[i][1].partition(" ")[2]))
        assert len(nops) == 2 and nops[0] < nops[1] < read, (cb, mt)
        for i in range(first, last):
            target = code[i][2]
            assert target is None or target <= code[nops[0]][0] or target > code[-1][0] or not any(
                re.search(r"\ba(\[|\d)", s.partition(" ")[2]) for a, s, _ in code if a >= target), (cb, mt, code[i])
