"""The wave sweeps keep loads in flight over several rows and wait for them by counting
(k_wave.h), which is right only for the operations the compiler emits.  Every instantiation's gfx950
assembly is followed over all paths: nothing reads or writes a register that a load still in flight
will write.  (Loads return in order, so that a load may write over an earlier one's result.)
"""
import os
import re
import subprocess

import pytest

from trans_amd import build

CSRC = os.path.dirname(build.SRC)
FORMS = [  # value type, equations, rows in flight, waves per SIMD
    ("double", 7, 2, 2), ("double", 5, 2, 2), ("double", 2, 3, 2),
    ("float", 7, 4, 2), ("float", 5, 4, 2), ("float", 2, 4, 2),
    ("float", 7, 2, 4), ("float", 5, 2, 4), ("float", 2, 2, 4)]
KERNEL = re.compile(r"k_lusgs_waveI([df])Lb([01])ELi(\d)ELi(\d)ELi(\d)ELb([01])E")
MEMORY = re.compile(r"(buffer|global|flat|scratch|image)_(load|store|atomic)")
REGISTERS = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _registers(text):
    out = set()
    for kind, lo, hi, one in REGISTERS.findall(text):
        out |= {(kind, r) for r in range(int(lo or one), int(hi or one) + 1)}
    return out


def _functions(text):
    """Instruction and label lines of every sweep kernel."""
    out, cur = {}, None
    for line in text.splitlines():
        line = line.split(";")[0].rstrip()
        m = re.match(r"(\w+):", line)
        if m and KERNEL.search(m.group(1)):
            cur = out.setdefault(m.group(1), [])
        elif line.startswith(".Lfunc_end"):
            cur = None
        elif cur is not None and (line.startswith(".LBB") or (line.startswith("\t") and line.strip()[:1] != ".")):
            cur.append(line.strip())
    return out


def _violations(lines):
    """Instructions that touch a register of a load that may still be in flight."""
    names, blocks, new = {}, [], True
    for line in lines:
        if line.endswith(":"):
            names[line[:-1]] = len(blocks)
            blocks.append([])
            new = False
            continue
        if new:
            blocks.append([])
            new = False
        blocks[-1].append(line)
        new = line.startswith(("s_cbranch", "s_branch", "s_endpgm"))

    def successors(i):
        last = blocks[i][-1].split() if blocks[i] else [""]
        if last[0] == "s_endpgm":
            return []
        to = [names[last[1]]] if last[0].startswith(("s_cbranch", "s_branch")) else []
        return to if last[0] == "s_branch" else to + [i + 1]

    # per register of a load in flight: how many operations at least have been issued since
    at = [None] * len(blocks)
    at[0] = {}
    todo, bad = [0], set()
    while todo:
        i = todo.pop()
        flying = dict(at[i])
        for n, line in enumerate(blocks[i]):
            op, _, rest = line.partition(" ")
            if op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", rest)
                if m:
                    flying = {r: c for r, c in flying.items() if c < int(m.group(1))}
                continue
            load = MEMORY.match(op) and "load" in op
            touched = _registers(rest.partition(",")[2] if load else rest)
            if any(r in flying for r in touched):
                bad.add((i, n, line))
            if MEMORY.match(op):
                flying = {r: min(c + 1, 64) for r, c in flying.items()}
                if load or ("atomic" in op and "sc0" in rest):
                    flying.update({r: 0 for r in _registers(rest.partition(",")[0])})
        for q in successors(i):
            old = at[q]
            if old is None:
                at[q] = dict(flying)
                todo.append(q)
                continue
            more = {r: c for r, c in flying.items() if r not in old or old[r] > c}
            if more:
                old.update(more)
                todo.append(q)
    return bad


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("sweeps")
    text = "#include <hip/hip_runtime.h>\n#include <climits>\n"
    text += "".join(f'#include "{CSRC}/{h}"\n' for h in ("dev_common.h", "k_time.h", "k_wave.h"))
    for r, neq, rows, waves in FORMS:
        for fwd in ("true", "false"):
            for alt in ("true", "false"):
                text += (f"template __global__ void k_lusgs_wave<{r}, {fwd}, {neq}, {rows}, {waves}, {alt}>"
                         f"(Fields, const BlkInfo*, const WaveTile*, int, int*, {r}*, int*, int);\n")
    src = tmp / "sweeps.hip"
    src.write_text(text)
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC", "-Wall")]
    subprocess.run([build.HIPCC, "--offload-device-only", "-S", "-w"] + flags + [str(src), "-o", str(tmp / "sweeps.s")],
                   check=True)
    return _functions((tmp / "sweeps.s").read_text())


def test_the_forms_are_the_ones_in_use(kernels):
    if not os.path.exists(build.OUT):
        pytest.skip("library not built")
    nm = subprocess.run(["nm", build.OUT], check=True, capture_output=True, text=True).stdout
    built = {m.groups() for line in nm.splitlines() if "device_stub" in line for m in [KERNEL.search(line)] if m}
    assert built == {KERNEL.search(f).groups() for f in kernels}


def test_no_register_of_a_load_in_flight_is_touched(kernels):
    assert len(kernels) == 4 * len(FORMS)
    for name, lines in kernels.items():
        assert not _violations(lines), name


def test_nothing_spills(kernels):
    """Scratch operations would count among those that the waits count."""
    for name, lines in kernels.items():
        assert not any(line.startswith("scratch_") for line in lines), name


def test_a_weaker_wait_is_seen(kernels):
    """The check itself: waits that let one more operation pass, or none at all, in the text."""
    for name, lines in list(kernels.items())[::4]:
        assert _violations([re.sub(r"vmcnt\(\d+\)", "", line) for line in lines]), name
        most = max(int(n) for line in lines for n in re.findall(r"vmcnt\((\d+)\)", line))
        seen = 0
        for n in range(1, most + 1):
            weaker = [re.sub(rf"vmcnt\({n}\)", f"vmcnt({n + 1})", line) for line in lines]
            seen += weaker != lines and bool(_violations(weaker))
        assert seen, name
