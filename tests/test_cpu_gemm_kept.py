"""CPU: the waits of gd_kernel (csrc/gemm_mid.hip) in the code that was built.  Its direct-to-LDS loads are counted by hand; a wait has to
cover the stage behind it whatever the compiler makes of the loads around it."""
import os
import re
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin/"
OBJ = os.path.join(os.path.dirname(__file__), "..", "voxcpm.cpp_amd", "lib", "obj", "gemm_mid.o")


@pytest.fixture(scope="module")
def device_object(tmp_path_factory):
    if not os.path.exists(OBJ) or not os.path.exists(LLVM + "llvm-objdump"):
        pytest.skip("the library was not built on this machine")
    d = tmp_path_factory.mktemp("gemm_mid")
    fat, dev = str(d / "fat"), str(d / "dev.o")
    subprocess.check_call([LLVM + "llvm-objcopy", "--dump-section=.hip_fatbin=" + fat, OBJ, str(d / "copy.o")])
    subprocess.check_call([LLVM + "clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + fat, "--output=" + dev])
    return dev


def instructions(dev, epi):
    """[(address, text, branch target or None)] of gd_kernel<epi>"""
    symbol = f"_ZN12_GLOBAL__N_19gd_kernelILi{epi}EEEvNS_7gm_argsE"
    text = subprocess.check_output([LLVM + "llvm-objdump", "-d", "--disassemble-symbols=" + symbol, dev], text=True)
    start = int(re.search(r"^([0-9a-f]+) <" + symbol + ">:", text, re.M).group(1), 16)
    out = []
    for m in re.finditer(r"^\t(\S.*?)\s*// ([0-9A-F]+):[^<\n]*(?:<" + symbol + r"(?:\+0x([0-9a-f]+))?>)?$", text, re.M):
        target = None
        if m.group(1).startswith(("s_branch", "s_cbranch")):
            target = start + int(m.group(3) or "0", 16)
        out.append((int(m.group(2), 16), m.group(1), target))
    return out


@pytest.mark.parametrize("epi", [0, 1])
def test_every_stage_wait_holds_by_itself(device_object, epi):
    """A stage is three direct-to-LDS loads of a wave.  Behind a barrier the waves read the stage that was requested before the last one
    (behind the first barrier: two before).  So the wait in front of the barrier may leave at most as many loads outstanding as were
    issued, on any path, behind that stage's third load."""
    code = instructions(device_object, epi)
    at = {a: i for i, (a, _, _) in enumerate(code)}
    barriers = [i for i, (_, t, _) in enumerate(code) if t.startswith("s_barrier")]
    assert len(barriers) >= 4
    # (loads of the stage begun, loads behind the last stage, behind the one before, behind the one before that, nothing of LDS in flight):
    # the least over the paths
    state, work = {0: (0, 0, 0, 0, True)}, [0]
    while work:
        i = work.pop()
        ph, *y, clean = state[i]
        text = code[i][1]
        if re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", text):
            y = [min(v + 1, 64) for v in y]
        if "_load_lds_" in text:
            ph, clean = ph + 1, False
            if ph == 3:
                ph, y = 0, [0, y[0], y[1]]
        if re.search(r"vmcnt\(0\)", text):
            clean = True
        nxt = [] if text.startswith(("s_endpgm", "s_branch")) else [i + 1]
        if code[i][2] is not None:
            nxt.append(at[code[i][2]])
        for k in nxt:
            new = (ph, *y, clean)
            if k in state:
                assert state[k][0] == ph, "a stage's loads are cut by a branch"
                new = (ph, *map(min, y, state[k][1:4]), clean and state[k][4])
            if state.get(k) != new:
                state[k] = new
                work.append(k)
    for i in barriers:
        _, _, before, before2, clean = state[i]
        if clean:
            continue
        wait = re.match(r"s_waitcnt vmcnt\((\d+)\)", code[i - 1][1])
        assert wait, code[i - 1]
        behind = before2 if i == barriers[0] else before
        assert int(wait.group(1)) <= behind, f"{code[i][0]:#x}: {wait.group(1)} loads may be outstanding, {behind} were issued behind the stage"
