"""The register-weight GEMM items (kern_k3h_moe_gemm3_*) wait for their loads by count, so a
K step that meets at a barrier under a counted wait has to issue every load the count
assumes: a load the compiler drops (its data unused past the last step) would let the wait
pass before the activation rows that the other waves read have landed.  Checked on the CPU
in the built code object: the listing's loads between barriers."""
import os
import re
import subprocess

import pytest

import k3h

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
ENTRIES = ("kern_k3h_moe_gemm3_situ_mx", "kern_k3h_moe_gemm3_acc", "kern_k3h_moe_gemm3_bf16")


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """Entry name -> its instructions, in address order."""
    tools = [os.path.join(LLVM, t) for t in ("clang-offload-bundler", "llvm-objdump")]
    if not all(os.path.exists(t) for t in tools):
        pytest.skip("no LLVM tools to list the built code object with")
    obj = str(tmp_path_factory.mktemp("waits") / "gemm.o")
    subprocess.run([tools[0], "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    f"--input={os.path.join(k3h.BUILD, 'k3h_moe_gemm.hsaco')}", f"--output={obj}"],
                   check=True)
    text = subprocess.run([tools[1], "-d", "--no-show-raw-insn", obj], check=True,
                          stdout=subprocess.PIPE, text=True).stdout
    out = {}
    for line in text.splitlines():
        m = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if m:
            cur = out.setdefault(m.group(1), [])
        elif line.startswith("\t"):
            cur.append(line.split("//")[0].strip())
    return out


def _segments(ins):
    """Per barrier, what comes between it and the one before: the loads into LDS, the loads
    into registers and the MFMAs up to its last vector-memory wait, and that wait's count;
    and the loads that follow it before the next wait, branch or barrier."""
    segs, lds, reg, mfma, wait = [], 0, 0, 0, None
    after = None
    for s in ins:
        load = re.match(r"(global|buffer)_load", s)
        if load and "lds" in s.split()[0]:
            lds += 1
        elif load:
            reg += 1
        elif s.startswith("v_mfma"):
            mfma += 1
        elif s.startswith(("s_cbranch", "s_branch")):
            after = None
        elif "vmcnt(" in s:
            after = None
            wait = int(re.search(r"vmcnt\((\d+)\)", s).group(1))
        elif s.startswith("s_barrier"):
            after = [0, 0]
            segs.append((lds, reg, mfma, wait, after))
            lds = reg = mfma = 0
            wait = None
        if load and after is not None:
            after[0] = lds
            after[1] = reg
    return segs


@pytest.mark.parametrize("entry", ENTRIES)
def test_counted_waits_count_issued_loads(listing, entry):
    segs = _segments(listing[entry])
    loops = []  # runs of counted barriers: a K loop's steps
    prev = False
    for lds, reg, mfma, wait, after in segs:
        counted = bool(wait)
        if counted and (not prev or reg == 2):
            loops.append([])
        if counted:
            loops[-1].append((lds, reg, mfma, wait, after))
        prev = counted
    assert loops
    for steps in loops:
        first, mt = steps[0], steps[0][2] // 2
        # the loop's first barrier: two of the five register loads, none of the LDS loads
        assert mt in (1, 2, 4) and first[:2] == (0, 2), steps
        for lds, reg, mfma, wait, _ in steps[1:]:
            assert (lds, reg, mfma) == (mt, 5, 4 * mt), f"m tiles {mt}: a step issues {lds} + {reg} loads"
        # the turn's last step: its loads are issued before the branch back
        assert steps[-1][4] == [mt, 3], steps
        # its own second weights are among the loads of len(steps) - 1 whole steps and two
        assert {w for *_, w, _ in steps} == {first[3]} and first[3] <= 2 + (len(steps) - 1) * (5 + mt)
    assert sorted(s[0][2] // 2 for s in loops) == [1, 1, 2, 2, 4, 4]


@pytest.mark.parametrize("entry", ENTRIES)
def test_every_tile_height_has_both_weight_policies(listing, entry):
    """Non-temporal weights up to 1.25 tiles per expert, cacheable ones above, for tiles of
    one, two and four m tiles alike."""
    bodies, mfma, loads, nt = set(), 0, 0, 0
    for s in listing[entry]:
        if s.startswith("v_mfma"):
            mfma += 1
        elif s.startswith("global_load_dwordx4"):
            loads += 1
            nt += s.endswith(" nt")
        elif s.startswith("s_barrier"):
            if mfma in (4, 8, 16) and loads == 4:  # a whole step of the K loop
                bodies.add((mfma // 4, nt > 0))
            mfma = loads = nt = 0
    assert bodies == {(mt, policy) for mt in (1, 2, 4) for policy in (False, True)}, bodies
