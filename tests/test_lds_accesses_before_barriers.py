"""No kernel may reach a barrier with an LDS access of its own outstanding: behind the barrier another wave is free to write what
a read has yet to fetch, and to read what a write has yet to leave.  A release fence says so in the source, but the compiler drops
the wait where the accesses reach the barrier over a loop's back edge, so the compiled kernels themselves are followed: every .hip
source is compiled to assembly with the library's own flags, and the youngest LDS access that may be outstanding is carried along
every path of the control flow."""
import concurrent.futures
import os
import re
import subprocess

import pytest

from pypto_amd import build

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
KERNELS = [s for s in build.SOURCES if s.endswith(".hip")]
NONE = 64  # more than the counter holds: nothing is outstanding
PERMUTES = ("ds_permute", "ds_bpermute", "ds_swizzle")  # among the lanes: no memory


def outstanding_at_barriers(body):
    """[(block, instruction)] of the barriers that a path reaches with an LDS access outstanding."""
    names, blocks = ["entry"], {"entry": []}
    for line in body.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"(\.LBB\w+):", line)
        if label:
            names.append(label.group(1))
            blocks[names[-1]] = []
        elif line and not line.startswith("."):
            blocks[names[-1]].append(line)
    after = {"entry": NONE}  # LDS operations issued since the youngest access that may be outstanding, at a block's start
    todo, found = ["entry"], set()
    while todo:
        name = todo.pop()
        d, ends = after[name], []
        for i, ins in enumerate(blocks[name]):
            op = ins.split()[0]
            if op.startswith(PERMUTES):
                d = min(d + 1, NONE)
            elif op.startswith("ds_"):  # (scalar loads overtake, and count for none)
                d = 0
            elif op == "s_waitcnt":
                assert re.fullmatch(r"s_waitcnt( (lgkmcnt|vmcnt|expcnt)\(\d+\))+", ins), ins
                left = re.search(r"lgkmcnt\((\d+)\)", ins)
                if left and d >= int(left.group(1)):
                    d = NONE
            elif op == "s_barrier":
                if d < NONE:
                    found.add((name, i))
            elif op.startswith("s_cbranch"):
                ends.append((ins.split()[1], d))
            elif op == "s_branch":
                ends.append((ins.split()[1], d))
                break
            elif op in ("s_endpgm", "s_setpc_b64"):
                break
        else:
            at = names.index(name) + 1
            if at < len(names):
                ends.append((names[at], d))
        for to, d in ends:
            if d < after.get(to, NONE + 1):
                after[to] = d
                todo.append(to)
    return sorted(found)


def functions(asm):
    return re.findall(r"^(\w+):\s*; @\S+\n(.*?)^\.Lfunc_end\d+:", asm, re.S | re.M)


@pytest.mark.parametrize("access", ["ds_read_b32 v2, v0", "ds_write_b32 v0, v1", "ds_add_u32 v0, v1"])
def test_the_check_follows_accesses_over_a_back_edge(access):
    loop = ".LBB0_1:\n {}\n s_barrier\n " + access + "\n s_cbranch_scc1 .LBB0_1\n s_waitcnt lgkmcnt(0)\n s_endpgm\n"
    assert outstanding_at_barriers(loop.format("v_nop")) == [(".LBB0_1", 1)]
    assert outstanding_at_barriers(loop.format("s_waitcnt lgkmcnt(1)")) == [(".LBB0_1", 1)]
    assert outstanding_at_barriers(loop.format("s_waitcnt vmcnt(3) lgkmcnt(0)")) == []
    permute = loop.replace("s_cbranch", "ds_bpermute_b32 v4, v3, v3\n s_cbranch")
    assert outstanding_at_barriers(permute.format("s_waitcnt lgkmcnt(1)")) == []


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("asm")
    flags = [f for f in build.HIPCC_FLAGS if f != "-shared"] + ["-I", build.INCLUDE, "-I", build.CSRC, "--cuda-device-only", "-S"]

    def compiled(src):
        path = out / (src + ".s")
        res = subprocess.run([HIPCC] + flags + [os.path.join(build.CSRC, src), "-o", str(path)], capture_output=True, text=True)
        assert res.returncode == 0, res.stderr
        return path.read_text()

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        return dict(zip(KERNELS, pool.map(compiled, KERNELS)))


@pytest.mark.parametrize("src", KERNELS)
def test_no_lds_access_is_outstanding_at_a_barrier(assembly, src):
    found = functions(assembly[src])
    assert found
    bad = {name: at for name, body in found if (at := outstanding_at_barriers(body))}
    assert not bad
