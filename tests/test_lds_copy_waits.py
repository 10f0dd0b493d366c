"""CPU check of the waits around direct memory -> LDS copies, on the gfx950
assembly the compiler writes for this repository's kernels.

global_load_lds counts in vmcnt and writes LDS behind the compiler's back: it
knows of no conflict between such a copy and an LDS read issued before it, so
it places no lgkmcnt wait between the two, and gfx950's s_barrier implies
none. A kernel that copies into a stage it has read must have those reads
complete: at the barrier in front of the copies (tile product, stages shared by
the block) or at the copies themselves (rings of one wave).

The check walks each kernel's control flow with the queue of LDS operations
that a wave may still have in flight (they return in order; lgkmcnt(n) leaves
the last n).
"""
import re

import pytest

from logan_amd import build

from _asm import compiled


def _kernels(name: str, pattern: str):
    """{mangled name: instruction and label lines} of the kernels matching."""
    out = compiled(name)[0]
    found, cur = {}, None
    with open(out) as f:
        for line in f:
            m = re.match(r"(_ZN\S+):", line)
            if m:
                cur = found.setdefault(m[1], []) if re.search(pattern, m[1]) else None
            elif line.startswith(".Lfunc_end"):
                cur = None
            elif cur is not None:
                cur.append(line.split(";")[0].rstrip())
    return found


def _blocks(lines):
    blocks, labels, cur = [], {}, []
    for line in lines:
        m = re.match(r"(\.L\S+):", line)
        if m:
            blocks.append(cur)
            cur = []
            labels[m[1]] = len(blocks)
            continue
        t = line.strip()
        if not t or t.startswith("."):
            continue
        cur.append(t)
        if t.startswith(("s_branch", "s_cbranch", "s_endpgm")):
            blocks.append(cur)
            cur = []
    blocks.append(cur)
    succ = []
    for i, b in enumerate(blocks):
        last = b[-1].split() if b else [""]
        nxt = [] if last[0] in ("s_branch", "s_endpgm") else [i + 1]
        if last[0].startswith(("s_branch", "s_cbranch")):
            nxt.append(labels[last[1]])
        succ.append([s for s in nxt if s < len(blocks)])
    return blocks, succ


def reads_in_flight(lines, at):
    """The most LDS reads a wave may have in flight where an instruction
    starting with `at` issues, and how many such instructions there are."""
    blocks, succ = _blocks(lines)
    seen = [set() for _ in blocks]
    seen[0].add(())
    work, most, sites = [0], 0, set()
    while work:
        i = work.pop()
        outs = set()
        for state in seen[i]:
            q = list(state)  # True: a read, False: another LDS operation
            for n, t in enumerate(blocks[i]):
                op = t.split()[0]
                if op.startswith(at):
                    sites.add((i, n))
                    most = max(most, sum(q))
                if op.startswith("ds_"):
                    q.append(op.startswith("ds_read"))
                m = re.search(r"lgkmcnt\((\d+)\)", t) if op == "s_waitcnt" else None
                if m:
                    q = q[len(q) - min(int(m[1]), len(q)):]
            outs.add(tuple(q))
        for s in succ[i]:
            if not outs <= seen[s]:
                seen[s] |= outs
                assert len(seen[s]) < 2000
                work.append(s)
    return most, len(sites)


@pytest.fixture
def hipcc():
    try:
        return build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")


def test_the_walk_itself():
    """A read in flight at a barrier reached through a loop's back edge only."""
    code = ["s_barrier", ".LBB0_1:", "ds_read_b32 v1, v2", "s_waitcnt lgkmcnt(1)", "s_cbranch_scc1 .LBB0_3",
            ".LBB0_2:", "s_waitcnt vmcnt(0) lgkmcnt(0)", ".LBB0_3:", "s_barrier", "s_cbranch_scc0 .LBB0_1",
            "s_endpgm"]
    assert reads_in_flight(code, "s_barrier") == (1, 2)
    code[3] = "s_waitcnt lgkmcnt(0)"
    assert reads_in_flight(code, "s_barrier") == (0, 2)


def test_qmm_tile_reads_complete_at_the_barriers(hipcc):
    """Of the tile product's LDS reads only the last ones, the MI reads of the
    next slice's x operands, may be in flight at a barrier: the copies behind
    it overwrite the codes just read, and x of a step before those."""
    ks = _kernels("gemm.hip", "affine_qmm_tile_kernel")
    assert ks
    bad = {}
    for name, lines in ks.items():
        mi = int(re.search(r"ILi\dELi(\d+)E", name)[1])
        most, sites = reads_in_flight(lines, "s_barrier")
        assert sites >= 5, name
        if most > mi:
            bad[name] = most
    assert not bad


def test_moe_ring_reads_complete_at_the_copies(hipcc):
    """A wave's reads of its ring complete before it copies the next batch
    into the slot it has read."""
    ks = _kernels("moe_mfma.hip", "(lds|wide)_kernel")
    assert ks
    bad = {}
    for name, lines in ks.items():
        most, sites = reads_in_flight(lines, "global_load_lds")
        assert sites, name
        if most:
            bad[name] = most
    assert not bad
