"""The prompt-pass kernels read LDS with loads issued from inline asm, some of them one step ahead of the
wait that retires them.  The compiler believes an asm statement's outputs valid as soon as the statement
ends, so until that wait nothing may touch the registers such a read targets.  This test compiles
the sources to assembly and walks the generated code: LDS reads complete in order, `s_waitcnt
lgkmcnt(N)` leaves at most the N newest under way, and no instruction in between may name a register
that a read still under way writes."""
import os
import re
import shutil
import subprocess

import pytest

from test_flow_asm import CSRC, ROOT, _regs


def _scan(path):
    bad, fn, pending, n_ahead = [], None, [], 0   # pending: [(line, regs)] oldest first
    for ln, line in enumerate(open(path), 1):
        t = line.strip()
        m = re.match(r"^(_Z\w+):", t)
        if m:
            fn, pending = m.group(1), []
        if not t or t[0] in ";.":
            continue
        if t.startswith("s_waitcnt"):
            m = re.search(r"lgkmcnt\((\d+)\)", t)
            if m:
                n = int(m.group(1))
                pending = pending[len(pending) - n:] if n else []
            continue
        live = set().union(*[r for _, r in pending]) if pending else set()
        if t.startswith("ds_read_b128"):
            ops = t.split(None, 1)[1].split(",")
            dst, rest = _regs(ops[0]), _regs(",".join(ops[1:]))
            hit = (dst | rest) & live
            if hit:
                bad.append((fn, ln, t, sorted(hit)))
            if pending:
                n_ahead += 1
            pending.append((ln, dst))
            continue
        hit = _regs(t) & live
        if hit:
            bad.append((fn, ln, t, sorted(hit)))
    return bad, n_ahead


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
@pytest.mark.parametrize("source", ["k_prefill", "k_tiles"])
def test_no_register_of_a_pending_lds_read_is_touched(tmp_path, source):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = tmp_path / (source + ".s")
    cmd = [hipcc, "-S", "--cuda-device-only", os.path.join(CSRC, source + ".hip"), "-o", str(out), "--offload-arch=gfx950",
           "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I", os.path.join(ROOT, "include"), "-I", CSRC]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    bad, n_ahead = _scan(str(out))
    assert n_ahead > 0, "no LDS reads issued ahead of a wait found: has the kernel changed?"
    assert not bad, bad[:5]


def _functions(path):
    """(name, [(line, instruction)], label -> index) of every kernel in an assembly file"""
    fn, body, labels = None, [], {}
    for ln, line in enumerate(open(path), 1):
        t = line.split(";")[0].strip()
        m = re.match(r"^(_Z\w+):", t)
        label = re.match(r"^(\.LBB\w+):", t)
        if m or t.startswith(".Lfunc_end"):
            if fn:
                yield fn, body, labels
            fn, body, labels = m.group(1) if m else None, [], {}
        elif label:
            labels[label.group(1)] = len(body)
        elif fn and t and t[0] != ".":
            body.append((ln, t))
    if fn:
        yield fn, body, labels


def _scan_paths(path):
    """The same along every path through the code, jumps taken and not, and how many jumps back a read is under way across"""
    bad, carried = [], 0
    for fn, body, labels in _functions(path):
        seen, work = [set() for _ in body], [(0, ())]
        while work:
            i, pending = work.pop()  # pending: registers of each read under way, oldest first
            while i < len(body) and pending not in seen[i]:
                seen[i].add(pending)
                assert len(seen[i]) <= 64, "reads pile up in %s" % fn
                ln, t = body[i]
                op = t.split()[0]
                live = set().union(*pending)
                i += 1
                if op == "s_waitcnt":
                    m = re.search(r"lgkmcnt\((\d+)\)", t)
                    if m:
                        pending = pending[max(0, len(pending) - int(m.group(1))):]
                elif op == "s_endpgm":
                    break
                elif op == "s_branch" or op.startswith("s_cbranch"):
                    to = labels[t.split()[1]]
                    carried += bool(pending) and to < i
                    if op == "s_branch":
                        i = to
                    else:
                        work.append((to, pending))
                else:
                    hit = _regs(t) & live
                    if hit:
                        bad.append((fn, ln, t, sorted(hit)))
                    if op == "ds_read_b128":
                        pending += (frozenset(_regs(t.split(None, 1)[1].split(",")[0])),)
    return bad, carried


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
@pytest.mark.parametrize("source", ["k_prefill", "k_tiles"])
def test_reads_under_way_across_a_jump(tmp_path, source):
    """The first reads of a stage are under way when the product loop jumps back: the registers are followed along the jumps too."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = tmp_path / (source + ".s")
    cmd = [hipcc, "-S", "--cuda-device-only", os.path.join(CSRC, source + ".hip"), "-o", str(out), "--offload-arch=gfx950",
           "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I", os.path.join(ROOT, "include"), "-I", CSRC]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    bad, carried = _scan_paths(str(out))
    assert carried > 0, "no read is under way across a jump back: has the loop changed?"
    assert not bad, bad[:5]
