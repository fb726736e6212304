"""Loads that the kernels issue by inline asm: the compiler takes their output
registers as written at once, so it may reuse one while its load is in flight
unless the source keeps the value alive up to a wait that covers the load. This
compiles the tile kernels to gfx950 assembly and follows every path: no
instruction touches a register whose load may still be outstanding.

Counted: vmcnt retires in issue order, each vector-memory instruction is one.
Branches on a flag that the path itself set to a constant (the loop's exits)
are followed one way only."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "unlimited-ocr.cpp_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _vregs(text):
    out = set()
    for a, b, c in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        out |= {int(c)} if c else set(range(int(a), int(b) + 1))
    return out


def _functions(asm):
    """{name: (instructions, {label: index})}"""
    out, name = {}, None
    for line in asm.split("\n"):
        line = line.split(";")[0].split("//")[0].rstrip()
        m = re.match(r"^(\.?\w+):", line)
        if m and m[1].startswith("_Z"):
            name = m[1]
            out[name] = ([], {})
        elif m and m[1].startswith(".Lfunc_end"):
            name = None
        elif name and m:
            out[name][1][m[1]] = len(out[name][0])
        elif name and line.strip() and not line.strip().startswith("."):
            out[name][0].append(line.strip())
    return out


def in_flight_uses(ins, labels):
    """Instructions that touch a VGPR with an outstanding load: [(index, text)]."""
    found, seen = {}, set()
    work = [(0, (), frozenset([("exec", -1)]))]
    while work:
        pc, queue, consts = work.pop()
        while pc < len(ins):
            if (pc, queue, consts) in seen:
                break
            seen.add((pc, queue, consts))
            assert len(seen) < 2_000_000, "state space"
            text = ins[pc]
            op, _, rest = text.partition(" ")
            args = [a.strip() for a in rest.split(",")]
            if op == "s_endpgm":
                break
            if op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", text)
                if m:
                    n = int(m[1])
                    queue = queue[max(0, len(queue) - n):] if n else ()
            elif op == "s_branch":
                pc = labels[args[0]]
                continue
            elif op.startswith("s_cbranch_"):
                known = dict(consts).get("vcc" if "vcc" in op else "exec" if "exec" in op else None)
                taken = None if known is None else (known != 0) == op.endswith("nz")
                if taken is not False:
                    if taken:
                        pc = labels[args[0]]
                        continue
                    work.append((labels[args[0]], queue, consts))
            else:
                used = _vregs(rest)
                if any(d & used for d in queue):
                    found[pc] = text
                c = dict(consts)
                # exec: some lane is on at the entry and after a region's end
                # (s_or_b64 exec, exec, saved), unknown inside one
                if "saveexec" in op:
                    c.pop("exec", None)
                elif args[0] == "exec":
                    c.pop("exec", None)
                    if op == "s_or_b64" or args[1:] == ["-1"]:
                        c["exec"] = -1
                # lane masks that are a constant: s_mov_b64 p, 0 / -1 and vcc = exec & [~]p
                if op == "s_mov_b64" and args[1] in ("0", "-1"):
                    c[args[0]] = int(args[1])
                elif op in ("s_and_b64", "s_andn2_b64") and args[:2] == ["vcc", "exec"] and args[2] in c:
                    c["vcc"] = c[args[2]] if op == "s_and_b64" else ~c[args[2]]
                elif args[0] != "exec" and not op.startswith(("s_cmp", "s_bitcmp", "s_barrier", "s_nop")):
                    c.pop(args[0], None)
                    if "vcc" in rest.split(",")[0] or op.endswith("_e32") and op.startswith("v_cmp"):
                        c.pop("vcc", None)
                    m = re.match(r"s\[?(\d+)(?::(\d+))?\]?$", args[0])  # a write of part of a known pair
                    if m:
                        lo, hi = int(m[1]), int(m[2] or m[1])
                        for k in [k for k in c if k[0] == "s"]:
                            a, b = map(int, re.match(r"s\[(\d+):(\d+)\]", k).groups())
                            if a <= hi and lo <= b:
                                c.pop(k)
                consts = frozenset(c.items())
                if re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", op):
                    dst = frozenset(_vregs(args[0])) if "_load" in op and "lds" not in text else frozenset()
                    queue = (queue + (dst,))[-64:]
            pc += 1
    return sorted(found.items())


def test_a_register_reused_under_its_load_is_seen():
    ins = ["global_load_dword v1, v[2:3], off", "s_mov_b64 s[0:1], -1", "s_and_b64 vcc, exec, s[0:1]",
           "s_cbranch_vccnz .E", "v_mov_b32_e32 v1, 0", "v_mov_b32_e32 v4, 0", "s_waitcnt vmcnt(0)",
           "v_mov_b32_e32 v1, 0", "s_endpgm"]
    assert in_flight_uses(ins, {".E": 5}) == []
    assert in_flight_uses(ins, {".E": 4}) == [(4, "v_mov_b32_e32 v1, 0")]
    ins[0:0] = ["global_load_dword v9, v[2:3], off"]
    assert in_flight_uses(ins[:2] + ["s_waitcnt vmcnt(1)", "v_mov_b32_e32 v9, 0", "s_endpgm"], {}) == []


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("unit", ["experts_tile_gu_z0", "experts_tile_gu_z1", "experts_tile_dn_z0", "experts_tile_dn_z1"])
def test_no_register_of_a_load_in_flight_is_touched(unit, tmp_path):
    out = tmp_path / f"{unit}.s"
    # (the Makefile's flags; the expf table header is a build product)
    subprocess.run(["make", "-s", "../_build/expf_exceptions.h"], cwd=CSRC, check=True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I../../include", "-I.", "-I../_build", "-S",
                    "--cuda-device-only", f"{unit}.hip", "-o", str(out)], cwd=CSRC, check=True, capture_output=True)
    kernels = {n: f for n, f in _functions(out.read_text()).items() if "int4_tile_kernel" in n}
    assert len(kernels) == 6
    for name, (ins, labels) in kernels.items():
        assert sum(i.startswith("global_load") for i in ins) > 20, name
        bad = in_flight_uses(ins, labels)
        assert not bad, (name, bad[:4])
