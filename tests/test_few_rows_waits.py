"""The few-row kernel's stage hand-over in compiled code, on the CPU.

A block's weight pieces are direct-to-LDS loads that other waves read after the
next barrier, so each wave must have waited for its own. It waits until at most
n of its loads are in flight, n being what the step before issued after them;
loads of a value that nothing reads are not in the compiled code, and a count
that includes them lets a block's own pieces still be in flight.
"""

from __future__ import annotations

import re
import subprocess

import pytest

import helpers

HIPCC = "/opt/rocm/bin/hipcc"


def hand_overs(body):
    """(fewest loads issued since the barrier before on any path, vmcnt allowed) of each
    barrier that an explicit wait leads up to."""
    at = {m.group(1): i for i, m in enumerate(re.match(r"(\.LBB\w+):", s) for s in body) if m}
    best, found, todo = {}, {}, [(0, 0, None)]
    while todo:
        i, issued, allowed = todo.pop()
        while i < len(body):
            if best.get((i, allowed), issued + 1) <= issued:
                break
            best[i, allowed] = issued
            s = body[i]
            op = s.split()[0] if s.split() else ""
            if re.match(r"(global|buffer)_load_", op):
                issued, allowed = issued + 1, None
            elif op == "s_waitcnt" and "vmcnt" in s:
                allowed = int(re.search(r"vmcnt\((\d+)\)", s).group(1))
            elif op == "s_barrier":
                if allowed is not None:
                    found[i] = min(found.get(i, (issued, allowed)), (issued, allowed))
                issued, allowed = 0, None
            elif op.startswith("s_cbranch"):
                todo.append((at[s.split()[1]], issued, allowed))
            elif op == "s_branch":
                i = at[s.split()[1]]
                continue
            elif op == "s_endpgm":
                break
            i += 1
    return [found[i] for i in sorted(found)]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "few_rows.s"
    csrc = helpers.PKG_DIR / "csrc"
    subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", f"-I{helpers.REPO / 'include'}", f"-I{csrc}", "-x", "hip",
         "--cuda-device-only", "-S", str(csrc / "kernels" / "few_rows.hip"), "-o", str(out)],
        check=True, capture_output=True, timeout=300)
    return {m.group(1): [s.strip() for s in m.group(2).splitlines()]
            for m in re.finditer(r"^(_Z\S*few_rows_nk_kernel\S*):(.*?)^\.Lfunc_end", out.read_text(),
                                 re.M | re.S)}


def test_every_hand_over_waits_for_the_block_it_hands_over(kernels):
    assert len(kernels) == 12, sorted(kernels)  # 3 row counts x 1 or 2 m-blocks x gain or none
    for name, body in kernels.items():
        steps = hand_overs(body)
        assert len(steps) >= 6, name  # three in the loop, three in the tail
        for i, (issued, allowed) in enumerate(steps):
            assert allowed <= issued, f"{name}, step {i}: {issued} loads issued, {allowed} allowed in flight"
