"""The waits in front of barriers, in the compiler's listing of the kernel: what is still in flight there is named by a count of
the youngest memory operations, so the count may cover none that the compiler is free to drop or to move."""

import os
import re
import subprocess

import pytest


def _events(listing: str) -> dict[str, list[str]]:
    """Per kernel, in the listing's order: block loads into LDS, other buffer loads, waits and barriers."""
    kernels, events = {}, None
    for line in listing.splitlines():
        text = line.strip()
        if re.match(r"_ZN\w+:", line):
            events = kernels.setdefault(line.split(":")[0], [])
        elif events is None:
            continue
        elif text.startswith("buffer_load"):
            events.append("block" if re.search(r"\blds\b", text) else "load")
        elif text.startswith("s_barrier"):
            events.append("barrier")
        elif text.startswith("s_waitcnt") and "vmcnt" in text:
            events.append(re.search(r"vmcnt\((\d+)\)", text).group(1))
        elif text.startswith("s_endpgm"):
            events = None
    return kernels


def _kernels(source: str, name: str, tmp_path) -> dict[str, list[str]]:
    from nunchaku_rocm_amd import build

    try:
        cmd = [build.hipcc(), *build.FLAGS]
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "listing.s"
    subprocess.run([*cmd, "-S", "--cuda-device-only", os.path.join(build.CSRC, source), "-o", str(out)], check=True, capture_output=True)
    return {kernel: ev for kernel, ev in _events(out.read_text()).items() if name in kernel}


def test_barriers_of_the_wide_gemm_leave_out_register_loads_only(tmp_path):
    """At a barrier of the loop a wavefront's own block loads have landed: what may still be in flight are the activations of
    the next stage's second group, 2 loads per row block, which the compiler waits for itself."""
    kernels = _kernels("gemm_w4a4_wide.hip", "gemm_w4a4_wide_kernel", tmp_path)
    assert len(kernels) == 8
    for name, events in kernels.items():
        counts = []
        for i, event in enumerate(events):
            if event == "barrier":
                waits = [j for j in range(i) if events[j].isdigit()]
                count = int(events[waits[-1]])
                issued = [e for e in events[: waits[-1]] if e in ("block", "load")]
                assert set(issued[len(issued) - count :] if count else []) <= {"load"}, (name, i)
                assert not {"block", "load"} & set(events[waits[-1] : i]), (name, i)
                counts.append(count)
        # tiles of either height: a barrier before the loop, one per stage of its body, and one with nothing in flight after it
        assert counts.count(2) == 5 and counts.count(4) == 5 and set(counts) == {0, 2, 4}, (name, counts)


def test_barriers_of_the_awq_gemm_leave_out_block_loads_only(tmp_path):
    kernels = _kernels("awq_gemm.hip", "awq_gemm_kernel", tmp_path)
    assert len(kernels) == 8
    for name, events in kernels.items():
        left_out = None  # by the latest wait
        first = True
        for i, event in enumerate(events):
            if event.isdigit():
                issued = [e for e in events[:i] if e in ("block", "load")]
                left_out = issued[len(issued) - int(event) :] if int(event) else []
            elif event == "barrier":
                assert left_out is not None and set(left_out) <= {"block"}, (name, i)
                if first:  # half of the block loads so far: the second stage's
                    assert 2 * len(left_out) == events[:i].count("block"), name
                else:
                    assert not left_out, (name, i)
                first = False
