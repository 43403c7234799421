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


def test_barriers_of_the_awq_gemm_leave_out_block_loads_only(tmp_path):
    from nunchaku_rocm_amd import build

    try:
        cmd = [build.hipcc(), *build.FLAGS]
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "awq_gemm.s"
    subprocess.run([*cmd, "-S", "--cuda-device-only", os.path.join(build.CSRC, "awq_gemm.hip"), "-o", str(out)], check=True, capture_output=True)
    kernels = {name: ev for name, ev in _events(out.read_text()).items() if "awq_gemm_kernel" in name}
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
