"""The order of the histogram's memory operations, in the gfx950 code compiled from its source (no GPU runs here)."""

import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def count_kernels(tmp_path_factory):
    """The instructions of every instantiation of count_kernel, comments taken off."""
    spec = importlib.util.spec_from_file_location("ck_build", os.path.join(ROOT, "cute-kernels_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    out = tmp_path_factory.mktemp("assembly") / "count_sort.s"
    subprocess.run(
        [build.HIPCC, *build.COMMON_FLAGS, *build.DEVICE_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "count_sort.hip"),
         "-o", str(out)],
        check=True, capture_output=True,
    )
    kernels, name = {}, None
    for line in out.read_text().splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            name = label[1]
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name is not None and "count_kernel" in name and line.startswith("\t") and not line.startswith("\t."):
            kernels.setdefault(name, []).append(line.split(";")[0].strip())
    return kernels


def test_a_block_takes_its_ticket_behind_its_own_atomics(count_kernels):
    """The block that takes the last ticket reads what the others added to the accumulators. Their additions return nothing and
    s_barrier waits for none of them: every wave has to wait for its own between the additions and the barrier."""
    assert len(count_kernels) == 8  # ids of 32 and 64 bits, counters in registers and in LDS, 512 and 1,024 threads
    for name, code in count_kernels.items():
        additions = [i for i, line in enumerate(code) if line.startswith("global_atomic_add") and not line.endswith("sc0")]
        assert additions, name
        barrier = next(i for i in range(additions[-1], len(code)) if code[i] == "s_barrier")
        tickets = [i for i, line in enumerate(code) if line.startswith("global_atomic_add") and line.endswith("sc0")]
        assert tickets and min(tickets) > barrier, name
        assert any("vmcnt(0)" in line for line in code[additions[-1] : barrier]), name
