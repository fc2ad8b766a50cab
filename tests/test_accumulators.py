"""Where the GEMMs keep their accumulators and how many registers they put in scratch, in the gfx950 code compiled from their
source (no GPU runs here)."""

import functools
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(None)
def _assembly(source):
    spec = importlib.util.spec_from_file_location("ck_build", os.path.join(ROOT, "cute-kernels_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    return subprocess.run(
        [build.HIPCC, *build.COMMON_FLAGS, *build.DEVICE_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", "-"],
        check=True, capture_output=True, text=True,
    ).stdout


def _kernels(source):
    """The instructions of every kernel of a source, comments taken off."""
    kernels, name = {}, None
    for line in _assembly(source).splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            name = label[1]
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name is not None and line.startswith("\t") and not line.startswith("\t."):
            kernels.setdefault(name, []).append(line.split(";")[0].strip())
    return kernels


@pytest.mark.parametrize("source,instantiations", [("grouped_gemm_line.hip", 20), ("grouped_gemm_fp8.hip", 6)])
def test_accumulators_stay_where_they_are_between_products(source, instantiations):
    """The products are asm to the compiler, which knows nothing of their latency: an accumulator that it moves or spills between
    two of them may be read before it is written. An instantiation that runs out of registers does that, without an error."""
    kernels = {name: code for name, code in _kernels(source).items() if re.search("gemm_(line|fp8)_kernel", name)}
    assert len(kernels) == instantiations
    for name, code in kernels.items():
        products = [i for i, line in enumerate(code) if line.startswith("v_mfma")]
        loop = code[products[0] : products[-1]]
        assert not [line for line in loop if "accvgpr" in line or re.match(r"scratch_\w+ .*\ba\[?\d", line)], name


@pytest.mark.parametrize("source,kernel,instantiations,most", [
    ("grouped_gemm_line.hip", "line", 20, 0), ("grouped_gemm_skinny.hip", "skinny", 96, 0), ("grouped_gemm_fp8.hip", "fp8", 6, 44),
])
def test_registers_in_scratch(source, kernel, instantiations, most):
    """None, but for 256-row e4m3 tiles, around the operands of their first step (the accumulators are looked at above)."""
    spills = re.findall(rf"\.symbol: +(\w*gemm_{kernel}_kernel\w*)\.kd.*?\.vgpr_spill_count: +(\d+)", _assembly(source), re.S)
    assert len(spills) == instantiations
    assert not {name: count for name, count in spills if int(count) > most}
