"""Wait states that the hardware does not enforce and the compiler's hazard pass cannot add inside inline assembly: on
gfx950 a scalar write of M0 needs one instruction (or s_nop) between it and a load into LDS that takes its address from M0.
Read from the assembly that this repository's own sources compile to."""
import os
import re
import subprocess

import pytest

from diffractom_amd import build as b

SOURCES = [s for s in b.SOURCES if "load_lds" in (b.CSRC / s).read_text()]


def _device_assembly(source, tmp_path):
    out = tmp_path / "device.s"
    try:
        hipcc = b.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not found")
    subprocess.run([hipcc, f"--offload-arch={b.ARCH}", "-O3", "-std=c++17", "--offload-device-only", "-S", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(b.PKG.parent / "include"),
                    str(b.CSRC / source), "-o", str(out)], check=True, stderr=subprocess.DEVNULL, env=dict(os.environ))
    return out.read_text()


def test_sources_with_lds_loads():
    assert SOURCES == ["radon_lines.hip"]


@pytest.mark.parametrize("source", SOURCES)
def test_wait_state_between_m0_write_and_lds_load(source, tmp_path):
    ins = [line.split(";")[0].strip() for line in _device_assembly(source, tmp_path).splitlines()]
    ins = [i for i in ins if i and not i.startswith(".") and not i.endswith(":")]
    loads = [k for k, i in enumerate(ins) if re.match(r"(global|buffer)_load_lds", i)]
    assert loads
    for k in loads:
        assert not re.match(r"s_\w+ m0,", ins[k - 1]), f"{ins[k - 1]} / {ins[k]}"
