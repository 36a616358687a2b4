"""The kernels that keep copies in flight through a loop of matrix instructions spill nothing
inside it: a reload from scratch memory waits for every copy issued before it."""
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build():
    spec = importlib.util.spec_from_file_location("hy3moe_build", os.path.join(ROOT, "hunyuan-image-3-80b.cpp_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _loops(asm):
    """{(kernel, loop header): lines} of the innermost loops of every function."""
    out, name, header = {}, None, None
    for line in asm.splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            name, header = m.group(1), None
        elif re.match(r"(\.LBB\d+_\d+:|; %bb\.\d+:)", line):  # a new basic block
            if "Inner Loop Header" in line:
                header = re.match(r"\.L(BB\d+_\d+)", line).group(1)
            else:
                m = re.search(r"in Loop: Header=(BB\d+_\d+)", line)
                header = m.group(1) if m else None
        if name and header:
            out.setdefault((name, header), []).append(line)
    return out


@pytest.mark.parametrize("src", ["hy_mfma", "hy_mfma_few", "hy_mfma_f32", "hy_gemm", "hy_flash"])
def test_no_scratch_in_matrix_loops(src, tmp_path):
    b = _build()
    asm = tmp_path / "k.s"
    subprocess.run([b.hipcc(), *b.COMMON, *b.DEVICE, "--cuda-device-only", "-S", os.path.join(b.CSRC, src + ".hip"),
                    "-o", str(asm)], check=True, capture_output=True)
    loops = {k: v for k, v in _loops(asm.read_text()).items() if any("v_mfma" in l for l in v)}
    assert loops
    bad = {k: [l.strip() for l in v if "scratch_" in l] for k, v in loops.items()}
    assert not {k: v for k, v in bad.items() if v}
