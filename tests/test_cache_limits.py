"""The sizes from which buffers bypass the caches (fcqt_abi_internal.hpp), per
layout: the lines lie where the measurements beside them put them."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
NCOEF = (132992, 99072)          # (3, 4, 2) x (8, 16, 32) and (4, 3) x (12, 48)


def _first(tmp_path, rule):
    """First batch of each layout at which `rule` (an expression of batch and ncoef) holds."""
    src = tmp_path / "limits.cpp"
    src.write_text('#include <cstdint>\n#include <cstdio>\n#include "fcqt_abi_internal.hpp"\nusing namespace fcqt;\n'
                   "int main() {\n    for (int64_t ncoef : {%s}) {\n        int64_t batch = 1;\n"
                   "        while (!(%s)) ++batch;\n        printf(\"%%ld\\n\", (long)batch);\n    }\n}\n"
                   % (", ".join(map(str, NCOEF)), rule))
    exe = tmp_path / "limits"
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'flash-cqt_amd' / 'csrc'}", str(src), "-o", str(exe), "-L/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath,/opt/rocm/lib"], check=True, timeout=300)
    return tuple(map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split()))


@pytest.mark.parametrize("rule,first", [("stream_planes_in(batch, ncoef)", (140, 165)),
                                        ("stream_planes_out(batch, ncoef)", (192, 224))])
def test_first_batch_past_the_caches(tmp_path, rule, first):
    assert _first(tmp_path, rule) == first
