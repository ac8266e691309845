# SPDX-License-Identifier: MPL-2.0
"""The persistent decode step's kernel on the CPU, wave by wave: its residual stream and KV cache must be the same
bits whichever wave of whichever workgroup runs last (persist_cpu.cpp), so that no two waves meet in LDS without a
barrier between them.  Parity is by the kernel's own in-order run; the GPU tests compare that with the oracle."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "bare.metal_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"

pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang++")


def _host_source(text):
    """Device source for the host: LDS arrays from the harness, no asm statements (all are empty)."""
    text = re.sub(r"__shared__ (?:__attribute__\(\(aligned\(16\)\)\) )?(\w+) (\w+)\[([^;]*)\];",
                  r"\1* \2 = (\1*)emu::lds(#\2, sizeof(\1) * (\3));".replace("#\\2", '"\\2"'), text)
    text = re.sub(r"__shared__ (\w+) (\w+);", r'\1& \2 = *(\1*)emu::lds("\2", sizeof(\1));', text)
    assert "__shared__" not in text
    assert all(a.startswith('""') for a in re.findall(r"\basm(?: volatile)?\((.*)", text))
    return re.sub(r"\basm(?: volatile)?\([^;]*\);", ";", text)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("persist_cpu")
    for src, dst in (("decode_persist.hip", "decode_persist.cpp"), ("q8_common.h", "q8_common.h"), ("bmk.h", "bmk.h"),
                     ("decode_state.h", "decode_state.h")):
        with open(os.path.join(CSRC, src)) as f:
            (d / dst).write_text(_host_source(f.read()))
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text("")
    exe = d / "persist_cpu"
    r = subprocess.run([CLANG, "-std=c++17", "-O2", "-mfma", "-mavx2", "-w", "-I", str(d),
                        os.path.join(HERE, "persist_cpu.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return str(exe)


# (sequences, query heads, KV heads, position): eight heads on two, whose merge shares end with a head; SmolLM2-135M's
# heads, one and two sequences; a position in the second 64-key sub-chunk of every piece
@pytest.mark.parametrize("nb,nh,nkv,pos", [(1, 8, 2, 20), (1, 9, 3, 20), (2, 9, 3, 20), (2, 6, 2, 5), (1, 4, 1, 700)])
def test_result_does_not_depend_on_wave_order(program, nb, nh, nkv, pos):
    n = min(8, os.cpu_count() or 1)
    runs = [subprocess.Popen([program, str(nb), str(nh), str(nkv), str(pos), str(k), str(n)], stdout=subprocess.PIPE,
                             stderr=subprocess.STDOUT, text=True) for k in range(n)]
    outs = [r.communicate(timeout=600)[0] for r in runs]
    assert all(r.returncode == 0 for r in runs), "".join(outs)[-2000:]
    assert sum(int(o.split("runs ")[1].split()[0]) for o in outs) == 128
