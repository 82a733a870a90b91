"""The reference-named C++ interface (include/mtg_reference.hpp) through the C++
test drivers in tests/cpp, built by __graft_entry__.build()."""
import glob
import json
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BIN = os.path.join(HERE, "cpp", "bin")


def _run(name, timeout):
    exe = os.path.join(BIN, name)
    if not os.path.exists(exe):
        import sys
        sys.path.insert(0, os.path.join(os.path.dirname(HERE), "moss-transcribe.cpp_amd"))
        import build
        build.build_cpp_tests()
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                       timeout=timeout)
    assert p.returncode == 0, p.stderr
    return json.loads(p.stdout.strip().splitlines()[-1])


def test_cpp_policy_controls():
    rec = _run("test_cpu_speculative", 60)
    assert rec == {"record": "speculativePolicy", "controls": 13, "passed": True}


@pytest.mark.gpu
def test_cpp_speculative_gate_on_gpu():
    print("C++ speculative gate: 2-layer q8_0 model, 40 tokens, forced rejections", flush=True)
    rec = _run("test_speculative_gate", 100)
    assert rec["passed"] and rec["tokens"] == 40


def test_erf_polynomials_round_as_the_series():
    rec = _run("test_erf_poly", 100)
    assert rec["differ"] == 0 and rec["floats"] > 17_000_000


def test_product_alone_takes_the_kernels_it_may():
    """csrc/kernels.hip launch_mul_mat on the fake HIP runtime: x and y that overlap,
    panels of which a CU holds few."""
    rec = _run("test_mul_mat_route", 60)
    assert rec == {"record": "mulMatRoute", "failures": 0}


def test_prompts_of_several_blocks_and_their_buffers():
    """The prefill's streams, copies and buffers on the fake HIP runtime, with and
    without memory for the second set of rows."""
    rec = _run("test_prefill_buffers", 60)
    assert rec == {"record": "prefillBuffers", "failures": 0}


def test_inline_asm_names_the_registers_it_writes():
    """m0 is the compiler's too (LDS addressing, indexed registers): an asm statement that
    writes it has to list it as clobbered."""
    found = 0
    for path in glob.glob(os.path.join(os.path.dirname(HERE), "moss-transcribe.cpp_amd", "csrc", "*.h*")):
        with open(path) as f:
            for text in re.findall(r"\basm\b[^;]*;", f.read()):
                if re.search(r"s_mov_b32 m0", text):
                    found += 1
                    assert re.search(r':[^:]*"m0"[^:]*\)\s*;$', text), (os.path.basename(path), text)
    assert found
