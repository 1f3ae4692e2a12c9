"""What llmp_hip_exl3_linear_static asks the HIP runtime for after llmp_hip_exl3_linear_static_prepare: launches and nothing
else, whatever the rows (include/llmp_hip.h: a capture may refuse any other call). The runtime's calls are counted by
tests/host/counted_runtime.cc; no GPU, and the operands are addresses that nothing reads."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import ctypes as C, sys
runtime = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from llmp_amd import _lib
lib = _lib.load()
launches, others = C.c_int.in_dll(runtime, "counted_launches"), C.c_int.in_dll(runtime, "counted_others")
for codebook in range(3):
    for bits in range(1, 9):
        op = _lib.Exl3Linear()
        op.weights.trellis, op.weights.suh, op.weights.svh = 0x1000000, 0x2000000, 0x2100000
        op.weights.k, op.weights.n, op.weights.bits, op.weights.codebook = 256, 128, bits, codebook
        op.x, op.a_had, op.y, op.f32, op.m = 0x3000000, 0x3100000, 0x3200000, 1, 1
        before = others.value
        _lib.check(lib.llmp_hip_exl3_linear_static_prepare(C.byref(op)))
        assert others.value > before, "the runtime's calls are not counted"
        for m in (1, 4, 5, 16, 17, 33, 81, 145):
            op.m = m
            before, launched = others.value, launches.value
            _lib.check(lib.llmp_hip_exl3_linear_static(C.byref(op), None))
            assert launches.value > launched
            assert others.value == before, (codebook, bits, m)
"""


def test_a_prepared_static_linear_asks_for_nothing_but_launches(tmp_path):
    shared = os.path.join(tmp_path, "counted_runtime.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", shared, os.path.join(ROOT, "tests", "host", "counted_runtime.cc")],
                   check=True, timeout=120)
    done = subprocess.run([sys.executable, "-c", PROGRAM, shared, ROOT], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout[-2000:] + done.stderr[-4000:]
