"""What the EXL3 linears and the stored encodings' matrix product ask the HIP runtime for. The runtime's calls are counted by
tests/host/counted_runtime.cc; no GPU, and the operands are addresses that nothing reads. The matrix product: which of its
forms it takes. llmp_hip_exl3_linear_static after llmp_hip_exl3_linear_static_prepare: launches and nothing else, whatever
the rows (include/llmp_hip.h: a capture may refuse any other call). The linears over a scratch larger than they need: which
passes they take."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SETUP = """
import ctypes as C, sys
runtime = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from llmp_amd import _lib
lib = _lib.load()
launches, others = C.c_int.in_dll(runtime, "counted_launches"), C.c_int.in_dll(runtime, "counted_others")
"""

STATIC = """
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


# One arena for the scratch and, behind the least that the passes of sixteen take, an operand: accepted, with the launches of
# those passes; the same arena with the operand past the wide passes' part: their fewer launches. An operand in the least
# part is refused either way.
ARENA = """
def linear(**kw):
    op = _lib.Exl3Linear()
    op.weights.trellis, op.weights.suh, op.weights.svh = 0x1000000, 0x2000000, 0x2100000
    op.weights.k, op.weights.n, op.weights.bits, op.weights.codebook = 512, 256, 4, 0
    op.x, op.a_had, op.y, op.f32, op.m = 0x3000000, 0x3100000, 0x3200000, 1, 77
    for name, value in kw.items():
        setattr(op, name, value)
    return op

def multi(**kw):
    one, op = linear(), _lib.Exl3MultiLinear()
    op.first, op.second = one.weights, one.weights
    op.x, op.a_had, op.y, op.f32, op.m = one.x, one.a_had, one.y, one.f32, one.m
    for name, value in kw.items():
        setattr(op, name, value)
    return op

arena, size = 0x4000000, 1 << 24
for make, name in ((linear, "linear"), (multi, "multi_linear")):
    call = getattr(lib, "llmp_hip_exl3_" + name)
    op = make()
    least = getattr(lib, f"llmp_hip_exl3_{name}_scratch")(C.byref(op))
    wide = getattr(lib, f"llmp_hip_exl3_{name}_wide_scratch")(C.byref(op))
    assert 0 < least < wide < size // 2

    def counted(op, given):
        before = launches.value
        _lib.check(call(C.byref(op), arena, given, None))
        return launches.value - before

    sixteens, together = counted(op, wide - 1), counted(op, wide)
    assert together < sixteens
    for field in ("x", "a_had", "y"):
        assert counted(make(**{field: arena + least}), size) == sixteens, (name, field)
        assert counted(make(**{field: arena + wide}), size) == together, (name, field)
        assert call(C.byref(make(**{field: arena + least - 8})), arena, size, None) > 0
        assert b"overlaps" in lib.llmp_hip_last_error()
"""

# (encoding, K, outputs, rows, launches): on both sides of the choice between the matrix product's one launch and its two, by
# the times of both on the device (256 compute units, which the library also takes where it cannot ask).
MATRIX = """
def launched(decoder, k, outputs, rows):
    w = _lib.DecodeOperand()
    w.data, w.scales, w.k, w.rows, w.rows_per_scale, w.row_bytes = 0x10000000, 0x8000000000, k, outputs, outputs, 2 * k
    if decoder == 11:
        w.group, w.bits, w.scale_type, w.scale_row_bytes = 32, 4, 1, k // 16
    size = lib.llmp_hip_decode_matrix_scratch(C.byref(w), outputs, rows)
    before = launches.value
    _lib.check(lib.llmp_hip_decode_matrix_staged(decoder, C.byref(w), 0, outputs, 0x9000000000, rows, k, 0xA000000000, outputs, 0,
                                                 0xB000000000, size, None))
    return launches.value - before

for case in CASES:
    assert launched(*case[:4]) == case[4], case
"""

CASES = [
    (3, 4096, 14336, 300, 2), (3, 1024, 14336, 300, 2), (3, 4096, 14336, 200, 2), (9, 4096, 4096, 1024, 2), (0, 768, 8192, 400, 2),
    (3, 4096, 4096, 17, 2), (7, 4096, 14336, 1024, 2), (0, 4096, 2048, 64, 2),
    # A full round of tiles of 256 by 256 or, at a short K, of 256 by 128.
    (3, 4096, 8192, 2048, 1), (1, 4096, 8192, 2048, 1), (0, 1024, 14336, 512, 1), (7, 768, 4096, 2048, 1),
    # Small tiles, one a compute unit, and a short K.
    (2, 1536, 2048, 17, 1), (9, 1536, 2048, 300, 1), (0, 1536, 14336, 17, 1),
    # Affine: only where the one launch leaves much of its round idle.
    (11, 4096, 14336, 17, 1), (11, 4096, 14336, 512, 1), (11, 4096, 14336, 2048, 1), (11, 2048, 2048, 300, 1),
    (11, 4096, 14336, 300, 2), (11, 4096, 4096, 1024, 2)]


def run(tmp_path, program):
    shared = os.path.join(tmp_path, "counted_runtime.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", shared, os.path.join(ROOT, "tests", "host", "counted_runtime.cc")],
                   check=True, timeout=120)
    done = subprocess.run([sys.executable, "-c", SETUP + program, shared, ROOT], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout[-2000:] + done.stderr[-4000:]


def test_a_prepared_static_linear_asks_for_nothing_but_launches(tmp_path):
    run(tmp_path, STATIC)


def test_an_arena_that_holds_operands_behind_the_least_scratch_is_accepted(tmp_path):
    run(tmp_path, ARENA)


def test_the_matrix_product_takes_the_faster_form(tmp_path):
    run(tmp_path, MATRIX.replace("CASES", repr(CASES)))
