"""What the entry points of elementwise.hip launch at sizes near the limits of a launch, without a GPU: the library runs in a process
of its own against a stand-in for the runtime's launch call, which refuses what the runtime refuses (2^32 threads and more in a
dimension) and hands grids and kernel arguments to the test."""
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

STAND_IN = r"""
#include <cstddef>
#include <cstdint>
struct dim3 { uint32_t x, y, z; };
static thread_local struct { dim3 grid, block; size_t smem; void* stream; } pending;
static thread_local int error = 0;
static void (*seen)(uint32_t, uint32_t, void**) = nullptr;
extern "C" {
void on_launch(void (*f)(uint32_t, uint32_t, void**)) { seen = f; }
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t smem, void* stream) { pending = {grid, block, smem, stream}; return 0; }
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* smem, void** stream) {
  *grid = pending.grid, *block = pending.block, *smem = pending.smem, *stream = pending.stream;
  return 0;
}
int hipLaunchKernel(const void*, dim3 grid, dim3 block, void** args, size_t, void*) {
  if (grid.x == 0 || (uint64_t)grid.x * block.x >> 32) return error = 9;   // hipErrorInvalidConfiguration
  seen(grid.x, block.x, args);
  return 0;
}
int hipGetLastError() { const int e = error; error = 0; return e; }
}
"""

PROLOGUE = """
import ctypes as C, os, sys
sys.path.insert(0, sys.argv[2])
shim = C.CDLL(sys.argv[1], os.RTLD_GLOBAL | os.RTLD_NOW)   # before the library: its calls bind to the stand-in
from odysseus_transformer_amd import _lib
assert "torch" not in sys.modules
launches = []
@C.CFUNCTYPE(None, C.c_uint32, C.c_uint32, C.POINTER(C.c_void_p))
def seen(grid, block, args):
    launches.append((grid, block, read(args)))
def value(args, k, kind):
    return C.cast(args[k], C.POINTER(kind)).contents.value
shim.on_launch(seen)
A = 1 << 20   # an aligned address; nothing is read or written
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    folder = tmp_path_factory.mktemp("stand_in")
    (folder / "launch.cpp").write_text(STAND_IN)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(folder / "launch.so"), str(folder / "launch.cpp")], check=True)
    return str(folder / "launch.so")


def run(stand_in, program):
    r = subprocess.run([sys.executable, "-c", PROLOGUE + textwrap.dedent(program), stand_in, str(ROOT)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("rows", [(1 << 24) - 1, 1 << 24, (1 << 26) - 4])
def test_rmsnorm_rows(stand_in, rows):
    """A block per row up to 2^24 - 1 rows, a wavefront per row from there: the most rows of that kernel are the most of the call."""
    run(stand_in, f"""
        read = lambda args: None
        _lib.call("ody_rmsnorm_fwd", A, A, A, 0, {rows}, 2048, 1e-6, _lib.ODY_BF16, 0)
        assert launches == [({rows} if {rows} < 1 << 24 else ({rows} + 3) // 4, 256, None)], launches
    """)


@pytest.mark.parametrize("B,L,D,dtype", [(1, 5, 128, 0), (3, 1 << 25, 128, 0), (2, (1 << 25) + 1, 64, 1), (1, (1 << 24) + 7, 1024, 1)])
def test_rope_tokens(stand_in, B, L, D, dtype):
    """One launch, or several that together take every token once."""
    run(stand_in, f"""
        read = lambda args: value(args, 12, C.c_int64)
        _lib.call("ody_rope", A, 0, 0, {B}, {L}, 2, {D}, {L} * 4 * {D}, 4 * {D}, {D}, 10000.0, 0, {dtype}, 0)
        tokens, at = max(1, 256 // ({D} // 2)), 0
        for grid, block, token0 in launches:
            assert token0 == at and block == 256, (token0, at)
            at += grid * tokens
        assert {B} * {L} <= at < {B} * {L} + tokens, (at, launches)
    """)


ADAMW = """
N = 48
class Table(C.Structure):
    _fields_ = [("p", C.c_uint64 * N), ("g", C.c_uint64 * N), ("m", C.c_uint64 * N), ("v", C.c_uint64 * N), ("n", C.c_int64 * N),
                ("step_size", C.c_float * N), ("inv_sqrt_bc2", C.c_float * N), ("end", C.c_uint32 * N)]
def read(args):
    return Table.from_buffer_copy(C.cast(args[0], C.POINTER(Table)).contents)
def step(dtype, tensors):   # (address of the parameter, elements, step); gradient and moments 1, 2 and 3 << 44 behind it
    n = len(tensors)
    p, e, s = ((C.c_int64 * n)(*c) for c in zip(*tensors))
    g, m, v = ((C.c_int64 * n)(*(t[0] + (k << 44) for t in tensors)) for k in (1, 2, 3))
    _lib.call("ody_adamw_many", p, g, m, v, e, s, n, 1e-3, 0.9, 0.99, 1e-8, 0.01, dtype, 0)
    covered = []   # per launch: (address, elements, step size) of its entries
    for grid, block, t in launches:
        size, first, entries = 2 if dtype == 0 else 4, 0, []
        for k in range(N):
            if t.end[k] == first:
                break
            assert t.end[k] - first == -(-t.n[k] * size // 4096) and t.p[k] % 16 == 0
            assert [t.g[k], t.m[k], t.v[k]] == [t.p[k] + (j << 44) for j in (1, 2, 3)]
            entries.append((t.p[k], t.n[k], t.step_size[k]))
            first = t.end[k]
        assert first == grid == t.end[N - 1] and block == 256
        covered.append(entries)
    return covered
"""


@pytest.mark.parametrize("dtype", [0, 1])
def test_adamw_elements(stand_in, dtype):
    """Tensors beyond a launch, alone and between small ones: every element in one launch, with its own tensor's step size."""
    run(stand_in, ADAMW + f"""
size, most = 2 if {dtype} == 0 else 4, ((1 << 24) - 1) * 4096
sizes = [7, most // size - 2048, 5, 2 * most // size + 11, 4096] + [9] * 60
tensors = [(A + (k << 38), n, k + 1) for k, n in enumerate(sizes)]
covered = sum(step({dtype}, tensors), [])
for p, n, s in tensors:
    at, own = p, [e for e in covered if p <= e[0] < p + (1 << 38)]
    for e in own:
        assert e[0] == at and abs(e[2] / (1e-3 / (1 - 0.9 ** s)) - 1) < 1e-6, (e, at)
        at += e[1] * size
    assert at == p + n * size, (at, p, n)
""")


def test_adamw_parameters_that_share_memory(stand_in):
    """Their updates follow each other: never two in one launch, and in the order of the call."""
    run(stand_in, ADAMW + """
whole, part, behind, again = (A, 4096, 1), (A + 4096, 512, 2), (A + 8192, 512, 3), (A, 4096, 4)
covered = [[e[0] for e in launch] for launch in step(0, [whole, behind, part, again])]
assert covered == [[A, A + 8192], [A + 4096], [A]], covered
""")
