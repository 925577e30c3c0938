"""What the host side launches and allocates, with a host-only HIP runtime: no GPU, no kernel runs."""
import shutil

import pytest

from tests import host_hip

pytestmark = pytest.mark.skipif(not shutil.which("/opt/rocm/bin/hipcc"), reason="needs hipcc")


@pytest.fixture(scope="module")
def hip(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


# A decode of 5000 vectors of 64-bit values by each expression: blocks of its last launch.
GRIDS = """
L = fa.lib()
x = np.cumsum(np.random.default_rng(1).integers(0, 1000, 5000 * 1024)).astype(np.int64)
x[::300] = 1 << 50
plans = {}
for e in EXPRS:
    enc = fa.encode_from_memory(x if e != 7 else x >> 14, e)
    plans[e] = fa.Plan(enc, x.dtype)
    assert plans[e].n_pages == 1
def grid(e, family=None, cap=0):
    if family is not None:
        fa.check(L.fls_gpu_tune_set(family, 64, 255, 64, 1, cap), "tune_set")
    launches()
    plans[e].decode(4096, 4096, x.nbytes)
    return launches()[-1][1:3]
def select(e):
    launches()
    plans[e].select(4096, "<", np.int64(5), 4096, 4096)
    return launches()[-1][1:3]
"""


def test_patched_pages_have_their_own_launch_shape(hip):
    """Patched pages of 64-bit values take the shape that the table or a caller names for them (no cap of their own besides),
    and follow an FFOR setting made after theirs, as before they had an entry."""
    got = host_hip.run(hip, GRIDS.replace("EXPRS", "(1, 2, 4, 5, 12)") + """
result = {"shipped": [grid(e) for e in (2, 4, 5, 12)], "predicate": select(2), "ffor": grid(1)}
result["own"] = [grid(e, 7, 600) for e in (2, 4, 5, 12)]
result["s and b"] = [grid(2, 9, 300), grid(4), grid(5), grid(12)]
result["ffor after own"] = grid(1)
result["by ffor"] = [grid(e, 2, 700) for e in (2, 4, 5, 12)]
""")
    assert got["shipped"] == [[1250, 64]] * 2 + [[1024, 64]] * 2 and got["predicate"] == [1024, 64] and got["ffor"] == [2500, 128]
    assert got["own"] == [[600, 64]] * 4 and got["s and b"] == [[300, 64]] * 2 + [[600, 64]] * 2
    assert got["ffor after own"] == [2500, 128]
    assert got["by ffor"] == [[700, 64]] * 4


def test_plain_position_pages_have_their_own_launch_shape(hip):
    """RLE pages of 64-bit values with plain positions, likewise."""
    got = host_hip.run(hip, GRIDS.replace("EXPRS", "(6, 7)") + """
result = {"shipped": [grid(6), grid(7)], "own": grid(7, 8, 300), "rle after own": grid(6), "by rle": grid(7, 4, 200)}
""")
    rle, pos = got["shipped"]
    assert pos == [2500, 64] and rle == [2500, 128]
    assert got["own"][0] == 300 and got["rle after own"] == rle and got["by rle"][0] == 200


ENCODE = """
L = fa.lib()
size = C.c_uint64()
def encode(fn, n_vec, stream=0):
    calls()
    fa.check(getattr(L, fn)(4096, n_vec * 1024, 8, 1, 4096, 1 << 40, C.byref(size), stream), fn)
    return calls()
def current():
    d = C.c_int(-1)
    _h.hipGetDevice(C.byref(d))
    return d.value
"""


def test_allocation_free_encoder_allocates_nothing(hip):
    """fls_gpu_encode_noalloc neither allocates device memory nor pins host memory, on its first call either."""
    got = host_hip.run(hip, ENCODE + """
result = [sorted({c[0] for c in encode("fls_gpu_encode_noalloc", n)}) for n in (1, 16384)]
""")
    assert got == [["launch", "symbol_on"], ["launch"]]


def test_encoder_scratch_is_on_the_streams_device(hip):
    """A stream of another device than the current one (0x201: device 2): its scratch and kernels are that device's, from the
    fixed scratch, a slot, or the stream's allocator; the current device stays what it was."""
    got = host_hip.run(hip, ENCODE + """
result = []
for fn, n in (("fls_gpu_encode_noalloc", 64), ("fls_gpu_encode", 64), ("fls_gpu_encode", 1 << 20)):
    c = encode(fn, n, 0x201)
    where = {int(x[1]) for x in c if x[0] in ("symbol_on", "malloc_async_on")} | {int(x[1].split()[-1]) for x in c if x[0] == "launch"}
    result.append([sorted(where), current()])
""")
    assert got == [[[2], 0]] * 3


def test_encoder_takes_the_special_streams(hip):
    """The null stream, hipStreamLegacy and hipStreamPerThread are the current device's (1 here)."""
    got = host_hip.run(hip, ENCODE + """
_h.hipSetDevice(1)
result = []
for s in (0, 1, 2):
    for fn in ("fls_gpu_encode_noalloc", "fls_gpu_encode"):
        result.append(sorted({int(x[1].split()[-1]) for x in encode(fn, 64, s) if x[0] == "launch"}) + [current()])
""")
    assert got == [[1, 1]] * 6
