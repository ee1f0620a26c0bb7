"""Host code of the batched queries when device memory runs out, without a GPU: the library on a
stand-in for the HIP runtime (hip_stub.c) whose allocations above a limit fail."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CHILD = """
import ctypes as C, json, sys
import numpy as np
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from ncollide_amd import _lib
lib = _lib.load()


class Ctx(C.Structure):  # ncx_ctx
    _fields_ = [("device", C.c_int), ("stream", C.c_void_p), ("num_cus", C.c_int)]


ctx = Ctx(0, None, 256)
limit = C.c_size_t.in_dll(stub, "stub_limit")
count = lambda name: C.c_int.in_dll(stub, name).value
rec = np.zeros((8, 8), np.uint32)  # balls
shapes = C.c_void_p()
assert lib.ncx_shapes_create(C.byref(ctx), rec.ctypes.data, 8, None, None, None, 0, C.byref(shapes)) == 0
poses = np.zeros((8, 8), np.float32)
p = poses.ctypes.data
error = lambda: lib.ncx_last_error().decode()


def contact(n):
    ix = np.zeros(n, np.uint32)
    out = np.zeros(12 * n, np.uint8)
    return lib.ncx_contact_batch(shapes, p, ix.ctypes.data, ix.ctypes.data, n, 0.0, None, *[out.ctypes.data] * 5, None)


def distance(n):
    ix = np.zeros(n, np.uint32)
    return lib.ncx_distance_batch(shapes, p, ix.ctypes.data, ix.ctypes.data, n, np.zeros(n, np.float32).ctypes.data, None)


def impact(n):
    ix = np.zeros(n, np.uint32)
    out = np.zeros(12 * n, np.uint8)
    return lib.ncx_time_of_impact_batch(shapes, p, p, ix.ctypes.data, ix.ctypes.data, n, 1.0, 0.0,
                                        *[out.ctypes.data] * 7)


def rays(n):
    ix = np.zeros(n, np.uint32)
    col = np.zeros(n, np.float32).ctypes.data
    out = np.zeros(12 * n, np.uint8)
    return lib.ncx_shapes_cast_rays(shapes, p, ix.ctypes.data, (C.c_void_p * 6)(*[col] * 6), n, 1.0, 1,
                                    *[out.ctypes.data] * 3)


"""


def run(tmp_path, body):
    stub = str(tmp_path / "hip_stub.so")
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-o", stub, os.path.join(HERE, "hip_stub.c")])
    r = subprocess.run([sys.executable, "-c", CHILD + body, stub], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.splitlines()[-1])


@pytest.mark.parametrize("query", ["distance", "contact"])
@pytest.mark.parametrize("npairs", [100, 20000])
def test_time_of_impact_after_a_refused_batch(tmp_path, npairs, query):
    """A batch whose lists cannot grow is refused and leaves the set usable: the next query's header is
    not at address zero."""
    out = run(tmp_path, f"""
limit.value = 1 << 22  # the lists of 2^19 pairs take 8 MiB
refused = {query}(1 << 19)
message = error()
limit.value = (1 << 64) - 1
rc = impact({npairs})
print(json.dumps([refused, message, rc, count("stub_null_fills"), count("stub_launches")]))
""")
    refused, message, rc, null_fills, launches = out
    assert refused != 0 and "hipMalloc" in message
    assert (rc, null_fills) == (0, 0) and launches > 0


@pytest.mark.parametrize("call,least,little", [("contact", 20, 27), ("rays", 12, 20), ("impact", 0, 20)])
def test_batches_of_little_memory(tmp_path, call, least, little):
    """Contacts take their pairs in parts, and rays theirs in chunks, where there is no memory for all of
    them at once; times of impact do without their order.  With none at all the first two are refused."""
    body = f"""
limit.value = 1 << {{}}
a = count("stub_launches")
print(json.dumps([{call}(1 << 20), count("stub_launches") - a]))
"""
    none, few, all_ = (run(tmp_path, body.format(k)) for k in (least, little, 62))
    assert (none[0] == 0) == (call == "impact")
    assert few[0] == all_[0] == 0
    assert few[1] < all_[1] if call == "impact" else few[1] > all_[1]


def test_counters_do_not_wrap(tmp_path):
    """The kernels' query counters are 32 bits wide and pass the number of queries by a few thousand before
    the last wavefront ends: 2^32 - 2 mesh distances go in chunks that leave room for that."""
    launches = run(tmp_path, """
pts = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
tri = np.array([[0, 1, 2]], np.uint32)
mesh = C.c_void_p()
assert lib.ncx_trimesh_create(C.byref(ctx), pts.ctypes.data, 3, tri.ctypes.data, 1, C.byref(mesh)) == 0, error()
a = count("stub_launches")
assert lib.ncx_mesh_distance_batch(mesh, p, shapes, p, p, (1 << 32) - 2, p) == 0, error()
print(json.dumps(count("stub_launches") - a))
""")
    assert launches == 4 * 2  # a fill and a search each
