"""A particle whose creation index is not one of its system's is reported.

Results leave the device in creation order, so such a particle would leave a
slot unwritten.  No public call makes one: the two kernels that order results
are launched on a table of their own, in pinned memory that host and device
share, whose index array the test fills.
"""
import ctypes
import os
import re

import numpy as np
import pytest

from conftest import PKG, uniform_box
from test_gpu_parity import mdpd_system

pytestmark = pytest.mark.gpu

N, NPAD = 200, 256


def _struct(name):
    """ctypes layout of a struct of csrc/common.hpp from its declarations."""
    text = re.sub(r"//[^\n]*", "", open(os.path.join(PKG, "csrc", "common.hpp")).read())
    const = {k: int(v) for k, v in re.findall(r"constexpr int (\w+) = (\d+);", text)}
    body = re.search(r"struct %s \{(.*?)\};" % name, text, re.S).group(1)
    kinds = {"int": ctypes.c_int, "float": ctypes.c_float, "double": ctypes.c_double, "uint32_t": ctypes.c_uint32,
             "long long": ctypes.c_longlong}
    fields = []
    for decl in filter(None, (" ".join(d.split()) for d in body.split(";"))):
        kind, rest = re.match(r"(long long|\w+) ?(.*)", decl).groups()
        for d in rest.split(","):
            star, field, dim = re.match(r" ?(\*?)(\w+)(?:\[(\w+)\])?$", d).groups()
            t = ctypes.c_void_p if star else kinds[kind]
            fields.append((field, t * int(const.get(dim, dim)) if dim else t))
    return type(name, (ctypes.Structure,), {"_fields_": fields})


class _Pinned:
    """Arrays of zeros that host and device share."""

    def __init__(self, engine):
        engine.load()
        path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line)
        self.hip, self.kept = ctypes.CDLL(path), []

    def __call__(self, n, dtype):
        p, size = ctypes.c_void_p(), n * np.dtype(dtype).itemsize
        assert self.hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), ctypes.c_uint(0)) == 0
        self.kept.append(p)
        ctypes.memset(p, 0, size)
        return p.value, np.frombuffer((ctypes.c_char * size).from_address(p.value), dtype)

    def close(self):
        for p in self.kept:
            self.hip.hipHostFree(p)


@pytest.mark.parametrize("index, want", [(None, 0), (0, 0), (-1, 1), (N, 1), (1 << 30, 1)])
@pytest.mark.parametrize("kernel", ["gather", "harvest"])
def test_creation_index_outside_the_system_is_reported(engine, kernel, index, want):
    lib = ctypes.CDLL(engine.library_path())
    pinned = _Pinned(engine)
    SysDev, PoolDev = _struct("SysDev"), _struct("PoolDev")
    sys_at, sys_mem = pinned(ctypes.sizeof(SysDev), np.uint8)
    d = SysDev.from_buffer(sys_mem.data)
    d.n, d.npad, d.ncell, d.phase = N, NPAD, 1, 3
    P = PoolDev()
    for b in range(2):
        for f in ("pos", "vel"):
            getattr(P, f)[b] = pinned(4 * NPAD, np.float32)[0]
        for f in ("tag", "mask", "image", "phi"):
            getattr(P, f)[b] = pinned(NPAD, np.int32)[0]
    for f, words in (("frc", 4), ("rho", 1), ("vir", 6), ("wave_sys", 1), ("cell_sys", 1)):
        setattr(P, f, pinned(words * NPAD, np.float32)[0])
    at, origin = pinned(NPAD, np.int32)
    origin[:N] = np.random.default_rng(1).permutation(N)
    P.origin[0] = P.origin[1] = at
    if index is not None:
        origin[77] = index
    at, tag = pinned(NPAD, np.int32)
    tag[:] = 100 + np.arange(NPAD)
    P.tag[0] = P.tag[1] = at
    P.sys, P.cap, P.nact, P.nsys, P.maxnbr, P.one = sys_at, NPAD, NPAD, 1, 32, 1
    P.nlist, rows = pinned(32 * NPAD, np.int32)
    out_at, out = pinned(NPAD, np.int32)
    bad_at, bad = pinned(1, np.int32)
    if kernel == "gather":
        rc = lib._ZN4mdpd13launch_gatherERKNS_7PoolDevEiPiS3_P12ihipStream_t(
            ctypes.byref(P), 7, ctypes.c_void_p(out_at), ctypes.c_void_p(bad_at), None)       # G_TAG
    else:
        rc = lib._ZN4mdpd14launch_harvestERKNS_7PoolDevEPKiiiPiP12ihipStream_t(
            ctypes.byref(P), (ctypes.c_int * 1)(0), 1, NPAD, ctypes.c_void_p(bad_at), None)
        out = rows[12 * NPAD:13 * NPAD]                                                       # after x, v, f
    assert rc == 0 and pinned.hip.hipDeviceSynchronize() == 0
    assert bad[0] == want
    ok = (origin[:N] >= 0) & (origin[:N] < N)
    if index is None:
        np.testing.assert_array_equal(out[origin[:N]], tag[:N])
    assert ok.sum() == N - want
    pinned.close()


def test_gather_of_a_handle_whose_device_is_not_current(engine):
    pinned, count = _Pinned(engine), ctypes.c_int()
    assert pinned.hip.hipGetDeviceCount(ctypes.byref(count)) == 0
    if count.value < 2:
        pytest.skip("one device")
    x, v = uniform_box(300, 4.0, 1)
    a, b = mdpd_system(engine, x, v, 4.0), mdpd_system(engine, x, v, 4.0)
    for s in (a, b):
        s.run(2)
    want = a.gather("x"), a.debug_sorted()[1]
    pinned.hip.hipSetDevice(1)
    np.testing.assert_array_equal(b.gather("x"), want[0])
    pinned.hip.hipSetDevice(1)
    np.testing.assert_array_equal(b.debug_sorted()[1], want[1])
    pinned.hip.hipSetDevice(0)
    a.close()
    b.close()
