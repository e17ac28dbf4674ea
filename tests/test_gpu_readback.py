"""Fields read in chunks: a whole field is what reads of its parts give, for
sizes below the directly written ones, of one chunk, of many with a remainder
and with a layer larger than a chunk."""
import ctypes
import threading

import numpy as np
import pytest

import tclb_amd
from test_gpu_parity import random_case, say

pytestmark = pytest.mark.gpu


def parts(lat, q, rows):
    """The field from reads of at most `rows` rows of a layer each."""
    return np.concatenate([np.concatenate([lat.quantity(q, region=(0, y, z, lat.nx, min(rows, lat.ny - y), 1))
                                           for y in range(0, lat.ny, rows)], axis=1) for z in range(lat.nz)])


@pytest.mark.parametrize("model,storage,nx,ny,nz", [
    ("d2q9", "f64", 37, 11, 1),           # a few kB
    ("d2q9_SRT", "f16s", 1501, 903, 1),   # U: 32 MB by rows, the last chunk shorter
    ("d3q19", "f64", 61, 48, 57),         # P: 1.3 MB, one chunk
    ("d3q27", "f32", 129, 97, 113),       # U: 34 MB by layers
    ("d3q19", "f16s", 1100, 1000, 3),     # a layer of U is 26 MB
    ("d2q9_SRT", "f64", 800011, 6, 1),    # a row of U is 19 MB
])
def test_whole_field_is_its_parts(model, storage, nx, ny, nz):
    say(f"reads {model} {storage} {nx}x{ny}x{nz}")
    lat = tclb_amd.Lattice(model, nx, ny, nz, storage)
    lat.set_flags(random_case(model, nx, ny, nz, seed=3).flags)
    lat.init()
    lat.iterate(3)
    for q in lat.quantities[:3]:
        whole = lat.quantity(q)
        step = max(1, 120000 // (nx * 24))   # rows of a read that is written directly
        assert np.array_equal(whole, parts(lat, q, step), equal_nan=True), q
        sub = lat.quantity(q, region=(1, 2, 0, nx - 2, ny - 3, nz), scale=2.0)
        assert np.array_equal(sub, 2.0 * whole[:, 2:ny - 1, 1:nx - 1], equal_nan=True), q


def test_threads_read_one_lattice():
    say("two threads read one lattice")
    case = random_case("d3q19", 150, 120, 90, seed=4)
    case.init_f = None
    lat = case.build("f32")
    lat.iterate(2)
    want = {q: lat.quantity(q) for q in ("P", "U")}
    got = {}
    threads = [threading.Thread(target=lambda k=k, q=q: got.__setitem__((k, q), lat.quantity(q)))
               for k in range(2) for q in ("P", "U")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 4
    for (_, q), a in got.items():
        assert np.array_equal(a, want[q]), q


def test_batch_reads():
    """Fields of a batch's cases against the same lattices read alone."""
    say("batch reads")
    for model, storage, shapes in [("d2q9_drag", "f16s", [(1024, 256, 1), (130, 70, 1)]),
                                   ("d3q19", "f16s", [(150, 110, 97), (48, 50, 33)])]:
        runs = []
        for k, s in enumerate(shapes):
            c = random_case(model, *s, seed=6 + k)
            c.init_f = None
            runs.append(c)
        batch = tclb_amd.Batch(model, storage, capacity_bytes=1 << 29)
        ids = [batch.add(c) for c in runs]
        batch.iterate(5)
        for i, c in zip(ids, runs):
            lat = c.build(storage)
            lat.iterate(5)
            for q in ("U", lat.quantities[0]):
                assert np.array_equal(batch.quantity(i, q), lat.quantity(q), equal_nan=True), q


def free_device_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_reads_keep_no_device_memory():
    """A read leaves no device memory behind beyond what a few kB of launches
    take, whatever the size of a layer: U of 1100x1000 is 26 MB a layer."""
    say("device memory of reads")
    tclb_amd.Lattice("d3q19", 8, 8, 8, "f16s").quantity("U")   # the runtime's own first needs
    shape = (1100, 1000, 3)
    batch = tclb_amd.Batch("d3q19", "f16s", capacity_bytes=1 << 29)
    cid = batch.add_case(*shape)
    lat = tclb_amd.Lattice("d3q19", *shape, "f16s")
    flags = np.full(shape[::-1], lat.spec.flag("MRT"), np.uint16)
    lat.set_flags(flags)
    lat.init()
    batch.set_flags(cid, flags)
    batch.init_case(cid)
    for x in (lat, batch):
        x.iterate(2)
    free = free_device_memory()
    u, v = lat.quantity("U"), batch.quantity(cid, "U")
    assert np.array_equal(u, v)
    assert free - free_device_memory() <= 4 << 20
