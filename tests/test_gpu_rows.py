"""Rows of every length through the curl kernels' quads (16 bytes of a row per lane): the CPU oracle's
fields, FP32 bit for bit and FP64 to 1e-12 of the largest value (the bound the parity scenarios
have), over row lengths that leave every remainder of a quad.  The nanoblock steps its TF/SF box's auxiliary world inside the main
world's launches and its objects in launches of their own; a read between two calls of a half step
makes the waiting launches run apart.
"""
import ctypes

import numpy as np
import pytest

from scenarios import ROOT

pytestmark = pytest.mark.gpu

LIBS = {"hip": ROOT / "alis_amd" / "libalis_workloads.so", "oracle": ROOT / "oracle" / "libwl_oracle.so"}
ENGINES = {"hip": ROOT / "alis_amd" / "libalis.so", "oracle": ROOT / "oracle" / "liboracle.so"}


def _fields(kind, name, cells, bits, steps, parted=None):
    w, e = ctypes.CDLL(str(LIBS[kind])), ctypes.CDLL(str(ENGINES[kind]))
    w.wl_create.restype = w.wl_device.restype = ctypes.c_void_p
    w.wl_create.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 3
    w.wl_step.argtypes = [ctypes.c_void_p, ctypes.c_int]
    w.wl_device.argtypes = w.wl_free.argtypes = [ctypes.c_void_p]
    w.wl_field.restype = ctypes.c_long
    w.wl_field.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_double), ctypes.c_long]
    for f in (e.alis_dev_core, e.alis_dev_ghosts):
        f.argtypes = [ctypes.c_void_p, ctypes.c_int]
    c = w.wl_create(name.encode(), cells, bits, 64)
    w.wl_step(c, steps)
    per = (cells + 4) ** 3
    buf = (ctypes.c_double * per)()
    out = []

    def read(h):
        for a in range(3):
            n = w.wl_field(c, 0, h, 0, a, buf, per)
            assert n > 0
            out.append(np.frombuffer(buf, dtype=np.float64, count=n).copy())
    if parted:
        dev = w.wl_device(c)
        for h in range(2):
            assert e.alis_dev_core(dev, h) == 0
            if parted == "core":
                read(h)
            assert e.alis_dev_ghosts(dev, h) == 0
            if parted == "ghosts":
                read(0)
        w.wl_step(c, 2)
    read(0), read(1)
    w.wl_free(c)
    return np.concatenate(out)


def _agree(name, cells, bits, steps, parted=None):
    print(f"[gpu] {name} {cells}^3 fp{bits}", flush=True)
    got, ref = _fields("hip", name, cells, bits, steps, parted), _fields("oracle", name, cells, bits, steps, parted)
    assert got.shape == ref.shape and np.abs(ref).max() > 0
    if bits == 32:
        assert np.array_equal(got, ref)
    else:
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("cells,bits", [(58, 32), (59, 32), (60, 32), (61, 32), (62, 32), (60, 64), (61, 64)])
def test_dipole_rows(cells, bits):
    _agree("dipole", cells, bits, 30)


@pytest.mark.parametrize("cells,bits", [(108, 32), (109, 32), (110, 32), (111, 32), (109, 64), (110, 64)])
def test_scatterer_rows(cells, bits):
    _agree("nanoblock", cells, bits, 12)


@pytest.mark.parametrize("name,cells,bits,parted", [("nanoblock", 109, 32, "core"), ("nanoblock", 109, 64, "core"), ("dipole", 59, 32, "core"),
                                                    ("dipole", 59, 32, "ghosts"), ("dipole", 60, 64, "ghosts")])
def test_half_step_in_parts(name, cells, bits, parted):
    _agree(name, cells, bits, 15, parted)


@pytest.mark.parametrize("worlds", [2])
def test_batch_half_step_in_parts(worlds):
    """A read between the core and the post of a batch (complex worlds, Bloch boundaries)."""
    out = {}
    for kind in LIBS:
        w, e = ctypes.CDLL(str(LIBS[kind])), ctypes.CDLL(str(ENGINES[kind]))
        w.wl_create.restype = w.wl_device_of.restype = ctypes.c_void_p
        w.wl_create.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 3
        w.wl_step.argtypes = w.wl_device_of.argtypes = [ctypes.c_void_p, ctypes.c_int]
        w.wl_free.argtypes = [ctypes.c_void_p]
        w.wl_field.restype = ctypes.c_long
        w.wl_field.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_double), ctypes.c_long]
        e.alis_dev_batch_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int, ctypes.POINTER(ctypes.c_void_p)]
        for f in (e.alis_dev_batch_core, e.alis_dev_batch_post):
            f.argtypes = [ctypes.c_void_p, ctypes.c_int]
        e.alis_dev_batch_release.argtypes = [ctypes.c_void_p]
        e.alis_dev_batch_release.restype = None
        c = w.wl_create(b"kpoints", worlds, 32, 64)
        w.wl_step(c, 3)
        dev = (ctypes.c_void_p * worlds)(*[w.wl_device_of(c, q) for q in range(worlds)])
        B = ctypes.c_void_p()
        assert e.alis_dev_batch_create(dev, worlds, ctypes.byref(B)) == 0
        buf = (ctypes.c_double * 2000000)()
        got = []

        def read():
            for q in range(worlds):
                for h in range(2):
                    for m in range(2):
                        for a in range(3):
                            n = w.wl_field(c, q, h, m, a, buf, len(buf))
                            assert n > 0
                            got.append(np.frombuffer(buf, dtype=np.float64, count=n).copy())
        for h in range(2):
            assert e.alis_dev_batch_core(B, h) == 0
            read()
            assert e.alis_dev_batch_post(B, h) == 0
        for h in range(2):
            assert e.alis_dev_batch_core(B, h) == 0 and e.alis_dev_batch_post(B, h) == 0
        read()
        e.alis_dev_batch_release(B)
        w.wl_free(c)
        out[kind] = np.concatenate(got)
    assert np.abs(out["oracle"]).max() > 0 and np.array_equal(out["hip"], out["oracle"])


@pytest.mark.parametrize("bits", [32, 64])
def test_whole_sync_over_many_chunks(bits):
    """The host fields of a world whose arrays take several chunks of the copy to the host (110^3: 10 of
    4 MiB, over all its threads): the sum of their squares is the oracle's (FP64: as rounded to float)."""
    sums = {}
    for kind in LIBS:
        w = ctypes.CDLL(str(LIBS[kind]))
        w.wl_create.restype = ctypes.c_void_p
        w.wl_create.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 3
        w.wl_step.argtypes = [ctypes.c_void_p, ctypes.c_int]
        w.wl_checksum.restype = ctypes.c_double
        w.wl_checksum.argtypes = w.wl_free.argtypes = [ctypes.c_void_p]
        c = w.wl_create(b"nanoblock", 110, bits, 64)
        sums[kind] = []
        for _ in range(2):
            w.wl_step(c, 15)                             # (the first steps are all zeros)
            sums[kind].append(w.wl_checksum(c))
        w.wl_free(c)
    assert sums["oracle"][0] > 0
    for got, ref in zip(sums["hip"], sums["oracle"]):
        assert got == ref if bits == 32 else abs(got - ref) <= 1e-7 * ref


@pytest.mark.parametrize("cells,bits", [(108, 32), (109, 32), (110, 32), (111, 32), (109, 64), (110, 64)])
def test_face_samples_of_the_curl(cells, bits, monkeypatch):
    """A phaser's z faces at every place of a quad, sampled by the H curl (the pair across the face in one
    quad, in the next lane's, or in the next wavefront's) and by k_phs_sample: the same accumulators."""
    w, e = ctypes.CDLL(str(LIBS["hip"])), ctypes.CDLL(str(ENGINES["hip"]))
    w.wl_create.restype = w.wl_device.restype = ctypes.c_void_p
    w.wl_create.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 3
    w.wl_step.argtypes = [ctypes.c_void_p, ctypes.c_int]
    w.wl_device.argtypes = w.wl_free.argtypes = [ctypes.c_void_p]
    e.alis_dev_phaser_size.restype = ctypes.c_long
    e.alis_dev_phaser_size.argtypes = [ctypes.c_void_p, ctypes.c_int]
    e.alis_dev_phaser_read.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.POINTER(ctypes.c_double), ctypes.c_long]
    got = []
    for mode in ("force", "0"):
        monkeypatch.setenv("ALIS_PRESAMPLE", mode)
        c = w.wl_create(b"nanoblock", cells, bits, 64)
        w.wl_step(c, 40)
        dev = w.wl_device(c)
        n = e.alis_dev_phaser_size(dev, 0)
        assert n > 0
        out = np.zeros(n)
        assert e.alis_dev_phaser_read(dev, 0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), n) == 0
        w.wl_free(c)
        got.append(out)
    assert np.abs(got[0]).max() > 0 and np.array_equal(got[0], got[1])
