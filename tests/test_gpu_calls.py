"""Batches of Bloch worlds (complex fields, CPML along z) in other ways than updateWorldsE/H: FP32 fields
bit for bit the CPU oracle's, after enough steps that the fields reach the ends of z."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from scenarios import ROOT

pytestmark = pytest.mark.gpu

LIBS = {"hip": (ROOT / "alis_amd" / "libalis_workloads.so", ROOT / "alis_amd" / "libalis.so"),
        "oracle": (ROOT / "oracle" / "libwl_oracle.so", ROOT / "oracle" / "liboracle.so")}
WORLDS, STEPS = 2, 90


def _fields(kind, program=None):
    """The fields of WORLDS k-point worlds after STEPS steps and then program(engine, batch, devices)."""
    w, e = (ctypes.CDLL(str(p)) for p in LIBS[kind])
    V, I = ctypes.c_void_p, ctypes.c_int
    w.wl_create.restype = w.wl_device_of.restype = V
    w.wl_create.argtypes = [ctypes.c_char_p] + [I] * 3
    w.wl_step.argtypes = w.wl_device_of.argtypes = [V, I]
    w.wl_free.argtypes = [V]
    w.wl_field.restype = ctypes.c_long
    w.wl_field.argtypes = [V] + [I] * 4 + [ctypes.POINTER(ctypes.c_double), ctypes.c_long]
    e.alis_dev_batch_create.argtypes = [ctypes.POINTER(V), I, ctypes.POINTER(V)]
    for f in (e.alis_dev_core, e.alis_dev_ghosts, e.alis_dev_batch_core, e.alis_dev_batch_post):
        f.argtypes = [V, I]
    e.alis_dev_batch_release.argtypes, e.alis_dev_batch_release.restype = [V], None
    c = w.wl_create(b"kpoints", WORLDS, 32, 64)
    w.wl_step(c, STEPS)
    if program:
        dev = (V * WORLDS)(*[w.wl_device_of(c, q) for q in range(WORLDS)])
        B = V()
        assert e.alis_dev_batch_create(dev, WORLDS, ctypes.byref(B)) == 0
        program(e, B, dev)
        e.alis_dev_batch_release(B)
        w.wl_step(c, 2)
    buf = (ctypes.c_double * 400000)()
    out = []
    for q in range(WORLDS):
        for h in range(2):
            for m in range(2):
                for a in range(3):
                    n = w.wl_field(c, q, h, m, a, buf, len(buf))
                    assert n > 0
                    out.append(np.frombuffer(buf, dtype=np.float64, count=n).copy())
    w.wl_free(c)
    return np.concatenate(out)


def test_parts_in_entries_of_their_own(monkeypatch):
    monkeypatch.setenv("ALIS_BATCH_PAIRS", "0")
    got, ref = _fields("hip"), _fields("oracle")
    assert np.abs(ref).max() > 0 and np.array_equal(got, ref)


def _cores_apart(e, B, dev):
    for h in range(2):
        for d in dev:
            assert e.alis_dev_core(d, h) == 0
        assert e.alis_dev_batch_post(B, h) == 0


def _ends_apart(e, B, dev):
    for h in range(2):
        assert e.alis_dev_batch_core(B, h) == 0
        for d in dev:
            assert e.alis_dev_ghosts(d, h) == 0


@pytest.mark.parametrize("program", [_cores_apart, _ends_apart])
def test_half_steps_of_single_and_shared_calls(program):
    got, ref = _fields("hip", program), _fields("oracle", program)
    assert np.abs(ref).max() > 0 and np.array_equal(got, ref)


WORLDS_OF = r'''
import ctypes, sys
import numpy as np
V, I = ctypes.c_void_p, ctypes.c_int
ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
ec = ctypes.CDLL(sys.argv[1])
ec.ec_beam.restype = ec.ec_plane.restype = ec.ec_objects.restype = V
ec.ec_field.restype = ctypes.c_long
ec.ec_step.argtypes, ec.ec_step_many.argtypes, ec.ec_step_read.argtypes = [V, I], [V, I, I], [V, I, I, I]
ec.ec_field.argtypes = [V, I, I, V, ctypes.c_long]
mode = sys.argv[4]
W = (V * 1)(ec.ec_plane(730)) if mode == "plane" else (V * 2)(*[ec.ec_objects(2 * n if "large" in mode else n, 3 if "large" in mode else 1) if "objects" in mode else ec.ec_beam(n, 20) for n in (40, 43)])
if "objects" in mode:
    ec.ec_step_read(W, 2, 31, "together" in mode)
elif mode == "together":
    ec.ec_step_many(W, 2, 45)
else:
    for w in W:
        ec.ec_step(w, 6 if mode == "plane" else 45)
out, buf = [], np.zeros(4000000)
for w in W:
    for h in range(2):
        for a in range(3):
            n = ec.ec_field(w, h, a, buf.ctypes.data, buf.size)
            assert n > 0
            out.append(buf[:n].copy())
np.save(sys.argv[3], np.concatenate(out))
'''


@pytest.mark.parametrize("mode", ["alone", "together", "plane"])
def test_sources_of_many_cells(tmp_path, mode):
    """Focused beams, whose core runs at its call while the source is on and waits once it has ended; a uniform
    source over a plane of 731 x 731 cells, which takes four cells per thread."""
    client = tmp_path / "engine_client.so"
    subprocess.run(["gcc", "-O1", "-std=gnu99", "-shared", "-fPIC", f"-I{ROOT / 'include'}", "-o", str(client),
                    str(ROOT / "tests" / "engine_client.c")], check=True)
    _compare(client, tmp_path, mode, "fp32")


@pytest.mark.parametrize("mode", ["objects", "objects together", "large objects", "large objects together"])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_current_updates_apart_and_with_the_next_step(tmp_path, mode, precision):
    """Overlapping objects: the current update runs beside the end of the H half step (small ones), with the
    next E half step, or by itself where the currents are read before."""
    client = tmp_path / "engine_client.so"
    subprocess.run(["gcc", "-O1", "-std=gnu99", "-shared", "-fPIC", f"-I{ROOT / 'include'}", "-o", str(client),
                    str(ROOT / "tests" / "engine_client.c")], check=True)
    _compare(client, tmp_path, mode, precision)


def _compare(client, tmp_path, mode, precision):
    """FP32 bit for bit, FP64 to 1e-12 of the largest value (the bound the parity scenarios have)."""
    got = {}
    for kind in LIBS:
        print(f"[gpu] {mode}, {kind}, {precision}", flush=True)
        subprocess.run([sys.executable, "-c", WORLDS_OF, str(client), str(LIBS[kind][1]), str(tmp_path / f"{kind}.npy"), mode],
                       check=True, timeout=100, env={**os.environ, "ALIS_PRECISION": precision})
        got[kind] = np.load(tmp_path / f"{kind}.npy")
    big = np.abs(got["oracle"]).max()
    assert big > 0
    if precision == "fp32":
        assert np.array_equal(got["hip"], got["oracle"])
    else:
        assert np.abs(got["hip"] - got["oracle"]).max() <= 1e-12 * big
