"""The probe-spectrum kernel against the CPU oracle's sums, where its workgroups (4 bins, 16 probes,
256 staged samples) end: the factors of both engines are correctly rounded to a few units in the
last place, so a bin differs by at most 4 eps of the sum of its samples' magnitudes."""
import ctypes

import numpy as np
import pytest

from scenarios import ROOT
from test_spectrum import _abi

pytestmark = pytest.mark.gpu


def _sums(path, probes, bins, v):
    lib = _abi(path)
    S = ctypes.c_void_p()
    assert lib.alis_dev_spectrum_create(probes, bins, bins + 3, ctypes.byref(S)) == 0, lib.alis_dev_error()
    dp = ctypes.POINTER(ctypes.c_double)
    for n, row in enumerate(v):
        assert lib.alis_dev_spectrum_add(S, (n + 1) / 512.0, row.ctypes.data_as(dp)) == 0
    out = np.zeros((probes, bins, 2))
    assert lib.alis_dev_spectrum_read(S, out.ctypes.data_as(dp)) == 0
    lib.alis_dev_spectrum_release(S)
    return out


@pytest.mark.parametrize("probes,bins,samples", [(1, 1, 1), (1, 5, 255), (3, 4, 256), (15, 7, 257), (16, 130, 300), (17, 3, 600), (40, 9, 256)])
def test_sums_at_workgroup_edges(probes, bins, samples):
    print(f"[gpu] spectrum of {probes} probes, {bins} bins, {samples} samples", flush=True)
    v = np.random.default_rng(probes * 1000 + bins).standard_normal((samples, probes))
    got = _sums(ROOT / "alis_amd" / "libalis.so", probes, bins, v)
    ref = _sums(ROOT / "oracle" / "liboracle.so", probes, bins, v)
    assert np.all(np.abs(got - ref) <= 4 * np.finfo(float).eps * np.abs(v).sum(axis=0)[:, None, None])
