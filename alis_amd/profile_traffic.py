"""HBM traffic per launch of the curl kernels from two rocprofv3 counter runs.

    rocprofv3 --pmc FETCH_SIZE -d DIR_F -o run --output-format csv -- python3 bench.py \\
        --steps 3 --warmup 1 --no-fp64 --cpu-steps 0 --copy-mib 256
    rocprofv3 --pmc WRITE_SIZE -d DIR_W -o run --output-format csv -- python3 bench.py \\
        --steps 3 --warmup 1 --no-fp64 --cpu-steps 0 --copy-mib 256
    python3 alis_amd/profile_traffic.py DIR_F DIR_W 256 16777216 > profiles/k_curl_nanoblock256_traffic.json

The last two arguments are the copy's MiB and the world's cells.

FETCH_SIZE and WRITE_SIZE (KiB per dispatch) are scaled by what they read for the
device-to-device copy of known size that bench.py makes first (the largest copy dispatch).
"""
import csv
import hashlib
import json
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def kernels_sha256():
    """SHA-256 of the device kernels of the engine (the "Kernels" section of engine.hip and
    the files of kernels it includes, alis_amd/csrc/*.inc): a traffic measurement stays
    valid while these are unchanged."""
    src = (ROOT / "alis_amd/csrc/engine.hip").read_text()
    a = src.index("// Kernels\n")
    b = src.index("// Device world\n", a)
    inc = "".join(f.read_text() for f in sorted((ROOT / "alis_amd/csrc").glob("*.inc")))
    return hashlib.sha256((src[a:b] + inc).encode()).hexdigest()


def rows(d):
    f = next(Path(d).rglob("*counter_collection.csv"))
    return list(csv.DictReader(f.open()))


def main():
    dF, dW, mib, cells = sys.argv[1], sys.argv[2], int(sys.argv[3]), int(sys.argv[4])
    F, W = rows(dF), rows(dW)
    nbytes = mib << 20
    cF = max(float(r["Counter_Value"]) for r in F if "copyBuffer" in r["Kernel_Name"])
    cW = max(float(r["Counter_Value"]) for r in W if "copyBuffer" in r["Kernel_Name"])
    fs, ws = nbytes / 1024 / cF, nbytes / 1024 / cW
    out = {"kernels_sha256": kernels_sha256(),
           "cells": cells, "fields": "fp32",
           "calibration": {"copy_bytes": nbytes, "FETCH_SIZE_kib": cF, "WRITE_SIZE_kib": cW,
                           "fetch_scale": round(fs, 5), "write_scale": round(ws, 5)}}
    # k_curl<float, HALF, ...> and k_curl_aux<float, HALF, ...>: HALF 0 is the E launch, 1 H
    # (the largest launches of each kind: the main world, not an auxiliary world)
    for name, half in (("E", "<float, 0,"), ("H", "<float, 1,")):
        def curl(r):
            return "k_curl" in r["Kernel_Name"] and half in r["Kernel_Name"]
        big = max(int(r["Grid_Size"]) for r in F if curl(r))

        def mine(r):
            return curl(r) and int(r["Grid_Size"]) == big
        f = [float(r["Counter_Value"]) for r in F if mine(r)]
        w = [float(r["Counter_Value"]) for r in W if mine(r)]
        fa, wa = sum(f) / len(f), sum(w) / len(w)
        out[name] = {"FETCH_SIZE_kib": round(fa, 1), "WRITE_SIZE_kib": round(wa, 1), "dispatches": len(f),
                     "traffic_bytes": round((fa * fs + wa * ws) * 1024)}
    print(json.dumps(out, indent=1))


if __name__ == "__main__":
    main()
