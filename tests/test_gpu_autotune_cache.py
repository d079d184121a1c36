"""Kept autotuner results (SP_AUTOTUNE_CACHE) where a split tile is the fastest: the fastest
one-launch tile is kept beside it, for calls that cannot split the step.  A file with the split line
alone is read as well.  Grouped batches run the built-in one-launch tile, whose shape problems
share.  Results are the same bits with every tile."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
import json, sys
import numpy as np
import stencilparareal_amd as sp
N, S = 32, 4
out = {}
for tuned in (True, False):
    b = sp.Batch([sp.Problem(N, S, 0.01, (1.0, -0.5, 0.25), 0.01, 64, 8)], kmax=2, coarse_dtype="f64", autotune=tuned)
    u, q = b.fields("u"), b.fields("q")
    u[0].set(np.random.default_rng(1).standard_normal((N, N, N)))
    b.run(u, q)
    i = b.info(0)
    out[tuned] = [i.fine_variant, i.fine_tx, i.fine_ty, i.fine_nthreads, i.fine_kchunk], q[0].get()
conv = sp.Convection(N, N, N, 1. / N, 0.01, 0.0, 1.0, -0.5, 0.25)
us = conv.autotune(S)
conv.autotune(1)
a, b = conv.field(), [conv.field() for _ in range(2)]
a.set(np.random.default_rng(2).standard_normal((N, N, N)))
conv.DoRK4Timestep(a, b[0], 0.0, 1e-4)
conv.set_tile(32, 16, 512, 0, variant="scalar")
conv.DoRK4Timestep(a, b[1], 0.0, 1e-4)
conv.set_tile()
equal = bool(np.array_equal(b[0].get(), b[1].get()) and np.array_equal(out[True][1], out[False][1]) and np.isfinite(out[True][1]).all())
print(json.dumps(dict(tuned=out[True][0], builtin=out[False][0], equal=equal, single=conv.get_tile(S), us=us)))
'''


@pytest.mark.gpu
@pytest.mark.parametrize("both_lines", [True, False])
def test_one_launch_tile_beside_a_split_one(tmp_path, both_lines):
    # device ni nj nk nslices in_dtype out_dtype variant tx ty nthreads kchunk microseconds
    cache = tmp_path / "tiles"
    lines = []
    for slices in (1, 4):
        if both_lines:
            lines.append(f"0 32 32 32 {slices} 0 0 0 24 24 1024 16 30.0")
        lines.append(f"0 32 32 32 {slices} 0 0 3 16 16 384 8 12.0")
    cache.write_text("\n".join(lines) + "\n")
    r = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True, timeout=120, cwd=ROOT,
                       env=dict(os.environ, SP_AUTOTUNE_CACHE=str(cache)))
    assert r.returncode == 0, r.stderr[-3000:]
    got = json.loads(r.stdout.strip().splitlines()[-1])
    assert got["equal"] and got["us"] == 12.0 and got["single"]["variant"] == "split"
    assert got["tuned"] == got["builtin"]


@pytest.mark.gpu
def test_tuning_keeps_both(tmp_path):
    cache = tmp_path / "tiles"
    r = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True, timeout=120, cwd=ROOT,
                       env=dict(os.environ, SP_AUTOTUNE_CACHE=str(cache)))
    assert r.returncode == 0, r.stderr[-3000:]
    got = json.loads(r.stdout.strip().splitlines()[-1])
    kept = [line.split() for line in cache.read_text().splitlines()]
    one = [k for k in kept if k[4] == "4" and k[7] != "3"]
    assert got["equal"] and len(one) == 1
    split = [k for k in kept if k[4] == "4" and k[7] == "3"]
    assert (got["single"]["variant"] == "split") == (len(split) == 1)
    assert all(float(k[12]) < float(one[0][12]) for k in split)
