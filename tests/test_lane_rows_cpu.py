"""The batched engine's lane rows, checked on the CPU (no GPU needed):
tests/lane_rows_check.hip replays their layout and sums, every index
bounds-checked, against the row groups' additions (see its header).  A run
with one first-piece length moved must fail."""
import os
import struct
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from osqp_amd import build as B
from osqp_amd import problems as pr

from .conftest import ROOT


def _short_rows(m, n, lens, seed):
    """A with the given row lengths cyclically, every column hit; P diagonal."""
    rng = np.random.default_rng(seed)
    ln = np.resize(lens, m)
    ci = np.concatenate([(r * 7 + np.sort(rng.choice(n, k, replace=False))) % n for r, k in enumerate(ln)])
    A = sp.csc_matrix((rng.standard_normal(ci.size), (np.repeat(np.arange(m), ln), ci)), shape=(m, n))
    A = A + 10.0 * sp.eye(m, n, format="csc")
    return dict(P=sp.diags(1.0 + rng.random(n), format="csc"), A=sp.csc_matrix(A))


def _circulant(n, per):
    """A with entry (r, (r + k) mod n) for k < per: rows and columns of `per` entries; P a band of the same."""
    rng = np.random.default_rng(n + per)
    r = np.repeat(np.arange(n), per)
    A = sp.csc_matrix((rng.standard_normal(n * per), (r, (r + np.tile(np.arange(per), n)) % n)), shape=(n, n))
    return dict(P=sp.diags([1.0 + rng.random(n - k) for k in range((per + 1) // 2)], list(range((per + 1) // 2)),
                           format="csc"), A=A)


def _problems():
    out = [(pr.mpc(N, seed=N), 1) for N in (1, 10, 33, 50)]
    out.append((_short_rows(1, 1, [1], 1), 1))
    out.append((_short_rows(64, 64, [1, 2, 3, 4], 2), 1))
    out.append((_short_rows(65, 65, [5, 1, 7], 3), 1))
    out.append((_short_rows(257, 300, [2], 4), 0))      # columns without entries
    out += [(pr.portfolio(n, seed=n), 1) for n in (500, 1000)]  # long rows of A
    out.append((pr.portfolio(3000, seed=5), 0))         # rows of A' of 18 entries and more
    p = _short_rows(100, 100, [3], 6)
    p["A"] = sp.vstack([p["A"], sp.csc_matrix((1, 100))], format="csc")
    out.append((p, 0))                                  # an empty row
    # past 2048 columns: FP32 alone, and rows that the lanes do not pad too much
    out += [(_circulant(2048, 9), 1), (_circulant(2049, 9), 2), (_circulant(4096, 5), 2), (_circulant(4097, 5), 0),
            (_circulant(2048, 3), 1), (_circulant(2049, 3), 0)]
    return out


def test_lane_rows_replay(tmp_path):
    objs = [os.path.join(B.BUILD, f) for f in sorted(os.listdir(B.BUILD))] if os.path.isdir(B.BUILD) else []
    objs = [o for o in objs if o.endswith(".o") and "serve_batch" not in o]
    if not os.path.exists(B.HIPCC) or not objs:
        pytest.skip("needs hipcc and the library's objects (python -m osqp_amd.build)")
    probs = tmp_path / "probs.bin"
    with open(probs, "wb") as f:
        ps = _problems()
        f.write(struct.pack("i", len(ps)))
        for p, want in ps:
            P, A = sp.csc_matrix(sp.triu(p["P"])), sp.csc_matrix(p["A"])
            f.write(struct.pack("iii", P.shape[0], A.shape[0], want))
            for M in (P, A):
                M.sort_indices()
                f.write(struct.pack("i", M.nnz))
                f.write(M.indptr.astype(np.int32).tobytes())
                f.write(M.indices.astype(np.int32).tobytes())
                f.write(M.data.astype(np.float64).tobytes())
    obj, exe = tmp_path / "check.o", tmp_path / "check"
    subprocess.run([B.HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Wno-unused-result", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "osqp_amd", "csrc"),
                    "-c", os.path.join(ROOT, "tests", "lane_rows_check.hip"), "-o", str(obj)],
                   check=True, capture_output=True)
    subprocess.run([B.HIPCC, "--offload-arch=gfx950", str(obj)] + objs +
                   ["-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lrocprofiler-sdk-roctx", "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe), str(probs)], capture_output=True, text=True)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
    bad = subprocess.run([str(exe), str(probs), "plant"], capture_output=True, text=True)
    assert bad.returncode == 1 and "FAILURES" in bad.stdout, bad.stdout[-2000:]
