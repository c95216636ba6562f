"""The stencil-lattice searches' own arithmetic on the CPU: the folded screen
(pyhea_amd/csrc/hea_screen.h) against the oracle's sequential FP64 updates
(its window bound, also the one taken for a whole round of accepts, and that a
bound shrunk 1e7-fold is caught), the step of a bounded sequence, and the
detection of stencil tables (hea_stencil.h): every shell set and edge it
takes, rows in any order, and tables it must refuse."""
import os
import subprocess

import numpy as np
import pytest

from pyhea_amd.problem import make_problem

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FCC, FCC_REF, BCC = 1, 2, 3

CASES = {
    "fcc3-k4-equimolar": (("FCC", 3, [0.25] * 4, "true", 1, [27] * 4), False),
    "bcc4-k4-zero-target": (("BCC", 4, [0.25] * 4, "pyhea", 3, [32] * 4), True),
    "fcc4-k5": (("FCC", 4, [0.3, 0.25, 0.2, 0.15, 0.1], "true", 4, None), False),
    "fcc3-k6": (("FCC", 3, [0.3, 0.2, 0.2, 0.1, 0.1, 0.1], "pyhea", 5, None), False),
    "bcc4-k2": (("BCC", 4, [0.5, 0.5], "pyhea", 2, [64, 64]), False),
}


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fold") / "fold_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "oracle"), "-I", os.path.join(ROOT, "pyhea_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "fold_check.cpp"), "-o", exe], check=True)
    return exe


def _write(path, spec, nbr=None, target=None):
    nbr = spec.nbr if nbr is None else nbr
    z = list(spec.shell_sizes[:spec.S]) + [0] * (3 - spec.S)
    with open(path, "wb") as f:
        f.write(np.array([nbr.shape[0], spec.K, spec.S] + z, np.int32).tobytes())
        f.write(np.ascontiguousarray(nbr, np.int32).tobytes())
        f.write(np.array(spec.counts, np.int32).tobytes())
        f.write(np.array(spec.weight, np.float64).tobytes())
        f.write(np.ascontiguousarray(spec.target if target is None else target,
                                     np.float64).tobytes())
    return str(path)


def _bound(harness, tmp_path, name, scale):
    (typ, cell, fr, shells, seed, counts), zero = CASES[name]
    spec = make_problem(typ, cell, fr, shells=shells, target_seed=seed, counts=counts)
    path = _write(tmp_path / f"{name}.bin", spec,
                  target=np.zeros_like(spec.target) if zero else None)
    return subprocess.run([harness, path, "3", "200", "7", repr(scale)], capture_output=True,
                          text=True), spec


@pytest.mark.parametrize("name", sorted(CASES))
def test_folded_window_bound(harness, tmp_path, name):
    r, spec = _bound(harness, tmp_path, name, 1.0)
    assert r.returncode == 0, r.stdout + r.stderr
    ok, pairs, ratio = r.stdout.split()
    assert ok == "ok" and int(pairs) > 3 * spec.n_sites and 0.0 < float(ratio) < 1.0


def test_shrunk_folded_window_is_caught(harness, tmp_path):
    assert all(_bound(harness, tmp_path, name, 1e-7)[0].returncode == 1 for name in CASES)


def test_step_of_a_bounded_sequence(harness):
    r = subprocess.run([harness, "--steps", "200000", "5"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    ok, cases, fast = r.stdout.split()
    assert ok == "ok" and int(cases) > 190000 and int(fast) > 1000000


def _detect(harness, path):
    r = subprocess.run([harness, "--detect", path], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return tuple(int(x) for x in r.stdout.split())


@pytest.mark.parametrize("typ,cell,shells,weights,want", [
    ("FCC", 3, "true", 3, (FCC, 3)), ("FCC", 3, "pyhea", 3, (FCC_REF, 3)),
    ("BCC", 3, "true", 3, (BCC, 3)), ("FCC", 7, "pyhea", 2, (FCC, 7)),
    ("BCC", 9, "true", 1, (BCC, 9)), ("FCC", 2, "true", 3, (0, 0)),
    ("BCC", 1, "true", 3, (0, 0)), ("FCC", 1, "pyhea", 2, (0, 0)),
])
def test_stencil_detection(harness, tmp_path, typ, cell, shells, weights, want):
    spec = make_problem(typ, cell, [0.5, 0.5], weight=[4.0, 1.0, 0.5][:weights], shells=shells)
    assert _detect(harness, _write(tmp_path / "p.bin", spec)) == want


def test_stencil_detection_takes_any_row_order_and_no_other_table(harness, tmp_path):
    spec = make_problem("FCC", 4, [0.5, 0.5], shells="true")
    rng = np.random.default_rng(3)
    z = np.cumsum([0] + list(spec.shell_sizes))
    shuffled = np.concatenate([rng.permuted(spec.nbr[:, z[s]:z[s + 1]], axis=1)
                               for s in range(3)], axis=1)
    assert _detect(harness, _write(tmp_path / "a.bin", spec, shuffled)) == (FCC, 4)
    # one neighbour listed twice, two shells exchanged in one row, sites renumbered
    twice = spec.nbr.copy()
    twice[17, 0] = twice[17, 1]
    mixed = spec.nbr.copy()
    mixed[200, [0, 12]] = mixed[200, [12, 0]]
    perm = rng.permutation(spec.n_sites)
    renamed = np.empty_like(spec.nbr)
    renamed[perm] = perm[spec.nbr]
    for k, bad in enumerate((twice, mixed, renamed)):
        assert _detect(harness, _write(tmp_path / f"b{k}.bin", spec, bad)) == (0, 0)
