"""The oracle libraries are the ones the sources in this tree produce: they
build from scratch with the host compiler (the product's portable pow is
compiled for the host there), and a library that is older than its sources is
built again before it is loaded, so that no comparison runs against an oracle
the tree cannot produce."""
import ctypes
import os
import subprocess

import numpy as np

import pyoracle


def test_oracle_builds_from_scratch(tmp_path):
    subprocess.run(["make", "-s", "-B", "-C", pyoracle.HERE, "BUILD=%s" % tmp_path], check=True)
    names = ("liboracle.so", "liboracle_bxpow.so", "liboracle_helm.so")
    libs = [ctypes.CDLL(os.path.join(str(tmp_path), n)) for n in names]
    # the fresh build computes what the loaded one does: one HLLC face, whose
    # wave-speed estimate takes both powers
    UL = np.array([1.0, 0.3, -0.2, 2.9])
    UR = np.array([0.4, 0.1, 0.5, 0.7])
    F = np.zeros((2, 4))
    for f, l in zip(F, (libs[1], pyoracle._load(True))):
        l.or_hllc_face.argtypes = pyoracle._SIGS["or_hllc_face"]
        args = [v.ctypes.data_as(pyoracle.D) for v in (UL, UR)]
        assert l.or_hllc_face(2, 0, *args, 1.4, 1.0, f.ctypes.data_as(pyoracle.D)) == 0
    assert F[0].any() and F[0].tobytes() == F[1].tobytes()


def test_loading_builds_what_is_stale(monkeypatch):
    calls = []
    monkeypatch.setattr(pyoracle, "_libs", {})
    monkeypatch.setattr(pyoracle, "build", lambda: calls.append(1))
    pyoracle._load(True)
    pyoracle._load(False)
    assert len(calls) == 2
