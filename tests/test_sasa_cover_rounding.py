"""The cover arcs formed in single precision, with the device's approximate
reciprocal and square root modelled on the host.

A cover arc decides that a circle's transitions are left out, so whatever it
claims must hold: at every angle of the arc and SA_COV_EPS (1e-5 rad) beyond
its ends the exact containment value is at least SA_COV_DELTA (1e-3).
"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
UNIT = 2.0 ** -23                       # a unit in the last place, relative to the smallest significand


@pytest.fixture(scope="module", params=[(0.0, 0.0), (1, 1), (1, -1), (-1, 1), (-1, -1)],
                ids=lambda p: "rcp%+g_sqrt%+g" % p)
def arcs_of(request, tmp_path_factory):
    so = str(tmp_path_factory.mktemp("cover") / "libcover.so")
    err = ["%.9ef" % (UNIT * k) for k in request.param]
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-DOG_COVER_RCP_ERR=" + err[0], "-DOG_COVER_SQRT_ERR=" + err[1], "-o", so,
                    os.path.join(HERE, "host", "sasa_core_host.cpp")], check=True)
    host = C.CDLL(so)
    dp = C.POINTER(C.c_double)

    def call(pairs):
        n = len(pairs)
        pairs = np.ascontiguousarray(pairs)
        arcs, basis = np.zeros((n, 2), np.float32), np.zeros((n, 6))
        host.host_cover_arcs(n, pairs.ctypes.data_as(dp), arcs.ctypes.data_as(C.POINTER(C.c_float)),
                             basis.ctypes.data_as(dp))
        return arcs, basis
    return call


def _unit(rng, n):
    v = rng.normal(size=(n, 3))
    return v / np.linalg.norm(v, axis=1)[:, None]


def _caps(rng, n, kind):
    n1, n2 = _unit(rng, n), _unit(rng, n)
    c1, c2 = rng.uniform(-0.99, 0.99, n), rng.uniform(-0.99, 0.99, n)
    if kind == "small circles":
        c1 = np.sqrt(1.0 - 10.0 ** rng.uniform(-5.5, -1.0, n)) * rng.choice([-1.0, 1.0], n)
    elif kind == "near axes":           # small amplitudes
        n2 = n1 * rng.choice([-1.0, 1.0], n)[:, None] + 10.0 ** rng.uniform(-3.2, -0.5, n)[:, None] * n2
        n2 /= np.linalg.norm(n2, axis=1)[:, None]
    # the other cap's cosine puts many arcs next to none, half and full circles
    t = np.sum(n1 * n2, axis=1)
    amp = np.sqrt((1.0 - c1 ** 2) * np.maximum(1.0 - t ** 2, 0.0))
    at = rng.random(n) < 0.7
    c2 = np.where(at, c1 * t - 1e-3 + amp * np.cos(np.pi * rng.random(n) ** 2), c2)
    ok = np.abs(c2) < 0.9999
    return np.concatenate([n1, c1[:, None], n2, c2[:, None]], axis=1)[ok]


@pytest.mark.parametrize("kind", ["any", "small circles", "near axes"])
def test_claimed_angles_are_covered(arcs_of, kind):
    pairs = _caps(np.random.default_rng(17), 60000, kind)
    arcs, basis = arcs_of(pairs)
    full = arcs[:, 1] >= 100.0
    part = (arcs[:, 1] > 0.0) & ~full
    assert part.sum() > 3000
    n1, c1, n2, c2 = pairs[:, :3], pairs[:, 3], pairs[:, 4:7], pairs[:, 7]
    s1 = np.sqrt(1.0 - c1 ** 2)
    worst = np.inf
    for f in np.linspace(0.0, 1.0, 9):
        a, w = arcs[:, 0].astype(np.float64) - 1e-5, arcs[:, 1].astype(np.float64) + 2e-5
        phi = np.where(full, 2.0 * np.pi * f, a + f * w)
        x = n1 * c1[:, None] + s1[:, None] * (np.cos(phi)[:, None] * basis[:, :3] + np.sin(phi)[:, None] * basis[:, 3:])
        worst = min(worst, (np.sum(x * n2, axis=1) - c2)[full | part].min())
    print("%s: least depth %.6e over %d arcs" % (kind, worst, (full | part).sum()))
    assert worst >= 1e-3
