"""CPU checks of the spreading kernels' constants and of the code that they
share with the host."""
import os
import re

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyiid_amd", "csrc")


def constants(header, name):
    text = open(os.path.join(CSRC, header)).read()
    body = re.search(r"constexpr float %s\[\d\]\[\d\] = \{(.*?)\n\};" % name, text, re.S).group(1)
    rows = re.findall(r"\{([^{}]*)\}", body)
    return np.array([[np.float32(v.strip().rstrip("f")) for v in r.split(",")] for r in rows])


def test_window_has_no_common_factor():
    """The F grid's window, averaged over a pair's place between the grid points,
    against its transform phihat: what is left multiplies F as a whole, where the
    errors at single places average out.  v_rcp_f32, which the weight 1/r comes
    from, is 6.8e-9 short on average.  Allowed: 4e-9, the least squares residue
    of the window (3.6e-9 r.m.s.)."""
    v = constants("fq_grid.h", "kFqVal").astype(np.float64)
    assert v.shape == (3, 6)
    y = (np.arange(4000) + 0.5) / 4000 - 0.5
    powers = y[None] ** np.arange(6)[:, None]
    mirror = (-y)[None] ** np.arange(6)[:, None]
    taps = np.concatenate([v @ powers, (v @ mirror)[::-1]])
    beta = 15.160
    for q in np.linspace(0.0, np.pi / 6, 33):
        a = np.sqrt(beta ** 2 - 9.0 * q * q)
        phihat = np.sinh(a) / a / (np.sinh(beta) / beta)
        z = (taps * np.exp(1j * q * (np.arange(6)[:, None] - 2.5 - y[None]))).sum(0) / phihat
        assert abs(z.mean() * (1.0 - 6.755e-9) - 1.0) < 4e-9, q
        assert np.sqrt((np.abs(z - 1.0) ** 2).mean()) < 1.2e-8, q
