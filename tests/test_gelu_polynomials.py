"""The two polynomials of the warm-start network's GELU, as rounded in the HIP
source, against scipy in double: Phi near zero and q(a) = erfcx(a / sqrt 2) / 2
beyond."""
import os
import re

import numpy as np
from scipy.special import erf, erfcx

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ipc_warp_amd", "csrc", "mlp.hip")


def _coefficients(name):
    body = re.search(name + r"\[\d+\] = \{([^}]*)\}", open(SRC).read()).group(1)
    return np.array([np.float32(v.strip().rstrip("f")) for v in body.split(",")], np.float64)


def test_centre_polynomial():
    z = np.linspace(0, 1.25, 100001)
    assert np.abs(z * np.polyval(_coefficients("kCentre"), z * z) - 0.5 * erf(z / np.sqrt(2))).max() <= 1.2e-9


def test_tail_polynomial():
    a = np.linspace(1.25, 14, 100001)
    t = 1 / (1 + np.float64(np.float32(0.3)) * a)
    assert np.abs(np.polyval(_coefficients("kTail"), t) * t / (0.5 * erfcx(a / np.sqrt(2))) - 1).max() <= 2.9e-8
