"""The relaxation polynomials of the electron diffusion kernels on the CPU:
x coth x of heatcap_poly.h, and the series of (e^u - 1)/u for |u| <= 1/4 as
spilady_amd/csrc/sld_dte.hip writes it, against long double."""
import os
import re

import numpy as np

from test_heatcap_poly import _consts, _horner

SRC = os.path.join(os.path.dirname(__file__), "..", "spilady_amd", "csrc", "sld_dte.hip")


def test_xcothx_fit():
    K = _consts()
    x = np.linspace(1e-6, K["kPolyXMax"], 20001)
    xl = x.astype(np.longdouble)
    ref = xl / np.tanh(xl)
    got = _horner(K["kXCothX"], x * x)
    assert np.max(np.abs((got - ref) / ref)) < 1e-15   # a few roundings of 1.1e-16


def test_expm1_series():
    body = re.search(r"kExpm1\[(\d+)\] = \{(.*?)\};", open(SRC).read(), re.S)
    c = [eval(v.strip()) for v in body.group(2).split(",")]
    assert len(c) == int(body.group(1))
    u = np.linspace(-0.25, 0.25, 20002)
    ul = u.astype(np.longdouble)
    ref = np.expm1(ul) / ul
    assert np.max(np.abs((_horner(c, u) - ref) / ref)) < 1e-15
