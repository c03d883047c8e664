"""The host's spectral norm (host_la.cpp, compiled here) over the range of magnitudes: numpy's to 1e-6 (the power
iteration's accuracy on random matrices) wherever the square of |A|^2 is finite, and not finite, never a
small number, where it is not (acceptance bars scale with the norm)."""
import ctypes
import subprocess

import numpy as np
import pytest

from conftest import PACKAGE_DIR

SHIM = """
#include "host_la.h"
extern "C" double norm(int n, const double* a) {
    rc::Mat m((size_t)n * n);
    for (size_t i = 0; i < m.size(); ++i) m[i] = rc::cd(a[2 * i], a[2 * i + 1]);
    return rc::opnorm2(n, m);
}
"""


@pytest.fixture(scope="module")
def norm(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_la")
    (d / "shim.cpp").write_text(SHIM)
    csrc = PACKAGE_DIR / "csrc"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{csrc}", "-o", str(d / "t.so"), str(d / "shim.cpp"),
                    str(csrc / "host_la.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))
    lib.norm.restype = ctypes.c_double
    lib.norm.argtypes = [ctypes.c_int, ctypes.c_void_p]
    return lambda a: lib.norm(len(a), np.ascontiguousarray(a, dtype=np.complex128).ctypes.data)


@pytest.mark.parametrize("n", [1, 2, 5, 33, 64])
def test_norm_over_magnitudes(norm, n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    for scale in (1e-60, 1e-3, 1.0, 1e3, 1e60):
        assert norm(scale * a) == pytest.approx(np.linalg.norm(scale * a, 2), rel=1e-6)
    assert norm(0 * a) == 0.0
    for scale in (1e80, 1e150):
        assert not np.isfinite(norm(scale * a))
    a[0, 0] = np.nan
    assert not np.isfinite(norm(a))
