"""Which f64 universes keep the library's logarithm, root and division: those whose noise holds a root that is not
shown to be steadied by the drift, wherever its argument vanishes (generated sources, no device needed)."""
import pytest

from conftest import GBM, HESTON, JUMP
from test_host import generate

HESTON_VARIANCE = HESTON[1]


@pytest.mark.parametrize("eqs,library", [
    (GBM, False),
    (HESTON, False),
    (JUMP, False),
    ([HESTON[0], HESTON_VARIANCE.replace("0.5 * max", "2.0 * max")], True),           # 4 a < s^2
    (["dX = (0.5 * (0.03125 - max(X, 0))) * dt + (0.25 * max(X, 0)^0.5) * dW1"], False),  # 4 a = s^2
    (["dX = (0.5 * (0.03125 - X)) * dt + (0.25 * X^0.5) * dW1"], False),
    (["dX = (0.5 * (0.03125 - X)) * dt + (0.2501 * max(0, X)^0.5) * dW1"], True),
    # Roots elsewhere than at 0.
    (["dX = (0.5 * (0.97 - X)) * dt + (0.8 * max(X * (1 - X), 0)^0.5) * dW1"], True),
    (["dX = (0.5 * (0.97 - X)) * dt + (0.8 * max(X, 0)^0.5 * max(1 - X, 0)^0.5) * dW1"], True),
    (["dv = (2.0 * (0.04 - v)) * dt + (0.3 * max(v - 0.01, 0)^0.5) * dW1"], True),
    (["dX = (1 - X) * dt + (abs(X - 2)^0.5) * dW1"], True),
    # A drift that depends on the time, on another process, or joins a jump.
    (["dv = (2.0 * (0.04 - t - max(v, 0))) * dt + (0.2 * max(v, 0)^0.5) * dW1"], True),
    (["dv = (2.0 * (m - max(v, 0))) * dt + (0.2 * max(v, 0)^0.5) * dW1", "dm = (0.04 - m) * dt + (0.1) * dW2"], True),
    (["dv = (2.0 * (0.04 - max(v, 0))) * dt + (0.2 * max(v, 0)^0.5) * dW1 + (-0.01) * dN1(3.0)"], True),
    # Another process's root, of a process that crosses 0.
    (["dS = (0.1 * S) * dt + (S * max(v, 0)^0.5) * dW1", "dv = (0.04 - v) * dt + (0.1) * dW2"], True),
    # A process whose noise vanishes like itself, with a drift that keeps it there or not.
    (["dS = (0.1 * S) * dt + (S * max(v, 0)^0.5) * dW1", "dv = (0.05 * v) * dt + (0.4 * v) * dW2"], False),
    (["dS = (0.1 * S) * dt + (S * v^0.5) * dW1", "dv = (2.0 * (0.04 - v)) * dt + (0.4 * v) * dW2"], False),
    (["dS = (0.1 * S) * dt + (S * v^0.5) * dW1", "dv = (2.0 * (-0.04 - v)) * dt + (0.4 * v) * dW2"], True),
    (["dX = (2.0 * (0.04 - X)) * dt + (0.4 * X * max(X, 0)^0.5) * dW1"], False),
    (["dS = (0.1 * S) * dt + (S * max(v, 0)^0.5) * dW1", "dv = (0.1) * dt + (0.4 * max(v, 0)^0.75) * dW2"], True),
    (["dS = (0.1 * S) * dt + (S * max(v, 0)^0.5) * dW1", "dv = (0.04 - v) * dt"], False),
    # Through an algebraic process, as another power, as a logarithm or an inverse function.
    (["dX = (0.5 * (0.97 - X)) * dt + (0.8 * R) * dW1", "R = max(X * (1 - X), 0)^0.5"], True),
    (["dX = (0.5 * (0.97 - X)) * dt + (0.8 * A^0.5) * dW1", "A = X * (1 - X)"], True),
    (["dX = (0.1 * X) * dt + (0.2 * max(X, 0)^0.7) * dW1"], True),
    (["dX = (0.1 * X) * dt + (0.2 * max(X, 0)^(0.4 + t)) * dW1"], True),
    (["dX = (0.1 * X) * dt + (0.2 * 2.718^(0.5 * log(2.718, X))) * dW1"], True),
    (["dX = (1 - X) * dt + (acosh(1 + X)) * dW1"], True),
    (["dX = (0.1) * dt + (max(X, 0)^0.5) * dN1(2.0)"], True),
    # No root of a process in the noise.
    (["dX = (0.1) * dt + (0.3 * t^0.5) * dW1"], False),
    (["dX = (0.1 * X) * dt + (0.2 * X^1.5 + X^2 + X^3) * dW1"], False),
    (["dX = (0.1 * X) * dt + (0.2 * X / (1 + X^2)) * dW1"], False),
    (["dX = (max(X, 0)^0.5) * dt + (0.3) * dW1"], False),
    (["dX = (0.1 * X) * dt + (0.3 * X) * dW1", "Y = max(X, 0)^0.5"], False),
    (["dX = (0.1 * X) * dt + (0.3 * A) * dW1", "A = B + X", "B = A"], False),
])
def test_library_form(eqs, library):
    f64, f32 = 0, 1
    for precision, rng, scramble in ((f64, 0, 0), (f64, 1, 0), (f64, 1, 1), (f32, 0, 0)):
        src = generate(eqs, 9, precision=precision, rng=rng, scramble=scramble, outputs=1)
        assert ("SDE_LIBRARY_F64" in src) == (library and precision == f64)
