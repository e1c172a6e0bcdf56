"""Kernels of universes whose noise is jumps alone draw no normals and load no table for them."""
import pytest

from conftest import GBM, JUMP
from test_host import generate


@pytest.mark.parametrize("eqs,wiener", [
    (["dX = (2.0 * (0.5 - X)) * dt + (0.1) * dN1(X)"], False),
    (["dX = (1.0) * dN1(X) + (0.5) * dN2(3.0)", "Y = X * X"], False),
    (JUMP, True),
    (GBM, True),
])
def test_generated_flag(eqs, wiener):
    for precision in (0, 1):
        for rng, scramble in ((0, 0), (1, 0), (1, 1)):
            src = generate(eqs, 9, precision=precision, rng=rng, scramble=scramble, outputs=1)
            assert ("WIENER = %s;" % ("true" if wiener else "false")) in src
