"""The device's inverse normal against the oracle's, one draw per path: dX = (1.0) * dW1 over one unit
step, so X_1 is the draw itself. Random draws of each generator, and XOR-scrambled points around
the words where the evaluation changes: both ends of the unit interval, its middle, powers of two
and the edges of the table's segments."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NOISE = ["dX = (1.0) * dW1"]
TIMES = [0.0, 1.0]


def _draws(paths, rng, precision, **kw):
    import sde_sim_rs
    plan = sde_sim_rs.Plan(NOISE, TIMES, paths, {"X": 0.0}, rng, "euler", precision=precision, **kw)
    f = plan.new_filtration()
    plan.run(f)
    torch.cuda.synchronize()
    return f[1, 0].cpu().numpy().astype(np.float64)


def _bound(z):
    """f64: t = sqrt(-2 ln q) carries half of its logarithm's 1 ulp and its own rounding, the rational
    R = t - |z| its own quotient's, with |dz/dt| <= 1, and the difference half an ulp of z: 2.5 ulp
    of max(t, R, 1) on each side (t <= |z| + 1.3 and R <= 2.6 over the whole range)."""
    return 2 * 2.5 * 2.0 ** -52 * (np.abs(z) + 2.6)


def _index_of(word, mask):
    """The point index whose scrambled first coordinate is `word`: dimension 0 is the bit reversal of
    the index's Gray code."""
    g = int("{:032b}".format(word ^ mask)[::-1], 2)
    i = 0
    while g:
        i ^= g
        g >>= 1
    return i


@pytest.mark.parametrize("rng,scramble", [("pseudo", "shift"), ("sobol", "shift"), ("sobol", "xor")])
def test_random_draws_match_the_oracle(oracle, rng, scramble):
    S = (1 << 16) + 37
    kw = dict(seed=9, scramble=scramble, scramble_seed=21)
    print("case: f64 inverse normal, %s %s" % (rng, scramble), flush=True)
    got = _draws(S, rng, "f64", **kw)
    ref = oracle.simulate(NOISE, TIMES, S, {"X": 0.0}, rng=rng, **kw)[:, 1, 0]
    assert np.all(np.abs(got - ref) <= _bound(ref)), np.max(np.abs(got - ref) / _bound(ref))


WORDS = [0, 1, 2, 1232, 1233, (1 << 16) - 1, 1 << 16, (1 << 22) - 1, 1 << 30, (1 << 30) + (1 << 22), (1 << 31) - 1]


@pytest.mark.parametrize("word", WORDS + [0xFFFFFFFF - w for w in WORDS])
def test_edge_words_match_the_oracle(oracle, word):
    """A few paths from the point whose scrambled word is exactly `word` (u = (word + 1/2) 2^-32)."""
    seed, S = 33, 3
    mask = int(oracle.xor_masks(seed, 1)[0])
    first = min(_index_of(word, mask), 2 ** 32 - S)
    kw = dict(scramble="xor", scramble_seed=seed, sobol_first=first)
    print("case: f64 inverse normal, word %d, index %d" % (word, first), flush=True)
    got = _draws(S, "sobol", "f64", **kw)
    ref = oracle.simulate(NOISE, TIMES, S, {"X": 0.0}, rng="sobol", **kw)[:, 1, 0]
    assert np.all(np.abs(got - ref) <= _bound(ref)), (got, ref)


@pytest.mark.parametrize("paths", [1, 65, (1 << 18) + 3])
def test_batched_f32_draws_match_the_oracle(oracle, paths):
    """One-step f32 OU instances with dX = 1 dW (kappa = 0, sigma = 1): the terminal value is the draw.
    2^18 draws reach the rare path (|z| > 4.17) about eight times. Bound: the f32 rational's of
    fp32_bounds, which the rare draws take, plus one rounding; the table's quadratics round less often and
    take the same q."""
    import sde_sim_rs
    import fp32_bounds as B
    print("case: batched f32 draws, %d paths" % paths, flush=True)
    inst = dict(kind=1, steps=1, paths=paths, x0=0.0, horizon=1.0, p0=0.0, p1=0.0, p2=1.0, seed=77)
    b = sde_sim_rs.Batch([inst], precision="f32", keep_terminal=True)
    b.run()
    got = b.terminal().astype(np.float64)
    u = np.array([oracle.pseudo_f64(77 + s, 1)[0] for s in range(paths)])
    z = B.inv_normal(u)
    bound = B.psi_error_words(u) + B.U * np.abs(z)
    assert np.all(np.abs(got - z) <= bound), np.max(np.abs(got - z) / bound)
