"""The PCG reduction's items against the left-to-right loop, bit for bit, where
they can go wrong: runs that end at tile and window edges, tiles with more
items than fit, predictions that miss because the running sum hovers at a
power of two, and values that no run can hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim_mod():
    from cloth_sim_self_collision_amd import _lib, sim
    if _lib.device_count() < 1:
        pytest.skip("no HIP device")
    return sim


def _sequential(t):
    with np.errstate(all="ignore"):
        return np.cumsum(t)[-1]  # numpy accumulates left to right


def _hover(rng, n):
    """A running sum within a few ulps of 1, above and below."""
    t = rng.choice([-3, -2, -1, 1, 2, 3], n) * 2.0 ** -53
    t[0] = 1.0
    return t


def _cancel(rng, n):
    """Products like (r, z): magnitudes over many orders, cancelling."""
    t = rng.standard_normal(n) * 10.0 ** np.linspace(60, 20, n)
    t[1::2] = -t[0::2][: len(t[1::2])] * (1 + 1e-10 * rng.standard_normal(len(t[1::2])))
    return t


def _waves(rng, n):
    """The running sum swings through zero every few addends."""
    return np.cos(np.arange(n) * rng.uniform(0.3, 2.5)) * np.exp2(rng.integers(-3, 4, n))


def _mostly_quiet(rng, n):
    """Long runs with a binade change here and there."""
    t = np.abs(rng.standard_normal(n)) * 1e-3
    at = rng.integers(0, n, max(1, n // 700))
    t[at] = rng.standard_normal(len(at)) * 10.0 ** rng.integers(0, 9, len(at))
    return t


KINDS = {"hover": _hover, "cancel": _cancel, "waves": _waves, "quiet": _mostly_quiet,
         "walk": lambda rng, n: rng.standard_normal(n),
         "falling": lambda rng, n: -np.exp2(-np.arange(n) * (900.0 / n)),
         "subnormal": lambda rng, n: rng.integers(-9, 10, n) * 5e-324,
         "zeros": lambda rng, n: np.where(rng.random(n) < 0.999, 0.0, rng.standard_normal(n))}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 3 * 1024 + 7, 4 * 1024, 4 * 1024 + 1,
                               63 * 1024 + 5, 64 * 1024,
                               65 * 1024 + 3, 200 * 1024 + 77])
def test_items_equal_the_loop(sim_mod, kind, n):
    rng = np.random.default_rng(n)
    t = KINDS[kind](rng, n)
    assert np.array_equal(sim_mod.ordered_sum(t), _sequential(t), equal_nan=True)


@pytest.mark.parametrize("name", ["at the cap", "past the cap", "full windows"])
def test_tiles_with_as_many_items_as_fit(sim_mod, name):
    from test_item_sum_emulation import crafted
    t = crafted()[name]
    assert sim_mod.ordered_sum(t) == _sequential(t)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 1.7e308])
@pytest.mark.parametrize("at", [0, 1023, 1500, 70000])
def test_special_values(sim_mod, bad, at):
    rng = np.random.default_rng(at)
    t = _cancel(rng, 70 * 1024 + 9)
    t[at:at + 2] = bad
    assert np.array_equal(sim_mod.ordered_sum(t), _sequential(t), equal_nan=True)
