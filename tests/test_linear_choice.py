"""Which kernel the table of measured products takes."""

import pytest

from fastgen_amd.kernels import linear


@pytest.fixture
def ask(monkeypatch):
    """Asks for one product of 64 rows, with the given measurements instead of the GPU's."""
    for table in ("choices", "timings", "_samples"):
        monkeypatch.setattr(linear, table, {})
    monkeypatch.setattr(linear, "force", None)
    recording = [False]
    monkeypatch.setattr(linear, "_capturing", lambda: recording[0])

    def run(names, measured=None, capturing=False, library_ties=False):
        recording[0] = capturing

        def measure(candidates, handicap, first):
            assert measured is not None, "measured once more"
            return dict(zip(names, measured))

        monkeypatch.setattr(linear, "_measure", measure)
        return linear._choose("silu_mul", 28672, 4096, 64, [(n, None) for n in names], library_ties=library_ties)

    return run


def test_one_matrix_that_lies_well_does_not_decide(ask):
    """The library's product is a fifth faster on some matrices than on others of the same shape."""
    names = ["wide", "library"]
    for measured in ((54.9, 48.6), (53.8, 60.1), (54.0, 61.0)):
        ask(names, measured)
    assert ask(names) == "wide" and ask(names, capturing=True) == "wide"


@pytest.mark.parametrize("wide,library", [(52.6, 58.6), (53.8, 54.0), (55.7, 53.8), (54.0, 58.6), (55.2, 53.5)])
def test_near_ties_go_to_the_same_kernel_in_every_process(ask, wide, library):
    """The times that different processes measured for one product: its kernel, and so its bits, must not depend on them."""
    for _ in range(4):
        assert ask(["wide", "library"], (wide, library)) == "wide"
    linear.choices.clear(), linear._samples.clear()
    for _ in range(4):
        assert ask(["wide", "library"], (library, wide), library_ties=True) == "library"


def test_a_lead_beyond_a_tie_decides_and_is_kept(ask):
    for _ in range(3):
        assert ask(["wide", "library"], (23.9, 19.8)) == "library"
    assert ask(["wide", "library"]) == "library" and not linear._samples


def test_a_clear_lead_is_not_measured_again(ask):
    assert ask(["wide", "library", "tiled"], (33.9, 19.8, 26.0)) == "library"
    assert ask(["wide", "library", "tiled"]) == "library" and not linear._samples
    assert ask(["wide", "tiled"], (33.9, 26.0)) == "tiled"  # the winner is not among the candidates: from the start
    assert ask(["wide", "tiled"]) == "tiled"


def test_the_fastest_of_several_wins(ask):
    assert linear._winner({"library": 50.0, "wide": 34.0, "tiled": 34.5}, ["library", "wide", "tiled"]) == "wide"


def test_nothing_is_measured_while_a_step_is_recorded(ask):
    assert ask(["wide", "library"], capturing=True) == "wide" and not linear.choices
    assert ask(["wide", "library"], (50.0, 40.0)) == "library"
    assert ask(["wide", "library"], capturing=True) == "library"  # not settled, but the best so far
    linear.choices.clear(), linear._samples.clear()
    linear.choices[("silu_mul", 28672, 4096, 64)] = "library"  # put there by a caller
    assert ask(["wide", "library"]) == "library"
