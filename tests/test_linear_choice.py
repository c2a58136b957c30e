"""Which kernel the table of measured products takes."""

import pytest
import torch

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


@pytest.mark.parametrize("times,winner", [([(54.9, 48.6), (53.8, 60.1), (54.0, 61.0)], "wide"),  # the first matrix lies well
                                          ([(50.0, 40.0), (50.0, 49.0), (50.0, 40.0)], "library")])
@pytest.mark.parametrize("n_matrices", [1, 2, 3, 5])
def test_a_product_is_settled_before_it_is_used(ask, monkeypatch, times, winner, n_matrices):
    """The first pass takes the kernel that later ones take, whatever it is and however few matrices a model has: a step that is
    recorded after one warm-up (two layers, one head) and the next engine's have the same bits.  The samples are of
    one matrix after the other."""
    ask(["wide"])  # (installs the fixture's table)
    left, on = list(times), []
    run = [("wide", lambda m: on.append(m)), ("library", lambda m: None)]

    def measure(candidates, handicap, first):
        candidates[0][1]()
        return dict(zip(("wide", "library"), left.pop(0)))

    monkeypatch.setattr(linear, "_measure", measure)
    settle = lambda: linear._settle("silu_mul", 28672, 4096, 64, run, lambda: list(range(n_matrices)))
    assert settle() == winner and not left and not linear._samples
    assert on == [i % n_matrices for i in range(3)]
    monkeypatch.setattr(linear, "_capturing", lambda: True)
    assert settle() == winner
    monkeypatch.setattr(linear, "_capturing", lambda: False)
    assert settle() == winner


def test_settling_ends_where_nothing_is_measured(ask, monkeypatch):
    ask(["wide"])
    two = [("wide", lambda m: None), ("library", lambda m: None)]
    settle = lambda names: linear._settle("silu_mul", 28672, 4096, 64, names, lambda: [0])
    assert settle(two[:1]) == "wide" and not linear.choices  # one candidate
    monkeypatch.setattr(linear, "force", "library")
    assert settle(two) == "library" and not linear.choices
    monkeypatch.setattr(linear, "force", None)
    monkeypatch.setattr(linear, "_capturing", lambda: True)
    assert settle(two) == "wide" and not linear.choices  # first met inside a recording


def test_matrices_that_are_measured_for_one_another():
    """The stored matrices of one shape, layout and alignment, as long as somebody holds them; of a part of a matrix the
    same parts."""
    make = lambda *shape: linear.streamed(torch.zeros(*shape, dtype=torch.bfloat16))
    a, b, other = make(48, 64), make(48, 64), make(64, 48)
    c = linear.StreamedMatrix(torch.zeros(48, 64, dtype=torch.bfloat16))  # stored by nobody
    assert [m is x for m, x in zip(a.alike(), (a, b))] == [True, True] and len(a.alike()) == 2
    assert other.alike() == [other] and len(c.alike()) == 3 and c.alike()[0] is c
    part = b.first_rows(16).alike()
    assert [m.rows.data_ptr() for m in part] == [b.rows.data_ptr(), a.rows.data_ptr()] and all(m.shape == (16, 64) for m in part)
    del a, part
    assert len(b.alike()) == 1
    assert len(linear._stored[linear._kind(make(48, 64))]) <= 2  # what is gone is not kept
