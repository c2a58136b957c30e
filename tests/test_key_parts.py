"""How the tile kernel's items are cut along their keys (host side, no GPU)."""

import random

import numpy as np
import pytest

from fastgen_amd.kernels import ops


@pytest.mark.parametrize("most", [None, 1, 3, 7])
def test_parts_cover_the_items(most):
    """Every item once, whole or in all of its parts; places and merges without gaps; results within their limit."""
    rng = random.Random(str(most))
    cuts = 0
    for _ in range(300):
        lens = [rng.randint(17, 3000) for _ in range(rng.randint(1, 4))]
        past = [rng.choice([0, 0, rng.randint(1, 20000)]) for _ in lens]
        n_kv, window = rng.choice([1, 2, 4, 8]), rng.choice([0, 0, 100, 4096])
        _, big = ops.attention_items(lens, np.concatenate([[0], np.cumsum(lens)]), past, rng.choice([1, 2, 3, 4, 8]), 128)
        cut = ops.cut_key_ranges(big, n_kv, 128, window, 256, most)
        if cut is None:
            continue
        cuts += 1
        items, parts, merges, n_places = cut
        assert n_places * n_kv * 128 * 136 * 4 <= ops.KEY_PART_MAX_BYTES
        seen = {}
        for it, (place, code) in zip(items.tolist(), parts.tolist()):
            seen.setdefault(tuple(it), []).append((place, code & 0xFFFF, code >> 16))
        assert set(seen) == {tuple(b) for b in big.tolist()}
        of = {(t, n): (place, k) for t, n, place, k in merges.tolist()}
        used = []
        for it, has in seen.items():
            if has[0][0] < 0:
                assert len(has) == 1
                continue
            place, k = of.pop((it[1], it[2]))
            assert k > 1 and sorted(has) == [(place + i, i, k) for i in range(k)]
            used += [p for p, _, _ in has]
        assert not of and sorted(used) == list(range(n_places))
    assert cuts > 20


def test_what_is_cut():
    """Long key ranges on few workgroups are cut; short ones, evenly loaded steps, block windows and wide heads are not."""
    def cut(lens, heads, n_kv, past=0, hd=128, window=0):
        _, big = ops.attention_items(lens, np.concatenate([[0], np.cumsum(lens)]), [past] * len(lens), heads // n_kv, 128)
        return ops.cut_key_ranges(big, n_kv, hd, window, 256)

    assert cut([100], 32, 8, past=8000) and cut([512], 32, 8, past=8000) and cut([611, 1437], 16, 4)
    assert cut([2048], 32, 8) is None and cut([2000], 16, 4) is None and cut([100], 32, 8) is None
    assert cut([512], 32, 8, past=8000, hd=192) is None and cut([512], 32, 8, past=8000, window=-4096) is None
    assert cut([512], 32, 8, past=8000, window=300) is None
    assert ops.cut_key_ranges(np.zeros((0, 4), np.int32), 8, 128, 0, 256) is None


def test_a_cut_beside_decoded_tokens_has_to_gain_more():
    """Decoded tokens' chunks fill the units that a long item leaves: prompts whose cut gains little alone stay whole beside them."""
    def cut(n, past, heads, n_kv, beside):
        _, big = ops.attention_items([n], [0, n], [past], heads // n_kv, 128)
        return ops.cut_key_ranges(big, n_kv, 128, 0, 256, beside=beside) is not None

    for n, past, heads, n_kv, worth_it in ((1500, 0, 16, 4, False), (1300, 0, 16, 4, False), (800, 1000, 16, 4, False), (500, 1500, 24, 8, False),
                                           (512, 2000, 32, 8, False), (512, 4000, 32, 8, True), (600, 3000, 16, 4, True), (100, 8000, 32, 8, True)):
        assert cut(n, past, heads, n_kv, False) and cut(n, past, heads, n_kv, True) == worth_it


@pytest.mark.parametrize("lens,heads,n_kv,rows,two,more", [
    ([300], 32, 8, 64, False, {}), ([512], 32, 8, 64, False, {}), ([513], 32, 8, 64, True, {}), ([380, 874], 24, 8, 64, True, {}),
    ([1280], 16, 4, 64, True, {}), ([1281], 16, 4, 128, None, {}), ([512] * 4, 16, 4, 64, True, {}), ([513] * 4, 16, 4, 128, False, {}),
    ([1280], 32, 8, 128, False, {}), ([1] * 8 + [896], 32, 8, 64, True, {}), ([1] * 8 + [897], 32, 8, 128, False, {}),
    ([1] * 8 + [768], 32, 8, 64, True, {}), ([1] * 8 + [1200], 16, 4, 64, True, {}), ([1] * 12 + [693, 1204], 16, 4, 128, False, {}),
    ([2048], 32, 8, 128, False, {}), ([1024], 32, 8, 128, False, dict(window=300)), ([1024], 32, 8, 64, True, dict(window=4096)),
    ([1024], 32, 8, 128, False, dict(page=32)), ([512], 32, 8, 64, False, dict(page=32)), ([1024], 32, 8, 128, False, dict(window=-64))])
def test_which_items_a_prompt_gets(monkeypatch, lens, heads, n_kv, rows, two, more):
    """Items of 64 rows where half of 256 units would stand idle, and, added up as the larger form does it, up to a workgroup a unit and ten
    passes (beside decoded tokens seven, or three workgroups for four units); from there on, where a window hides keys and on small pages the form of 128 rows, whose error against
    64 bits is smaller than that of 64 rows with one sum."""
    from types import SimpleNamespace

    import torch

    seen = []
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    monkeypatch.setattr(ops, "attention_tile_rows", lambda hd, small=False, exact=False, dist=False: 64 if small else 128)
    monkeypatch.setattr(ops, "upload", lambda values, dtype, device: torch.as_tensor(values))
    monkeypatch.setattr(ops, "attention_plan", lambda *a: None)
    lists, listed = ops.attention_items, []
    monkeypatch.setattr(ops, "attention_items", lambda *a: listed.append(a) or lists(*a))
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, tile_rows, key_parts, two_sums, **k: seen.append((a[6], tile_rows, key_parts, two_sums)))
    starts = np.concatenate([[0], np.cumsum(lens)])
    ctx = SimpleNamespace(q_lens=np.array(lens), n_cached=np.zeros(len(lens), int), q_start_host=starts, seq_records=None, scratch={})
    q = torch.empty(1, heads * 128, dtype=torch.bfloat16)
    pages = torch.empty(1, n_kv, more.get("page", 64), 128, dtype=torch.bfloat16)
    ops.paged_attention(q, q, pages, pages, SimpleNamespace(block_table=None), ctx, heads, 1.0, more.get("window", 0))
    (items, got, parts, sums), = seen
    assert got == rows and bool(sums) == bool(two) and (parts is not None) == (two is None)
    if two is None:  # (keys in parts)
        return
    assert len(listed) == 1  # (a step on new inputs waits for each list)
    assert int(items.view(-1, 4)[:, 2].max()) <= rows // (heads // n_kv)


def test_a_cut_takes_the_host_less_than_the_items_do():
    """A step on new inputs waits for the host: counting what a cut of its items gives is the lesser part of listing them."""
    import time

    lens = [611, 1437]
    starts = np.concatenate([[0], np.cumsum(lens)])
    _, big = ops.attention_items(lens, starts, [0, 0], 4, 128)
    assert ops.cut_key_ranges(big, 4, 128, 0, 256)

    def shortest(call):
        took = []
        for _ in range(200):
            t = time.perf_counter()
            call()
            took.append(time.perf_counter() - t)
        return min(took)

    assert shortest(lambda: ops.cut_key_ranges(big, 4, 128, 0, 256)) < shortest(lambda: ops.attention_items(lens, starts, [0, 0], 4, 128))


def test_a_second_stream_is_for_many_workgroups(monkeypatch):
    """The waits between two streams cost what the kernels gain beside each other up to about three workgroups a unit."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    assert [ops._tiles_beside(n) for n in (1, 273, 512, 764, 1000, 2000)] == [False] * 4 + [True] * 2
    monkeypatch.setattr(ops, "_ONE_STREAM", True)
    assert not ops._tiles_beside(2000)
