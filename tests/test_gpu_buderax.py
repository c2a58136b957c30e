"""Buderax on the GPU against the plain implementation (``tests/plain_buderax.py``): each new
mechanism alone, then whole models of several shapes under every way of cutting requests into steps,
with small pools so that pages and slots change hands, in float32 (strict) and bfloat16."""

from __future__ import annotations

from typing import Dict, List

import pytest
import torch

import traces
from helpers import assert_close, make_runner, run_trace, save_model_folder
from plain_buderax import (ALL_LOOP, ONE_PASS, PLAIN_STACK, SMALL_LOOP, plain_buderax_forward, plain_buderax_greedy,
                           plain_buderax_weights, plain_mixture, plain_route, plain_scaled_embedding,
                           plain_zero_centred_rmsnorm)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CONFIGS = {"small_loop": SMALL_LOOP, "plain_stack": PLAIN_STACK, "all_loop": ALL_LOOP, "one_pass": ONE_PASS}


def _tokens(config, lengths: Dict[str, int], seed: int) -> Dict[str, List[int]]:
    g = torch.Generator().manual_seed(seed)
    return {r: torch.randint(0, config["vocab"], (n,), generator=g).tolist() for r, n in lengths.items()}


def _mostly_close(got, want, noise, what):
    """bfloat16: a routing decision that lies within rounding of a tie may fall the other way than in the
    plain bfloat16 run, and the positions that read that token then differ by more than rounding.  Nine in
    ten positions of a request keep to the tolerance of ``assert_close`` (twice the plain bfloat16 run's
    worst error), none is off by more than a routing decision can explain, and all are finite."""
    for rid, w in want.items():
        g = got[rid]
        assert g.shape == w.shape and torch.isfinite(g).all(), f"{what} {rid}"
        err = (g - w).abs().amax(-1)
        tol = 2.0 * float((noise[rid] - w).abs().max()) + 1e-3 * float(w.abs().max())
        assert float((err <= tol).float().mean()) >= 0.9, f"{what} {rid}: {(err > tol).nonzero().flatten().tolist()} over {tol:.3e}"
        assert float(err.max()) <= 0.5 * float(w.abs().max()), f"{what} {rid}: {float(err.max()):.3e}"


# ------------------------------------------------------------ mechanisms alone
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding_scale_offset_norm_and_stream_additions(dtype):
    from fastgen_amd.config import PartSpec
    from fastgen_amd.kernels import ops
    from fastgen_amd.parts import build_part

    g = torch.Generator().manual_seed(0)
    V, D, T = 37, 72, 9
    table = (torch.randn(V, D, generator=g)).to(torch.bfloat16).float()
    tok = torch.randint(0, V, (T,), generator=g)
    emb = build_part("embedding", PartSpec("embedding", "embed", dict(vocab_size=V, dim=D, scale=3.5, names={"weight": ""})))
    emb.load({"embed": table}, dtype, DEV)
    h = emb.forward(tok.to(DEV, torch.int32))
    want = plain_scaled_embedding(table, tok, 3.5)
    torch.testing.assert_close(h.cpu(), want, rtol=0, atol=0)
    # the norm's weight is stored around zero
    w = (torch.randn(D, generator=g) * 0.3).to(torch.bfloat16).float()
    norm = build_part("norm", PartSpec("rmsnorm", "n", dict(dim=D, eps=1e-5, unit_offset=True, names={"weight": ""})))
    norm.load({"n": w}, dtype, DEV)
    delta = torch.randn(T, D, generator=g).to(dtype)
    out = norm.forward(h, delta.to(DEV), dtype)
    want_h = want + delta.float()
    torch.testing.assert_close(h.cpu(), want_h, rtol=1e-6, atol=1e-6)
    tol = dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(out.float().cpu(), plain_zero_centred_rmsnorm(want_h, w, 1e-5), **tol)
    # what enters the stream at the start of a pass: what was left to add, the embedding again, the pass's vector
    step = torch.randn(3, D, generator=g)
    loop = build_part("injection", PartSpec("loop_input", "loop", dict(dim=D, times=3)))
    loop.load({"loop.step": step}, dtype, DEV)
    parts = torch.randn(2, T, D, generator=g)
    for index, pending in ((0, None), (2, delta.to(DEV)), (1, parts.to(DEV))):
        hh = want_h.clone().to(DEV)
        loop.forward(hh, pending, want.to(DEV), index)
        ref = want_h.clone()
        if pending is not None:
            ref = ref + (delta.float() if pending.dim() == 2 else parts[0] + parts[1])
        if index > 0:
            ref = ref + want
        torch.testing.assert_close(hh.cpu(), ref + step[index], rtol=1e-6, atol=1e-5)
    # the gate on the heads' outputs, from columns of a wider tensor
    x, wide = torch.randn(T, 48, generator=g).to(dtype), torch.randn(T, 80, generator=g).to(dtype)
    xd = x.to(DEV)
    ops.gate_mul(xd, wide.to(DEV)[:, 32:])
    torch.testing.assert_close(xd.float().cpu(), (x.float() * torch.sigmoid(wide[:, 32:].float())).to(dtype).float(), **tol)
    a, b = torch.randn(T, D, generator=g).to(dtype), torch.randn(T, D, generator=g).to(dtype)
    torch.testing.assert_close(ops.add_rows(a.to(DEV), b.to(DEV)).cpu()[0], a.float() + b.float(), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,E,top,F,T", [(64, 5, 2, 24, 70), (96, 4, 1, 20, 7), (40, 6, 6, 16, 33), (128, 3, 2, 64, 300),
                                         (64, 70, 3, 8, 1), (72, 4, 2, 44, 230), (64, 2, 1, 40, 90), (48, 3, 2, 20, 400)])
def test_routed_experts_alone(dtype, D, E, top, F, T):
    """Router, sort, the experts' products and the weighted sum against the plain mixture: few rows (tiles of
    16) and many rows an expert (larger tiles, and those that go through LDS), all experts chosen, one
    chosen, more experts than a wave has lanes, widths that are no multiple of 8 or of 32."""
    from fastgen_amd.config import PartSpec
    from fastgen_amd.kernels import ops
    from fastgen_amd.parts import build_part

    config = {"width": D, "vocab": 8, "layers": [{"mixer": dict(heads=1, kv_heads=1, dim=8, vdim=8),
                                                   "mlp": {"router": {"experts": E, "top": top}, "expert": {"ff": F}}}]}
    w = plain_buderax_weights(config, D + E)
    g = torch.Generator().manual_seed(T)
    n = torch.randn(T, D, generator=g).to(torch.bfloat16).float()
    plus = torch.randn(T, D, generator=g).to(torch.bfloat16).float()
    part = build_part("feed_forward", PartSpec("moe", "l0.mlp", dict(
        dim=D, hidden_dim=F, n_experts=E, top=top,
        names={"router.weight": "router", "router.bias": "router.b", "expert": "e{}", "gate_proj.weight": "gate",
               "up_proj.weight": "up", "down_proj.weight": "down"})))
    part.load(w, dtype, DEV)
    choice, weight = ops.moe_route(n.to(DEV, dtype), part.router, part.bias, top)
    idx, wt = plain_route(n, w["l0.mlp.router"], w["l0.mlp.router.b"], top)
    assert torch.equal(choice.cpu().long(), idx)
    torch.testing.assert_close(weight.cpu(), wt, rtol=1e-5, atol=1e-6)
    got = part.forward(n.to(DEV, dtype), plus=plus.to(DEV, dtype)).cpu()[0]
    want = plain_mixture(n, w, "l0.mlp", config["layers"][0]["mlp"]) + plus
    if dtype == torch.float32:
        torch.testing.assert_close(got, want, rtol=2e-5, atol=2e-5)
    else:
        low = plain_mixture(n.to(dtype), {k: v.to(dtype) for k, v in w.items()}, "l0.mlp", config["layers"][0]["mlp"]) + plus
        assert float((got - want).abs().max()) <= 2.0 * float((low - want).abs().max()) + 1e-3 * float(want.abs().max())
    alone = part.forward(n.to(DEV, dtype)).cpu()[0]
    torch.testing.assert_close(alone + plus, got, rtol=1e-5, atol=1e-5)


# ----------------------------------------------------------------- whole models
LENGTHS = {"a": 150, "b": 37, "c": 2, "d": 1, "e": 70, "f": 19}


@pytest.fixture(scope="module")
def cases(tmp_path_factory):
    out = {}
    for name, config in CONFIGS.items():
        weights = plain_buderax_weights(config, seed=len(name), sharpen=5.0)
        folder = save_model_folder(tmp_path_factory.mktemp(name), config, weights)
        toks = _tokens(config, LENGTHS, seed=7)
        out[name] = (config, weights, folder, toks, {r: plain_buderax_forward(weights, config, t) for r, t in toks.items()})
    return out


def _all_traces(lengths):
    return {"whole": traces.whole(lengths), "tail": traces.tail(lengths, 40), "chunks": traces.chunks(lengths),
            "mixed": traces.mixed(lengths, seed=3), "mixed2": traces.mixed(lengths, max_live=3, seed=11, budget=23)}


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_float32_every_cut_batch_and_reuse(cases, name):
    """Whole prompts, prompts then single tokens, portions down to two tokens and one, mixed batches of
    unequal requests: the same logits as the plain run, and the same bits whatever the cut.  Pages of 16
    tokens and a pool that holds the live requests only: pages and slots are used again."""
    config, weights, folder, toks, want = cases[name]
    runner = make_runner(folder, torch.float32, page_size=16, max_tokens=304, max_requests=4)
    first = None
    for kind, tr in _all_traces(LENGTHS).items():
        got = run_trace(runner, tr, toks)
        assert_close(got, want, torch.float32, None, f"buderax {name} {kind}")
        if first is None:
            first = got
        else:
            for r in got:
                assert torch.equal(got[r], first[r]), f"{name} {kind}: request {r} depends on the cut"
        assert runner.cache.free_pages() == 304 // 16 and runner.cache.free_slots() == 4


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_bfloat16_every_cut_batch_and_reuse(cases, name):
    config, weights, folder, toks, want = cases[name]
    noise = {r: plain_buderax_forward(weights, config, t, torch.bfloat16) for r, t in toks.items()}
    runner = make_runner(folder, torch.bfloat16, page_size=16, max_tokens=304, max_requests=4)
    for kind, tr in _all_traces(LENGTHS).items():
        _mostly_close(run_trace(runner, tr, toks), want, noise, f"buderax {name} {kind} bfloat16")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_streams_after_every_layer_run(cases, dtype):
    """The residual stream after each run of a layer (a looped layer counts each time), read from the
    engine by stopping the run order there."""
    import dataclasses

    from fastgen_amd.engine import Model, ModelRunner, StepEntry
    from fastgen_amd.weights.source import SafetensorsSource

    config, weights, folder, toks, _ = cases["small_loop"]
    streams: list = []
    plain_buderax_forward(weights, config, toks["b"], dtype, streams=streams)
    full = Model.from_folder(folder, dtype, DEV)
    for n_runs in range(1, len(full.layout.order) + 1):
        layout = dataclasses.replace(full.layout, order=full.layout.order[:n_runs])
        model = Model(layout, dtype, DEV, args=full.args, architecture=full.architecture)
        model.load(SafetensorsSource(folder))
        seen = {}
        norm = model.parts.final_norm
        keep = norm.forward
        norm.forward = lambda h, pending, dt, rows=None: (seen.update(h=h.clone(), pending=pending), keep(h, pending, dt, rows))[1]
        runner = ModelRunner(model, page_size=16, max_tokens=64, max_requests=1)
        runner.step([StepEntry("b", toks["b"], [0])])
        h, pending = seen["h"], seen["pending"]
        h = h + (pending.sum(0) if pending.dim() == 3 else pending.float())
        want = streams[n_runs - 1]
        tol = 2e-5 if dtype == torch.float32 else 4e-2
        assert float((h.cpu() - want).abs().max()) <= tol * float(want.abs().max()), f"after {n_runs} layer runs"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_decoding_across_pages(cases, dtype):
    """A short prompt, then 140 tokens one by one over nine pages (bfloat16: from recorded steps)."""
    config, weights, folder, _, _ = cases["one_pass"]
    toks = _tokens(config, {"z": 150}, seed=5)
    want = {"z": plain_buderax_forward(weights, config, toks["z"])}
    runner = make_runner(folder, dtype, page_size=16, max_tokens=160, max_requests=2)
    got = run_trace(runner, traces.tail({"z": 150}, 140), toks)
    if dtype == torch.float32:
        assert_close(got, want, dtype, None, "buderax long decoding")
    else:
        _mostly_close(got, want, {"z": plain_buderax_forward(weights, config, toks["z"], torch.bfloat16)}, "long decoding")
        assert runner.use_graphs and runner.graphs, "decode steps of this model are recorded"


def test_a_far_key_decides(tmp_path):
    """One query and one key, hundreds of tokens apart and on different pages, are scaled so that their
    score stands out: the logits at the query follow that key's value, in a prompt, in portions and
    decoded alone; losing the key would change them by far more than the tolerance."""
    config = {"architecture": "Buderax", "width": 32, "vocab": 50, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6},
              "layers": [{"type": "attention", "mlp": None,
                          "mixer": {"heads": 2, "kv_heads": 1, "dim": 16, "vdim": 16, "scale": 0.25,
                                    "rot": {"base": 10000.0, "dims": 4, "scaling": {"factor": 2.0}}}}]}
    w = plain_buderax_weights(config, 9)
    # token 1 is the far key, token 2 the query.  The key's embedding has one large component, which only
    # the key projection reads, the query's another, which only the query projection reads, both into the
    # head dimensions that are not rotated: their score towers over all others, the query's own included
    w["embed"][1] = 0.0
    w["embed"][1, 1] = 6.0
    w["embed"][2] = 0.0
    w["embed"][2, 0] = 6.0
    w["l0.norm1"][:] = 0.0
    w["l0.mix.q"][:, :2] = 0.0
    w["l0.mix.k"][:, :2] = 0.0
    w["l0.mix.q"][4:16, 0] = 3.0
    w["l0.mix.q"][20:32, 0] = 3.0
    w["l0.mix.k"][4:16, 1] = 3.0
    n = 420
    toks = torch.randint(3, 50, (n,), generator=torch.Generator().manual_seed(2)).tolist()
    toks[33] = 1          # just behind a page's edge (pages of 16 tokens)
    toks[400] = toks[419] = 2
    want = {"s": plain_buderax_forward(w, config, toks)}
    without = list(toks)
    without[33] = 7
    gap = float((plain_buderax_forward(w, config, without)[400] - want["s"][400]).abs().max())
    assert gap > 0.05 * float(want["s"].abs().max()), "the test's weights do not make the far key count"
    folder = save_model_folder(tmp_path / "m", config, w)
    for dtype in (torch.float32, torch.bfloat16):
        runner = make_runner(folder, dtype, page_size=16, max_tokens=432, max_requests=1)
        for tr in (traces.whole({"s": n}), traces.tail({"s": n}, 25), traces.chunks({"s": n})):
            got = run_trace(runner, tr, {"s": toks})
            if dtype == torch.float32:
                assert_close(got, want, dtype, None, "far key")
            else:
                assert float((got["s"] - want["s"]).abs().max()) < 0.2 * gap


def test_greedy_generation_through_the_engine(cases):
    from fastgen_amd.engine import Engine
    from fastgen_amd.sampling import SamplingParams

    config, weights, folder, toks, _ = cases["small_loop"]
    prompts = [toks["b"], toks["f"], toks["c"], toks["e"][:40], toks["d"]]
    want = [plain_buderax_greedy(weights, config, p, 9) for p in prompts]
    engine = Engine.from_folder(folder, torch.float32, DEV, page_size=16, max_tokens=320, max_batch=3, max_step_tokens=24)
    assert engine.generate(prompts, SamplingParams(temperature=0.0, max_new_tokens=9)) == want
    low = Engine.from_folder(folder, torch.bfloat16, DEV, page_size=16, max_tokens=320, max_batch=3, max_step_tokens=24)
    got = low.generate(prompts, SamplingParams(temperature=0.0, max_new_tokens=9))
    assert [len(g) for g in got] == [9] * len(prompts)


def test_command_lines(cases, tmp_path):
    """The trace runner and the chat tool take the model by its folder, as they take any other."""
    import json
    import subprocess
    import sys
    from pathlib import Path

    config, weights, folder, toks, want = cases["plain_stack"]
    root = Path(__file__).resolve().parents[1]
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": toks["b"][:20], "want": [19]}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": toks["b"][20:], "want": [0, 16]}], "end": ["x"]}]
    out = tmp_path / "out"
    run = subprocess.run([sys.executable, str(root / "bin" / "trace_run"), "--model", str(folder), "--dtype", "float32",
                          "--out", str(out), "--max-tokens", "64"], input="\n".join(json.dumps(s) for s in steps) + "\n",
                         capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stderr[-2000:]
    assert [l for l in run.stdout.splitlines() if l.startswith("done")] == ["done 0", "done 1"]
    import numpy as np
    got = np.fromfile(out / "1.f32", dtype="<f4").reshape(2, -1)
    assert np.abs(got - want["b"][[20, 36]].numpy()).max() <= 2e-5 * float(want["b"].abs().max())
    chat = subprocess.run([sys.executable, str(root / "bin" / "fgchat"), str(folder), "--prompt-ids", "1,2,3", "--max-tokens",
                           "5", "--temperature", "0"], capture_output=True, text=True, timeout=600)
    assert chat.returncode == 0, chat.stderr[-2000:]


@pytest.mark.parametrize("pairs,E", [(1, 3), (255, 32), (256, 256), (256, 257), (257, 32), (1025, 7), (8192, 32), (8193, 32), (9001, 300),
                                     (1024, 300), (2048, 5), (2049, 32), (4096, 300), (4097, 32)])
def test_sort_at_the_edges_of_its_forms(pairs, E):
    """Pairs that a thread holds, one more, and more experts than the small form counts: every pair once, among its expert's
    places, and tiles that cover them."""
    from fastgen_amd.kernels import ops

    torch.manual_seed(pairs)
    choice = torch.randint(0, E, (pairs, 1), dtype=torch.int32)
    choice[choice == E // 2] = 0  # (one without pairs)
    sorted_, tiles = (t.cpu() for t in ops.moe_sort(choice.cuda(), E, 16))
    assert torch.equal(sorted_.sort().values, torch.arange(pairs, dtype=torch.int32))
    assert torch.equal(choice[sorted_.long(), 0], choice[:, 0].sort().values)
    assert int(tiles[:, 2].sum()) == pairs and int(tiles[:, 2].max()) <= 16
    for e, first, rows, _ in tiles[tiles[:, 2] > 0].tolist():
        assert (choice[sorted_[first : first + rows].long(), 0] == e).all()


@pytest.mark.parametrize("counts,D,F", [((0, 64, 65, 128, 129, 256, 300, 1, 513), 192, 72 * 8), ((700,), 64, 64), ((3,) * 70 + (260,), 128, 136 * 8),
                                        ((1,) * 9, 320, 64), ((5,) * 3 + (0, 128) * 9 + (64, 1), 64, 136 * 8)])
@pytest.mark.parametrize("tile_rows", [128, 256])
def test_large_tiles_of_experts_give_the_rows_bits(counts, D, F, tile_rows):
    """Packed experts with sizes in multiples of 64 (the large tiles) against matrices stored row by row, where experts have as
    many rows as a tile of 64, 128 or 256, one more, none, more than one tile, and where there are more than 64 tiles."""
    from fastgen_amd.kernels import ops

    E, T = len(counts), sum(counts)
    torch.manual_seed(T)
    x = torch.full((T, D + 8), float("nan"), device="cuda").bfloat16()[:, :D]  # (the rows lie apart, with NaN between)
    x.copy_(torch.randn(T, D))
    wg, wu = ((torch.randn(E, F, D, device="cuda") / D ** 0.5).bfloat16() for _ in range(2))
    wd = (torch.randn(E, D, F, device="cuda") / F ** 0.5).bfloat16()
    choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T)].int()[:, None].cuda()
    sorted_, tiles = ops.moe_sort(choice, E, tile_rows)
    act = ops.moe_gate_up(x, wg, wu, sorted_, tiles, 1, tile_rows)
    assert torch.equal(ops.moe_gate_up(x, ops.pack_experts(wg), ops.pack_experts(wu), sorted_, tiles, 1, tile_rows), act)
    assert torch.equal(ops.moe_down(act, ops.pack_experts(wd), sorted_, tiles, tile_rows),
                       ops.moe_down(act, wd, sorted_, tiles, tile_rows))


@pytest.mark.parametrize("E,top,T,D,F", [(3, 2, 40, 40, 24), (5, 1, 700, 2048, 136), (4, 3, 300, 104, 520), (32, 4, 257, 64, 32)])
@pytest.mark.parametrize("tile_rows", [16, 32, 64, 128, 256])
def test_packed_experts_give_the_rows_bits(E, top, T, D, F, tile_rows):
    """The routed products from packed experts and from matrices stored row by row, for every tile: the same bits whatever
    the storage and the tile (k in steps of 32, ascending), at sizes that end inside a block of 16 rows, a step of 32 k
    and a wave's columns; and the products themselves, against fp32 with one rounding of the activation to bfloat16."""
    from fastgen_amd.kernels import ops

    torch.manual_seed(T)
    x = torch.randn(T, D, device="cuda").bfloat16()
    wg, wu = ((torch.randn(E, F, D, device="cuda") / D ** 0.5).bfloat16() for _ in range(2))
    wd = (torch.randn(E, D, F, device="cuda") / F ** 0.5).bfloat16()
    choice = torch.stack([torch.randperm(E, device="cuda")[:top] for _ in range(T)]).int()
    if F < 32 and tile_rows >= 128:
        pytest.skip("tiles through LDS take sizes from 32 on")
    sorted_, tiles = ops.moe_sort(choice, E, tile_rows)
    act = ops.moe_gate_up(x, wg, wu, sorted_, tiles, top, tile_rows)
    y = ops.moe_down(act, wd, sorted_, tiles, tile_rows)
    packed_act = ops.moe_gate_up(x, ops.pack_experts(wg), ops.pack_experts(wu), sorted_, tiles, top, tile_rows)
    assert torch.equal(packed_act, act)
    assert torch.equal(ops.moe_down(act, ops.pack_experts(wd), sorted_, tiles, tile_rows), y)
    small, small_tiles = ops.moe_sort(choice, E, 16)
    small_act = ops.moe_gate_up(x, wg, wu, small, small_tiles, top, 16)
    assert torch.equal(ops.moe_down(small_act, wd, small, small_tiles, 16), y)
    pair = sorted_.long()
    expert, rows = choice.reshape(-1)[pair].long(), x[pair // top].float()
    # a value at a time: the matrices of all pairs would not be small
    gate, up = torch.empty(2, T * top, F, device="cuda").unbind(0)
    want = torch.empty(T * top, D, device="cuda")
    for e in range(E):
        at = expert == e
        gate[at], up[at] = rows[at] @ wg[e].float().T, rows[at] @ wu[e].float().T
        want[pair[at]] = act[at].float() @ wd[e].float().T
    torch.testing.assert_close(act.float(), torch.nn.functional.silu(gate) * up, rtol=2 ** -7, atol=1e-4)
    torch.testing.assert_close(y, want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("T", [3, 200])
def test_routed_experts_take_rows_anywhere(T):
    """Rows of x whose stride is no multiple of 8: what the same rows give from memory of their own (the experts are packed,
    and only the matrix-core kernels, which read x 16 bytes at a time, read them).  The router adds such rows' 64
    products in another order, 64 roundings of 2^-24 each in its logits and so in the experts' weights."""
    from fastgen_amd.config import PartSpec
    from fastgen_amd.parts import build_part

    D, E, top, F = 64, 4, 2, 40
    config = {"width": D, "vocab": 8, "layers": [{"mixer": dict(heads=1, kv_heads=1, dim=8, vdim=8),
                                                   "mlp": {"router": {"experts": E, "top": top}, "expert": {"ff": F}}}]}
    part = build_part("feed_forward", PartSpec("moe", "l0.mlp", dict(
        dim=D, hidden_dim=F, n_experts=E, top=top,
        names={"router.weight": "router", "router.bias": "router.b", "expert": "e{}", "gate_proj.weight": "gate",
               "up_proj.weight": "up", "down_proj.weight": "down"})))
    part.load(plain_buderax_weights(config, 3), torch.bfloat16, DEV)
    x = torch.randn(T, D).to(DEV, torch.bfloat16)
    want = part.forward(x)
    for wide in (D + 3, D + 4):
        rows = torch.zeros(T, wide, dtype=torch.bfloat16, device=DEV)[:, :D]
        rows.copy_(x)
        torch.testing.assert_close(part.forward(rows), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("E,top,T,D,F", [(3, 2, 40, 72, 40), (4, 2, 300, 296, 168)])
@pytest.mark.parametrize("tile_rows", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("packed", [False, True])
def test_routed_experts_infinite_weights_stay_infinite(E, top, T, D, F, tile_rows, packed):
    """An infinity among an expert's weights, in the first k (which the kernels read again where a step ends behind k):
    its output is infinite with the sign of what it meets, not a number that is none; every other output is finite."""
    from fastgen_amd.kernels import ops

    torch.manual_seed(D)
    x = torch.randn(T, D, device="cuda").bfloat16()
    wu, wd = torch.randn(E, F, D, device="cuda").bfloat16(), torch.randn(E, D, F, device="cuda").bfloat16()
    wg = (torch.randn(E, F, D, device="cuda") / D ** 0.5).bfloat16()
    wu[:, 5, 0] = float("inf")
    wd[:, 7, 3] = float("inf")
    stored = ops.pack_experts if packed else (lambda w: w)
    choice = torch.stack([torch.randperm(E, device="cuda")[:top] for _ in range(T)]).int()
    sorted_, tiles = ops.moe_sort(choice, E, tile_rows)
    act = ops.moe_gate_up(x, stored(wg), stored(wu), sorted_, tiles, top, tile_rows)
    assert torch.isinf(act[:, 5]).all()
    other = torch.arange(F, device="cuda") != 5
    assert torch.isfinite(act[:, other]).all()
    clean = act.clone()
    clean[:, 5] = 1
    y = ops.moe_down(clean, stored(wd), sorted_, tiles, tile_rows)
    met = torch.empty(T * top, device="cuda")
    met[sorted_.long()] = clean[:, 3].float()
    assert torch.equal(y[:, 7], met * float("inf"))
    other = torch.arange(D, device="cuda") != 7
    assert torch.isfinite(y[:, other]).all()


@pytest.mark.parametrize("tile_rows", [128, 256])
def test_packed_experts_wide_tiles_give_the_rows_bits(tile_rows):
    """The same where the tiles through LDS are wide (128 x 256 a workgroup of a product, from 170 of them on), at sizes that
    end inside a wave's columns (32 of gate and up, 64 of down), a step of 32 k and a round of four steps."""
    from fastgen_amd.kernels import ops

    E, top, T, D, F = 32, 4, 700, 1048, 520
    tiles = ops.moe_max_tiles(T * top, E, tile_rows)
    assert tiles * -(-F // 128) >= 170 and tiles * -(-D // 256) >= 170
    test_packed_experts_give_the_rows_bits(E, top, T, D, F, tile_rows)


@pytest.mark.parametrize("dim,top", [(8, 1), (264, 3), (2048, 4), (2056, 5), (4096, 9), (4104, 2), (100, 2)])
@pytest.mark.parametrize("kind", ["bf16", "bf16 none", "bf16 sums", "fp32", "fp32 weight"])
def test_expert_sum_inside_the_norm_gives_the_bits_of_the_two_kernels(dim, top, kind):
    """A routed feed-forward's sum added up by the norm that follows it: every type a step has, whole and gathered rows
    (which leave h as it is), sizes at the edges of a workgroup's share and beyond what the kernel takes."""
    from fastgen_amd.kernels import ops
    torch.manual_seed(dim + top)
    T = 7
    act = torch.float32 if kind.startswith("fp32") and kind != "fp32 weight" else torch.bfloat16
    y, weight = torch.randn(T * top, dim, device="cuda"), torch.rand(T, top, device="cuda")
    plus = None if kind == "bf16 none" else torch.randn(3, T, dim, device="cuda") if kind == "bf16 sums" else (
        torch.randn(T, dim, device="cuda").to(act))
    w = torch.randn(dim, device="cuda").to(torch.float32 if kind == "fp32 weight" else act)
    h0 = torch.randn(T, dim, device="cuda")
    pending = ops.ExpertSum(y, weight, plus)
    for rows in (None, torch.tensor([6, 0, 6], dtype=torch.int32, device="cuda")):
        n = T if rows is None else 3
        h, want_h = h0.clone(), h0.clone()
        out, want = torch.empty(n, dim, dtype=act, device="cuda"), torch.empty(n, dim, dtype=act, device="cuda")
        pending.add_norm(h, w, 1e-6, out, rows)
        ops.add_rmsnorm(want_h, pending.total(), w, 1e-6, want, rows)
        assert torch.equal(out, want) and torch.equal(h, want_h)


@pytest.mark.parametrize("hd", [16, 80, 128, 192, 256])
@pytest.mark.parametrize("lens", [[1, 1, 1], [1, 300, 2], [130]])  # split alone and in chunks; beside tiles; tiles
def test_output_gate_inside_the_attention(hd, lens):
    """Both forms of the gate, rows with strides of their own, one that cannot be read in fours: the bits that the two kernels
    give."""
    from types import SimpleNamespace

    import numpy as np

    from fastgen_amd.kernels import ops
    torch.manual_seed(hd + sum(lens))
    H, KV, P, cached = 6, 2, 16, [20, 700, 1500][: len(lens)]
    pages = [-(-(n + c) // P) for n, c in zip(lens, cached)]
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages)).int()
    for i, n in enumerate(pages):
        table[i, :n], order = order[:n], order[n:]
    k = torch.randn(sum(pages), KV, P, hd, device="cuda").bfloat16()
    v = torch.randn(sum(pages), KV, hd, P, device="cuda").bfloat16()
    T = sum(lens)
    q = torch.randn(T, H * hd, device="cuda").bfloat16()
    wide = (4 * torch.randn(T, H * hd + 12, device="cuda")).bfloat16()
    wide[:, :13] = torch.tensor([0.0, -0.0, 90.0, -87.0, -88.5, -104.0, 1e-30, float("inf"), -float("inf"), 17.0, -17.0, 300.0, -300.0])
    starts = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)

    def run(**gate):
        ctx = SimpleNamespace(scratch={}, seq_records=None, q_lens=np.array(lens, dtype=np.int32), q_start_host=starts,
                              n_cached=np.array(cached, dtype=np.int32), graph_capacity=0)
        return ops.paged_attention(q, torch.empty_like(q), k, v, SimpleNamespace(block_table=table.cuda()), ctx, H,
                                   hd ** -0.5, **gate)

    plain = run()
    for gate in (wide[:, 8:], wide[:, : H * hd], wide[:, 3 : 3 + H * hd], wide[:, : H * hd].float()):
        for sigmoid in (True, False):
            assert torch.equal(run(gate=gate, gate_sigmoid=sigmoid), ops.gate_mul(plain.clone(), gate, sigmoid))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,dim,extra", [(5, 40, 0), (16, 264, 0), (16, 512, 1), (33, 2048, 0), (130, 1000, 2)])
def test_route_forms_give_the_same_bits(E, dim, extra, dtype):
    """A token's experts and weights beside 1, 256, 257, 512, 513, 1280, 1281 tokens (workgroups of one token, four, eight;
    the last ones partly filled)."""
    from fastgen_amd.kernels import ops
    torch.manual_seed(E + dim)
    x = torch.randn(1299, dim, device="cuda").to(dtype)
    router, bias = torch.randn(E + extra, dim, device="cuda"), torch.randn(E, device="cuda")
    whole = ops.moe_route(x, router, bias, 3, n_extra=extra)
    for n in (1, 255, 256, 257, 511, 512, 513, 1279, 1280, 1281):
        for got, want in zip(ops.moe_route(x[:n], router, bias, 3, n_extra=extra), whole):
            assert torch.equal(got, want[:n])
