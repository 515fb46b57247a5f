"""The work that a user of this framework has it do, as cases that can be timed and compared.

Most of it is the integer SpiralCore/FBS step: batched greedy decode, prefill of prompts,
teacher-forced scoring and serving sessions over device slots, at the configurations of
``uor_fbs.synth.CONFIGS``. Beside it stand the Hamming reads in the step, the discrete M1 panel
scorer, the CSR drawer index and the copy heads' read. Everything is whole numbers, and every
output has to be the same, bit for bit.

The weights of a model are seeded by its configuration (a program loads one model and gives it
many inputs); prompts, rows, tables, queries and streams come from the case's seed. Each prepared
state has a model handle and device buffers of its own.
"""

from __future__ import annotations

import ctypes as C
import functools
import os
import sys
from dataclasses import replace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "uor-r4_amd"))

from uor_fbs import copy as copy_heads  # noqa: E402
from uor_fbs import d11, hip, index, session, synth  # noqa: E402

WEIGHTS = 2026120203
SERVE_ROWS = 61  # rows of user tokens that a serving state goes through in turn
PANEL_CONTEXT = 192


def listed():
    return [
        # One interactive user: a single sequence of the smallest configuration continues a
        # 256-token prompt. A latency: one block on the whole card.
        dict(name="decode_w128_single", kind="decode", config="c1", batch=1, prompt=256, gen=64),
        # Batched generation at width 128: most sequences settle, and the layer chain sets the step.
        dict(name="decode_w128_b1024", kind="decode", config="c2", batch=1024, prompt=128, gen=128),
        # The headline workload's shape: width 256, vocabulary 32,768, Zipf drawers, 1,024 sequences.
        dict(name="decode_w256_b1024", kind="decode", config="c3", batch=1024, prompt=256, gen=256),
        # The largest model (width 512, int8 codes, 32-row window, 1,024 drawers) with more
        # sequences than the card holds blocks.
        dict(name="decode_w512_i8_b4096", kind="decode", config="c5", batch=4096, prompt=48, gen=48),
        # Prompts taken in before generation: an odd batch and length, no choice but the last.
        dict(name="prefill_w256_b300", kind="prefill", config="c3", batch=300, prompt=509),
        # Evaluation: rows scored teacher-forced, every position's choice wanted.
        dict(name="score_w256_8192x128", kind="score", config="c4", rows=8192, length=128, full=False),
        # The serving loop over device slots: 1,024 sessions take a user token and reply with 31
        # more, one launch a token.
        dict(name="serve_w256_b1024", kind="serve", config="c3", sessions=1024, launches=32),
        # A few live sessions through the Python session API, one token each a call.
        dict(name="sessions_w128_b8", kind="sessions", config="c1", sessions=8, prompt=40),
        # The step with Hamming reads over each session's past (copy and type heads at two hooks).
        dict(name="decode_hamming_w256_b256", kind="hamming", batch=256, prompt=256, gen=64, typed=True),
        # A panel of the discrete M1 scorer: rows of 186-192 tokens with the sparse trunk.
        dict(name="m1_panel_14287", kind="m1", rows=14287, min_len=186, mode="relation", trunk=True),
        # A codebook change: the drawer index of a 65,536-token table is built again and a batch of
        # queries probes it.
        dict(name="index_build_probe_65536", kind="index", tokens=65536, queries=65536, k=8),
        # The copy heads' read at the end of 4,096 streams.
        dict(name="copy_read_4096x1024", kind="copy", streams=4096, length=1024, kept=16, rule="mean"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "score", "serve", "serve",
                       "sessions", "hamming", "m1", "index", "copy"])
    if kind == "decode":
        config = rng.choice(["c1", "c2", "c3", "c3", "c5", "w96", "nearest"])
        batch = _log(rng, 1, 2048)
        return dict(kind=kind, config=config, batch=batch, prompt=_log(rng, 1, 200),
                    gen=_log(rng, 1, 24 if config in ("c5", "nearest") else 120),
                    snapped=rng.random() < 0.2 and config in ("c1", "c2", "w96"))
    if kind == "prefill":
        return dict(kind=kind, config=rng.choice(["c1", "c3", "c3", "c5"]), batch=_log(rng, 1, 700),
                    prompt=_log(rng, 2, 300))
    if kind == "score":
        return dict(kind=kind, config=rng.choice(["c1", "c4", "c5"]), rows=_log(rng, 1, 1500),
                    length=_log(rng, 2, 128), full=rng.random() < 0.3)
    if kind == "serve":
        return dict(kind=kind, config=rng.choice(["c2", "c3", "c3", "c5"]), sessions=_log(rng, 1, 1500),
                    launches=rng.choice([1, 1, 8]))
    if kind == "sessions":
        return dict(kind=kind, config=rng.choice(["c1", "c3"]), sessions=_log(rng, 1, 40),
                    prompt=_log(rng, 1, 100))
    if kind == "hamming":
        return dict(kind=kind, batch=_log(rng, 1, 300), prompt=_log(rng, 8, 250), gen=_log(rng, 1, 48),
                    typed=rng.random() < 0.7)
    if kind == "m1":
        return dict(kind=kind, rows=_log(rng, 1, 14000), min_len=_log(rng, 1, PANEL_CONTEXT),
                    mode=rng.choice(["relation", "relation", "flock", "route"]), trunk=rng.random() < 0.7)
    if kind == "index":
        return dict(kind=kind, tokens=_log(rng, 64, 1 << 20), queries=_log(rng, 1, 4096),
                    k=rng.choice([1, 8, 16]))
    return dict(kind=kind, streams=_log(rng, 1, 4096), length=_log(rng, 2, 1024),
                kept=rng.choice([1, 8, 16, 32]),
                rule=rng.choice(["mean", "mean", "latest-exact", "latest-nearest", "longest-exact"]))


# ---------------------------------------------------------------------------------------------
# Models.


def _spec(case):
    """The case's model: a configuration at a context that holds the case's positions."""
    if case["kind"] == "hamming":
        return replace(synth.CONFIGS["c3"], context=case["prompt"] + case["gen"] + 1,
                       hamming=synth.HammingSpec(heads=8, depths=(3, 6), kept=16, typed=case["typed"]))
    config = case["config"]
    if config == "w96":  # a width that is not a power of two, Zipf drawers, a 5-row window
        spec = synth.Spec(vocab=700, width=96, mlp=160, layers=2, context=512, kept=3, window=5,
                          drawers=48, probes=6, zipf_drawers=1.3, max_drawer=40)
    elif config == "nearest":  # the whole-table head in the writer's place
        spec = replace(synth.CONFIGS["c2"], head=1)
    else:
        spec = synth.CONFIGS[config]
    if case.get("snapped"):
        spec = replace(spec, raw_gates=False, raw_transition=False)
    return spec


@functools.lru_cache(maxsize=6)
def _weights(spec):
    return synth.make_artifact(spec, WEIGHTS)


def _tokens(spec, count, length, seed):
    make = synth.zipf_prompts if spec.zipf_drawers else synth.uniform_prompts
    return make(spec.vocab, count, length, 2 * seed + 1)


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _u32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.uint32).view(np.int32)).cuda()


def _zeros(shape, dtype=torch.int32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _check(code):
    if code:
        raise hip.FbsError(code, hip.lib().uor_fbs_last_error().decode())


class _Sessions:
    """A batch's state, window and position on the device."""

    def __init__(self, model, n):
        self.state = _zeros((n, model.state_words), torch.int64)
        self.history = _zeros((n, model.history_words))
        self.position = _zeros(n)

    def all(self):
        return self.state, self.history, self.position


def _take_in(model, prompts, sessions):
    """The prompts from fresh sessions into `sessions`; each prompt's choice."""
    n, length = prompts.shape
    first, status = _zeros((n, 1)), _zeros(n)
    _check(hip.lib().uor_fbs_decode_async(
        model.handle, _ptr(prompts), n, length, 0, _ptr(first), None, None, None,
        *[_ptr(t) for t in sessions.all()], _ptr(status), _stream()))
    return first, status


# ---------------------------------------------------------------------------------------------
# What a program has in hand.


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_decode(case, seed):
    spec = _spec(case)
    model = hip.Model(_weights(spec))
    n = case["batch"]
    prompts = _u32(_tokens(spec, n, case["prompt"], seed))
    before = _Sessions(model, n)
    first, _ = _take_in(model, prompts, before)
    return dict(kind="decode", model=model, n=n, gen=case["gen"], first=first, before=before,
                after=_Sessions(model, n), reply=_zeros((n, case["gen"] + 1)), status=_zeros(n))


def _prepare_prefill(case, seed):
    spec = _spec(case)
    model = hip.Model(_weights(spec))
    return dict(kind="prefill", model=model, sessions=_Sessions(model, case["batch"]),
                prompts=_u32(_tokens(spec, case["batch"], case["prompt"], seed)))


def _prepare_score(case, seed):
    spec = _spec(case)
    model = hip.Model(_weights(spec))
    n, length = case["rows"], case["length"]
    s = dict(kind="score", model=model, n=n, length=length, full=case["full"],
             rows=_u32(_tokens(spec, n, length, seed)), choices=_zeros((n, length)), status=_zeros(n))
    if case["full"]:  # every position's kept drawers and query too
        s.update(kept=_zeros((n, length, model.probes)), query=_zeros((n, length, model.width)))
    else:
        s.update(matches=_zeros(1, torch.int64))
    return s


def _prepare_serve(case, seed):
    spec = _spec(case)
    model = hip.Model(_weights(spec))
    n = case["sessions"]
    slots = _Sessions(model, n)
    one = torch.ones(n, dtype=torch.uint8, device="cuda")
    cache = _zeros((n, int(hip.lib().uor_fbs_slot_cache_bytes(model.handle))), torch.uint8)
    order = _u32(np.random.default_rng(seed).permutation(n))
    s = dict(kind="serve", model=model, n=n, launches=case["launches"], slots=slots, order=order,
             slide=one, cache=cache, user=_u32(_tokens(spec, SERVE_ROWS, n, seed)), turn=0,
             served=_zeros((case["launches"], n)), status=_zeros(n))
    prompts = _u32(_tokens(spec, n, 40, seed + 1))
    _serve(s, prompts, 40, s["served"][0])  # each session's prompt, in its slot
    return s


def _prepare_sessions(case, seed):
    spec = _spec(case)
    pool = session.SessionPool(hip.Model(_weights(spec)), case["sessions"])
    live = [session.Session(pool) for _ in range(case["sessions"])]
    for s, prompt in zip(live, _tokens(spec, case["sessions"], case["prompt"], seed + 1)):
        s.set_context_slide(True)
        s.feed(prompt.tolist())
    return dict(kind="sessions", live=live, turn=0,
                user=_tokens(spec, SERVE_ROWS, case["sessions"], seed).tolist())


def _prepare_hamming(case, seed):
    spec = _spec(case)
    model = hip.Model(_weights(spec))
    n, length, gen = case["batch"], case["prompt"], case["gen"]
    s = dict(kind="hamming", model=model, n=n, gen=gen, before=_Sessions(model, n), after=_Sessions(model, n),
             reply=_zeros((n, gen + 1)), status=_zeros(n), stream=_zeros((n, model.stream_words)),
             after_stream=_zeros((n, model.stream_words)), first=_zeros((n, 1)),
             payloads=_zeros((n, model.payload_words), torch.int64) if model.payload_words else None)
    prompts = _u32(_tokens(spec, n, length, seed))
    _check(hip.lib().uor_fbs_decode_stream_async(
        model.handle, _ptr(prompts), n, length, 0, _ptr(s["first"]), None, None, None, None, None,
        *[_ptr(t) for t in s["before"].all()], _ptr(s["stream"]), _ptr(s["payloads"]), _ptr(s["status"]),
        _stream()))
    return s


@functools.lru_cache(maxsize=4)
def _panel_weights(mode, trunk):
    return d11.synthetic(context=PANEL_CONTEXT, read_mode=mode, trunk=trunk, seed=WEIGHTS,
                         trunk_entries=600_000)


def _prepare_m1(case, seed):
    art = _panel_weights(case["mode"], case["trunk"])
    rows = case["rows"]
    prefixes, lengths, targets = d11.panel_rows(art, rows, seed, min_len=case["min_len"])
    return dict(kind="m1", model=d11.IntegerDiscreteModel(art), rows=rows, prefixes=_u32(prefixes),
                lengths=torch.from_numpy(lengths).cuda(), targets=_u32(targets),
                out=_zeros((rows, d11.ROW_DTYPE.itemsize // 4)))


def _random_table(count, gen):
    """Width-32 token rows whose first and last blocks are roots, the middle ones any values."""
    roots = torch.from_numpy(index.CODEBOOK).cuda()
    t = torch.randint(-(1 << 31), (1 << 31) - 1, (count, 32), dtype=torch.int32, device="cuda", generator=gen)
    cells = torch.randint(0, 256, (count,), device="cuda", generator=gen)
    t[:, :8] = roots[cells // 16]
    t[:, 24:] = roots[cells % 16]
    return t


def _prepare_index(case, seed):
    n, q = case["tokens"], case["queries"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return dict(kind="index", n=n, q=q, k=case["k"], table=_random_table(n, gen), queries=_random_table(q, gen),
                roots=torch.from_numpy(index.CODEBOOK).cuda(), offsets=_zeros(257), members=_zeros(n),
                cells=_zeros(n), absent=_zeros(1), built=_zeros(1),
                work=_zeros(int(hip.lib().uor_fbs_index_workspace_bytes(n)) // 4), prediction=_zeros(q),
                admitted=_zeros((q, 16)), top8=_zeros((q, 8)), status=_zeros(q))


def _prepare_copy(case, seed):
    heads = copy_heads.synthetic(kept=case["kept"], rule=case["rule"], seed=WEIGHTS)
    rng = np.random.default_rng(seed)
    n, length = case["streams"], case["length"]
    tokens = rng.integers(0, heads.codes.shape[0], (n, length)).astype(np.uint32)
    # Half of the streams say again something that they said before, as text does.
    for i in range(0, n, 2):
        if length >= 16:
            a = int(rng.integers(1, length - 8))
            tokens[i, -6:] = tokens[i, a:a + 6]
    lengths = np.full(n, length, np.int32)
    lengths[n // 2:] = rng.integers(1, length + 1, n - n // 2)
    return dict(kind="copy", heads=copy_heads.CopyHeads(heads), n=n, length=length, tokens=_u32(tokens),
                lengths=torch.from_numpy(lengths).cuda(), out=_zeros((n, heads.table.shape[1]), torch.int64),
                found=_zeros(n, torch.uint8), chosen=_zeros((n, heads.codes.shape[1], case["kept"])))


# ---------------------------------------------------------------------------------------------
# One pass.


def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_decode(s):
    _check(hip.lib().uor_fbs_decode_async(
        s["model"].handle, _ptr(s["first"]), s["n"], 1, s["gen"], _ptr(s["reply"]),
        *[_ptr(t) for t in s["before"].all()], *[_ptr(t) for t in s["after"].all()], _ptr(s["status"]),
        _stream()))
    return (s["reply"], s["status"], *s["after"].all())


def _run_prefill(s):
    first, status = _take_in(s["model"], s["prompts"], s["sessions"])
    return (first, status, *s["sessions"].all())


def _run_score(s):
    lib, h = hip.lib(), s["model"].handle
    if s["full"]:
        _check(lib.uor_fbs_sequences_async(h, _ptr(s["rows"]), s["n"], s["length"], _ptr(s["choices"]),
                                           _ptr(s["kept"]), _ptr(s["query"]), _ptr(s["status"]), _stream()))
        return s["choices"], s["kept"], s["query"], s["status"]
    s["matches"].zero_()
    _check(lib.uor_fbs_score_async(h, _ptr(s["rows"]), s["n"], s["length"], _ptr(s["choices"]),
                                   _ptr(s["matches"]), _ptr(s["status"]), _stream()))
    return s["choices"], s["matches"], s["status"]


def _serve(s, tokens, length, reply):
    _check(hip.lib().uor_fbs_serve_slots_async(
        s["model"].handle, _ptr(s["order"]), s["n"], s["n"], _ptr(tokens), length, 0, _ptr(reply),
        *[_ptr(t) for t in s["slots"].all()], _ptr(s["cache"]), _ptr(s["slide"]), None, None, None,
        _ptr(s["status"]), _stream()))


def _run_serve(s):
    tokens = s["user"][s["turn"] % SERVE_ROWS]
    s["turn"] += 1
    for k in range(s["launches"]):
        _serve(s, tokens, 1, s["served"][k])
        tokens = s["served"][k]
    return (s["served"], s["status"], *s["slots"].all())


def _run_sessions(s):
    tokens = s["user"][s["turn"] % SERVE_ROWS]
    s["turn"] += 1
    chosen = session.serve_steps(s["live"], tokens)
    return np.array(chosen, np.int64), np.stack([x.last_query_q12() for x in s["live"]])


def _run_hamming(s):
    _check(hip.lib().uor_fbs_decode_stream_async(
        s["model"].handle, _ptr(s["first"]), s["n"], 1, s["gen"] - 1, _ptr(s["reply"]),
        *[_ptr(t) for t in s["before"].all()], _ptr(s["stream"]), _ptr(s["payloads"]),
        *[_ptr(t) for t in s["after"].all()], _ptr(s["after_stream"]), _ptr(s["payloads"]), _ptr(s["status"]),
        _stream()))
    out = (s["reply"], s["status"], *s["after"].all(), s["after_stream"])
    return out if s["payloads"] is None else (*out, s["payloads"])


def _run_m1(s):
    code = d11.lib().uor_d11_score_rows_async(s["model"].handle, _ptr(s["prefixes"]), _ptr(s["lengths"]),
                                              _ptr(s["targets"]), s["rows"], PANEL_CONTEXT, _ptr(s["out"]),
                                              _stream())
    if code:
        raise d11.DiscreteError(d11.lib().uor_d11_last_error().decode())
    return s["out"]


def _run_index(s):
    lib, at = hip.lib(), _stream()
    _check(lib.uor_fbs_index_build_async(_ptr(s["table"]), s["n"], 32, _ptr(s["roots"]), 0, _ptr(s["offsets"]),
                                         _ptr(s["members"]), _ptr(s["cells"]), _ptr(s["absent"]),
                                         _ptr(s["work"]), _ptr(s["built"]), at))
    _check(lib.uor_fbs_index_probe_async(_ptr(s["table"]), s["n"], 32, _ptr(s["roots"]), _ptr(s["queries"]),
                                         s["q"], s["k"], _ptr(s["offsets"]), _ptr(s["members"]),
                                         _ptr(s["prediction"]), _ptr(s["admitted"]), _ptr(s["top8"]),
                                         _ptr(s["status"]), at))
    return [s[k] for k in ("built", "offsets", "members", "cells", "absent", "prediction", "admitted", "top8",
                           "status")]


def _run_copy(s):
    code = copy_heads.lib().uor_copy_mean_rows_async(
        s["heads"].handle, _ptr(s["tokens"]), _ptr(s["lengths"]), None, s["n"], s["length"], _ptr(s["out"]),
        _ptr(s["found"]), _ptr(s["chosen"]), _stream())
    if code:
        raise copy_heads.CopyError(copy_heads.lib().uor_copy_last_error().decode())
    return s["out"], s["found"], s["chosen"]


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, and what its outputs may differ by.


def _layer_ops(spec):
    """Multiplies and adds of one position's layers: the window's taps, the transition's, the output
    gate's and the feed-forward gates' quaternion products (28 each), the norms and requantizes."""
    d = spec.width
    return spec.layers * (2 * d * (spec.window + 1) + 2 * 28 * (d // 4) + 28 * (spec.mlp // 4) + 12 * d)


def _scan_rows(spec):
    """Candidate rows that a choice looks at on average."""
    return spec.vocab if spec.head else spec.vocab * (spec.probes or spec.kept) // (spec.drawers or 256)


def _table_bytes(spec):
    return spec.vocab * spec.width * (1 if spec.table == "i8" else 2)


def _session_bytes(spec):
    return spec.layers * spec.width * (8 + 4 * spec.window) + 4


def _step_work(spec, sequences, steps, choices, sessions_moved, outputs=0):
    """Every table row that a choice may look at is read once by the whole pass (never more rows
    than the choices look at), each session's state in and out, the tokens and other outputs."""
    rows = min(spec.vocab, choices * _scan_rows(spec))
    return {"bytes": rows * _table_bytes(spec) // spec.vocab + sessions_moved * _session_bytes(spec)
            + 8 * sequences * steps + outputs,
            "flops": sequences * steps * _layer_ops(spec) + 3 * choices * _scan_rows(spec) * spec.width}


def work(case):
    kind = case["kind"]
    if kind in ("decode", "hamming"):
        spec, n, steps = _spec(case), case["batch"], case["gen"] + (kind == "decode")
        w = _step_work(spec, n, steps, n * steps, 2 * n)
        if kind == "hamming":  # a popcount per head, read and earlier position; the kept rows' sums
            reads, mean = 2, case["prompt"] + steps // 2
            w["flops"] += n * steps * reads * 8 * (3 * mean + 2 * 16 * spec.width)
            w["bytes"] += (n * mean * reads * 8 * spec.width if case["typed"] else 0) + 4 * n * mean
        return w
    if kind == "prefill":
        return _step_work(_spec(case), case["batch"], case["prompt"], case["batch"], case["batch"])
    if kind == "score":
        spec, at = _spec(case), case["rows"] * case["length"]
        return _step_work(spec, case["rows"], case["length"], at, 0,
                          at * 4 * (spec.width + spec.probes) if case["full"] else 0)
    if kind in ("serve", "sessions"):
        n, steps = case["sessions"], case.get("launches", 1)
        return _step_work(_spec(case), n, steps, n * steps, 2 * n)
    if kind == "m1":  # the prefixes and targets in, the records out; the read's levels over the prefix
        tokens = case["rows"] * (case["min_len"] + PANEL_CONTEXT) // 2
        return {"bytes": 4 * tokens + case["rows"] * (8 + d11.ROW_DTYPE.itemsize), "flops": tokens * 4 * 5 * 8}
    if kind == "index":  # the endpoint blocks, cells and members of a build; the rows that queries look at
        n, q = case["tokens"], case["queries"]
        looked = q * n * case["k"] // 256
        return {"bytes": 76 * n + min(n, looked) * 64 + q * (128 + 104), "flops": 3 * 32 * looked + q * 16 * 2 * 24}
    width, heads, kept = 256, 4, case["kept"] if case["rule"] == "mean" else 1
    tokens = case["streams"] * case["length"] * 3 // 4  # half of the streams are shorter
    return {"bytes": 4 * tokens + case["streams"] * (width * 8 + 5 + 4 * heads * case["kept"]) + 32768 * heads * 8,
            "flops": tokens * heads * 3 + case["streams"] * heads * kept * width * 2}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Nothing to give: every output is whole numbers, held to equality."""
    return None
