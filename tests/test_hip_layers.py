"""Teacher-forced tokens layer by layer (fbs_layers.hip) against the step kernels (a model created with
one wavefront a sequence, which takes no layer by layer launch) and the oracle: prompts and scored rows at
the edges of the stretches, widths and windows, fresh and resumed sessions, refused tokens and full
contexts. Every output is an integer and equal."""

import ctypes as C
from contextlib import contextmanager
from dataclasses import replace

import numpy as np
import pytest

import oracle
from uor_fbs import hip, synth
from uor_fbs.hipmem import DeviceArray, runtime

pytestmark = pytest.mark.gpu

SHAPES = {
    # One quaternion a lane: half the lanes, a ragged width (24 quaternions; its norm is no power of
    # two's), the full wavefront with a window of 16.
    "w128": replace(synth.CONFIGS["c2"], context=96, layers=3),
    "w96": synth.Spec(vocab=2048, width=96, mlp=160, layers=2, context=96, kept=4, window=5, drawers=40, probes=4),
    "w256": replace(synth.CONFIGS["c3"], context=96, layers=3),
    # Two and four a lane, int8 codes, windows whose tap words take two positions a round and one.
    "w512i8": replace(synth.CONFIGS["c5"], context=224, layers=2),
    "w320": synth.Spec(vocab=2048, width=320, mlp=512, layers=2, context=96, kept=4, window=40, drawers=33, probes=3),
    "w768": synth.Spec(vocab=2048, width=768, mlp=1024, layers=2, context=96, kept=4, window=24, drawers=64, probes=4),
    # The shortest window over the reference's cells, and the whole-table head.
    "w64": synth.Spec(vocab=4096, width=64, mlp=96, layers=2, context=96, kept=8, window=1),
    # Taps of up to 4, whose words do not fit the chain's shortest form, over several rounds of taps.
    "w256t": replace(synth.CONFIGS["c3"], context=96, layers=3, tap_fields=(59, 66)),
    "w320t": synth.Spec(vocab=2048, width=320, mlp=512, layers=2, context=96, kept=4, window=40, drawers=33, probes=3,
                        tap_fields=(59, 66)),
}
DEEP = synth.Spec(vocab=512, width=1024, mlp=1024, layers=16, context=96, kept=4, window=64, drawers=32, probes=3)


@pytest.fixture(scope="module")
def models():
    made = {}

    def get(name, monkeypatch):
        if name not in made:
            art = synth.make_artifact(SHAPES[name], 31)
            monkeypatch.setenv("UOR_FBS_BLOCK_WAVES", "1")
            steps = hip.Model(art)
            monkeypatch.delenv("UOR_FBS_BLOCK_WAVES")
            made[name] = art, hip.Model(art), steps
        return made[name]

    return get


def _up(a, t):
    d = DeviceArray(np.shape(a), t)
    d.upload(np.ascontiguousarray(a, t))
    return d


def decode(model, prompts, gen, resume=None):
    n, length = prompts.shape
    tok = _up(prompts, np.uint32)
    ins = [None] * 3 if resume is None else [_up(a, t) for a, t in zip(resume, (np.int64, np.int32, np.uint32))]
    out = [DeviceArray((n, gen + 1), np.uint32), DeviceArray((n, model.state_words), np.int64),
           DeviceArray((n, model.history_words), np.int32), DeviceArray(n, np.uint32), DeviceArray(n, np.int32)]
    p = lambda d: None if d is None else d.ptr  # noqa: E731
    hip._check(hip.lib().uor_fbs_decode_async(model.handle, tok.ptr, n, length, gen, out[0].ptr, *map(p, ins),
                                              *[o.ptr for o in out[1:]], None))
    assert runtime().hipDeviceSynchronize() == 0
    return [o.download() for o in out]


def rows(model, tokens):
    """The rows' choices, kept drawers, queries and statuses, and their next-token matches, without and
    with the choices written out."""
    n, length = tokens.shape
    tok = _up(tokens, np.uint32)
    out = [DeviceArray((n, length), np.uint32), DeviceArray((n, length, model.probes), np.uint32),
           DeviceArray((n, length, model.width), np.int32), DeviceArray(n, np.int32)]
    hip._check(hip.lib().uor_fbs_sequences_async(model.handle, tok.ptr, n, length, *[o.ptr for o in out], None))
    assert runtime().hipDeviceSynchronize() == 0
    got = [o.download() for o in out]
    for argmin in (False, True):
        matches, status = DeviceArray(1, np.uint64), DeviceArray(n, np.int32)
        best = DeviceArray((n, length), np.uint32) if argmin else None
        hip._check(hip.lib().uor_fbs_score_async(model.handle, tok.ptr, n, length,
                                                 best.ptr if argmin else None, matches.ptr, status.ptr, None))
        assert runtime().hipDeviceSynchronize() == 0
        got += [matches.download(), status.download()] + ([best.download()] if argmin else [])
    return got


@contextmanager
def by_layers(model, calls):
    """The calls inside all ran by layers."""
    before = model.layer_calls
    yield
    assert model.layer_calls == before + calls


def tokens_for(name, n, length, seed):
    spec = SHAPES[name]
    make = synth.zipf_prompts if spec.zipf_drawers else synth.uniform_prompts
    return make(spec.vocab, n, length, seed).copy()


@pytest.mark.parametrize("name", list(SHAPES))
@pytest.mark.parametrize("n,length", [(1, 9), (3, 10), (2, 40), (5, 64)])
def test_prompts_equal_the_step_kernels(models, monkeypatch, name, n, length):
    art, layers, steps = models(name, monkeypatch)
    print(f"prompts {name}: {n} of {length}", flush=True)
    a = tokens_for(name, n, length, 5)
    with by_layers(layers, 1):
        first = decode(layers, a, 3)
    for got, want in zip(first, decode(steps, a, 3)):
        np.testing.assert_array_equal(got, want)
    # The sessions resumed by a second prompt, whose choices the oracle makes in one pass.
    b = tokens_for(name, n, 12, 6)
    with by_layers(layers, 1):
        second = decode(layers, b, 0, first[1:4])
    for got, want in zip(second, decode(steps, b, 0, first[1:4])):
        np.testing.assert_array_equal(got, want)
    if name in ("w128", "w96"):
        fed = np.concatenate([a, first[0][:, :3], b], axis=1)
        st, want_tok, _, _ = oracle.sequences(art, fed, threads=2)
        assert st == 0
        np.testing.assert_array_equal(second[0][:, 0], want_tok[:, -1])


@pytest.mark.parametrize("name", list(SHAPES))
@pytest.mark.parametrize("n,length", [(1, 8), (7, 31), (3, 96)])
def test_rows_equal_the_step_kernels(models, monkeypatch, name, n, length):
    art, layers, steps = models(name, monkeypatch)
    print(f"rows {name}: {n} of {length}", flush=True)
    t = tokens_for(name, n, length, 7)
    with by_layers(layers, 3):
        got = rows(layers, t)
    for g, w in zip(got, rows(steps, t)):
        np.testing.assert_array_equal(g, w)
    if name in ("w128", "w96"):
        st, want_tok, want_kept, want_query = oracle.sequences(art, t, threads=2)
        assert st == 0
        for g, w in zip(got, (want_tok, want_kept, want_query)):
            np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("name", ["w128", "w512i8"])
def test_refused_sequences(models, monkeypatch, name):
    # A token outside the vocabulary at the first, a middle and the last position, a context that ends
    # within the prompt (and under a bad token): the others are served, the refused export nothing.
    art, layers, steps = models(name, monkeypatch)
    vocab, context = SHAPES[name].vocab, SHAPES[name].context
    t = tokens_for(name, 8, 24, 8)
    for r, at in ((0, 0), (2, 11), (3, 23), (4, 22), (6, 20)):
        t[r, at] = vocab + r
    with by_layers(layers, 4):
        served, fresh = rows(layers, t), decode(layers, t, 2)
    for g, w in zip(served, rows(steps, t)):
        np.testing.assert_array_equal(g, w)
    for g, w in zip(fresh, decode(steps, t, 2)):
        np.testing.assert_array_equal(g, w)
    assert [int(s) for s in fresh[4]] == [1, 0, 1, 1, 1, 0, 1, 0]
    warm = decode(steps, tokens_for(name, 8, 10, 9), 0)
    position = np.array([10, context - 24, context - 24, context, context - 20, context - 12, context - 3, context - 26],
                        np.uint32)
    resume = (warm[1], warm[2], position)
    with by_layers(layers, 1):
        held = decode(layers, t, 2, resume)
    for g, w in zip(held, decode(steps, t, 2, resume)):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("name", ["w128", "w96", "w320", "w512i8", "w256t", "w320t"])
def test_sessions_at_the_ends_of_their_range(models, monkeypatch, name):
    # States and window rows over all of their types' values: the transport leaves its fast form's ranges
    # (at the first positions, in some quaternions only) and comes back to them.
    art, layers, steps = models(name, monkeypatch)
    n, rng = 6, np.random.default_rng(12)
    state = rng.integers(-2**63, 2**63 - 1, (n, layers.state_words), dtype=np.int64)
    state >>= rng.integers(0, 63, state.shape)
    state[0], state[1, ::7], state[2, 5] = 2**63 - 1, -2**63, 2**62 + 9
    state[3:5] >>= 40
    history = rng.integers(-2**31, 2**31 - 1, (n, layers.history_words), dtype=np.int32)
    history[3] = 2**31 - 1
    history[4] >>= 12
    resume = (state, history, np.arange(n, dtype=np.uint32))
    t = tokens_for(name, n, 43, 13)
    with by_layers(layers, 1):
        got = decode(layers, t, 1, resume)
    for g, w in zip(got, decode(steps, t, 1, resume)):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("n,length", [(2600, 72), (1000, 200)])
def test_parts_and_stretches_of_a_large_launch(models, monkeypatch, n, length):
    # More positions than the workspace holds at once: the sequences run in parts, or in stretches.
    art, layers, steps = models("w512i8", monkeypatch)
    t = tokens_for("w512i8", n, length, 10)
    t[n - 100, 3] = t[n - 5, length - 7] = SHAPES["w512i8"].vocab
    print(f"rows {n} of {length}", flush=True)
    with by_layers(layers, 4):
        got = rows(layers, t)
        print("prompts", flush=True)
        fed = decode(layers, t, 1)
    pick = [0, 700, n - 577, n - 576, n - 101, n - 100, n - 5, n - 1]
    for i, w in enumerate(rows(steps, t[pick])[:4]):
        np.testing.assert_array_equal(got[i][pick], w)
    for g, w in zip(fed, decode(steps, t[pick], 1)):
        np.testing.assert_array_equal(g[pick], w)
    # The matches of all rows: the choices against the next tokens of the positions served.
    served = np.cumsum(t >= SHAPES["w512i8"].vocab, axis=1) == 0
    assert got[4][0] == ((got[0][:, :-1] == t[:, 1:]) & served[:, :-1]).sum() == got[6][0]


@pytest.mark.parametrize("name,window", [("w128", 16), ("w96", 5), ("w320", 40)])
@pytest.mark.parametrize("beyond", [False, True])
def test_layers_with_the_smallest_and_largest_taps(monkeypatch, name, window, beyond):
    # Codes whose shifts have no word of the common form (1 and 29 to 37) in the second layer, which alone
    # takes the other form: the model still goes by layers, and equals the one-wavefront kernels and the oracle.
    # Beyond: the third layer has codes without any word (shifts of 0 and 63), and no call goes by layers.
    spec = replace(SHAPES[name], window=window, layers=3)
    art = synth.make_artifact(spec, 33)
    rng = np.random.default_rng(25)
    for layer, fields in ((1, [67] + list(range(31, 40))), (2, [68, 5])):
        taps = art.layers[layer].wide_taps
        at = rng.permutation(taps.size)[:taps.size // 3]
        if layer == 1 or beyond:
            field = np.array(fields)[rng.integers(0, len(fields), at.size)]
            taps[at] = (field * 16 + rng.integers(0, 16, at.size)) * rng.choice([-1, 1], at.size)
    layers = hip.Model(art)
    monkeypatch.setenv("UOR_FBS_BLOCK_WAVES", "1")
    steps = hip.Model(art)
    monkeypatch.setenv("UOR_FBS_BLOCK_WAVES", "0")
    monkeypatch.setenv("UOR_FBS_LAYER_BYTES", "0")
    pairs = hip.Model(art)
    t = synth.uniform_prompts(spec.vocab, 3, 43, 26)
    st, want_tok, want_kept, want_query = oracle.sequences(art, t, threads=2)
    assert st == 0
    for model in (layers, steps, pairs):
        got = rows(model, t)
        for g, w in zip(got, (want_tok, want_kept, want_query)):
            np.testing.assert_array_equal(g, w)
    # States over all their values, so that the window's largest terms meet the transport's wide form.
    state = rng.integers(-2**63, 2**63 - 1, (3, layers.state_words), dtype=np.int64) >> 30
    history = rng.integers(-2**31, 2**31 - 1, (3, layers.history_words), dtype=np.int32)
    resume = (state, history, np.arange(3, dtype=np.uint32))
    want = decode(steps, t, 2, resume)
    for model in (layers, pairs):
        for g, w in zip(decode(model, t, 2, resume), want):
            np.testing.assert_array_equal(g, w)
    assert layers.layer_calls == (0 if beyond else 4) and steps.layer_calls == pairs.layer_calls == 0


def test_the_workspace_keeps_to_its_bound(models, monkeypatch):
    # 2 MiB hold some 600 positions of width 128: 50 sequences of 90 run in parts or in stretches of 64.
    art, _, steps = models("w128", monkeypatch)
    t = tokens_for("w128", 50, 90, 23)
    monkeypatch.setenv("UOR_FBS_LAYER_BYTES", str(2 << 20))
    small = hip.Model(art)
    for g, w in zip(decode(small, t, 1), decode(steps, t, 1)):
        np.testing.assert_array_equal(g, w)
    assert small.layer_calls == 1 and 0 < small.layer_bytes <= 2 << 20
    for g, w in zip(rows(small, t), rows(steps, t)):
        np.testing.assert_array_equal(g, w)
    assert small.layer_calls == 4
    # A sequence at a time would cost more than the steps: none goes by layers.
    monkeypatch.setenv("UOR_FBS_LAYER_BYTES", str(300 << 10))
    tiny = hip.Model(art)
    for g, w in zip(decode(tiny, t, 1) + rows(tiny, t), decode(steps, t, 1) + rows(steps, t)):
        np.testing.assert_array_equal(g, w)
    assert tiny.layer_calls == tiny.layer_bytes == 0
    monkeypatch.setenv("UOR_FBS_LAYER_BYTES", "0")
    none = hip.Model(art)
    with pytest.raises(hip.FbsError):
        hip._check(hip.lib().uor_fbs_decode_async(none.handle, None, 1, 1, 0, *[None] * 9))
    error = hip.lib().uor_fbs_last_error()
    for g, w in zip(decode(none, t, 1), decode(steps, t, 1)):
        np.testing.assert_array_equal(g, w)
    assert none.layer_calls == none.layer_bytes == 0 and hip.lib().uor_fbs_last_error() == error


def test_the_workspace_grows_in_few_steps(models, monkeypatch):
    # Prompts and rows that get longer call by call (the larger sizes allocate by doubling).
    art = models("w128", monkeypatch)[0]
    for call in (lambda m, t: decode(m, t, 0), lambda m, t: m.score(t)):
        model = hip.Model(art)
        held = []
        for length in range(16, 64):
            call(model, tokens_for("w128", 8, length, 24))
            held.append(model.layer_bytes)
        assert model.layer_calls == len(held) and held == sorted(held) and len(set(held)) <= 5


@pytest.mark.parametrize("n,length", [(3, 96), (2, 600)])
def test_scored_rows_take_their_choices_in_place(n, length):
    # A score call whose choices go over its rows counts the matches of the rows as they came in, at
    # the edges of wavefronts and of rounds of 256 positions.
    model = hip.Model(synth.make_artifact(replace(SHAPES["w128"], context=600), 31))
    t = synth.uniform_prompts(SHAPES["w128"].vocab, n, length, 22)
    for _ in range(12):  # every other token the choice before it, as far as twelve rounds settle them
        t[:, 1::2] = model.sequences(t)[0][:, :-1:2]
    want_choices = model.sequences(t)[0]
    want = int((want_choices[:, :-1] == t[:, 1:]).sum())
    assert 0 < want < n * (length - 1)
    tok, matches, status = _up(t, np.uint32), DeviceArray(1, np.uint64), DeviceArray(n, np.int32)
    hip._check(hip.lib().uor_fbs_score_async(model.handle, tok.ptr, n, length, tok.ptr, matches.ptr, status.ptr, None))
    assert runtime().hipDeviceSynchronize() == 0
    np.testing.assert_array_equal(tok.download(), want_choices)
    assert int(matches.download()[0]) == want and not status.download().any()


def _capture(stream, call):
    """`call` recorded on `stream`, as an executable graph."""
    rt = runtime()
    graph, run = C.c_void_p(), C.c_void_p()
    assert rt.hipStreamBeginCapture(stream, 0) == 0  # global mode: an allocation ends the capture
    try:
        call()
    finally:
        ended = rt.hipStreamEndCapture(stream, C.byref(graph))
    assert ended == 0
    assert rt.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    assert rt.hipGraphDestroy(graph) == 0
    return run


@pytest.mark.parametrize("call", ["score", "sequences", "decode", "decode in parts"])
def test_calls_captured_after_a_warm_up(call):
    # The warm-up goes by layers, the captured call by the step kernels, whose buffers the warm-up left:
    # nothing is allocated under capture, and every replay equals the direct call.
    parts = call == "decode in parts"  # the workspace holds fewer of DEEP's sessions than run together
    spec, n, length = (DEEP, 500, 70) if parts else (SHAPES["w128"], 40, 24)
    model = hip.Model(synth.make_artifact(spec, 31))
    rt, lib, h = runtime(), hip.lib(), model.handle
    t = synth.uniform_prompts(spec.vocab, n, length, 21)
    tok, status = _up(t, np.uint32), DeviceArray(n, np.int32)
    if call == "score":
        outs = [DeviceArray((n, length), np.uint32), DeviceArray(1, np.uint64), status]
        launch = lambda st: lib.uor_fbs_score_async(h, tok.ptr, n, length, *[o.ptr for o in outs], st)  # noqa: E731
    elif call == "sequences":
        outs = [DeviceArray((n, length), np.uint32), DeviceArray((n, length, model.probes), np.uint32),
                DeviceArray((n, length, model.width), np.int32), status]
        launch = lambda st: lib.uor_fbs_sequences_async(h, tok.ptr, n, length, *[o.ptr for o in outs], st)  # noqa: E731
    else:
        outs = [DeviceArray((n, 2), np.uint32), status]
        launch = lambda st: lib.uor_fbs_decode_async(h, tok.ptr, n, length, 1, outs[0].ptr, *[None] * 6,  # noqa: E731
                                                     status.ptr, st)
    stream = C.c_void_p()
    assert rt.hipStreamCreate(C.byref(stream)) == 0
    print(f"{call}: warm-up", flush=True)
    hip._check(launch(stream))
    assert rt.hipStreamSynchronize(stream) == 0
    want = [o.download() for o in outs]
    print("capture", flush=True)
    run = _capture(stream, lambda: hip._check(launch(stream)))
    for _ in range(3):
        for o in outs:
            o.zero()
        assert rt.hipDeviceSynchronize() == 0
        assert rt.hipGraphLaunch(run, stream) == 0
        assert rt.hipStreamSynchronize(stream) == 0
        for o, w in zip(outs, want):
            np.testing.assert_array_equal(o.download(), w)
        rows(model, t[:3])  # the program's own calls between the replays
    assert rt.hipGraphExecDestroy(run) == 0
    assert rt.hipStreamDestroy(stream) == 0
