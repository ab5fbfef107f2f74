"""Batches that run at once share no stream that a library keeps a workspace by: over a stand-in for torch's pool of
streams, which hands 32 of them out in turn."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from macllm_infer_amd.engine import engine as engine_module
from macllm_infer_amd.engine import graphs as graphs_module
from macllm_infer_amd.parts import block, streams

POOL = 32
DEVICE = torch.device("cuda", 0)


class FakeStream:
    turn = 0

    def __init__(self, device=None, number=None):
        if number is None:
            number = FakeStream.turn % POOL
            FakeStream.turn += 1
        self.number, self.device, self.cuda_stream = number, DEVICE, 1000 + number

    def __eq__(self, other):
        return self.number == other.number

    def __hash__(self):
        return self.number

    def wait_stream(self, other):
        pass


@pytest.fixture()
def cuda(monkeypatch):
    """torch.cuda's streams and captures without a GPU; ``current`` is the stream that work would be queued on."""
    state = SimpleNamespace(current=FakeStream(number=-1), capturing=False, recorded=set())

    @contextlib.contextmanager
    def on(stream):
        before, state.current = state.current, stream
        try:
            yield
        finally:
            state.current = before

    class FakeGraph:
        default_capture_stream = None

        def __init__(self, graph, pool=None, stream=None):
            if stream is None and FakeGraph.default_capture_stream is None:
                FakeGraph.default_capture_stream = FakeStream()
            self.on = on(stream if stream is not None else FakeGraph.default_capture_stream)

        def __enter__(self):
            state.capturing = True
            return self.on.__enter__()

        def __exit__(self, *error):
            state.capturing = False
            return self.on.__exit__(*error)

    FakeStream.turn = 0
    for name, value in (("Stream", FakeStream), ("stream", on), ("graph", FakeGraph), ("CUDAGraph", object),
                        ("current_stream", lambda device=None: state.current), ("synchronize", lambda device=None: None),
                        ("graph_pool_handle", object), ("current_device", lambda: 0)):
        monkeypatch.setattr(torch.cuda, name, value)
    monkeypatch.setattr(block, "_side_streams", {})
    monkeypatch.setattr(streams, "_of_device", {})
    return state


def captures(state, kind, drawn_between=0):
    """A function that captures a graph of ``kind`` and returns the streams worked on so far, warm-up and fork included."""
    used = set()

    def forward(context, cache):
        used.add(state.current)
        if state.capturing:                                  # (only what is recorded forks)
            used.add(block.side_stream(DEVICE, state.current))
            state.recorded |= {state.current, block.side_stream(DEVICE, state.current)}
    bank = graphs_module.DecodeGraphs(SimpleNamespace(forward=forward, blocks=[], step_layout={}), None, DEVICE, 4096)

    def capture():
        for _ in range(drawn_between):
            FakeStream()
        bank._capture(0, SimpleNamespace(capacity=kind == "portions", context=None))
        return used
    return capture


@pytest.mark.parametrize("drawn_between", [0, 1, 2, 5])
def test_no_capture_of_portions_works_on_a_stream_of_the_single_tokens(cuda, drawn_between):
    """33 captures in a row, other parts of the program drawing streams in between, while single tokens may be under way: their
    graph works on the streams that it was recorded and forked on."""
    captures(cuda, "singles")()
    singles = set(cuda.recorded)
    capture = captures(cuda, "portions", drawn_between)
    for _ in range(POOL + 1):
        assert not singles & capture()


@pytest.mark.parametrize("kind", ["singles", "portions"])
def test_a_recording_says_whether_it_forked(cuda, kind):
    """By the second stream that was handed out during it, not by its size or by what other kinds of batches do."""
    for forks in (True, False, True):
        def forward(context, cache):
            if forks:                                        # (a warm-up, on another stream, forks as well)
                block.side_stream(DEVICE, cuda.current)
        bank = graphs_module.DecodeGraphs(SimpleNamespace(forward=forward, blocks=[], step_layout={}), None, DEVICE, 4096)
        static = SimpleNamespace(capacity=kind == "portions", context=None)
        assert bank._capture(0, static)[0] is static and static.forks == forks


def test_every_kind_of_batch_has_streams_of_its_own(cuda):
    of_device = streams.batch_streams(DEVICE)
    assert streams.batch_streams(DEVICE) is of_device
    own = [stream for kind in streams.KINDS for stream in (of_device.recording[kind], of_device.side[kind])]
    assert len(set(own + of_device.beside)) == len(own) + len(of_device.beside)
    assert of_device.recording[streams.SINGLES] == torch.cuda.graph.default_capture_stream
    for _ in range(2 * POOL):
        assert of_device.apart() not in own + of_device.beside
    for kind in streams.KINDS:
        assert block.side_stream(DEVICE, of_device.recording[kind]) == of_device.side[kind]
    for number in range(POOL):                           # work on any other stream forks to none of a kind's
        main = FakeStream(number=number)
        side = block.side_stream(DEVICE, main)
        assert side != main and (of_device.side_of(main) is not None or side not in own)


def engine_on(monkeypatch, asked):
    bank = SimpleNamespace(streams=streams.batch_streams(DEVICE), bucket_key=lambda lanes, lowered: "key",
                           ask_beside=lambda keys, candidates: asked.append(keys), stream_beside=lambda key, candidates: candidates[0])
    monkeypatch.setattr(engine_module.ops, "stream_beside", lambda main, candidates: candidates[-1])
    engine = SimpleNamespace(graphs=bank, device=DEVICE, _beside={})
    engine._streams_beside = lambda: engine_module.Engine._streams_beside(engine)
    return engine


def test_single_tokens_run_beside_portions_only_where_their_streams_are_apart(cuda, monkeypatch):
    """Whatever stream of the pool the caller is on: beside it only if it is none of the single tokens' own (a portion
    that is launched kernel by kernel works on the caller's), on a stream that is neither the caller's nor a kind's."""
    asked = []
    engine = engine_on(monkeypatch, asked)
    of_device = engine.graphs.streams
    for number in [-1] + list(range(POOL)):
        cuda.current = FakeStream(number=number)
        asked.clear()
        stream = engine_module.Engine._stream_for_singles(engine, [object()], None)
        if of_device.belongs_to(streams.SINGLES, cuda.current):
            assert stream is None and not asked
        else:
            assert stream != cuda.current and stream in of_device.beside and asked == [["key"]]
    assert len(engine._beside) <= engine_module.CALLERS_STREAMS


def test_the_streams_of_a_callers_stream_begin_with_the_one_the_clock_found(cuda, monkeypatch):
    engine = engine_on(monkeypatch, [])
    found = engine._streams_beside()
    assert found[0] == engine.graphs.streams.beside[-1] and set(found) == set(engine.graphs.streams.beside)
    monkeypatch.setattr(engine_module.ops, "stream_beside", None)               # not asked again
    assert engine._streams_beside() is found


def test_an_attention_rides_beside_a_scan_in_chunks_where_their_workgroups_share_the_chip():
    """Behind long contexts the number of workgroups decides, whichever of heads, chunks and tokens they come from: a model with four
    times the heads stops at a quarter of the tokens.  Behind short ones the tokens do, a little earlier where the scan's heads
    are more than the compute units hold."""
    from macllm_infer_amd.kernels import ops

    def rides(tokens, longest, heads=24, query_heads=8, kv_heads=2, dh=64, lanes=1):
        chunks, tiles = -(-tokens // 128) + lanes - 1, -(-tokens // 64) + lanes          # (of a captured step)
        return bool(ops._fn("ssd", "mi_ssd_chunks_beside")(128, heads, 64, 128, chunks, tokens, query_heads, kv_heads, dh, tiles, longest))
    assert [rides(tokens, 4096) for tokens in (150, 256, 640, 896)] == [True, True, True, False]
    assert [rides(tokens, 4096, 48, 16, 4) for tokens in (150, 256, 512, 640)] == [True, True, False, False]
    assert [rides(tokens, 4096, 96, 32, 8) for tokens in (64, 150, 256, 640)] == [True, False, False, False]
    assert [rides(tokens, 4096, 96) for tokens in (256, 448, 640)] == [True, False, False]
    assert [rides(tokens, 4096, query_heads=32) for tokens in (129, 256, 640)] == [True, False, False]
    assert [rides(tokens, 2048) for tokens in (150, 768, 896, 1024)] == [True, True, True, False]
    assert [rides(tokens, 2048, 48) for tokens in (150, 768, 896, 1024)] == [True, True, False, False]
    assert [rides(tokens, 2048, query_heads=32) for tokens in (150, 896, 1024)] == [True, True, False]
    assert not rides(768, 2048, query_heads=32, lanes=16) and not rides(768, 2048, 192, 32, 8)      # far more than the chip holds
    assert not any(rides(tokens, 0, dh=128) for tokens in (129, 300))        # heads of 128 behind contexts of unknown length
