"""Decode-graph capture through torch's nccl process group waits for the group's watchdog first: the engine's own agreements
(the consistency check, the capture's) are eager collectives that the watchdog thread tracks until its next pass, and a query of
their end events while the capture holds the communicator's stream ends the process. CPU only: the group and the capture are
stand-ins that record the order of things."""
import contextlib
import types

import pytest
import torch
import torch.distributed as dist

from llmss_amd.engine import LLMEngine
from llmss_amd.engine.engine import _DecodeBuffers
from llmss_amd.models.config import get_preset
from llmss_amd.models.decoder import DecoderLM
from llmss_amd.models.weights import random_weights
from llmss_amd.parallel.dist import TPGroup


class TrackedGroup:
    """The watchdog's list: eager collectives stay on it until waited for."""

    def __init__(self, log):
        self.log, self.pending = log, 0

    def _wait_for_pending_works(self):
        self.log.append("wait")
        self.pending = 0


class TorchTP(TPGroup):
    """Rank 0 of two on a stand-in nccl group; collectives leave the values alone."""

    def __init__(self, group):
        super().__init__(0, 2, group=group)

    def _eager(self):
        if not self._suspend and not self.group.capturing:
            self.group.pending += 1

    def all_reduce(self, t):
        self._eager()
        return t

    def all_gather_last_dim(self, t):
        self._eager()
        return torch.cat([t, t], -1)

    def all_gather_object(self, obj):
        self._eager()
        return [obj, obj]

    def all_reduce_int(self, v, op="min"):
        self._eager()
        return int(v)


@pytest.fixture
def engine(monkeypatch):
    log = []
    group = TrackedGroup(log)
    group.capturing = False
    monkeypatch.setattr(dist, "get_backend", lambda g=None: "nccl")
    nothing = types.SimpleNamespace(wait_stream=lambda s: None)

    @contextlib.contextmanager
    def graph(g, **kw):
        assert group.pending == 0, "a capture starts while the watchdog tracks collectives"
        log.append("capture")
        group.capturing = True
        yield
        group.capturing = False

    for name, v in (("Stream", lambda: nothing), ("current_stream", lambda: nothing), ("synchronize", lambda: None),
                    ("stream", lambda s: contextlib.nullcontext()), ("empty_cache", lambda: None), ("graph", graph),
                    ("graph_pool_handle", lambda: None), ("CUDAGraph", lambda: types.SimpleNamespace(replay=lambda: None))):
        monkeypatch.setattr(torch.cuda, name, v)
    cfg = get_preset("tiny-llama", hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=256, num_layers=2)
    m = DecoderLM(cfg, random_weights(cfg, 2, 0, dtype=torch.float32, seed=5, std=0.05), TorchTP(group))
    e = LLMEngine(m, max_num_seqs=8, block_size=16, num_blocks=64, use_graphs=False, autotune=False, graph_buckets=[1, 8])
    e.buf = _DecodeBuffers(e.buckets[-1], e.max_blocks, torch.device("cpu"))
    return e, group, log


def test_capture_waits_for_the_watchdog(engine):
    e, group, log = engine
    assert e.tp.torch_pg and group.pending > 0  # the constructor's consistency checks
    e.capture_graphs()
    assert log.index("wait") < log.index("capture")
    assert log.count("capture") == len(e.buckets) * len(e._decode_modes())


def test_schedule_captures_wait_for_the_watchdog(engine, monkeypatch):
    e, group, log = engine
    e.capture_graphs()
    e._tbo_cands = [8]
    log.clear()

    class Event:
        def __init__(self, **kw): pass
        def record(self): pass
        def synchronize(self): pass
        def elapsed_time(self, o): return 1.0
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(e.model, "overlap_split", lambda b: 0)  # (the second stream's own calls are not the point)
    e._schedule_ab(e._graph_pool, e._graph_modes)
    assert "capture" in log and log.index("wait") < log.index("capture")


def test_settle_waits_on_nccl_groups_only(monkeypatch):
    log = []
    g = TrackedGroup(log)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: log.append("sync"))
    monkeypatch.setattr(dist, "get_backend", lambda g=None: "nccl")
    TPGroup(0, 2, group=g).settle()
    assert log == ["sync", "wait"]
    log.clear()
    TPGroup(0, 2, fake=True).settle()
    TPGroup(0, 1).settle()
    TPGroup(0, 2, group=g, comm=object()).settle()  # native communicator: no watchdog
    monkeypatch.setattr(dist, "get_backend", lambda g=None: "gloo")
    TPGroup(0, 2, group=g).settle()
    assert log == []
