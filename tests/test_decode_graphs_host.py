"""Lifetime of captured decode graphs (CPU): no collection inside a capture, and a dropped
manager takes its executor (and graphs) along without the collector."""

import gc
import weakref
from contextlib import contextmanager
from types import SimpleNamespace

import torch

from tokserve_amd.batching import execution, graphs
from tokserve_amd.batching.metadata import SequenceWork
from tokserve_amd.engine.config import LlamaConfig
from tokserve_amd.engine.model import LlamaModel
from tokserve_amd.engine.paged.manager import PagedKVCacheManager


class Cycle:
    """Garbage that only the collector finds; reports when it goes."""

    def __init__(self, gone: list) -> None:
        self.me = self
        self.gone = gone

    def __del__(self) -> None:
        self.gone.append(True)


def test_no_garbage_is_collected_inside_a_capture(monkeypatch) -> None:
    gone: list = []
    state = {"capturing": False, "inside": None}

    @contextmanager
    def capture(graph):
        state["capturing"] = True
        yield
        state["capturing"] = False

    def forward_packed(batch, storage):
        if state["capturing"]:  # enough tracked objects for several automatic collections
            kept = [[i] for i in range(50_000)]
            state["inside"] = (len(kept), len(gone), gc.isenabled())
        return torch.zeros(batch.num_tokens, 4)

    monkeypatch.setattr(torch.cuda, "graph", capture)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: SimpleNamespace(replay=lambda: None))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: Cycle(gone))
    monkeypatch.setattr(graphs.ops, "greedy_argmax", lambda x: x.argmax(-1, keepdim=True))
    monkeypatch.setattr(graphs.DecodeGraphs, "_upload", lambda self, *args: None)
    storage = SimpleNamespace(block_size=2, device=torch.device("cpu"))
    runner = graphs.DecodeGraphs(SimpleNamespace(forward_packed=forward_packed), storage)
    assert gc.isenabled()
    runner.run([SequenceWork((1,), 0, (0,))])
    assert state["inside"] == (50_000, 0, False)
    assert gc.isenabled()
    gc.collect()
    assert gone == [True]


def test_a_dropped_manager_frees_its_executor_without_the_collector() -> None:
    config = LlamaConfig(vocab_size=32, hidden_size=16, intermediate_size=24,
                         num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=1,
                         max_position_embeddings=16)
    model = LlamaModel(config)
    manager = PagedKVCacheManager(num_layers=1, num_blocks=4, num_key_value_heads=1,
                                  block_size=2, head_dim=8, device=torch.device("cpu"),
                                  dtype=torch.float32)
    gc.collect()
    gc.disable()
    try:
        executor = weakref.ref(execution._executor_for(model, manager))
        assert executor() is execution._executor_for(model, manager)
        assert executor().manager is manager
        alive = weakref.ref(manager)
        del manager
        assert alive() is None and executor() is None
    finally:
        gc.enable()
    own = execution.BatchExecutor(model, PagedKVCacheManager(
        num_layers=1, num_blocks=4, num_key_value_heads=1, block_size=2, head_dim=8,
        device=torch.device("cpu"), dtype=torch.float32))
    assert own.manager.storage.num_layers == 1  # an executor of the caller's own holds it
