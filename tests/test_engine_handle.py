"""An engine's native half lives exactly as long as something that can use it (no GPU: a stand-in for the library)."""
import gc

import pytest

from mini_llm_amd import Engine, EngineOptions, native


class Library:
    def __init__(self):
        self.destroyed = []

    def mllm_engine_runner(self, handle):
        return handle + 1

    def mllm_engine_destroy(self, handle):
        self.destroyed.append(handle)

    def mllm_runner_info(self, handle, buf, cap):
        text = b'{"vocab_size": 5}\0'
        if buf is not None and cap >= len(text):
            buf[:len(text)] = text
        return len(text) - 1


@pytest.fixture
def library(monkeypatch):
    lb = Library()
    monkeypatch.setattr(native, "_lib", lb)
    gc.collect()
    gc.disable()                       # nothing here may wait for the collector of cycles
    yield lb
    gc.enable()


def test_an_engine_let_go_is_destroyed_at_once(library):
    e = Engine(10, EngineOptions())
    del e
    assert library.destroyed == [10]


def test_a_runner_in_use_keeps_its_engine(library):
    r = Engine(10, EngineOptions()).runner
    assert library.destroyed == []
    del r
    assert library.destroyed == [10]


def test_close_destroys_once(library):
    e = Engine(10, EngineOptions())
    e.close()
    assert library.destroyed == [10]
    e.close()
    del e
    assert library.destroyed == [10]
