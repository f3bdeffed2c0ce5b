"""Scratch memory on a GPU that is too full for it: a failed allocation makes
torch give back its cached blocks, so it is not tried again by every call."""
import pytest
import torch

from rocm_qlora import ops

DEV = torch.device("cpu", 0)


@pytest.fixture
def memory(monkeypatch):
    """Requests of `n` bytes (the size query's argument) fail above state["room"]."""
    state = {"room": 100, "tried": 0, "failed": 0}

    def scratch(fn, dev, n):
        state["tried"] += 1
        if n > state["room"]:
            state["failed"] += 1
            raise torch.OutOfMemoryError("full")
        return torch.empty(n, dtype=torch.uint8)

    monkeypatch.setattr(ops, "_bytes", lambda fn, index, n: n)
    monkeypatch.setattr(ops, "_scratch", scratch)
    monkeypatch.setattr(ops, "_FULL", {}, raising=False)
    return state


def _got(n):
    t = ops._spare("size", DEV, n)
    return 0 if t is None else t.numel()


def test_failures_back_off(memory):
    assert all(_got(1000) == 0 for _ in range(2000))
    assert memory["failed"] <= 16  # 1, 2, 4 .. 256 calls apart


def test_smaller_requests_are_still_met(memory):
    for _ in range(20):
        assert _got(1000) == 0 and _got(80) == 80
    assert memory["tried"] - memory["failed"] == 20


def test_room_again(memory):
    for _ in range(500):
        _got(1000)
    memory["room"] = 2000
    assert any(_got(1000) for _ in range(257))
    assert all(_got(1000) == 1000 for _ in range(5))


def test_one_failure_costs_one_call(memory):
    assert _got(1000) == 0
    memory["room"] = 2000
    assert [_got(1000) for _ in range(3)] == [0, 1000, 1000]


def test_devices_are_apart(memory):
    assert _got(1000) == 0
    memory["room"] = 2000
    assert ops._spare("size", torch.device("cpu", 1), 1000).numel() == 1000


def test_nothing_asked_for(memory):
    assert _got(0) == 0
