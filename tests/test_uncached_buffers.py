"""Buffers of the peer-to-peer all-reduce: never freed, used again by the next all-reduce of the process once every rank has closed the
one before, and not at all where a peer may still write to them; a peer's, once mapped, are never unmapped."""
import os

import pytest
import torch

from minivllm_amd.parallel import custom_allreduce as ca


class _Lib:
    """The library's memory functions on a counter."""

    def __init__(self):
        self.top, self.cleared, self.freed, self.closed, self.opened = 4096, [], [], [], []

    def mvl_car_alloc(self, out, nbytes, uncached):
        assert uncached
        out._obj.value = self.top
        self.top += nbytes
        return 0

    def mvl_car_clear(self, p, nbytes):
        self.cleared.append((nbytes, p.value))
        return 0

    def mvl_car_free(self, p):
        self.freed.append(p)
        return 0

    def mvl_car_ipc_open(self, handle, out):
        self.opened.append(handle)
        out._obj.value = 1 << 40 | len(self.opened)
        return 0 if handle else 1

    def mvl_car_ipc_close(self, p):
        self.closed.append(p)
        return 0

    def mvl_car_set_loopback(self, on):
        pass


@pytest.fixture
def idle(monkeypatch):
    monkeypatch.setattr(ca, "_IDLE", {}, raising=False)
    monkeypatch.setattr(ca, "_MAPPED", {}, raising=False)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)


def _reduce(lib, sizes=(512, 64, 256), device=0):
    car = object.__new__(ca.CustomAllReduce)
    car._lib, car.device, car.loopback, car.group = lib, torch.device("cuda", device), True, None
    car._buffers = [ca._take_buffer(lib, device, n) for n in sizes] if hasattr(ca, "_take_buffer") else []
    car._own, car._mapped = [p for _, p in car._buffers] or [4096], [7]             # (_mapped: what a close would unmap)
    return car


def test_a_closed_one_frees_nothing_and_the_next_takes_over(idle, monkeypatch):
    monkeypatch.setattr(ca.dist, "barrier", lambda group=None: None)
    lib = _Lib()
    first = _reduce(lib)
    own = list(first._own)
    first.close()
    assert not lib.freed and not lib.closed and first._own == []
    first.close()                                               # (once closed, nothing is given back twice)
    top = lib.top
    second = _reduce(lib, (64, 200, 512))                       # the smallest that holds each; all of it cleared
    assert second._own == [own[1], own[2], own[0]] and lib.top == top
    assert lib.cleared == [(64, own[1]), (256, own[2]), (512, own[0])]
    third = _reduce(lib)                                        # two at a time: buffers of their own
    assert not set(third._own) & set(own) and lib.top > top
    other = _reduce(lib, device=1)
    third.close()
    assert not set(_reduce(lib, device=1)._own) & set(third._own) and other._own


def test_what_a_peer_may_still_write_to_is_not_used_again(idle, monkeypatch):
    lib = _Lib()
    dead = _reduce(lib)
    own = set(dead._own)
    dead._release()

    def gone(group=None):
        raise RuntimeError("a peer is gone")
    monkeypatch.setattr(ca.dist, "barrier", gone)
    alone = _reduce(lib)
    own |= set(alone._own)
    alone.close()
    assert not lib.freed and not set(_reduce(lib)._own) & own


def test_a_peers_buffer_is_mapped_once_and_stays(idle):
    lib, a, b = _Lib(), (11, b"a", 4096), (11, b"b", 4096)          # (a later process of the same number)
    at = ca._map_peer(lib, 0, a, b"one")
    assert ca._map_peer(lib, 0, a, b"two") == at and lib.opened == [b"one"]
    others = {ca._map_peer(lib, 0, b, b"one"), ca._map_peer(lib, 1, a, b"one"), ca._map_peer(lib, 0, (12, b"a", 4096), b"one")}
    assert len(others | {at}) == 4 and len(lib.opened) == 4
    with pytest.raises(RuntimeError, match="ipc_open"):
        ca._map_peer(lib, 0, (13, b"a", 0), b"")
    assert len(ca._MAPPED) == 4


@pytest.mark.gpu
def test_the_next_one_works_on_the_same_memory():
    import torch.distributed as dist
    dist.init_process_group("gloo", init_method=f"tcp://127.0.0.1:{29433 + os.getpid() % 200}", rank=0, world_size=1)
    try:
        seen = None
        for _ in range(3):
            car = ca.CustomAllReduce(dist.group.WORLD, 1, 4, torch.device("cuda", 0), max_bytes=1 << 20, loopback=True)
            own = sorted(car._own)
            assert car.healthy() and car.self_test()
            car.close()
            assert seen in (None, own)
            seen = own
    finally:
        dist.destroy_process_group()
