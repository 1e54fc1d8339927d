"""The workspaces that matmul2 keeps with parameter objects (cumm_amd/gemm/main.py _Slots): who shares one,
who must not, how many wait for an owner.  Host memory stands for the device's."""
import copy
import gc
import threading

import pytest

from cumm_amd import tensorview as tv
from cumm_amd.gemm import main
from cumm_amd.tensorview.gemm import GemmParams

SIZE = 1 << 17


@pytest.fixture
def device(monkeypatch):
    now, made = [0], []

    def empty(shape, dtype, where):
        made.append(shape[0])
        return tv.Tensor(shape, dtype)
    monkeypatch.setattr(main, "empty", empty)
    monkeypatch.setattr(main._Slots, "_device", staticmethod(lambda: now[0]))
    monkeypatch.setattr(main._Slots, "_spare", {})
    return now, made


def _params(stream=0):
    p = GemmParams()
    p.stream = stream
    return p


def _address(p, nbytes=SIZE):
    return main._Slots.of(p, nbytes).byte_pointer()


def test_an_object_keeps_its_buffer_and_leaves_it_to_the_next_on_its_stream(device):
    now, made = device
    p = _params()
    first = _address(p)
    p.alpha = 2.0
    assert _address(p) == first and _address(p, 100) == first and len(made) == 1
    del p
    gc.collect()
    for stream, dev in ((7, 0), (0, 1)):        # another stream, another device
        now[0] = dev
        assert _address(_params(stream)) != first
    now[0] = 0
    count = len(made)
    assert _address(_params()) == first and len(made) == count
    larger = _params()
    assert main._Slots.of(larger, SIZE + 1).nbytes > SIZE and len(made) == count + 1
    assert _address(_params()) == first          # (the small one is still there)


def test_live_objects_copies_and_other_streams_have_buffers_of_their_own(device):
    a, b = _params(), _params()
    assert _address(a) != _address(b)
    c = copy.copy(a)
    c.alpha = 2.0
    assert _address(c) != _address(a)
    before = _address(a)
    a.stream = 5
    assert _address(a) != before
    a.stream = 0
    assert _address(a) not in (_address(b), _address(c))


def test_few_buffers_wait_for_an_owner(device):
    many = [_params(stream) for stream in range(50)] + [_params() for _ in range(50)]
    for p in many:
        _address(p)
    del p, many
    gc.collect()
    assert 0 < len(main._Slots._spare) <= main._Slots._MOST


def test_threads_on_one_stream_never_share_a_buffer(device):
    held, clashes, lock = set(), [], threading.Lock()

    def work():
        for _ in range(300):
            p = _params()
            at = _address(p)
            with lock:
                clashes.extend([at] if at in held else [])
                held.add(at)
            with lock:
                held.discard(at)
            del p
    threads = [threading.Thread(target=work) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert clashes == [] and len(main._Slots._spare) <= main._Slots._MOST
