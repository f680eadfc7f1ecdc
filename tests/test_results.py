"""Results of the producers as objects: copied, saved, and done with the words that their totals landed in (ops.CompressedKV)."""
import copy
import ctypes
import gc
import io
import pickle
import weakref

import pytest
import torch


def landed(total, ws=None, words=None):
    """A result of values whose total landed in two words, and the words."""
    from mustafar_amd import ops
    pair = (ctypes.c_int64 * 2)(7, total)
    landing = ops._LandingPair(ctypes.addressof(pair), 0, ws, words)
    c = ops.CompressedKV(torch.arange(2).view(1, 2), torch.tensor([[0, 1, 2]], dtype=torch.int32), torch.ones(16, dtype=torch.float16),
                         torch.zeros(1, dtype=torch.int32), 64, 128, True, torch.tensor([max(total, -1)]), landing)
    return c, pair


@pytest.mark.parametrize("read_first", [False, True])
def test_results_are_copied_and_saved(read_first):
    c, pair = landed(8)
    if read_first:
        assert c.used_halfs() == 8
    file = io.BytesIO()
    torch.save(c, file)
    file.seek(0)
    for other in (copy.copy(c), copy.deepcopy(c), pickle.loads(pickle.dumps(c)), torch.load(file, weights_only=False)):
        assert torch.equal(other.bmp, c.bmp) and torch.equal(other.nz, c.nz) and other.is_value and other.tokens == 64
        assert other.used_halfs() == 8 and other.packed().numel() == 8 and other.nbytes() == c.nbytes()
    assert c.used_halfs() == 8


def test_a_result_saved_without_the_attribute():
    from mustafar_amd import ops
    c = ops.CompressedKV.__new__(ops.CompressedKV)
    c.__dict__.update(bmp=None, idx=None, nz=torch.ones(8), nz_off=None, tokens=64, head_dim=128, is_value=False,
                      total_halfs=torch.tensor([4]))
    assert c.used_halfs() == 4


def test_workspaces_are_saved_and_read_back():
    from mustafar_amd import ops
    ws = ops.Workspace("cpu", 512)
    for old in (False, True):
        if old:                                     # saved before it held status words
            del ws._status
        other = pickle.loads(pickle.dumps(ws))
        assert other.tensor.numel() == 512 and not other._spoilt and len(other._status) == 0
        other.status_spoilt(None)
        assert copy.deepcopy(ws).tensor.numel() == 512


def test_status_words_of_growing_calls_are_bounded(monkeypatch):
    from mustafar_amd import ops
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ws = ops.Workspace("cpu", 256)
    for words in range(64, 60000, 64):
        t = ws.status(words)
        assert t.numel() >= words and t is ws._status[-1]
    assert sum(t.numel() for t in ws._status) <= 4 * 60000
    before = len(ws._status)
    ws.status_spoilt(ws._status[-1])
    assert ws.status(64).numel() >= 59968 and len(ws._status) == before + 1 and ws.status(59968) is ws._status[-1]


def test_a_known_total_gives_the_words_back_and_holds_no_workspace():
    from mustafar_amd import ops
    ws = ops.Workspace("cpu", 256)
    ws._status.append(torch.zeros(8, dtype=torch.int64))
    c, pair = landed(8, ws, ws._status[-1])
    landing, alive = c._landing, weakref.ref(ws)
    given = []
    landing._give = given.append
    del landing
    assert c.used_halfs() == 8 and given == [ctypes.addressof(pair)]
    pair[1] = 5                                     # another call's by now
    assert c.used_halfs() == 8
    c, pair = landed(8, ws, ws._status[-1])
    del ws
    gc.collect()
    assert alive() is None and c.used_halfs() == 8


def test_a_give_up_marks_the_words_that_the_call_had():
    from mustafar_amd import ops
    ws = ops.Workspace("cpu", 256)
    ws._status.append(torch.zeros(8, dtype=torch.int64))
    c, pair = landed(-1, ws, ws._status[-1])
    old, pair2 = landed(-1, ws, torch.zeros(8, dtype=torch.int64))
    for bad, spoils in ((old, False), (c, True)):
        with pytest.raises(RuntimeError, match="gave up"):
            bad.packed()
        assert ws._spoilt == spoils


def test_a_total_is_waited_for_on_the_device_of_its_call(monkeypatch):
    from mustafar_amd import ops
    c, pair = landed(8)
    c._landing.device, current = 3, [0]

    class Device:
        def __init__(self, index):
            self.index = index

        def __enter__(self):
            current.append(self.index)

        def __exit__(self, *e):
            current.pop()

    class Library:
        def mstf_landing_wait(self, stream, word, value):
            assert current[-1] == 3 and word == ctypes.addressof(pair) + 8
            ctypes.c_int64.from_address(value).value = 8
            return 0

    pair[1] = ops._LandingPair.EMPTY
    monkeypatch.setattr(torch.cuda, "device", Device)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current[-1], raising=False)
    monkeypatch.setattr(ops, "lib", Library)
    assert c.used_halfs() == 8 and current == [0]


def test_status_words_stay_with_the_current_device(monkeypatch):
    from mustafar_amd import ops
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    ws = ops.Workspace("cpu", 256)
    monkeypatch.setattr(ws, "device", torch.device("cuda", 1))
    assert ops._own_workspace(ws, torch.device("cuda", 1)) is None
    assert ops._own_workspace(ws, torch.device("cuda", 0)) is ws


@pytest.mark.gpu
def test_a_word_that_never_comes_is_an_error():
    from mustafar_amd import ops
    from mustafar_amd._lib import lib
    word, value = torch.empty(1, dtype=torch.int64, pin_memory=True), ctypes.c_int64()
    word[0] = ops._LandingPair.EMPTY
    assert lib().mstf_landing_wait(ops._stream(), word.data_ptr(), ctypes.addressof(value)) == -5
    word[0] = 6
    assert lib().mstf_landing_wait(ops._stream(), word.data_ptr(), ctypes.addressof(value)) == 0 and value.value == 6


@pytest.mark.gpu
def test_a_pair_is_given_back_once():
    from mustafar_amd._lib import lib
    L = lib()
    pair = L.mstf_landing_take()
    for p in (pair, pair, pair + 8, pair + 4):      # twice, and what is no pair
        L.mstf_landing_give(p)
    held = []
    while True:
        p = L.mstf_landing_take()
        if not p:
            break
        held.append(p)
        assert len(held) <= 1024
    assert len(set(held)) == len(held) and pair in held
    for p in held:
        L.mstf_landing_give(p)


@pytest.mark.gpu
def test_more_results_than_pairs():
    from mustafar_amd import ops
    x = torch.randn((1, 64, 128), device="cuda", dtype=torch.float16)
    results = []
    for _ in range(1100):
        c = ops.compress_kv(x, x, 89, 89, capacity_halfs=4096)
        assert c[0]._landing is not None
        assert all(side.used_halfs() == int(side.total_halfs) for side in c)    # (keys' and values' tiles are padded each on their own)
        results.append(c)
