"""The marshalling of the Python face: segments packed as bytes, the current stream's handle."""
import ctypes as C

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("patched", [True, False])
@pytest.mark.parametrize("P", [0, 3, None])
@pytest.mark.parametrize("shape", [(5,), (2, 5), (2, 9)])
def test_segments_are_what_the_structures_hold(t12, patched, P, shape):
    i16, i32 = torch.int16, torch.int32
    lists = [None] * 4 if P is None else [torch.zeros(6, dtype=i32), torch.zeros(P, dtype=i32), torch.zeros(P, dtype=i16), torch.zeros(P, dtype=i16)]
    ts = [t12.DeviceTensor12(5, 64, e, torch.zeros(320, dtype=torch.uint8), torch.zeros(160, dtype=torch.uint8), *lists) for e in (-1, 112)]
    outs = [torch.zeros(shape)[..., :5] for _ in ts]
    want = t12._seg_array([t.segment(o, patched) for t, o in zip(ts, outs)])
    assert bytes(t12._segments(ts, outs, patched)) == bytes(want)

    class Other(t12.DeviceTensor12):                                   # a tensor that makes its segments itself
        def segment(self, out, patched=True):
            s = super().segment(out, patched)
            s.base_exp = 7
            return s

    o = Other(5, 64, 1, ts[0].sm, ts[0].gr)
    assert t12._segments([o], outs[:1], patched)[0].base_exp == 7


@pytest.mark.parametrize("name", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_current_stream_without_torchs_private_calls(t12, monkeypatch, name):
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _Stream(17))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 5, raising=False)
    assert t12.current_stream() == 5
    monkeypatch.delattr(torch._C, name)
    assert t12.current_stream() == 17


class _Stream:
    """A stream whose work is done when another one waits for it."""

    def __init__(self, handle):
        self.cuda_stream, self.todo = handle, []

    def wait_stream(self, other):
        while other.todo:
            other.todo.pop(0)()


@pytest.mark.parametrize("base_exp", [None, 111])
@pytest.mark.parametrize("handle", [0, 5])
def test_the_packer_reads_behind_the_stream_it_is_given(t12, monkeypatch, base_exp, handle):
    """The number of escapes and the base exponent, which the host reads, are there only once torch's current stream has waited for the one
    the kernels run on, and so are the planes and the list when the call returns."""
    here, other, w = _Stream(11), _Stream(handle), torch.zeros((3, 64), dtype=torch.int16)
    empty, seen = torch.empty, []

    class Lib:
        def _later(self, stream, at, *words):
            assert stream == handle
            data = np.array(words, np.int32)
            other.todo.append(lambda: C.memmove(at, data.ctypes.data, data.nbytes))
            return 0

        def t12_pack_begin(self, w, M, K, hist, base, sm, gr, cnt, off, st):
            return self._later(st, off, 0, 1, 1, 2, 112)

        def t12_pack_planes(self, w, M, K, base, sm, gr, cnt, st):
            return self._later(st, cnt, 1, 0, 1)

        def t12_pack_row_offsets(self, cnt, M, off, st):
            return self._later(st, off, 0, 1, 1, 2)

        def t12_pack_escapes_plane(self, w, gr, M, K, base, off, cols, correct, wrong, st):
            seen.append(base)
            return self._later(st, cols, 7, 9)

        def t12_pack_histogram(self, w, n, hist, st):
            return self._later(st, hist, 192)

        def t12_pack_base_exp(self, hist):
            return int(hist[0])

    monkeypatch.setattr(t12, "lib", Lib())
    monkeypatch.setattr(t12, "current_stream", lambda: here.cuda_stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: here)
    monkeypatch.setattr(torch.cuda, "default_stream", lambda device=None: other if handle == 0 else None)
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda h, device=None: other if h else None)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **k).fill_(33))
    d = t12.pack_device(w, base_exp, stream=handle)
    assert (d.P, d.base_exp, d.row_off.tolist(), d.cols.tolist()) == (2, base_exp or 112, [0, 1, 1, 2], [7, 9])
    assert seen == [d.base_exp] and not other.todo
    assert t12.find_base_exp_device(w, stream=handle) & 0xFFFFFFFF == 192


@pytest.mark.gpu
@pytest.mark.parametrize("base_exp", [None, 110])
def test_pack_on_a_stream_that_is_behind(t12, base_exp):
    g = torch.Generator(device="cuda").manual_seed(3)
    w = (torch.randn((1000, 992), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    w[::7, ::31] = 8.0
    want = t12.pack_device(w, base_exp)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)                                  # (some milliseconds)
    got = t12.pack_device(w, base_exp, stream=side.cuda_stream)
    assert (got.P, got.base_exp) == (want.P, want.base_exp) and got.P > 0
    for name in ("sm", "gr", "row_off", "cols", "correct", "wrong"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
    assert base_exp or t12.find_base_exp_device(w, stream=side.cuda_stream) == want.base_exp


@pytest.mark.gpu
def test_current_stream_is_torchs(t12):
    torch.zeros(1, device="cuda")
    assert t12.current_stream() == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert t12.current_stream() == s.cuda_stream
    assert t12.current_stream() == torch.cuda.current_stream().cuda_stream
