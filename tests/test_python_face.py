"""The marshalling of the Python face: segments packed as bytes, the current stream's handle."""
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


@pytest.mark.gpu
def test_current_stream_is_torchs(t12):
    torch.zeros(1, device="cuda")
    assert t12.current_stream() == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert t12.current_stream() == s.cuda_stream
    assert t12.current_stream() == torch.cuda.current_stream().cuda_stream
