"""GPU parity: the GPU-side packer emits byte-identical arrays to the oracle's
(reference-pinned) packer."""
import importlib

import numpy as np
import pytest
import torch

from gpu_util import to_dev_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def synth(t12):
    return importlib.import_module("turbo_lossless_amd.synth")


def check_same(t12, oracle, w, base_exp=None):
    wd = to_dev_bits(w).reshape(w.shape)
    if base_exp is None:
        assert t12.find_base_exp_device(wd) == oracle.find_base_exp(w)
    d = t12.pack_device(wd, base_exp)
    p = oracle.pack(w, base_exp)
    torch.cuda.synchronize()
    assert d.base_exp == p.base_exp
    for f in ("sm", "gr", "row_off", "cols", "correct", "wrong"):
        assert np.array_equal(getattr(d, f).cpu().numpy(), getattr(p, f)), f
    return d, p


def test_golden_cases(t12, oracle, golden):
    for name, g in golden.items():
        forced = int(g["base_exp"]) if int(g["base_exp"]) != int(g["found_base_exp"]) else None
        check_same(t12, oracle, g["w"], forced)


@pytest.mark.parametrize("M,K", [(4096, 4096), (1280, 5120), (333, 1001), (1, 15), (7, 17), (128256 // 8, 4096)])
def test_shapes(t12, oracle, synth, M, K):
    gen = synth.weights_diffusion if K == 5120 else synth.weights_llm
    d, p = check_same(t12, oracle, gen(M, K, seed=M * 7 + K))
    # and the packed tensor decodes back on the GPU
    out = t12.decompress(d, patched=True)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint16), oracle.decode(p))


def test_all_patterns_and_forced_base(t12, oracle):
    w = np.arange(65536, dtype=np.uint16).reshape(256, 256)
    for be in (None, -1, 0, 100, 127, 240):
        check_same(t12, oracle, w, be)


@pytest.mark.parametrize("K", [32, 64, 2016, 2048, 2080, 4096, 4128, 6176])
@pytest.mark.parametrize("share", [0.0, 3e-4, 0.3])
def test_escapes_from_the_nibble_plane(t12, oracle, K, share):
    """Rows of 32 to three steps of 2048 columns and a bit: without escapes, with few, with many per lane, all of them, at both ends; and the
    entry point that reads the weights gives the same list."""
    rng = np.random.default_rng(K)
    w = (0x3C00 + rng.integers(0, 0x700, size=(11, K))).astype(np.uint16)          # exponents of one window
    esc = rng.random((11, K)) < share
    esc[1] = True
    esc[2], esc[3] = False, False
    esc[2, 0], esc[3, K - 1] = True, True
    w[esc] = (rng.integers(0, 2, size=int(esc.sum())) << 15 | 0x4100 | rng.integers(0, 128, size=int(esc.sum()))).astype(np.uint16)
    base = int(oracle.find_base_exp(w)) if share < 0.1 else 0x78 - 1
    d, p = check_same(t12, oracle, w, base)
    wd, n = to_dev_bits(w).reshape(w.shape), int(d.cols.numel())
    other = [torch.empty(n, dtype=t.dtype, device=t.device) for t in (d.cols, d.correct, d.wrong)]
    t12.check(t12.lib.t12_pack_escapes(wd.data_ptr(), 11, K, base, d.row_off.data_ptr(), *(o.data_ptr() for o in other), t12.current_stream()))
    for a, b in zip(other, (d.cols, d.correct, d.wrong)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("M", [1, 3, 4095, 4096, 4097, 8192, 12301])
def test_row_offsets(t12, M):
    c = torch.randint(0, 9, (M,), dtype=torch.int32, device="cuda")
    off = torch.full((M + 2,), -7, dtype=torch.int32, device="cuda")
    t12.check(t12.lib.t12_pack_row_offsets(c.data_ptr(), M, off.data_ptr(), t12.current_stream()))
    assert off[0] == 0 and off[M + 1] == -7 and torch.equal(off[1:M + 1].long(), torch.cumsum(c.long(), 0))


@pytest.mark.parametrize("M", [2 ** 31 - 8193, 2 ** 31 - 1])
def test_row_offsets_up_to_the_largest_row_count(t12, M):
    c = torch.zeros(M, dtype=torch.int32, device="cuda")
    at = [0, 5, 2 ** 30, M - 8192, M - 1]
    for i, r in enumerate(at):
        c[r] = 10 ** i
    off = torch.full((M + 2,), -7, dtype=torch.int32, device="cuda")
    t12.check(t12.lib.t12_pack_row_offsets(c.data_ptr(), M, off.data_ptr(), t12.current_stream()))
    assert off[0] == 0 and off[M + 1] == -7
    ends = at[1:] + [M]
    for i, (r, end) in enumerate(zip(at, ends)):                       # constant between the rows that count
        assert off[r + 1] == off[end] == int("1" * (i + 1)), (i, r)


def test_base_exponent_on_the_device(t12, oracle):
    """The window rule where windows tie (the first wins), where nothing is in a window's reach, and at both ends of the exponents."""
    for exps in ([0], [255], [1, 200], [15, 100], [254, 255], [16, 31, 46], list(range(256))):
        w = np.repeat(np.array(exps, np.uint16) << 7, 64).reshape(len(exps), 64)
        check_same(t12, oracle, w)
