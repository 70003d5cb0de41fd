"""GPU: the medium-batch decode+GEMM (3 .. 64 rows, planes and activations copied global -> LDS in rings of 128-column
windows) against float64 products of the matrices the tensors were packed from, at the sizes where it can go wrong: fewer
windows than the ring holds, windows that the K waves share unevenly, K slices, rows past a tile, slices begun in the
middle, batch tiles with one row, escape lists the LDS holds, overflowing ones, several entries of a row in one window.

Tolerance: products of bf16 are exact in fp32 and the sums are fp32, at most K terms in any order: K 2^-24 of
sum_k |w||x| bounds them; a tenth of that is asserted."""
import ctypes as C

import pytest
import torch

from gpu_util import dev

pytestmark = pytest.mark.gpu


def weight(M, K, seed, p_out, sigma=0.02):
    g = torch.Generator(device=dev()).manual_seed(seed)
    w = torch.randn((M, K), generator=g, device=dev()) * sigma
    if p_out:
        m = torch.rand((M, K), generator=g, device=dev()) < p_out
        w = torch.where(m, torch.randn((M, K), generator=g, device=dev()) * 8, w)
    return w.to(torch.bfloat16)


def acts(B, K, seed):
    return torch.randn((B, K), generator=torch.Generator(device=dev()).manual_seed(seed), device=dev()).to(torch.bfloat16)


def check(t12, Ms, K, B, p_out):
    Ws = [weight(M, K, 10 + i, p_out, 0.02 * 4 ** i) for i, M in enumerate(Ms)]
    X = acts(B, K, 5)
    pad = torch.zeros((B, K + 64), dtype=torch.int16, device=dev())
    pad[:, :K] = X.view(torch.int16)
    total = sum(Ms)
    big = torch.full((B, total + 8), float("nan"), device=dev())
    outs, c = [], 0
    for M in Ms:
        outs.append(big[:, c:c + M])
        c += M
    t12.gemm([t12.pack_device(w) for w in Ws], pad[:, :K], outs=outs)
    torch.cuda.synchronize()
    assert bool(big[:, total:].isnan().all())                  # nothing written past the last tensor
    for w, o in zip(Ws, outs):
        want, scale = X.double() @ w.double().T, X.double().abs() @ w.double().abs().T
        assert bool(((o.double() - want).abs() <= 0.1 * K * 2.0 ** -24 * scale + 1e-30).all()), (Ms, K, B)


@pytest.mark.parametrize("B", [33, 48, 64])
@pytest.mark.parametrize("Ms,K,p_out", [([1], 128, 0), ([17, 300], 256, 2e-3), ([129], 384, 2e-2), ([65, 1, 63], 640, 2e-3), ([1023], 1152, 3e-4),
                                        ([2300], 1024, 2e-3), ([4097], 2048, 3e-4), ([300], 14336, 2e-3), ([700], 4096, 5e-2)])
def test_four_batch_tiles(t12, Ms, K, p_out, B):
    check(t12, Ms, K, B, p_out)


@pytest.mark.parametrize("B", [17, 32])
@pytest.mark.parametrize("Ms,K,p_out", [([40], 14336, 2e-3), ([9000], 384, 2e-3), ([9000, 5001], 1280, 2e-2), ([20001], 128, 0), ([33000], 1024, 3e-4),
                                        ([16385], 256, 0.2), ([1000, 1000], 11008, 1e-2)])
def test_two_batch_tiles(t12, Ms, K, p_out, B):
    check(t12, Ms, K, B, p_out)


@pytest.mark.parametrize("B", [3, 5, 8, 9, 16])
@pytest.mark.parametrize("Ms,K,p_out", [([40], 14336, 2e-3), ([1100], 14336, 2e-2), ([28000], 384, 2e-3), ([33000], 1024, 3e-4), ([4097], 8192, 3e-4),
                                        ([7000, 7001], 2176, 1e-2), ([30000], 128, 0.2)])
def test_one_batch_tile(t12, Ms, K, p_out, B):
    check(t12, Ms, K, B, p_out)


def test_planes_that_are_not_aligned_take_the_general_kernels(t12):
    """A tensor whose planes start off a 16-byte boundary: the same product."""
    M, K, B = 300, 512, 40
    w = weight(M, K, 3, 2e-3)
    p = t12.pack_device(w)
    for name in ("sm", "gr"):
        plane = getattr(p, name)
        shifted = torch.empty(plane.numel() + 16, dtype=torch.uint8, device=dev())
        shifted[4:4 + plane.numel()] = plane
        setattr(p, name, shifted[4:4 + plane.numel()])
    X = acts(B, K, 6)
    (out,) = t12.gemm([p], X.view(torch.int16))
    want, scale = X.double() @ w.double().T, X.double().abs() @ w.double().abs().T
    assert bool(((out.double() - want).abs() <= 0.1 * K * 2.0 ** -24 * scale).all())


def test_infinite_and_nan_weights_stay_in_their_rows(t12):
    M, K, B = 200, 1024, 40
    w = weight(M, K, 4, 2e-3)
    w[7, 3], w[60, 1000], w[61, 127] = float("inf"), float("-inf"), float("nan")
    X = acts(B, K, 7)
    (out,) = t12.gemm([t12.pack_device(w)], X.view(torch.int16))
    want = X.double() @ w.double().T
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf()) and torch.equal(out[:, [7, 60]].sign(), want[:, [7, 60]].float().sign())
    assert bool(out[:, [i for i in range(M) if i not in (7, 60, 61)]].isfinite().all())


@pytest.mark.parametrize("M,K,B,p_out", [(14400, 2048, 9, 2e-3), (14337, 1152, 16, 3e-4), (14336, 1024, 33, 2e-3), (13001, 384, 64, 2e-2), (16000, 384, 24, 0.2),
                                         (15001, 256, 40, 2e-3), (600, 14336, 8, 2e-3), (3000, 11008, 5, 3e-4), (14336, 4096, 7, 3e-4)])
def test_gated_epilogue_is_bit_identical_to_unfused(t12, M, K, B, p_out):
    gate, up = t12.pack_device(weight(M, K, 1, p_out)), t12.pack_device(weight(M, K, 2, p_out, 0.3))
    X = acts(B, K, 3).view(torch.int16)
    st = t12.current_stream()
    og, ou = t12.gemm([gate, up], X)
    want = torch.empty((B, M), dtype=torch.int16, device=dev())
    t12.lib.launch_silu_mul_bf16_batch(og.data_ptr(), ou.data_ptr(), want.data_ptr(), M, B, st)
    got = torch.full((B, M + 8), -1, dtype=torch.int16, device=dev())
    rc = t12.lib.t12_gemm_swiglu(t12._seg_array([gate.segment(None)]), t12._seg_array([up.segment(None)]), X.data_ptr(), K, K, B, got.data_ptr(),
                                 M + 8, st)
    assert rc == 0, t12.lib.t12_last_error()
    assert torch.equal(got[:, :M], want) and bool((got[:, M:] == -1).all())


def test_deferred_partial_sums_add_up_to_the_same_bits(t12):
    M, K, B = 4096, 14336, 48
    p = t12.pack_device(weight(M, K, 8, 3e-4))
    X = acts(B, K, 9).view(torch.int16)
    (want,) = t12.gemm([p], X)
    out = torch.empty((B, M), device=dev())
    part = t12.GemmPartials()
    t12.check(t12.lib.t12_gemm_deferred(t12._seg_array([p.segment(out)]), 1, X.data_ptr(), K, M, K, B, C.byref(part), t12.current_stream()))
    assert part.nsplit > 1
    ws = torch.empty(part.nsplit * part.split_stride, device=dev())
    torch.cuda.synchronize()
    assert t12._hip_memcpy_d2d(ws.data_ptr(), part.ws, ws.numel() * 4) == 0
    tot = torch.zeros((B, M), device=dev())
    for z in range(part.nsplit):
        tot += ws.view(part.nsplit, B, part.ld)[z, :, :M]
    assert torch.equal(tot, want)


@pytest.mark.parametrize("T,K,ff,one", [(9, 128, 257, False), (24, 384, 1000, False), (70, 640, 384, False), (20, 256, 2100, True), (64, 1152, 300, True)])
def test_experts(t12, T, K, ff, one):
    """The launch over experts, whose rows are counted on the device: 1 / 2 / 4 batch tiles by the hint, experts without
    rows, every token at one expert (several passes of its batch tiles).  Gate and up sums are as above; their unit is
    rounded to bf16, where a value may differ by one place: 2^-8 of the output's norm."""
    from turbo_lossless_amd import moe
    E, k = 8, 2
    Ws = [[weight(M, Kc, 100 * e + i, 2e-3 if e % 2 else 2e-2, 0.05) for i, (M, Kc) in enumerate(((ff - ff % 64 + 64, K),) * 2 + ((K, ff - ff % 64 + 64),))]
          for e in range(E)]
    X = acts(T, K, T)
    g = torch.Generator(device=dev()).manual_seed(7 + T)
    ids = torch.stack([torch.randperm(E - 1, generator=g, device=dev())[:k] for _ in range(T)])         # the last expert has none
    if one:
        ids[:, 0], ids[:, 1] = 3, 4 * torch.arange(T, device=dev()) % 7
        ids[:, 1] = torch.where(ids[:, 1] == 3, 5, ids[:, 1])
    w = torch.rand((T, k), generator=g, device=dev())
    layer = moe.MoeLayer([moe.Expert(*[t12.pack_device(m) for m in e]) for e in Ws])
    got = layer(X.view(torch.int16), ids, w).double()
    want = torch.zeros((T, K), dtype=torch.float64, device=dev())
    for e in range(E):
        a, b = X.double() @ Ws[e][0].double().T, X.double() @ Ws[e][1].double().T
        h = (torch.nn.functional.silu(a) * b).to(torch.bfloat16).double()
        share = torch.where(ids == e, w, torch.zeros_like(w)).sum(1).double()
        want += share[:, None] * (h @ Ws[e][2].double().T)
    assert float((got - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.parametrize("Ms,K,B", [([8192, 64], 2048, 200), ([4224], 4096, 130), ([4224], 4096, 100), ([8576], 2048, 300), ([1100, 3124], 1152, 128)])
def test_splits_that_would_be_a_few_workgroups_more_than_the_chip(t12, Ms, K, B):
    """More than 64 rows, where the usual K split comes to 257 .. 288 workgroups: fewer slices, odd counts of them."""
    check(t12, Ms, K, B, 2e-3)
