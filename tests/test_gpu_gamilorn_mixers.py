"""GPU: every mechanism of the Gamilorn layers through the C ABI, alone, against the float64 oracle: windowed attention on
the ring cache (prompt kernel, decode kernel, general kernel, 32-bit form), the delta rule (scan and step), learned
positions, norm, activations, the 32-bit linear, the activation epilogue of the decode-GEMV."""
import ctypes as C
import importlib

import numpy as np
import pytest
import torch

from gamilorn_util import bits_and_values
from gpu_util import dev, rel_err
from oracle import gamilorn_oracle as go

pytestmark = pytest.mark.gpu


def up(x, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev()).to(dtype)


def bf16(x):
    return bits_and_values(x)[1]


class Attention:
    """One region set of the windowed attention, fed with given q, k, v row by row or run by run."""

    def __init__(self, t12, heads, kv, dim, vdim, window, keep, scale=0.1, bias=None, fp32=False, regions=1, rows=64, positions=4096):
        self.t12, self.H, self.G, self.d, self.e, self.fp32 = t12, heads, kv, dim, vdim, fp32
        self.bias = np.full(heads, -1.0) if bias is None else bias
        a = self.a = t12.WindowAttn()
        a.heads, a.kv_heads, a.dim, a.vdim, a.window, a.keep_first, a.scale = heads, kv, dim, vdim, window, keep, scale
        a.elem_bytes = 4 if fp32 else 2
        t12.check(t12.lib.t12_window_plan(C.byref(a), positions, rows))
        dt = torch.float32 if fp32 else torch.int16
        self.k = torch.zeros(regions * a.k_elems, dtype=dt, device=dev())
        self.v = torch.zeros(regions * a.v_elems, dtype=dt, device=dev())
        self.hb = up(self.bias)
        a.k, a.v, a.head_bias = self.k.data_ptr(), self.v.data_ptr(), self.hb.data_ptr()
        a.q_off, a.k_off, a.v_off = 0, heads * dim, heads * dim + kv * dim
        self.ld = heads * dim + kv * (dim + vdim)
        self.ws = torch.empty(t12.lib.t12_parallel_step_ws_floats(), dtype=torch.float32, device=dev())
        self.cnt = torch.zeros(t12.STEP_MAX_ITEMS, dtype=torch.int32, device=dev())

    def feed(self, q, k, v, pos, region, step=False, scale=1.0):
        """q [n, H, d], ... at positions pos [n]; region: one number (a run) or a list (rows of their own)."""
        n, t12, lib = len(q), self.t12, self.t12.lib
        rng = np.random.default_rng(9)
        x = np.concatenate([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], 1)
        b = np.round(rng.standard_normal(self.ld) * 4) / 4                # a bias the kernels add back
        xi, bi = up(x - b), up(b)
        run = not isinstance(region, (list, tuple))
        rows = (t12.Row * n)(*[t12.Row(int(p), 2 * r) for p, r in zip(pos, [region] * n if run else region)])
        dr = torch.empty(2 * n, dtype=torch.int32, device=dev())
        st = t12.current_stream()
        t12.check(lib.t12_rows_list(dr.data_ptr(), rows, n, st))
        out = torch.zeros((n, self.H * self.e), dtype=torch.float32 if self.fp32 else torch.bfloat16, device=dev())
        args = (C.byref(self.a), xi.data_ptr(), bi.data_ptr(), self.ld, dr.data_ptr(), n)
        if step:
            rc = lib.t12_parallel_step(C.byref(self.a), None, *args[1:], int(max(pos)), scale, 0.0, out.data_ptr(), None,
                                       self.H * self.e, self.ws.data_ptr(), self.cnt.data_ptr(), st)
            assert rc == 0, rc
            assert int(self.cnt.abs().sum()) == 0
        else:
            t12.check(lib.t12_window_store(*args, int(run), st))
            t12.check(lib.t12_window_attention(*args, int(run), scale, out.data_ptr(), int(self.fp32), self.H * self.e, st))
        torch.cuda.synchronize()
        return out.float().cpu().numpy().astype(np.float64).reshape(n, self.H, self.e)


def qkv(rng, n, H, G, d, e, gain=1.0):
    return (bf16(rng.standard_normal((n, H, d)) * gain), bf16(rng.standard_normal((n, G, d)) * gain),
            bf16(rng.standard_normal((n, G, e))))


SHAPES = [  # heads, kv, dim, vdim, window, keep
    (4, 4, 32, 32, 7, 0), (6, 2, 64, 96, 33, 5), (8, 1, 48, 80, 32, 40), (5, 1, 128, 64, 1, 2), (4, 2, 16, 128, 100, 1),
    (20, 1, 32, 48, 64, 33), (2, 2, 136, 200, 31, 0), (3, 1, 24, 20, 500, 9), (2, 1, 256, 256, 50, 64),
    (4, 2, 64, 160, 8, 4), (3, 1, 96, 176, 40, 0), (2, 1, 128, 208, 20, 3), (4, 1, 160, 40, 12, 7), (6, 3, 200, 112, 45, 0)]
LARGE = [(2, 1, 72, 300, 24, 5), (3, 3, 288, 64, 17, 2)]      # no matrix-core instance


@pytest.mark.parametrize("shape", SHAPES + LARGE)
@pytest.mark.parametrize("fp32", [False, True])
def test_attention_in_runs_matches_the_oracle(t12, shape, fp32):
    H, G, d, e, window, keep = shape
    rng = np.random.default_rng(d + e)
    n = 150
    q, k, v = qkv(rng, n, H, G, d, e)
    bias = rng.standard_normal(H) - 1.0
    scale = 1.3 / np.sqrt(d)
    want = go.sigmoid_window_attention(q, k, v, bias, scale, window, keep)
    for cuts in ([64, 64, 22], [2, 31, 33, 1, 50, 33], [5] * 30):
        at = Attention(t12, H, G, d, e, window, keep, scale, bias, fp32)
        pos = 0
        for c in cuts:
            s = slice(pos, pos + c)
            got = at.feed(q[s], k[s], v[s], range(pos, pos + c), 0)
            assert rel_err(got, want[s]) < (1e-5 if fp32 else 5e-3), (cuts, pos)
            pos += c


@pytest.mark.parametrize("shape", SHAPES)
def test_decode_steps_match_the_oracle_and_the_general_kernel(t12, shape):
    H, G, d, e, window, keep = shape
    rng = np.random.default_rng(d + 2 * e)
    n, first = 130, 60
    q, k, v = qkv(rng, n, H, G, d, e)
    scale, bias = 1.3 / np.sqrt(d), rng.standard_normal(H) - 1.0
    want = go.sigmoid_window_attention(q, k, v, bias, scale, window, keep)
    step, plain = (Attention(t12, H, G, d, e, window, keep, scale, bias, rows=60) for _ in range(2))
    for at in (step, plain):
        at.feed(q[:first], k[:first], v[:first], range(first), 0)
    for i in range(first, n):
        s = slice(i, i + 1)
        assert rel_err(step.feed(q[s], k[s], v[s], [i], [0], step=True), want[s]) < 5e-3, i
        assert rel_err(plain.feed(q[s], k[s], v[s], [i], [0]), want[s]) < 5e-3, i


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("window, keep", [(32, 0), (33, 4), (64, 32), (5, 33), (96, 31), (1, 0)])
def test_each_window_and_kept_edge_shows_alone(t12, window, keep, fp32):
    """All weights are nearly zero except that of one key the query points at: its value must come out when the key is
    visible and nothing when it is not, at both sides of both edges, in a run and decoded."""
    H, G, d, e = 2, 1, 32, 32
    rng = np.random.default_rng(window)
    n = 170
    bias = np.full(H, -30.0)
    k = bf16(rng.standard_normal((n, G, d)))
    v = bf16(1.0 + rng.random((n, G, e)))
    k /= np.linalg.norm(k, axis=2, keepdims=True)
    k = bf16(k)
    targets = {}
    for i in range(n):
        edges = {0, keep - 1, keep, i, i - 1, i - window + 1, i - window, i - window - 1, i - 31, i - 32, i - 33}
        cand = sorted(j for j in edges if 0 <= j <= i)
        targets[i] = cand[i % len(cand)]
    q = np.zeros((n, H, d))
    for i in range(n):
        q[i, :] = 60.0 * k[targets[i], 0]
    q = bf16(q)
    want = go.sigmoid_window_attention(q, k, v, bias, 1.0, window, keep)
    seen = np.array([go.visible(i, targets[i], window, keep) for i in range(n)])
    # (float32 of the oracle's own reading: visible targets stand at weight ~1, the rest is noise far below it)
    assert (want[seen].min() > 0.9) and (~seen).any()
    ran = Attention(t12, H, G, d, e, window, keep, 1.0, bias, fp32, rows=64)
    got = np.concatenate([ran.feed(q[s:s + 64], k[s:s + 64], v[s:s + 64], range(s, min(s + 64, n)), 0) for s in range(0, n, 64)])
    tol = 1e-4 if fp32 else 2e-2
    assert np.abs(got - want).max() < tol * np.abs(want).max()
    dec = Attention(t12, H, G, d, e, window, keep, 1.0, bias, fp32, rows=2)       # the tightest ring
    for i in range(n):
        s = slice(i, i + 1)
        got = dec.feed(q[s], k[s], v[s], [i], [0], step=not fp32)
        assert np.abs(got - want[s]).max() < tol * np.abs(want).max(), i


def test_rows_of_their_own_use_their_own_regions(t12):
    """A batch of unequal sequences, decoded together and each alone, with a region freed and used again in between."""
    H, G, d, e, window, keep, B = 4, 2, 32, 48, 20, 3, 3
    rng = np.random.default_rng(4)
    lens = [50, 7, 33]
    seqs = [qkv(rng, m + 6, H, G, d, e) for m in lens]
    at = Attention(t12, H, G, d, e, window, keep, 0.2, regions=B)
    old = qkv(rng, 60, H, G, d, e, 3.0)
    at.feed(*old, range(60), 1)                                        # somebody was in region 1 before
    for b in range(B):
        m = lens[b]
        at.feed(*(x[:m] for x in seqs[b]), range(m), b)
    for s in range(6):
        q, k, v = (np.concatenate([seqs[b][x][lens[b] + s][None] for b in range(B)]) for x in range(3))
        got = at.feed(q, k, v, [lens[b] + s for b in range(B)], list(range(B)), step=True)
        for b in range(B):
            i = lens[b] + s
            want = go.sigmoid_window_attention(seqs[b][0][i:i + 1], seqs[b][1][:i + 1], seqs[b][2][:i + 1], at.bias, 0.2, window, keep, i)
            assert rel_err(got[b:b + 1], want) < 5e-3, (b, s)


@pytest.mark.parametrize("heads, kv, keep", [(8, 2, 0), (4, 4, 70), (40, 1, 3)])
def test_long_windows_split_over_workgroups(t12, heads, kv, keep):
    """A window of many blocks: the decode kernel splits it and adds the partial sums; same result as one stretch."""
    d, e, window, n = 64, 64, 1500, 2100
    rng = np.random.default_rng(5)
    q, k, v = qkv(rng, n + 3, heads, kv, d, e)
    at = Attention(t12, heads, kv, d, e, window, keep, 0.2, rows=700)
    for s in range(0, n, 700):
        at.feed(q[s:s + 700], k[s:s + 700], v[s:s + 700], range(s, s + 700), 0)
    for i in range(n, n + 3):
        s = slice(i, i + 1)
        want = go.sigmoid_window_attention(q[s], k[:i + 1], v[:i + 1], at.bias, 0.2, window, keep, i)
        a = at.feed(q[s], k[s], v[s], [i], [0], step=True)
        b = at.feed(q[s], k[s], v[s], [i], [0], step=True)
        assert rel_err(a, want) < 5e-3 and np.array_equal(a, b)
        ws, at.ws = at.ws, torch.empty(0, device=dev())               # no workspace: one stretch
        c = at.feed(q[s], k[s], v[s], [i], [0], step=True)
        at.ws = ws
        assert rel_err(c, want) < 5e-3


# ---------------------------------------------------------------------------------------------------- delta rule
class Delta:
    def __init__(self, t12, heads, dim, rank, regions=1, seed=0):
        self.t12, self.N, self.D, self.rank = t12, heads, dim, rank
        rng = np.random.default_rng(seed)
        hd = heads * dim
        self.w2, self.w0, self.norm = rng.standard_normal((hd, rank)) / np.sqrt(rank), rng.standard_normal(hd) * 2 - 2, 1 + 0.3 * rng.standard_normal(hd)
        self.w2t_d, self.w0_d, self.norm_d = up(self.w2.T), up(self.w0), up(self.norm)
        d = self.d = t12.DeltaRule()
        d.heads, d.dim, d.rank, d.unit_eps, d.decay_rate, d.out_eps = heads, dim, rank, 1e-6, float(np.exp(-0.5)), 1e-5
        d.w2t, d.w0, d.norm_w = self.w2t_d.data_ptr(), self.w0_d.data_ptr(), self.norm_d.data_ptr()
        for i, name in enumerate(("r_off", "k_off", "v_off", "a_off", "g_off", "w1_off")):
            setattr(d, name, i * hd)
        t12.check(t12.lib.t12_delta_plan(C.byref(d)))
        self.ld = 5 * hd + rank
        self.state = torch.zeros(regions * 2 * d.state_elems, dtype=torch.float32, device=dev())
        self.state += 7.0                                              # what a region holds before position 0 must not matter
        d.state = self.state.data_ptr()
        self.parity = [0] * regions

    def rows(self, pos, regions):
        n = len(pos)
        r = (self.t12.Row * n)(*[self.t12.Row(int(p), 2 * g + self.parity[g]) for p, g in zip(pos, regions)])
        dr = torch.empty(2 * n, dtype=torch.int32, device=dev())
        self.t12.check(self.t12.lib.t12_rows_list(dr.data_ptr(), r, n, self.t12.current_stream()))
        return dr

    def feed(self, x, pos, region, fp32=True, scale=1.0):
        n, t12 = len(x), self.t12
        run = not isinstance(region, (list, tuple))
        dr = self.rows(pos, [region] * n if run else region)
        xi, bi = up(x - 0.25), up(np.full(self.ld, 0.25))
        work = torch.empty(n * self.d.work_elems, dtype=torch.float32, device=dev())
        out = torch.zeros((n, self.N * self.D), dtype=torch.float32 if fp32 else torch.bfloat16, device=dev())
        t12.check(t12.lib.t12_delta_rule(C.byref(self.d), xi.data_ptr(), bi.data_ptr(), self.ld, dr.data_ptr(), n, int(run), scale,
                                         work.data_ptr(), out.data_ptr(), int(fp32), self.N * self.D, t12.current_stream()))
        torch.cuda.synchronize()
        for g in {region} if run else set(region):
            self.parity[g] ^= 1
        return out.float().cpu().numpy().astype(np.float64)

    def oracle(self, x, S=None, rate=np.exp(-0.5)):
        n, hd, heads = len(x), self.N * self.D, lambda y: y.reshape(len(x), self.N, self.D)
        r, k, v, a, g = (x[:, i * hd:(i + 1) * hd] for i in range(5))
        w = np.exp(-rate * go.sigmoid(np.tanh(x[:, 5 * hd:]) @ self.w2.T + self.w0))
        S = np.zeros((self.N, self.D, self.D)) if S is None else S
        o, S = go.delta_scan(heads(r), heads(k), heads(v), heads(w), heads(go.sigmoid(a)), S)
        return go.delta_output(o, g, self.norm, 1e-5), S


@pytest.mark.parametrize("heads, dim, rank", [(2, 64, 16), (3, 32, 8), (1, 48, 5), (2, 128, 33), (1, 200, 64), (1, 16, 1), (1, 300, 12)])
def test_delta_scan_matches_the_oracle_in_any_portions(t12, heads, dim, rank):
    D = Delta(t12, heads, dim, rank)
    n = 60
    x = np.random.default_rng(dim).standard_normal((n, D.ld))
    want, _ = D.oracle(x)
    for cuts in ([60], [17, 1, 2, 40], [2] * 30):
        pos = 0
        for c in cuts:
            got = D.feed(x[pos:pos + c], range(pos, pos + c), 0)
            assert rel_err(got, want[pos:pos + c]) < 1e-4, (cuts, pos)
            pos += c


@pytest.mark.parametrize("heads, dim", [(2, 64), (1, 128), (24, 64), (25, 64), (40, 24)])
@pytest.mark.parametrize("n", [1, 4, 5, 15, 16, 17, 20, 21, 31, 32, 33, 36, 37, 47, 63, 101])
def test_delta_scan_of_runs_that_end_inside_a_chunk(t12, heads, dim, n):
    """Token by token: sixteen at a time through LDS, then up to four last tokens from memory or more of them through LDS.  In chunks (52
    tokens and more of heads of 64): a last chunk of fewer tokens.  Then one more call on the state that is left."""
    D = Delta(t12, heads, dim, 3)
    x = np.random.default_rng(n).standard_normal((n + 6, D.ld))
    want, _ = D.oracle(x)
    assert rel_err(D.feed(x[:n], range(n), 0), want[:n]) < 1e-4
    assert rel_err(D.feed(x[n:], range(n, n + 6), 0), want[n:]) < 1e-4


@pytest.mark.parametrize("heads, dim, rank", [(2, 64, 64), (3, 48, 65), (1, 32, 5), (2, 33, 1), (1, 31, 3), (1, 64, 512), (1, 40, 449)])
@pytest.mark.parametrize("n", [39, 40, 48, 49, 51, 52, 64, 65, 81, 100, 113])
@pytest.mark.parametrize("decay", [0.0, float(np.exp(-0.5)), 1.0, 1.5])
def test_delta_chunks_equal_the_tokens_one_by_one(t12, heads, dim, rank, n, decay):
    """Runs of 52 tokens and more of heads of 32 to 64 channels go through the chunked kernels at decay rates up to one, portions of
    13 token by token: same outputs, same state, from a state that is not zero."""
    x = np.random.default_rng(n + dim).standard_normal((n + 7, Delta(t12, heads, dim, rank).ld))
    x[20, dim * heads] = 30.0                                          # a key that dwarfs the others
    got = []
    for cuts in ([n], [13] * (n // 13) + [n % 13] * (n % 13 > 0)):
        D = Delta(t12, heads, dim, rank)
        D.d.decay_rate = decay
        D.feed(x[:7], range(7), 0)
        out, pos = [], 7
        for c in cuts:
            out.append(D.feed(x[pos:pos + c], range(pos, pos + c), 0))
            pos += c
        got.append((np.concatenate(out), D.state.view(2, -1)[D.parity[0]].cpu().numpy()))
    # (32-bit sums of up to 64 terms, state and outputs of the order of their terms: some 1e-7 each)
    assert rel_err(got[0][1], got[1][1]) < 1e-5
    assert rel_err(got[0][0], got[1][0]) < 1e-5


@pytest.mark.parametrize("alike, removal", [(0.0, 0.0), (0.9, 0.0), (0.9, 3.0), (0.99, 3.0), (0.999, 8.0)])
@pytest.mark.parametrize("rate", [0.0, float(np.exp(-0.5)), 1.0])
@pytest.mark.parametrize("dim", [32, 64])
def test_delta_chunks_are_as_exact_as_the_tokens_one_by_one(t12, dim, rate, alike, removal):
    """Against 64 bits, for keys that resemble each other and removal rates near one as well: there a token takes away most of what the one
    before it put in, and a sum over a chunk's tokens is much larger than what is left of it."""
    n, heads = 304, 4
    rng = np.random.default_rng(dim)
    D = Delta(t12, heads, dim, 16)
    hd = heads * dim
    x = rng.standard_normal((n, D.ld))
    base = rng.standard_normal((heads, dim))
    x[:, hd:2 * hd] = (np.sqrt(alike) * base + np.sqrt(1 - alike) * x[:, hd:2 * hd].reshape(n, heads, dim)).reshape(n, hd)
    x[:, 3 * hd:4 * hd] += removal
    x = np.round(x * 4096) / 4096                                      # (what the kernels add a bias of a quarter back to, exactly)
    D.w2, D.w0, D.norm = (y.astype(np.float32).astype(np.float64) for y in (D.w2, D.w0, D.norm))
    want, S = D.oracle(x, rate=rate)
    err = []
    for cuts in ([n], [38] * 8):
        D = Delta(t12, heads, dim, 16)
        D.d.decay_rate = rate
        got = np.concatenate([D.feed(x[i * cuts[0]:i * cuts[0] + c], range(i * cuts[0], i * cuts[0] + c), 0) for i, c in enumerate(cuts)])
        state = D.state.view(2, heads, dim, -1)[D.parity[0]].cpu().numpy()[:, :, :dim].transpose(0, 2, 1).astype(np.float64)
        err.append([np.linalg.norm(got - want) / np.linalg.norm(want), np.linalg.norm(state - S) / np.linalg.norm(S)])
    # (the inputs' own rounding, in both; the recurrence's share is 0.5 to 0.9 of that of the tokens one by one)
    print("outputs %.2e %.2e state %.2e %.2e" % (err[0][0], err[1][0], err[0][1], err[1][1]))
    assert err[0][0] <= 1.05 * err[1][0] and err[0][1] <= 1.05 * err[1][1], err


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("dim, at", [(64, 37), (40, 47), (64, 48)])
def test_a_value_channel_that_is_not_finite_keeps_to_its_column(t12, dim, at, value):
    """A column of the state never meets another one: only that of the value channel is lost, as token by token."""
    n, states = 64, []
    x = np.random.default_rng(7).standard_normal((n, Delta(t12, 2, dim, 8).ld))
    x[at, 2 * 2 * dim + dim + 5] = value
    for cuts in ([n], [32, 32]):
        D, pos = Delta(t12, 2, dim, 8), 0
        for c in cuts:
            D.feed(x[pos:pos + c], range(pos, pos + c), 0)
            pos += c
        states.append(D.state.view(2, 2, dim, -1)[D.parity[0]].cpu().numpy()[:, :, :dim])
    assert np.array_equal(np.isfinite(states[0]), np.isfinite(states[1]))
    lost = ~np.isfinite(states[0])
    assert lost[1, 5].all() and lost.sum() == dim
    assert rel_err(states[0][~lost], states[1][~lost]) < 1e-5


def test_large_finite_tokens_leave_those_before_them_alone(t12):
    """Keys and values whose products 32 bits cannot hold: what they put into the state is not finite, the outputs before them are."""
    D, n, at = Delta(t12, 2, 64, 8), 64, 37
    x = np.random.default_rng(6).standard_normal((n, D.ld))
    want = D.feed(x, range(n), 0)
    x[at, D.d.k_off + 64:D.d.k_off + 128] *= 1e15
    x[at, D.d.v_off + 64:D.d.v_off + 128] *= 1e25
    got = D.feed(x, range(n), 0)
    assert np.array_equal(got[:at], want[:at]) and np.array_equal(got[:, :64], want[:, :64])
    assert not np.isfinite(got[at + 1, 64:]).all()


@pytest.mark.parametrize("field", ["k", "v", "a", "w1", "r"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_token_that_is_not_finite_leaves_those_before_it_alone(t12, field, value):
    D, n, at = Delta(t12, 2, 64, 8), 60, 37
    x = np.random.default_rng(5).standard_normal((n, D.ld))
    want = D.feed(x, range(n), 0)
    col = getattr(D.d, field + "_off") + (0 if field == "w1" else 64 + 3)
    x[at, col] = value
    got = D.feed(x, range(n), 0)
    if field in ("a", "w1") and value == float("inf"):
        assert np.isfinite(got).all()                                  # a removal rate of one; a tanh of one
        assert np.array_equal(got[:at], want[:at])
        return
    hit = slice(0, 128) if field == "w1" else slice(64, 128)           # (W2 takes w1 to every head)
    assert np.array_equal(got[:at], want[:at])
    assert np.isnan(got[at, hit]).any() and np.isnan(got[at:, hit]).any(axis=1).sum() == (1 if field == "r" else n - at)
    if field != "w1":
        assert np.array_equal(got[:, :64], want[:, :64])               # the other head


def test_delta_state_survives_long_sequences_and_restarts_at_zero(t12):
    D = Delta(t12, 2, 64, 16)
    x = np.random.default_rng(1).standard_normal((700, D.ld))
    want, _ = D.oracle(x)
    got = np.concatenate([D.feed(x[:650], range(650), 0)] + [D.feed(x[i:i + 1], [i], [0]) for i in range(650, 700)])
    assert rel_err(got, want) < 1e-4
    assert rel_err(D.feed(x[5:30], range(25), 0), D.oracle(x[5:30])[0]) < 1e-4


def test_taking_a_step_back_is_turning_the_pair_around(t12):
    D = Delta(t12, 2, 32, 4)
    x = np.random.default_rng(2).standard_normal((12, D.ld))
    D.feed(x[:10], range(10), 0)
    D.feed(x[11:12], [10], [0])                                        # a token that is then taken back
    D.parity[0] ^= 1
    got = D.feed(x[10:11], [10], [0])
    assert rel_err(got, D.oracle(x[:11])[0][10:]) < 1e-4


@pytest.mark.parametrize("heads, dim, rank", [(2, 64, 16), (3, 32, 8), (1, 48, 5), (2, 128, 33), (2, 16, 1), (1, 96, 500)])
def test_fused_step_equals_the_separate_calls(t12, heads, dim, rank):
    """t12_parallel_step with both mixers: three sequences at their own positions, one of them at its first token."""
    B, H, G, d, e = 3, 4, 2, 32, 64
    rng = np.random.default_rng(rank)
    at = Attention(t12, H, G, d, e, 10, 2, 0.2, regions=B)
    D = Delta(t12, heads, dim, rank, regions=B, seed=3)
    lens = [11, 0, 40]
    past = []
    for b in range(B):
        q, k, v = qkv(rng, lens[b] + 4, H, G, d, e)
        x = rng.standard_normal((lens[b] + 4, D.ld))
        if lens[b]:
            at.feed(q[:lens[b]], k[:lens[b]], v[:lens[b]], range(lens[b]), b)
            D.feed(x[:lens[b]], range(lens[b]), b)
        past.append((q, k, v, x))
    off = at.ld
    for name in ("r_off", "k_off", "v_off", "a_off", "g_off", "w1_off"):
        setattr(D.d, name, getattr(D.d, name) + off)
    for s in range(4):
        rows = []
        for b in range(B):
            q, k, v, x = past[b]
            i = lens[b] + s
            rows.append(np.concatenate([q[i].ravel(), k[i].ravel(), v[i].ravel(), x[i]]))
        xi, bi = up(np.stack(rows) - 0.5), up(np.full(at.ld + D.ld, 0.5))
        pos = [lens[b] + s for b in range(B)]
        dr = D.rows(pos, list(range(B)))
        old = max(H * e, heads * dim)
        left = torch.zeros((B, old), dtype=torch.bfloat16, device=dev())
        right = torch.zeros((B, old), dtype=torch.bfloat16, device=dev())
        rc = t12.lib.t12_parallel_step(C.byref(at.a), C.byref(D.d), xi.data_ptr(), bi.data_ptr(), at.ld + D.ld, dr.data_ptr(), B, max(pos),
                                       1.5, 0.5, left.data_ptr(), right.data_ptr(), old, at.ws.data_ptr(), at.cnt.data_ptr(), t12.current_stream())
        assert rc == 0
        D.parity = [p ^ 1 for p in D.parity]
        lo, ro = (y.float().cpu().numpy() for y in (left, right))
        for b in range(B):
            q, k, v, x = past[b]
            i = pos[b]
            want = 1.5 * go.sigmoid_window_attention(q[i:i + 1], k[:i + 1], v[:i + 1], at.bias, 0.2, 10, 2, i)
            assert rel_err(lo[b, :H * e], want.ravel()) < 5e-3, (s, b)
            assert rel_err(ro[b, :heads * dim], 0.5 * D.oracle(x[:i + 1])[0][i]) < 5e-3, (s, b)


# ------------------------------------------------------------------------------------------------- layer pieces
def test_embedding_with_positions(t12):
    rng = np.random.default_rng(0)
    (tb, tv), (pb, pv) = bits_and_values(rng.standard_normal((11, 50))), bits_and_values(rng.standard_normal((9, 50)))
    tok, pos = np.array([3, 10, 0, 11, -1], np.int32), [8, 0, 4, 2, 9]
    rows = (t12.Row * 5)(*[t12.Row(p, 0) for p in pos])
    dr = torch.empty(10, dtype=torch.int32, device=dev())
    out = torch.empty((5, 50), dtype=torch.float32, device=dev())
    tt, pt, tk = up(tb.view(np.int16), torch.int16), up(pb.view(np.int16), torch.int16), up(tok, torch.int32)
    t12.check(t12.lib.t12_rows_list(dr.data_ptr(), rows, 5, t12.current_stream()))
    t12.check(t12.lib.t12_embed_positions(tt.data_ptr(), 11, pt.data_ptr(), 9, tk.data_ptr(), dr.data_ptr(), out.data_ptr(), 50, 5,
                                          t12.current_stream()))
    got = out.cpu().numpy()
    assert np.allclose(got[:3], go.embed(tok[:3], pos[:3], tv, pv), atol=1e-6)
    assert np.allclose(got[3], pv[2]) and np.allclose(got[4], 0.0)            # outside their tables: zeros


def test_rows_run_table(t12):
    dr = torch.empty((300, 2), dtype=torch.int32, device=dev())
    t12.check(t12.lib.t12_rows_run(dr.data_ptr(), 1000, 5, 300, t12.current_stream()))
    got = dr.cpu().numpy()
    assert np.array_equal(got[:, 0], np.arange(1000, 1300)) and (got[:, 1] == 5).all()


@pytest.mark.parametrize("n", [64, 100, 777])
def test_norm_in_32_bit(t12, n):
    rng = np.random.default_rng(n)
    x, w = rng.standard_normal((5, n)) * 3, rng.standard_normal(n)
    out = torch.empty((5, n), dtype=torch.float32, device=dev())
    xd, wd = up(x), up(1.0 + w)
    t12.check(t12.lib.t12_rms_norm_f32(xd.data_ptr(), wd.data_ptr(), out.data_ptr(), n, 1e-3, 5, t12.current_stream()))
    assert rel_err(out.cpu().numpy(), go.norm_zero_centred(x, w, 1e-3)) < 1e-6


@pytest.mark.parametrize("n", [4096, 1023, 3])
def test_activations(t12, n):
    rng = np.random.default_rng(n)
    z = np.concatenate([rng.standard_normal(n - 3) * 4, [0.0, -1e-5, 1e-5]]) if n > 3 else np.array([0.0, -40.0, 60.0])
    p, q, lib, st = 0.3, -0.7, t12.lib, t12.current_stream()
    xie = t12.Act(t12.ACT_XIELU, float(go.softplus(p)), float(0.5 + go.softplus(q)))
    zd, o32, o16 = up(z), torch.empty(n, device=dev()), torch.empty(n, dtype=torch.bfloat16, device=dev())
    t12.check(lib.t12_act(zd.data_ptr(), xie, o32.data_ptr(), 1, n, st))
    t12.check(lib.t12_act(zd.data_ptr(), xie, o16.data_ptr(), 0, n, st))
    want = go.xielu(z, p, q)
    assert rel_err(o32.cpu().numpy(), want) < 1e-6 and np.allclose(o16.float().cpu().numpy(), want, rtol=4e-3, atol=1e-7)
    t12.check(lib.t12_act(zd.data_ptr(), t12.Act(t12.ACT_SOFTCAP, 5.0, 0.0), zd.data_ptr(), 1, n, st))          # in place
    assert rel_err(zd.cpu().numpy(), go.softcap(z, 5.0)) < 1e-6


def packed(t12, oracle, M, K, seed, p_outlier=2e-3):
    synth = importlib.import_module("turbo_lossless_amd.synth")
    w = synth.weights_llm(M, K, seed=seed, p_outlier=p_outlier)
    return t12.DeviceTensor12.from_packed(oracle.pack(w), dev()), synth.bf16_bits_to_f32(w).astype(np.float64)


@pytest.mark.parametrize("M, K, B", [(70, 96, 1), (64, 128, 33), (5, 37, 3), (200, 1031, 40)])
def test_linear_in_32_bit(t12, oracle, M, K, B):
    t, w = packed(t12, oracle, M, K, M + K, 2e-2)
    x = np.random.default_rng(B).standard_normal((B, K)).astype(np.float32)
    xd, out = up(x), torch.full((B, M), 2.0, device=dev())
    seg = (t12.Segment * 1)(t.segment(out))
    want = x.astype(np.float64) @ w.T
    for acc in (0, 1):
        t12.check(t12.lib.t12_gemm_f32(seg, 1, xd.data_ptr(), K, M, K, B, acc, t12.current_stream()))
        assert rel_err(out.cpu().numpy(), want * (1 + acc)) < 2e-6


@pytest.mark.parametrize("M, K", [(96, 64), (130, 1024), (64, 2064), (1000, 4096)])
def test_decode_gemv_with_activation(t12, oracle, M, K):
    t, w = packed(t12, oracle, M, K, M)
    rng = np.random.default_rng(K)
    xb, xv = bits_and_values(rng.standard_normal(K))
    lib, st = t12.lib, t12.current_stream()
    xd, x32, nw = up(xb.view(np.int16), torch.int16), up(rng.standard_normal(K)), up(1 + 0.2 * rng.standard_normal(K))
    out = torch.empty(M, device=dev())
    o16 = torch.empty(M, dtype=torch.bfloat16, device=dev())
    seg = (t12.Segment * 1)(t.segment(out))
    xie, cap = t12.Act(t12.ACT_XIELU, 0.8, 1.1), t12.Act(t12.ACT_SOFTCAP, 3.0, 0.0)
    # the epilogue is the plain product followed by the function
    for norm in (False, True):
        args = (None, x32.data_ptr(), nw.data_ptr(), 1e-5, K) if norm else (xd.data_ptr(), None, None, 0.0, K)
        plain = torch.empty(M, device=dev())
        pseg = (t12.Segment * 1)(t.segment(plain))
        if norm:
            t12.check(lib.t12_gemv_norm(pseg, 1, x32.data_ptr(), None, nw.data_ptr(), 1e-5, None, K, st))
        else:
            t12.check(lib.t12_gemv(pseg, 1, xd.data_ptr(), K, st))
            assert rel_err(plain.cpu().numpy(), w @ xv) < 1e-4
        ref16, ref32 = torch.empty_like(o16), torch.empty_like(out)
        t12.check(lib.t12_act(plain.data_ptr(), xie, ref16.data_ptr(), 0, M, st))
        t12.check(lib.t12_act(plain.data_ptr(), cap, ref32.data_ptr(), 1, M, st))
        t12.check(lib.t12_gemv_act(seg, *args, xie, o16.data_ptr(), st))
        t12.check(lib.t12_gemv_act(seg, *args, cap, None, st))
        # (a last-bit difference in the norm can move the bf16 rounding of an activation)
        tol = 1e-3 if norm else 1e-6
        assert rel_err(out.cpu().numpy(), ref32.cpu().numpy()) < tol
        assert rel_err(o16.float().cpu().numpy(), ref16.float().cpu().numpy()) < max(tol, 4e-3)
    assert lib.t12_gemv_act(seg, xd.data_ptr(), None, None, 0.0, K, t12.Act(7, 0, 0), None, st) == -1


@pytest.mark.parametrize("M, K, B", [(12400, 128, 70), (12416, 192, 300), (24700, 64, 128), (300, 256, 100), (2048, 2048, 64), (12416, 1088, 300), (1000, 4096, 33), (514, 100, 9)])
def test_linear_with_activation_over_a_batch(t12, oracle, M, K, B):
    """The epilogue form where the shape has one, the deferred form (function in the sum over the K splits) elsewhere."""
    t, w = packed(t12, oracle, M, K, M + B)
    xb, xv = bits_and_values(np.random.default_rng(B).standard_normal((B, K)))
    lib, st = t12.lib, t12.current_stream()
    xd, out = up(xb.view(np.int16), torch.int16), torch.empty((B, M), device=dev())
    o16 = torch.zeros((B, M), dtype=torch.bfloat16, device=dev())
    seg = (t12.Segment * 1)(t.segment(out))
    xie = t12.Act(t12.ACT_XIELU, 0.8, 1.1)
    z = xv @ w.T
    want = np.where(z > 0, 0.8 * z * z + 0.5 * z, 1.1 * (np.expm1(np.minimum(z, 0)) - np.minimum(z, 0)) + 0.5 * z)
    rc = lib.t12_gemm_act(seg, xd.data_ptr(), K, K, B, xie, o16.data_ptr(), M, st)
    assert rc == (0 if B > 64 else 1)
    if rc == 1:
        part = t12.GemmPartials()
        t12.check(lib.t12_gemm_deferred(seg, 1, xd.data_ptr(), K, M, K, B, part, st))
        assert (part.nsplit > 1) == ((M, K, B) in ((2048, 2048, 64), (1000, 4096, 33)))
        if part.nsplit > 1:
            t12.check(lib.t12_act_partials(part, xie, o16.data_ptr(), M, B, st))
        else:
            t12.check(lib.t12_act(out.data_ptr(), xie, o16.data_ptr(), 0, B * M, st))
    assert rel_err(o16.float().cpu().numpy(), want) < 5e-3


def test_gather_rows(t12):
    x = torch.arange(600 * 24, dtype=torch.int16, device=dev()).reshape(600, 24)
    pick = list(range(599, 0, -2))
    out = torch.empty((len(pick), 24), dtype=torch.int16, device=dev())
    t12.check(t12.lib.t12_util_gather_rows(out.data_ptr(), x.data_ptr(), 48, (C.c_int * len(pick))(*pick), len(pick), t12.current_stream()))
    assert torch.equal(out, x[pick])


def test_host_side_refusals(t12):
    a, lib = t12.WindowAttn(), t12.lib
    a.heads, a.kv_heads, a.dim, a.vdim, a.window, a.elem_bytes = 4, 3, 32, 32, 8, 2
    assert lib.t12_window_plan(C.byref(a), 100, 8) == -1               # heads not a multiple of kv_heads
    a.kv_heads, a.window = 2, 0
    assert lib.t12_window_plan(C.byref(a), 100, 8) == -1
    a.window = 8
    assert lib.t12_window_plan(C.byref(a), 100, 8) == 0 and a.ring_blocks == 1
    assert lib.t12_window_attention(C.byref(a), None, None, 0, None, 1, 0, 1.0, None, 0, 0, None) == -1
    d = t12.DeltaRule()
    d.heads, d.dim, d.rank = 1, 1000, 4
    assert lib.t12_delta_plan(C.byref(d)) == -1
