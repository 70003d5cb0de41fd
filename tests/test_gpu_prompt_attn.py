"""The prompt passes' attention kernel (64 (row, head) pairs of a KV group per workgroup, steps of 128 positions) against the
generic row by row kernel, through one layer's logits for every prompt position.

Both round the same attention outputs to bf16, so an output differs by at most one unit there (2^-8 of itself) and nearly
none do; the O projection and the rest of the layer keep that relative to the row's norm, where the attention's part
dominates (weights of sigma 0.02 on unit rows against embeddings of 0.02), and round to bf16 twice more.  Bound: 2^-7 of each
row's norm.  One position too many or too few at n positions would change a row by about 1 / sqrt(n) >= 4 %."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_head,n_kv,head_dim,chunks,own_region", [
    (32, 32, 64, (128, 129, 7), True),            # ratio 1: 64 tokens per workgroup; exact tiles, one more, a pass for the old kernel
    (64, 8, 64, (65, 64, 191), False),            # ratio 8: 8 tokens; a ragged last workgroup, the reference's cache layout
    (32, 8, 128, (128, 256), True),               # ratio 4
    (32, 16, 128, (200, 133), False),             # ratio 2: ragged; positions past 256 in three steps
    (16, 4, 128, (257, 300), True),
])
def test_prompt_attention_equals_the_row_by_row_kernel(t12, n_head, n_kv, head_dim, chunks, own_region):
    V = 512
    cfg = dict(n_vocab=V, n_embd=n_head * head_dim, n_head=n_head, n_head_kv=n_kv, n_layer=1, n_ff=512, n_ctx=640,
               rope_theta=10000.0, rms_norm_eps=1e-5)
    gen = torch.Generator().manual_seed(n_head + n_kv)
    rows = [torch.randint(3, V, (n,), generator=gen).tolist() for n in chunks]

    def logits():
        # region 1 of several (head-major), or the model's one region (the reference's layout)
        eng = t12.Engine.synthetic(cfg, seed=77, max_seq=640, batch=max(chunks), p_outlier=0.0, per_sequence=640 if own_region else 0)
        try:
            return torch.cat([torch.as_tensor(eng.prefill_logits(1 if own_region else 0, r)) for r in rows]).double()
        finally:
            eng.close()

    try:
        t12.lib.t12_tune_attention(0)
        want = logits()
    finally:
        t12.lib.t12_tune_attention(1)
    got = logits()
    assert torch.isfinite(got).all()
    err = ((got - want).norm(dim=1) / want.norm(dim=1)).max()
    assert err < 2.0 ** -7, float(err)
