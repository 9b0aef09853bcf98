"""CPU validation of the reference op implementations themselves.

The paged references are checked against dense (non-paged) attention so the
GPU kernel tests compare against a trustworthy baseline.
"""

import pytest
import torch

from production_stack_amd import ops
from production_stack_amd.ops import reference


def test_rms_norm_matches_manual():
    x = torch.randn(5, 64, dtype=torch.bfloat16)
    w = torch.randn(64, dtype=torch.bfloat16)
    out = reference.rms_norm(x, w, 1e-6)
    xf = x.float()
    want = xf / (xf.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.float()
    torch.testing.assert_close(out.float(), want, atol=2e-2, rtol=2e-2)


def test_paged_decode_matches_dense_attention():
    torch.manual_seed(0)
    S, qh, kh, hd, bs = 3, 8, 2, 64, 16
    seq_lens = torch.tensor([5, 33, 16], dtype=torch.int32)
    max_blocks = 4
    nb = S * max_blocks + 1
    k_cache = torch.randn(nb, kh, bs, hd, dtype=torch.bfloat16)
    v_cache = torch.randn(nb, kh, bs, hd, dtype=torch.bfloat16)
    bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(S, max_blocks)
    q = torch.randn(S, qh, hd, dtype=torch.bfloat16)
    out = reference.paged_attn_decode(q, k_cache, v_cache, bt, seq_lens, 0.125)

    for s in range(S):
        ctx = int(seq_lens[s])
        k = reference._gather_kv(k_cache, bt[s], ctx).float()
        v = reference._gather_kv(v_cache, bt[s], ctx).float()
        for h in range(qh):
            kvh = h // (qh // kh)
            attn = torch.softmax((k[:, kvh] @ q[s, h].float()) * 0.125, dim=-1)
            want = attn @ v[:, kvh]
            torch.testing.assert_close(
                out[s, h].float(), want, atol=2e-2, rtol=2e-2
            )


def test_prefill_is_causal():
    """A prefill token at position p must ignore cache entries > p."""
    torch.manual_seed(0)
    qh, kh, hd, bs = 2, 2, 64, 16
    nb, max_blocks = 5, 4
    k_cache = torch.randn(nb, kh, bs, hd, dtype=torch.bfloat16)
    v_cache = torch.randn(nb, kh, bs, hd, dtype=torch.bfloat16)
    bt = torch.arange(1, 5, dtype=torch.int32).reshape(1, max_blocks)
    q = torch.randn(2, qh, hd, dtype=torch.bfloat16)
    token_seq = torch.zeros(2, dtype=torch.int32)
    token_pos = torch.tensor([3, 7], dtype=torch.int32)
    out = reference.paged_attn_prefill(
        q, k_cache, v_cache, bt, token_seq, token_pos, 0.125
    )
    # poisoning cache entries beyond each token's position must not change it
    k2, v2 = k_cache.clone(), v_cache.clone()
    k2[bt[0, 1].long(), :, :] = 1e4  # tokens 16.. (beyond pos 7)
    v2[bt[0, 1].long(), :, :] = -1e4
    out2 = reference.paged_attn_prefill(
        q, k2, v2, bt, token_seq, token_pos, 0.125
    )
    torch.testing.assert_close(out, out2)


def test_rope_preserves_tail_dims():
    """rot_dim < head_dim leaves the tail dims untouched."""
    T, qh, kh, hd, rot = 4, 2, 1, 64, 32
    pos = torch.arange(T, dtype=torch.int32)
    inv = 1.0 / (10000.0 ** (torch.arange(0, rot, 2).float() / rot))
    freqs = torch.outer(torch.arange(16).float(), inv)
    cos_sin = torch.cat([freqs.cos(), freqs.sin()], -1)
    q = torch.randn(T, qh * hd, dtype=torch.bfloat16)
    k = torch.randn(T, kh * hd, dtype=torch.bfloat16)
    q2, k2 = reference.rotary_embedding(pos, q, k, cos_sin, hd)
    torch.testing.assert_close(
        q2.view(T, qh, hd)[..., rot:], q.view(T, qh, hd)[..., rot:]
    )
    # position 0 is the identity rotation
    torch.testing.assert_close(
        q2.view(T, qh, hd)[0, :, :rot].float(),
        q.view(T, qh, hd)[0, :, :rot].float(),
        atol=1e-2,
        rtol=1e-2,
    )


def test_gemm_policy_limits():
    """The dispatch's idea of what fits in LDS is the kernel's."""
    from production_stack_amd import ops
    from production_stack_amd.ops import gemm_policy

    if not ops.HAVE_EXT:
        pytest.skip("extension not built")
    assert ops._C.skinny_limits() == (gemm_policy._LDS_X,
                                      gemm_policy._LDS_NORM_X)


@pytest.mark.parametrize("rule,shape,own", [
    # rows, rows of W, entries of each: on either side of each line
    ("few_rows", (1, 28672, 512), True), ("few_rows", (1, 28672, 256), False),
    ("few_rows", (1, 16384, 256), True), ("few_rows", (1, 16384, 192), False), ("few_rows", (3, 50304, 1536), True),
    ("few_rows", (4, 50304, 1536), False), ("few_rows", (16, 50304, 2048), True),
    ("few_rows", (8, 1024, 8192), True), ("few_rows", (8, 512, 8192), False),
    ("few_rows", (5, 512, 8192), True), ("few_rows", (16, 6144, 4096), True),
    ("few_rows_alone", (16, 6144, 4096), False),
    ("few_rows_alone", (12, 6144, 4096), True),
    ("few_rows_alone", (16, 4096, 4096), True),
    ("few_rows_alone", (16, 8256, 4096), True),
    ("few_rows_alone", (16, 6144, 3072), True),
    ("few_rows_alone", (17, 4096, 2048), False),
    ("rows_before_norm", (60, 2048, 1280), False),
    ("rows_before_norm", (60, 2048, 2048), True),
    ("rows_before_norm", (63, 2048, 3584), True),
    ("rows_before_norm", (63, 4096, 4096), False),
    ("rows_before_norm", (64, 4096, 4096), True),
    ("rows_before_norm", (32, 4096, 4096), True),
    ("rows_before_norm", (32, 4096, 3584), False),
    ("rows_before_norm", (63, 2560, 8192), False),
    ("rows_before_norm", (64, 2560, 8192), True),
    ("rows_before_norm", (96, 4096, 4096), True),
    ("rows_before_norm", (112, 4096, 4096), False),
    ("rows_before_norm", (129, 4096, 4096), True),
    ("rows_before_norm", (112, 4096, 6144), True),
    ("rows_before_norm", (80, 5120, 6144), False),
    ("rows_before_norm", (112, 5120, 4096), True),
    ("rows_before_norm", (144, 5120, 6144), False),
    ("rows_before_norm", (144, 6144, 4096), True),
    ("rows_before_norm", (176, 6144, 4096), False),
    ("rows_before_norm", (176, 6144, 5120), True),
    ("rows_before_norm", (176, 5120, 8192), True),
    ("rows_before_norm", (24, 4096, 12288), False),
    ("rows_before_norm", (24, 4096, 14336), True),
    ("rows_before_norm", (24, 8192, 13824), False),
    ("rows_before_norm", (32, 8192, 13824), True),
    ("rows_before_norm", (104, 1024, 10240), False),
    ("rows_before_norm", (104, 1024, 14336), True),
    ("rows_before_norm", (80, 5376, 5120), False),
    ("rows_before_norm", (80, 5632, 5120), True),
    ("rows_before_norm", (24, 2048, 1024), False),
    ("rows_before_norm", (24, 2560, 1024), True),
    ("rows_before_norm", (64, 3584, 3328), False),
    ("rows_before_norm", (64, 3584, 3584), True),
    ("rows_before_norm", (32, 4096, 12288), True),
    ("rows_before_rope", (144, 6144, 4096), True),
    ("rows_before_rope", (176, 6144, 4096), False),
    ("rows_before_rope", (176, 6144, 5120), True),
    ("rows_before_rope", (144, 5120, 4096), False),
    ("rows_before_rope", (160, 8192, 4096), False),
    ("rows_before_rope", (160, 8192, 5120), True),
    ("rows_before_rope", (144, 8192, 8192), True),
    ("rows_before_rope", (144, 5376, 8192), False),
    ("rows_before_gate", (48, 28288, 2048), True),
    ("rows_before_gate", (48, 28224, 2048), False),
    ("rows_before_rope", (128, 9216, 3584), False),
    ("rows_before_rope", (160, 9216, 3584), True)])
def test_gemm_policy_lines(rule, shape, own):
    """Which untuned products are in-house, by the lines that were measured."""
    from production_stack_amd.ops import gemm_policy

    assert getattr(gemm_policy, "_" + rule)(*shape) == own


def test_window_attention_plan():
    """Shares of portions' keys: of a sequence's rows alone behind many keys, of many
    short sequences behind some, none where nothing is gained; never more than
    records are merged of or than two rounds of the CUs."""
    def plan(rows, keys, runs, H=32, G=8, D=128):
        return ops._window_shares(rows, H, G, D, D, keys, runs)

    assert plan(70, 2570, 1) >= 8 and 4 <= plan(250, 2750, 1) <= 8
    assert plan(100, 100, 1) == plan(300, 300, 1) == plan(200, 400, 1) == 1
    # as many keys of one sequence are less than those of each of many
    assert plan(32, 602, 16) > plan(32, 602, 1) > 1
    assert plan(128, 302, 64) > plan(128, 302, 1) == 1
    assert plan(1419, 3419, 1) == plan(4000, 4000, 2) == 1
    for H, G, D in ((32, 8, 128), (40, 1, 64), (300, 2, 8), (1, 1, 128)):
        for rows in (1, 2, 31, 32, 33, 500, 5000):
            for keys in (0, 1, 63, 200, 5000, 100000):
                for runs in {1, 2, rows // 2 or 1, rows}:
                    n = plan(rows, keys, min(runs, rows), H, G, D)
                    heads = min(H // G, 128)
                    groups = (-(-rows // (128 // heads)) * G
                              * -(-(H // G) // 128))
                    assert n == 1 or 1 < n <= min(16, 512 // groups)
