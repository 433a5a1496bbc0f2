"""GPU parity of the rotary step of many tokens (k_qk_rope_heads, from 65,536
(token, head) rows: four heads of a token per wavefront) against the oracle:
64 and 66 heads (whole groups of four, and a last one of two; Q, K
and V heads in one group), head dimensions of 64 and 128.  Bar 1e-5, as the F32
attention shapes of test_gpu_attn; bit for bit against the kernel of fewer
rows, and on a projection's reduction slices."""
import numpy as np
import pytest

from conftest import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,kv,hd,rd,N", [(60, 2, 64, 32, 1024), (62, 2, 128, 128, 1000), (64, 1, 64, 64, 1001)])
def test_rope_many_rows(ctx, O, nh, kv, hd, rd, N):
    from dmoe import synth
    H = 256
    print(f"case: attention half, {nh}/{kv} heads of {hd}, N={N}", flush=True)
    # F32 projections, so that the rotary step and the attention set the error
    w = synth.host_attn(0, 5, O.quantize_rows, n_embd=H, n_head=nh, n_head_kv=kv, head_dim=hd, rotary_dim=rd,
                        block_length=32)
    layer = ctx.attn_upload(w)
    h = synth.normal(77, synth.S_X, N * H).reshape(N, H)
    y, x = ctx.attn_forward(layer, h)
    yr, xr = O.attn_forward(w, h)
    assert max_rel_err(y, yr) <= 1e-5 and max_rel_err(x, xr) <= 1e-5
    layer.free()


@pytest.mark.parametrize("nh,kv,hd,rd,qk", [(60, 2, 64, 32, True), (62, 2, 128, 128, True), (64, 1, 64, 64, False),
                                            (60, 1, 128, 64, False)])
def test_rope_kernels_agree_bit_for_bit(ctx, O, nh, kv, hd, rd, qk):
    """The first token count that takes k_qk_rope_heads against one token
    fewer, which takes k_qk_rope: with block-causal attention a token's output
    depends on the tokens up to the end of its block only, so every token of a
    block that is whole in both has the same bits."""
    from dmoe import synth
    H, heads = 256, nh + 2 * kv
    N = -(-65536 // heads)
    print(f"case: attention half, {nh}/{kv} heads of {hd}, N={N} and {N - 1}, qk_norm={qk}", flush=True)
    w = synth.host_attn(0, 6, O.quantize_rows, n_embd=H, n_head=nh, n_head_kv=kv, head_dim=hd, rotary_dim=rd,
                        block_length=32, qk_norm=qk)
    layer = ctx.attn_upload(w)
    h = synth.normal(78, synth.S_X, N * H).reshape(N, H)
    many, few = ctx.attn_forward(layer, h), ctx.attn_forward(layer, h[:N - 1])
    whole = (N - 1) // 32 * 32
    for a, b in zip(many, few):
        assert np.array_equal(a[:whole].view(np.uint32), b[:whole].view(np.uint32))
    layer.free()


@pytest.mark.parametrize("qk", [True, False])
def test_rope_many_rows_of_slices(ctx, O, qk):
    """Q4_K: the fused projection leaves two reduction slices (test_plan pins
    that), which the rotary step of many rows adds."""
    from dmoe import synth
    H, nh, kv, hd, N = 2048, 60, 2, 64, 1030
    print(f"case: attention half, {nh}/{kv} heads of {hd}, Q4_K H={H}, N={N}, qk_norm={qk}", flush=True)
    w = synth.host_attn(12, 7, O.quantize_rows, H, nh, kv, hd, 32, block_length=32, qk_norm=qk)
    layer = ctx.attn_upload(w)
    h = (synth.normal(79, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    y, x = ctx.attn_forward(layer, h)
    yr, xr = O.attn_forward(w, h)
    assert max_rel_err(y, yr) <= 1e-4 and max_rel_err(x, xr) <= 1e-4
    layer.free()
