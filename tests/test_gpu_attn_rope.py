"""GPU parity of the rotary step of many tokens (k_qk_rope_heads, from 65,536
(token, head) rows: four heads of a token per wavefront) against the oracle:
64 and 66 heads (whole groups of four, and a last one of two; Q, K
and V heads in one group), head dimensions of 64 and 128.  Bar 1e-5, as the F32
attention shapes of test_gpu_attn."""
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
