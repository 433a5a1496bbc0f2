"""GPU parity of Q6_K matrices past 32 tokens in chunks of the few-token
kernel (whole ones and a last one partly filled, one workspace reused chunk
after chunk): shapes that the grouped GEMM does not take (n_embd or n_ff of
256, a vocabulary that is no multiple of 256) or where the chunks are faster
(an odd number of super-blocks), against the oracle.  Bar 5e-4, as the other
Q6_K projections."""
import numpy as np
import pytest

from conftest import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,FF,N", [(256, 768, 40), (256, 768, 72), (768, 256, 64), (768, 256, 72), (512, 2816, 40),
                                    (512, 2816, 64)])
def test_dense_q6k_chunks(ctx, O, H, FF, N):
    from dmoe import synth
    print(f"case: dense MLP H={H} n_ff={FF} Q6_K N={N}", flush=True)
    w = synth.host_dense(H, FF, 14, 90 + N, O.quantize_rows)
    x = synth.normal(91 + N, synth.S_X, N * H).reshape(N, H)
    layer = ctx.dense_upload(w)
    assert max_rel_err(ctx.forward(layer, x), O.dense_forward(w, x)) <= 5e-4
    layer.free()


@pytest.mark.parametrize("H,V", [(512, 1296), (256, 1280), (2816, 1024)])
@pytest.mark.parametrize("N", [33, 64, 72])
def test_head_q6k_chunks(ctx, O, H, V, N):
    from dmoe import synth
    print(f"case: LM head H={H} V={V} Q6_K N={N}", flush=True)
    w = synth.host_head(H, V, 14, 95 + N, O.quantize_rows)
    h = (synth.normal(96 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    head = ctx.head_upload(w)
    assert max_rel_err(ctx.head_forward(head, h, 1e-6, logits=True)[2], O.head_forward(w, h, 1e-6)[2]) <= 5e-4
    head.free()
