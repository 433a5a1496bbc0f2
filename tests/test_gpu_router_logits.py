"""GPU parity of the router logits of many tokens (k_logits_mfma: f32 MFMA
tiles of 32 tokens x 32 experts): the oracle's bits, with a last tile of
tokens and of experts that is partly filled, and one, two and three 256-value
steps of the hidden size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [256, 512, 768])
@pytest.mark.parametrize("E,N", [(256, 768), (200, 901)])
def test_logits_many_tokens(ctx, O, H, E, N):
    from dmoe import synth
    print(f"case: router logits H={H} E={E} N={N}", flush=True)
    cfg = synth.LayerConfig("logits", H, E, 256, 48, 2, 32, 0, 0, 0, N, -0.05, 0.05)
    w = synth.host_layer(cfg, 17, O.quantize_rows)
    x = synth.make_x(cfg, 17, N)
    x[5, ::3] *= np.float32(1e-38)          # subnormal products and sums
    layer = ctx.upload(w)
    dg = ctx.forward(layer, x, debug=True)[1]
    dr = O.layer_forward(w, x, debug=True)[1]
    for k in ("logits", "probs", "idx", "weights", "counts", "perm"):
        assert np.array_equal(np.asarray(dg[k]).view(np.uint8), np.asarray(dr[k]).view(np.uint8)), k
    layer.free()
