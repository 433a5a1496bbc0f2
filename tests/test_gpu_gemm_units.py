"""GPU parity of the grouped GEMM over units of tokens (projections past the
few-token kernel: the LM head, the dense MLP): units of 64 tokens in two
blocks of 32, the last a half block of 16, each partly filled, whole, or just
begun.

Bars (max|y - y_oracle| / max|y_oracle|): as the projections' other tests,
exact weights times the activations as two int8 digits: 5e-4."""
import numpy as np
import pytest

from conftest import max_rel_err

pytestmark = pytest.mark.gpu

TOL = 5e-4
WTYPES = [12, 14, 8]


@pytest.mark.parametrize("wtype", WTYPES)
@pytest.mark.parametrize("N", [33, 48, 63, 64, 65, 97, 128])
def test_head_units(ctx, O, wtype, N):
    from dmoe import synth
    H, V = 512, 1280            # two super-blocks: the shortest reduction; five row groups
    print(f"case: LM head H={H} V={V} type={wtype} N={N}", flush=True)
    w = synth.host_head(H, V, wtype, 20 + N, O.quantize_rows)
    h = (synth.normal(21 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    head = ctx.head_upload(w)
    lg = ctx.head_forward(head, h, 1e-6, logits=True)[2]
    err = max_rel_err(lg, O.head_forward(w, h, 1e-6)[2])
    print(f"  max rel err {err:.3e}", flush=True)
    assert err <= TOL
    head.free()


@pytest.mark.parametrize("N", [1, 7, 16, 17, 32])
def test_head_q80_few_tokens(ctx, O, N):
    """Q8_0 projections of few tokens on the GEMM (half blocks, one token):
    this shape takes it at each of these counts."""
    from dmoe import synth
    H, V = 1024, 1280
    print(f"case: LM head H={H} V={V} Q8_0 N={N}", flush=True)
    w = synth.host_head(H, V, 8, 60 + N, O.quantize_rows)
    h = (synth.normal(61 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    head = ctx.head_upload(w)
    lg = ctx.head_forward(head, h, 1e-6, logits=True)[2]
    err = max_rel_err(lg, O.head_forward(w, h, 1e-6)[2])
    print(f"  max rel err {err:.3e}", flush=True)
    assert err <= TOL
    head.free()


@pytest.mark.parametrize("wtype", [12, 14])
@pytest.mark.parametrize("N", [33, 64, 90, 129])
def test_dense_units(ctx, O, wtype, N):
    from dmoe import synth
    H, FF = 1024, 1536          # twelve row groups of h, a down reduction in slices
    print(f"case: dense MLP H={H} n_ff={FF} type={wtype} N={N}", flush=True)
    w = synth.host_dense(H, FF, wtype, 30 + N, O.quantize_rows)
    x = synth.normal(31 + N, synth.S_X, N * H).reshape(N, H)
    layer = ctx.dense_upload(w)
    err = max_rel_err(ctx.forward(layer, x), O.dense_forward(w, x))
    print(f"  max rel err {err:.3e}", flush=True)
    assert err <= TOL
    layer.free()


@pytest.mark.parametrize("H", [512, 1024])
@pytest.mark.parametrize("N", [16, 17, 31, 32])
def test_head_q6k_few_tokens(ctx, O, H, N):
    """Q6_K heads of more than 32,768 rows: the GEMM's units of 32 tokens from
    17 tokens on (one half block more than a whole one, whole blocks), the
    few-token kernel below."""
    from dmoe import synth
    V = 33024                   # 129 row groups
    print(f"case: LM head H={H} V={V} Q6_K N={N}", flush=True)
    w = synth.host_head(H, V, 14, 40 + N, O.quantize_rows)
    h = (synth.normal(41 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    head = ctx.head_upload(w)
    lg = ctx.head_forward(head, h, 1e-6, logits=True)[2]
    err = max_rel_err(lg, O.head_forward(w, h, 1e-6)[2])
    print(f"  max rel err {err:.3e}", flush=True)
    assert err <= TOL
    head.free()
