"""GPU parity of Q8_0 projections on the grouped GEMM and on the item kernel:
the attention half (the norm hands the projection its digits with a scale per
32 values, the rotary step and the residual norm add its reduction slices)
and an LM head, at units of 64 tokens begun, in half blocks and whole, one
reduction slice (512 values) and several; DMOE_PROJ_GEMM pins the kernel, the
default is the size rule's.

Bars (max|y - y_oracle| / max|y_oracle|) as for the other Q8_0 projections:
1e-4 for the attention half, 5e-4 for the head's logits."""
import numpy as np
import pytest

from conftest import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["0", "1", ""], ids=["items", "gemm", "rule"])
def pinned(request):
    import os
    import dmoe
    if request.param:
        os.environ["DMOE_PROJ_GEMM"] = request.param
    c = dmoe.Context(0)
    os.environ.pop("DMOE_PROJ_GEMM", None)
    yield c
    c.close()


@pytest.mark.parametrize("H,nh,kv,N", [(512, 4, 4, 1), (512, 4, 4, 33), (512, 4, 4, 100), (1024, 8, 2, 17),
                                       (1024, 8, 2, 64), (1024, 8, 2, 97), (2048, 16, 4, 48)])
def test_attn_q80(pinned, O, H, nh, kv, N):
    from dmoe import synth
    print(f"case: attention half H={H} {nh}/{kv} heads of 128 Q8_0 N={N}", flush=True)
    w = synth.host_attn(8, 30 + N, O.quantize_rows, H, nh, kv, 128, 64, block_length=32)
    layer = pinned.attn_upload(w)
    h = (synth.normal(31 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    y, x = pinned.attn_forward(layer, h)
    yr, xr = O.attn_forward(w, h)
    assert max_rel_err(y, yr) <= 1e-4 and max_rel_err(x, xr) <= 1e-4
    layer.free()


@pytest.mark.parametrize("H,N", [(512, 33), (512, 65), (2048, 16), (2048, 48), (2048, 63), (2048, 128)])
def test_head_q80(pinned, O, H, N):
    from dmoe import synth
    V = 1280
    print(f"case: LM head H={H} V={V} Q8_0 N={N}", flush=True)
    w = synth.host_head(H, V, 8, 20 + N, O.quantize_rows)
    h = (synth.normal(21 + N, synth.S_X, N * H).reshape(N, H) * 2).astype(np.float32)
    head = pinned.head_upload(w)
    assert max_rel_err(pinned.head_forward(head, h, 1e-6, logits=True)[2], O.head_forward(w, h, 1e-6)[2]) <= 5e-4
    head.free()
