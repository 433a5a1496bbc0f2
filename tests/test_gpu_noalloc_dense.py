"""GPU: a Q6_K dense MLP through the allocation-free forward at token counts
whose grouped-GEMM workspace exceeds the fixed scratch: it is not refused, it
runs in the few-token kernel's chunks of 32 tokens (room for 32 at any
count), bit for bit what a context with that GEMM switched off computes.
Smaller counts take the GEMM as the allocating forward does."""
import numpy as np
import pytest

from conftest import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [40, 16384])
def test_noalloc_dense_q6k(ctx, O, monkeypatch, N):
    import torch
    import dmoe
    from dmoe import synth
    H, FF = 512, 768
    print(f"case: allocation-free forward, dense MLP H={H} n_ff={FF} Q6_K N={N}", flush=True)
    # bytes a token needs on the GEMM: two digit rows of x and h, h in f32
    assert (16384 * (2 * (H + FF) + 4 * FF) > dmoe.NOALLOC_SCRATCH_BYTES)
    w = synth.host_dense(H, FF, 14, 70, O.quantize_rows)
    x = synth.normal(71, synth.S_X, N * H).reshape(N, H)
    xd = torch.from_numpy(x).cuda()
    s = torch.cuda.current_stream().cuda_stream
    if N > 40:
        monkeypatch.setenv("DMOE_PROJ_GEMM", "0")
    other = dmoe.Context(0)
    monkeypatch.delenv("DMOE_PROJ_GEMM", raising=False)
    try:
        out = []
        for c, call in ((ctx, "forward_device_noalloc"), (other, "forward_device")):
            layer = c.dense_upload(w)
            yd = torch.full_like(xd, float("nan"))
            getattr(c, call)(layer, xd, N, yd, s)
            torch.cuda.synchronize()
            out.append(yd.cpu().numpy())
            layer.free()
    finally:
        other.close()
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    pick = np.r_[0:40, N - 40:N]                    # the oracle on the first and last chunks' rows
    assert max_rel_err(out[0][pick], O.dense_forward(w, x[pick])) <= 5e-4
