"""GPU parity of the per-token top-k among 65 to 256 candidates (k_route):
every ragged call (no block routing: all experts) and block routing that
admits more than 64 experts.  Bit-exact with the oracle, as all routing is."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("probs", "bmax", "thr", "allowed", "idx", "weights", "counts", "offsets", "perm")


def _same(dg, dr):
    assert dg["use_block_routing"] == dr["use_block_routing"]
    for k in KEYS:
        a, b = np.asarray(dg[k]), np.asarray(dr[k])
        assert a.shape == b.shape and np.array_equal(a.view(np.uint8), b.view(np.uint8)), k


# E, top_k, capacity, tokens: one group and several, a last group of one token,
# experts that do not fill the wavefront's four candidates per lane, a
# capacity of more than 64 experts (candidates restricted to the allowed ones)
SHAPES = [(256, 8, 48, 1), (256, 8, 48, 20), (256, 8, 48, 33), (256, 8, 48, 77), (200, 6, 40, 45),
          (65, 32, 16, 17), (256, 8, 100, 32), (256, 8, 100, 96), (256, 32, 200, 64)]


@pytest.mark.parametrize("E,K,cap,N", SHAPES, ids=lambda v: str(v))
@pytest.mark.parametrize("kind", ["normal", "ties", "extremes"])
def test_topk_many_candidates(ctx, O, E, K, cap, N, kind):
    import dmoe
    print(f"case: top-{K} of {E}, capacity {cap}, N={N}, {kind}", flush=True)
    rng = np.random.default_rng(E + N)
    hp = dmoe.hparams_of(4096, E, K, cap, 32)
    logits = (rng.standard_normal((N, E)) * 1.28).astype(np.float32)
    bias = rng.uniform(-0.1, 0.1, E).astype(np.float32)
    if kind == "ties":          # a handful of values: most candidates tie with others
        logits = rng.choice(np.array([-1.0, 0.0, 0.5, 2.0], np.float32), size=(N, E))
        bias = None
    elif kind == "extremes":    # saturated and infinite scores, a bias outside the restricted path's bound
        logits[rng.random((N, E)) < 0.2] = np.float32(np.inf)
        logits[rng.random((N, E)) < 0.2] = np.float32(-np.inf)
        bias[::7] = np.float32(-3e30)
        bias[3::7] = np.float32(-3.4028235e38)
    _same(ctx.route_logits(hp, logits, bias), O.route(hp, logits, bias))
