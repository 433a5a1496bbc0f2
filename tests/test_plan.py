"""CPU: the choice of kernels for projections, LM heads, dense MLPs and routed
Q4_K experts (csrc/dmoe_plan.h, pure host functions) over every type, the corners of each
kernel's range and the sizes around the 32-bit limits: the workspace is
planned for the tokens that the chosen kernel converts, and the chosen kernel
takes the type and the shape."""
import itertools
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
GEMV, Q4K, Q80, F16, Q6K = range(5)

PROBE = r"""
#include <cstdio>
#include "%s"
using namespace dmoe;
int main() {
  char kind; int path, rows, K, N, force;
  while (scanf(" %%c %%d %%d %%d %%d %%d", &kind, &path, &rows, &K, &N, &force) == 6) {
    KernelSwitches sw;
    sw.proj_gemm = force;
    if (kind == 'm') {      // a routed layer: top_k, experts, moe_ff, tokens, block routing (2: no tile kernels)
      printf("%%d 0 0\n", moe_gemm_pays(N, path, rows, K, true, force & 1, force < 2, 256));
      continue;
    }
    const ProjRoute r = kind == 'p' ? proj_route(sw, path, rows, K, N) : dense_route(sw, path, rows, K, N);
    printf("%%d %%d %%d\n", r.few, r.gemm_ks, r.chunk);
  }
}
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src = d / "probe.cpp"
    src.write_text(PROBE % (ROOT / "diffuse-cpp_amd" / "csrc" / "dmoe_plan.h"))
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(d / "probe"), str(src)], check=True)

    def ask(cases):
        """[(kind, path, rows, K, N, DMOE_PROJ_GEMM or -1)] -> [(few, gemm_ks, chunk)];
        a dense MLP's rows and K are its n_embd and n_ff"""
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "probe")], input=text, capture_output=True, text=True, check=True).stdout
        got = [tuple(map(int, line.split())) for line in out.splitlines()]
        assert len(got) == len(cases)
        return got
    return ask


def _fits(kind, path, rows, K, N, few, ks, chunk):
    """The kernel of the route takes the call, in the chunk that is planned."""
    if few:
        # converted activations: one chunk, reused; only Q6_K runs in several
        ok = path in (Q4K, Q6K) and 0 < chunk <= 32 and rows % 16 == 0 and K % 256 == 0 and ks == 0
        return ok and (chunk == N or path == Q6K)
    if ks:
        # 32-bit offsets into the converted activations (two digit rows a token)
        widest = max(rows, K) if kind == "d" else K
        steps = K // 256 // ks
        return (path in (Q4K, Q6K, Q80) and chunk == N and 2 * N * widest < 2 ** 31 and rows % 256 == 0
                and K % 256 == 0 and K // 256 % ks == 0 and (steps >= 2))
    return path in (Q4K, Q80) and chunk == N        # the item kernels


def test_a_route_fits_what_is_planned(routes):
    rows = [16, 256, 272, 512, 1024, 32768, 33024, 33040, 157184]
    ks = [256, 512, 2816, 4096, 8192, 16640]
    ns = [1, 8, 9, 16, 17, 24, 25, 32, 33, 64, 65, 2048, 64528, 64529, 131071, 131072, 262143, 262144, 300000]
    cases = [("p",) + c for c in itertools.product((Q4K, Q6K, Q80), rows, ks, ns, (-1, 0, 1))]
    cases += [("d",) + c for c in itertools.product((Q4K, Q6K, Q80), (256, 512, 4096, 16640), ks, ns, (-1, 0, 1))]
    for c, r in zip(cases, routes(cases)):
        kind, path, R, K, N, _ = c
        assert _fits(kind, path, R, K, N, *r), (c, r)


@pytest.mark.parametrize("N,K", [(262144, 4096), (131072, 8192), (64529, 16640)])
def test_q6k_head_past_the_gemm_runs_in_chunks(routes, N, K):
    """A Q6_K head of more tokens than the GEMM's 32-bit offsets reach: chunks
    of the few-token kernel, although the GEMM takes such a chunk by itself."""
    assert routes([("p", Q6K, 157184, K, N, -1)]) == [(1, 0, 32)]
    assert routes([("p", Q6K, 157184, K, 2 ** 31 // (2 * K) - 1, -1)])[0][1] > 0


@pytest.mark.parametrize("top_k,E,FF,N,block,gemm", [
    (8, 256, 1024, 1023, 0, 0), (8, 256, 1024, 1024, 1, 1), (8, 256, 1024, 1025, 0, 0), (8, 256, 1024, 1409, 0, 1),
    (8, 256, 512, 992, 1, 0), (8, 256, 512, 1024, 1, 1), (8, 128, 512, 512, 1, 1), (8, 128, 512, 705, 0, 0),
    (2, 16, 1024, 256, 1, 0), (2, 16, 1024, 480, 1, 0), (2, 16, 1024, 512, 1, 1), (4, 32, 512, 384, 1, 0),
    (6, 64, 1024, 352, 1, 1), (6, 64, 1024, 342, 0, 0), (2, 8, 2048, 128, 2, 1), (2, 8, 2048, 112, 2, 0)])
def test_routed_q4k_gemm(routes, top_k, E, FF, N, block, gemm):
    """Between 32 and 64 pairs per expert the grouped GEMM only where it
    measured ahead of the tile kernels: enough items, and with plain top-k
    more pairs per expert."""
    assert routes([("m", top_k, E, FF, N, block)])[0][0] == gemm


@pytest.mark.parametrize("rows,K,N,gemm", [
    (2048, 512, 16, 1), (1536, 512, 32, 0), (2048, 512, 64, 0), (16384, 512, 200, 1), (4096, 1024, 32, 1),
    (4096, 1024, 48, 0),
    (4096, 2048, 64, 1), (4096, 2816, 16, 1), (4096, 2816, 32, 0), (16384, 2816, 64, 0), (16384, 2816, 96, 1),
    (1024, 4096, 1, 1), (4096, 4096, 512, 1), (157184, 4096, 8, 0), (157184, 4096, 9, 1)])
def test_q80_gemm_or_items(routes, rows, K, N, gemm):
    """Q8_0 projections: the GEMM where it measured ahead of the items of 8
    tokens (few rows and short reductions keep those); DMOE_PROJ_GEMM pins it."""
    ask = [("p", Q80, rows, K, N, f) for f in (-1, 0, 1)]
    got = [r[1] > 0 for r in routes(ask)]
    assert got == [bool(gemm), False, True]


@pytest.mark.parametrize("kind,rows,K,N,gemm", [
    # heads of 17 to 24 tokens by the model, from 25 on always
    ("p", 157184, 4096, 16, 0), ("p", 157184, 2048, 17, 0), ("p", 157184, 2048, 24, 0), ("p", 157184, 2048, 25, 1),
    ("p", 65536, 4096, 17, 1), ("p", 100352, 2048, 20, 1), ("p", 81920, 1024, 20, 0), ("p", 33024, 2048, 17, 0),
    # past 32 tokens: an odd number of super-blocks is one slice
    ("p", 1024, 2816, 33, 0), ("p", 1024, 2816, 65, 0), ("p", 1024, 2816, 160, 1), ("p", 16384, 2816, 33, 1),
    ("p", 1024, 4096, 32, 0), ("p", 1024, 4096, 33, 1), ("p", 512, 512, 33, 1),
    # dense MLPs (n_embd, n_ff)
    ("d", 4096, 11008, 33, 0), ("d", 4096, 11008, 200, 1), ("d", 1024, 2816, 64, 0), ("d", 1024, 2816, 200, 1),
    ("d", 4096, 9216, 33, 1), ("d", 512, 1536, 33, 1)])
def test_q6k_gemm_or_chunks(routes, kind, rows, K, N, gemm):
    """Q6_K: the grouped GEMM where it measured ahead of the few-token kernel
    and its chunks of 32 tokens; DMOE_PROJ_GEMM = 0 keeps those."""
    (few, ks, chunk), off = routes([(kind, Q6K, rows, K, N, f) for f in (-1, 0)])
    assert (few, ks > 0, chunk) == ((0, True, N) if gemm else (1, False, min(N, 32)))
    assert off == (1, 0, min(N, 32))


def test_routes_of_the_gpu_tests(routes):
    """What GPU tests say of their shapes: the projection of the rotary step's
    slices, the Q6_K chunks, the Q8_0 heads of few tokens."""
    assert routes([("p", Q4K, 4096, 2048, 1030, -1)]) == [(0, 2, 1030)]
    chunks = [("d", Q6K, 256, 768, 72, -1), ("d", Q6K, 768, 256, 72, -1), ("d", Q6K, 512, 2816, 64, -1)]
    chunks += [("p", Q6K, 1296, 512, 72, -1), ("p", Q6K, 1280, 256, 72, -1), ("p", Q6K, 1024, 2816, 72, -1)]
    assert all(r == (1, 0, 32) for r in routes(chunks))
    gemm = [("p", Q80, 1280, 1024, n, -1) for n in (1, 7, 16, 17, 32)] + [("p", Q6K, 4096, 512, 72, -1)]
    gemm += [("p", Q6K, 33024, K, n, -1) for K in (512, 1024) for n in (17, 31, 32)]
    gemm += [("p", Q6K, 5120, 4096, 96, -1), ("p", Q6K, 4096, 4096, 96, -1)]
    gemm += [("d", Q6K, 1024, 1536, n, -1) for n in (33, 64, 90, 129)]
    gemm += [("p", Q6K, 1280, 512, n, -1) for n in (33, 48, 63, 64, 65, 97, 128)]
    assert all(r[1] > 0 for r in routes(gemm))
