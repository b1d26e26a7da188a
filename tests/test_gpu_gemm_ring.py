"""GPU parity of the GEMM's short-token kernel (one tile per workgroup, K stages in a deep
ring) at the edges of its tiles and of its ring, and the same bits from every tile size that
the dispatch chooses between."""
import numpy as np
import pytest
import torch

from oracle import linear as ol
from oracle.numerics import bf16_round
from tests.helpers import bf16_randn, to_gpu, with_outliers
from tests.test_gemm_tiles import EVERY_TILE

pytestmark = pytest.mark.gpu


def _operands(rng, M, N, K):
    from minimaxh3_amd import ops
    x = with_outliers(rng, bf16_randn(rng, (M, K)))
    w, b = bf16_randn(rng, (N, K), 0.02), bf16_randn(rng, (N,), 0.01)
    return x, w, b, ops.quant_rows(to_gpu(x)), ops.quant_rows(to_gpu(w))


@pytest.mark.parametrize("M,N,K", [
    (1, 40, 16), (33, 72, 272), (65, 136, 144),   # one stage; a stage whose second part is past K; both tails
    (129, 36, 400), (31, 520, 1024),              # rows of 8 bytes (element stores); exactly one ring of stages
    (257, 64, 1040), (64, 1000, 1168),
])
def test_ring_tiles_equal_the_instruction_model(M, N, K):
    """Bit-identical to the oracle with the fp8 instruction's accumulation, as the other tiles."""
    print(f"gemm ring M={M} N={N} K={K}", flush=True)
    from minimaxh3_amd import ops
    rng = np.random.default_rng(M + N + K)
    x, w, b, (x8, sa), (w8, sw) = _operands(rng, M, N, K)
    out = ops.gemm_rowwise(x8, w8, sa, sw.view(1, -1), to_gpu(b), 0, None, None, 0.0).float().cpu().numpy()
    x8c, sac = ol.quantize_rows(x)
    w8c, swc = ol.quantize_rows(w)
    np.testing.assert_array_equal(out, bf16_round(ol.scaled_mm(x8c, w8c, sac, swc, b, dot="mfma")))


@pytest.mark.parametrize("N,K,r,gelu", [
    (3072, 400, 0, False), (3072, 256, 0, True), (3072, 3072, 64, False), (3072, 144, 144, True), (1544, 2048, 128, False),
])
def test_prefixes_have_the_same_bits_on_every_tile(N, K, r, gelu):
    """A row's outputs do not depend on the rows beside it, so prefixes of one x, which take
    the ring's tiles (1 to 1000 rows), 128 x 128 and 256 x 256 ones, give the same bits."""
    from minimaxh3_amd import ops
    rng = np.random.default_rng(N + K + r)
    M = 12000
    _, _, b, (x8, sa), (w8, sw) = _operands(rng, M, N, K)
    bias = to_gpu(b)
    t = B = None
    if r:
        t, B = to_gpu(bf16_randn(rng, (M, r))), to_gpu(bf16_randn(rng, (N, r), 0.05))

    def gemm(m):
        return ops.gemm_rowwise(x8[:m], w8, sa[:m], sw.view(1, -1), bias, int(gelu), None if t is None else t[:m], B,
                                0.75 if r else 0.0).view(torch.int16)

    full = gemm(M)
    for m in (1, 32, 65, 130, 300, 513, 1000, 2048, 3100):
        print(f"gemm prefix {m} N={N} K={K} r={r} gelu={gelu}", flush=True)
        assert torch.equal(gemm(m), full[:m])


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("shape", EVERY_TILE)
def test_every_tile_has_the_same_bits(shape, gelu):
    """Prefixes of one x that take each of the six tiles, with ragged tokens, a K tail and a LoRA staged
    in LDS or read from global memory."""
    from minimaxh3_amd import ops
    N, K, r = shape
    rng = np.random.default_rng(N + K + r)
    M = max(EVERY_TILE[shape])
    _, _, b, (x8, sa), (w8, sw) = _operands(rng, M, N, K)
    bias = to_gpu(b)
    t = B = None
    if r:
        t, B = to_gpu(bf16_randn(rng, (M, r))), to_gpu(bf16_randn(rng, (N, r), 0.05))

    def gemm(m):
        return ops.gemm_rowwise(x8[:m], w8, sa[:m], sw.view(1, -1), bias, int(gelu), None if t is None else t[:m], B,
                                0.75 if r else 0.0).view(torch.int16)

    full = gemm(M)
    for m in EVERY_TILE[shape]:
        print(f"gemm tile {EVERY_TILE[shape].index(m)}: {m} x {N} x {K} r={r} gelu={gelu}", flush=True)
        assert torch.equal(gemm(m), full[:m])


@pytest.mark.parametrize("M", [1000, 1024, 1536])
def test_kv_statistics_of_a_block_do_not_depend_on_the_rows_after_it(M):
    """The key sums of a 128-row block are added in the order of the 128 x 128 tiles below 512
    tiles of 256 x 256, also where the plain product takes one round of those."""
    from minimaxh3_amd import ops
    rng = np.random.default_rng(M)
    C, K = 3072, 1024
    _, _, b, (x8, sa), (w8, sw) = _operands(rng, M, 3 * C, K)

    def stats(m):
        return ops.gemm_rowwise_kv_stats(x8[:m], w8, sa[:m], sw, to_gpu(b), m, C, 2 * C, C)[1]

    print(f"gemm K/V statistics M={M}", flush=True)
    assert torch.equal(stats(M)[:, :1], stats(128))
