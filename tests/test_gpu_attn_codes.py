"""GPU parity of the P codes where their rounding and flush can go wrong.

The kernel makes 8 S + 56 - 8 m near the bottom of the fp32 range, where the flush of codes
below 8 is the hardware's flush of denormal results (attn_codes_tile).  Here Q8 and K8 hold
few small integers and the scales are powers of two, so every score is exact, many lie on
the flush boundary (8 S + 56 - 8 m = 8) and on rounding ties: one code beside its place in a row moves the row by whole steps of the
output.  The bar is assert_attn_model's (the codes are exact; the fp8 products of P V are the
instruction's).  A pair of scales with the same product, far apart, must give the same bits.
"""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle.numerics import bf16_round, e4m3_encode
from tests.helpers import assert_attn_model, to_gpu

pytestmark = pytest.mark.gpu


def _fwd(q, k, v, sq, sk, mask, bias, kv_mode, dtype):
    """ops.attn_fwd and the oracle on integer-valued q, k, v [1, H, S, D] with block scales sq, sk."""
    from minimaxh3_amd import ops
    _, H, Sq, D = q.shape
    Sk = k.shape[2]
    nq, nk = -(-Sq // 128), -(-Sk // 128)
    q8, k8, v8t = e4m3_encode(q), e4m3_encode(k), e4m3_encode(np.ascontiguousarray(v.transpose(0, 1, 3, 2)))
    sqa, ska = np.full((1, H, nq), sq, np.float32), np.full((1, H, nk), sk, np.float32)
    sv = np.full((1, H, D), 0.25, np.float32)
    ref = oa.attn_fwd(q8, k8, v8t, sqa, ska, sv, mask, bias, dot="mfma")
    ref = bf16_round(ref) if dtype == torch.bfloat16 else ref.astype(np.float16).astype(np.float32)

    def e4m3(a, axis, n):
        w = [(0, 0)] * 4
        w[axis] = (0, n - a.shape[axis])
        return to_gpu(np.pad(a, w), torch.uint8).view(torch.float8_e4m3fn)

    out = ops.attn_fwd(e4m3(q8, 2, nq * 128), e4m3(k8, 2, nk * 128), e4m3(v8t, 3, nk * 128),
                       to_gpu(sqa, torch.float32), to_gpu(ska, torch.float32), to_gpu(sv, torch.float32),
                       None if mask is None else to_gpu(mask.astype(np.uint8), torch.bool),
                       None if bias is None else to_gpu(bias, torch.float32), -1.0,
                       torch.empty((1, H, Sq, D), dtype=dtype, device="cuda"), Sk, kv_mode)
    return out.float().cpu().numpy(), ref


@pytest.mark.parametrize("D,Sk,kv_mode,mask,bias,dtype", [
    (128, 500, 0, False, False, torch.bfloat16),   # all K/V in LDS
    (128, 500, 1, True, False, torch.bfloat16),    # K/V tiles streamed
    (64, 1100, 0, False, False, torch.float16),
    (128, 700, 0, False, True, torch.bfloat16),
    (64, 130, 0, True, True, torch.bfloat16),
])
def test_codes_on_the_flush_boundary(D, Sk, kv_mode, mask, bias, dtype):
    print(f"attn codes D={D} Sk={Sk} kv_mode={kv_mode} mask={mask} bias={bias} {dtype}", flush=True)
    rng = np.random.default_rng(D + Sk)
    H, Sq = 2, 200
    q, k = np.zeros((1, H, Sq, D), np.float32), np.zeros((1, H, Sk, D), np.float32)
    q[..., 0] = rng.integers(1, 5, (1, H, Sq))
    q[..., 1] = 1.0
    # scores q0 k0 + k1 in steps of 1/16 after the scales' 2^-4: 8 S in halves, so ties too
    k[..., 0] = rng.integers(-14, 15, (1, H, Sk))
    k[..., 1] = rng.integers(-8, 9, (1, H, Sk))
    v = rng.integers(-8, 9, (1, H, Sk, D)).astype(np.float32)
    km = rng.random((1, Sk)) < 0.7 if mask else None
    kb = (rng.integers(-3, 4, (1, Sk)) / 4.0).astype(np.float32) if bias else None
    out, ref = _fwd(q, k, v, 2.0 ** -2, 2.0 ** -2, km, kb, kv_mode, dtype)
    kind = "bf16" if dtype == torch.bfloat16 else "fp16"
    assert_attn_model(out, ref, kind, -1.0)
    if not bias:  # (with a bias S is formed from dot sq first, whose rounding the scales move)
        for sq, sk in ((2.0 ** -40, 2.0 ** 36), (2.0 ** 50, 2.0 ** -54)):
            far, _ = _fwd(q, k, v, sq, sk, km, kb, kv_mode, dtype)
            np.testing.assert_array_equal(far, out)
    # scores too small to count, down to the quantizers' smallest scales, and large ones: one
    # key (or ties) per row
    for sq, sk in ((2.0 ** -48, 2.0 ** -48), (2.0 ** -8, 2.0 ** -40), (1.0, 8.0)):
        out, ref = _fwd(q, k, v, sq, sk, km, kb, kv_mode, dtype)
        assert_attn_model(out, ref, kind, -1.0)
