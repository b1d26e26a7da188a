"""attn_quant_kv where its statistics are folded in the quantizing blocks and where a launch of
its own folds them (kv_split): the separate quantizers' bits either way."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,S,D,dtype", [
    (1, 1, 1, 128, torch.bfloat16), (2, 3, 129, 64, torch.float16), (1, 24, 1024, 128, torch.bfloat16),
    (1, 2, 65536, 128, torch.bfloat16),   # 2048 blocks, 8 per CU: the last with K and V split and folded
    (1, 2, 65537, 128, torch.bfloat16),   # the first with a fold launch and one block for both
    (2, 2, 66000, 64, torch.bfloat16), (4, 24, 1400, 128, torch.float16),   # few keys, more blocks than that
])
def test_fold_in_blocks_or_launch_gives_the_same_bits(B, H, S, D, dtype):
    print(f"kv fold B={B} H={H} S={S} D={D} {dtype}", flush=True)
    from minimaxh3_amd import ops
    g = torch.Generator(device="cuda").manual_seed(S)
    kv = torch.randn((B, S, 2, H, D), device="cuda", generator=g).to(dtype)
    k, v = (kv[:, :, i].permute(0, 2, 1, 3) for i in range(2))
    k8, sk, v8t, sv, mean = ops.attn_quant_kv(k, v)
    mean_s = ops.attn_kmean(k)
    k8_s, sk_s = ops.attn_quant_k(k, mean_s)
    v8t_s, sv_s = ops.attn_quant_v(v)
    for a, b in ((mean, mean_s), (sk, sk_s), (sv, sv_s)):
        assert torch.equal(a, b)
    assert torch.equal(k8.view(torch.uint8), k8_s.view(torch.uint8))
    assert torch.equal(v8t.view(torch.uint8), v8t_s.view(torch.uint8))
