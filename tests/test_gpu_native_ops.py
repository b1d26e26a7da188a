"""The hot ops' native dispatcher kernels (csrc/torch_ops.cpp): what the Python declarations of
the ops promise besides the launches themselves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _linear():
    from minimaxh3_amd.kernels import fp8_linear as fl
    torch.manual_seed(0)
    mod = fl.FP8Linear.from_linear(torch.nn.Linear(64, 32, device="cuda", dtype=torch.bfloat16))
    return mod, torch.randn(5, 64, device="cuda", dtype=torch.bfloat16)


def test_no_derivative():
    """Outputs of inputs that require grad require grad and refuse their backward; with grad
    mode off, or for inputs that do not, nothing is recorded; tangents are dropped."""
    from minimaxh3_amd import ops
    mod, x = _linear()
    xg = x.clone().requires_grad_()
    y = mod(xg)
    assert y.requires_grad and all(t.requires_grad for t in ops.quant_rows(xg))
    with pytest.raises(RuntimeError, match="no autograd formula"):
        y.float().sum().backward()
    with torch.no_grad():
        assert not mod(xg).requires_grad
    assert not mod(x).requires_grad
    with torch.inference_mode():
        assert mod(x).is_inference()
    out, tangent = torch.func.jvp(mod, (x,), (x,))
    assert torch.equal(out, mod(x)) and not tangent.any()


def test_refusals_keep_their_types():
    from minimaxh3_amd import ops
    from minimaxh3_amd._native import NativeError
    mod, x = _linear()
    x8, sa = ops.quant_rows(x)
    with pytest.raises(ValueError, match="expected a GPU tensor"):
        ops.quant_rows(x.cpu())
    with pytest.raises(ValueError, match="unsupported dtype"):
        ops.quant_rows(x.double())
    with pytest.raises(NativeError, match="bad act"):
        ops.gemm_rowwise(x8, mod.w8, sa, mod.w_scale, None, 7, None, None, 0.0)
    with pytest.raises(ValueError, match="w8 must be on"):
        ops.gemm_rowwise(x8, mod.w8.cpu(), sa, mod.w_scale, None, 0, None, None, 0.0)


def test_views_vmap_and_graph_replay_equal_plain_calls():
    from minimaxh3_amd.kernels.fp8_attention import fp8_attention
    mod, x = _linear()
    # a query off a 16-byte boundary takes the two launches
    q = torch.randn(2 * 200 * 128 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(1, 2, 200, 128)
    k = torch.randn(1, 2, 200, 128, device="cuda", dtype=torch.bfloat16)
    ref_a, ref_y = fp8_attention(q.clone(), k, k), mod(x)
    assert torch.equal(fp8_attention(q, k, k), ref_a)
    assert torch.equal(mod(x.t().contiguous().t()), ref_y)  # rows without unit stride
    xs = torch.stack([x, x + 1])
    assert torch.equal(torch.vmap(mod)(xs), torch.stack([mod(t) for t in xs]))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, a = mod(x), fp8_attention(q, k, k)
    for _ in range(3):
        y.zero_(), a.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref_y) and torch.equal(a, ref_a)
        assert torch.equal(mod(x), ref_y)


@pytest.mark.parametrize("r,k,dtype", [(16, 48, torch.bfloat16), (16, 80, torch.bfloat16), (16, 64, torch.float16),
                                       (16, 64, torch.float32), (16, 64, torch.float8_e4m3fn)])
def test_lora_operands_of_other_widths_or_types_are_refused(r, k, dtype):
    """The kernels read x, A, t and B as bf16 and take A's width from x: anything else is refused on the
    host (narrower or smaller operands would be read past their end)."""
    from minimaxh3_amd import ops
    mod, x = _linear()
    x8, sa = ops.quant_rows(x)
    a = torch.zeros((r, k), device="cuda").to(dtype)
    with pytest.raises(ValueError, match="bf16 x"):
        ops.lora_down(x, a)
    if dtype != torch.bfloat16:
        with pytest.raises(ValueError, match="bf16 x"):
            ops.lora_down(x.to(dtype), torch.zeros((r, 64), device="cuda", dtype=torch.bfloat16))
        t, b = (torch.zeros((n, r), device="cuda", dtype=torch.bfloat16) for n in (5, 32))
        for tt, bb in ((t.to(dtype), b), (t, b.to(dtype))):
            with pytest.raises(ValueError, match="LoRA operands"):
                ops.gemm_rowwise(x8, mod.w8, sa, mod.w_scale, None, 0, tt, bb, 1.0)


def test_missing_dimensions_raise_index_errors():
    """As indexing the missing dimension of x does; too many dimensions stay ValueErrors."""
    from minimaxh3_amd import ops
    _, x = _linear()
    a = torch.zeros((16, 64), device="cuda", dtype=torch.bfloat16)
    for call in (ops.quant_rows, lambda t: ops.lora_down(t, a)):
        for bad, err in ((x[0], IndexError), (x[0, 0], IndexError), (x[None], ValueError)):
            with pytest.raises(err):
                call(bad)


def test_both_attention_ops_refuse_the_same_operands():
    """attn_fwd checks its codes and key operands in Python, attn_fwd_q natively: the same calls are
    refused, with the operand's name, and the same accepted."""
    from minimaxh3_amd import ops
    B, H, S, D, Sk = 2, 2, 130, 64, 200
    q, k, v = (torch.randn((B, H, n, D), device="cuda", dtype=torch.bfloat16) for n in (S, Sk, Sk))
    c = ops.softmax_c(None, D)
    q8, sq = ops.attn_quant_q(q, c)
    k8, sk, v8t, sv, _ = ops.attn_quant_kv(k, v)
    mask, bias = torch.ones((B, Sk), device="cuda", dtype=torch.bool), torch.zeros((B, Sk), device="cuda")

    def both(Sk=Sk, mask=None, bias=None, **codes):
        a = {"k8": k8, "v8t": v8t, "sk": sk, "sv": sv, **codes}
        for call in (lambda: ops.attn_fwd(q8, a["k8"], a["v8t"], sq, a["sk"], a["sv"], mask, bias, -1.0, q, Sk),
                     lambda: ops.attn_fwd_q(q, c, a["k8"], a["v8t"], a["sk"], a["sv"], mask, bias, -1.0, Sk)):
            yield call

    for kw, name in [({"Sk": 300}, "k8"), ({"Sk": 100}, "k8"), ({"k8": k8.view(torch.uint8)}, "k8"),
                     ({"k8": k8.transpose(2, 3)}, "k8"), ({"v8t": v8t[..., :128]}, "v8t"), ({"v8t": v8t.cpu()}, "v8t"),
                     ({"sk": sk.double()}, "sk"), ({"sk": sk[:, :1]}, "sk"), ({"sv": sv[..., :32]}, "sv"),
                     ({"sv": sv.half()}, "sv"), ({"mask": mask[:, :7]}, "key_mask"), ({"mask": mask.cpu()}, "key_mask"),
                     ({"bias": bias[:, 1:]}, "key_bias"), ({"bias": bias.cpu()}, "key_bias")]:
        for call in both(**kw):
            with pytest.raises(ValueError, match=name):
                call()
    ref = None
    for kw in ({}, {"mask": mask}, {"mask": mask[0]}, {"mask": mask.float()}, {"bias": bias}, {"bias": bias[:1]},
               {"bias": bias.half()}, {"mask": mask.view(B, 1, 1, Sk)}):
        outs = [call() for call in both(**kw)]
        ref = outs[0] if ref is None else ref
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], ref)


def test_the_fused_layout_is_the_one_the_caller_tests():
    """ops.attn_fwd_q_supported, which the Python caller asks, and the native op agree on q's layouts."""
    from minimaxh3_amd import ops
    B, H, S, D = 1, 2, 40, 64
    k = torch.randn((B, H, S, D), device="cuda", dtype=torch.bfloat16)
    k8, sk, v8t, sv, _ = ops.attn_quant_kv(k, k)
    qs = [k, k.half(), k.float(), k[0], k.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2),
          torch.randn((B, S, H, D), device="cuda").bfloat16().permute(0, 2, 1, 3),
          torch.randn((B, H, S, D + 4), device="cuda").bfloat16()[..., :D],
          torch.randn((B, H, S, D + 8), device="cuda").bfloat16()[..., :D],
          torch.randn((B, H, S, 2 * D), device="cuda").bfloat16()[..., ::2]]
    for q in qs:
        if ops.attn_fwd_q_supported(q):
            assert ops.attn_fwd_q(q, 0.1, k8, v8t, sk, sv, None, None, -1.0, S).shape == q.shape
        else:
            with pytest.raises(ValueError, match="q must be"):
                ops.attn_fwd_q(q, 0.1, k8, v8t, sk, sv, None, None, -1.0, S)
    assert [ops.attn_fwd_q_supported(q) for q in qs] == [True, True, False, False, False, True, False, True, False]


def test_a_key_mean_of_another_size_is_refused():
    """The kernel reads B*H*D values of it: a shorter one would be read past its end."""
    from minimaxh3_amd import ops
    k = torch.randn((2, 3, 40, 64), device="cuda", dtype=torch.bfloat16)
    mean = ops.attn_kmean(k)
    for bad in (mean[:1], mean[..., :32], mean.cpu()):
        with pytest.raises(ValueError, match="mean must"):
            ops.attn_quant_k(k, bad)
    k8, sk = ops.attn_quant_k(k, mean)
    k8f, skf = ops.attn_quant_k(k, mean.view(-1))
    assert torch.equal(k8.view(torch.uint8), k8f.view(torch.uint8)) and torch.equal(sk, skf)
