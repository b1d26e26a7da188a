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
