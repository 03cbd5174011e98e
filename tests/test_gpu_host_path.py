"""The native host path against the Python classes it stands in for: same bits, same autograd behaviour."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(kind, q, k, v, e, bm, cls, use_native):
    from flash_mi355 import api
    args = {"plain": (None, None, 0, 0, 0, None), "window": (None, None, 0, 37, 0, None), "doc": (e, e, 1, 0, 0, None),
            "pos": (e, e, 1, 0, 0, torch.arange(q.shape[2], device="cuda", dtype=torch.int32)[None]), "block": (bm, bm, 2, 0, 0, None)}[kind]
    want_lse = cls is api.FlashAttentionWithLse
    if use_native:
        out = api._host().attention(q, k, v, True, None, *args, want_lse)
        assert out is not None, "the native path takes the usual calls"
    else:
        out = cls.apply(q, k, v, True, None, *args)
    return out if want_lse else (out,)


@pytest.mark.parametrize("layout", ["bhld", "blhd"])
@pytest.mark.parametrize("lse", [False, True])
@pytest.mark.parametrize("kind", ["plain", "window", "doc", "pos", "block"])
def test_native_path_gives_the_bits_of_the_python_path(kind, lse, layout):
    from flash_mi355 import api, workloads as W
    B, H, Hk, L, D = 2, 4, 2, 200, 64
    g = torch.Generator().manual_seed(1)
    def t(h):
        x = torch.randn(B, L, h, D, generator=g).bfloat16().cuda()
        return x.transpose(1, 2) if layout == "blhd" else x.transpose(1, 2).contiguous()
    q, k, v, do = t(H), t(Hk), t(Hk), t(H)
    ids = torch.from_numpy(np.stack([W.doc_ids_uniform(np.random.default_rng(2), L, 8, 60, 0.1) for _ in range(B)])).cuda()
    e = ids[:, None].expand(B, H, L)
    bm = (torch.rand(B, 1, 4, 4, generator=g) < 0.5).cuda() | torch.eye(4, dtype=torch.bool, device="cuda")
    cls = api.FlashAttentionWithLse if lse else api.FlashAttention
    w = torch.randn(B, H, L, generator=g).cuda()
    got = []
    for native in (True, False):
        x = [z.detach().requires_grad_(True) for z in (q, k, v)]
        out = _call(kind, *x, e, bm, cls, native)
        grads = torch.autograd.grad(out, x, (do, w)[:len(out)])
        assert all(z.shape == y.shape and z.stride(-1) == 1 for z, y in zip(grads, x))
        got.append([*[z.detach() for z in out], *grads])
    for a, b in zip(*got):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


def test_autograd_behaviour_of_the_native_node():
    from flash_mi355 import attention
    q, k, v = (torch.randn(1, 2, 64, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    with torch.no_grad():
        assert not attention(q, k, v, True).requires_grad
    out = attention(q, k, v, True)
    out.sum().backward(retain_graph=True)          # an expanded gradient (stride 0)
    first = q.grad.clone()
    out.sum().backward()
    assert torch.equal(q.grad, 2 * first)
    with pytest.raises(RuntimeError, match="second time"):
        out.sum().backward()
    out = attention(q, k.detach(), v.detach(), True)   # one operand wants a gradient
    (gq,) = torch.autograd.grad(out.sum(), q)
    assert torch.equal(gq, first)
    out = attention(q, k, v, True)
    with torch.no_grad():
        k.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def test_calls_the_native_path_leaves_to_python():
    """Everything that needs a conversion or an error message comes back as None and then works, or raises, as before."""
    from flash_mi355 import api, attention
    q = torch.randn(1, 2, 70, 64, device="cuda", dtype=torch.bfloat16)
    n = api._host().attention
    none = [(q, q, q, False, None, None, None, 1, 0, 0, None, False), (q.cpu(), q, q, False, None, None, None, 0, 0, 0, None, False),
            (q, q[:, :, :10], q[:, :, :10], True, None, None, None, 0, 0, 0, None, False), (q[:, :, :, ::2],) * 3 + (False, None, None, None, 0, 0, 0, None, False),
            (q, q, q, False, None, None, None, 0, 5, 0, None, False), (q[:, :, :0], q, q, False, None, None, None, 0, 0, 0, None, False)]
    assert all(n(*a) is None for a in none)
    odd = torch.randn(1, 2, 70, 72, device="cuda", dtype=torch.bfloat16)[:, :, :, 3:67]   # base not 16-byte aligned
    assert torch.equal(attention(odd, odd, odd, True), attention(odd.contiguous(), odd.contiguous(), odd.contiguous(), True))
    ids = torch.zeros(1, 2, 70, dtype=torch.int16, device="cuda") - 1
    assert torch.equal(attention(q, q, q, True, None, ids, ids, 1), attention(q, q, q, True, None, ids.int(), ids.int(), 1))


def test_transforms_tracers_and_subclasses_stay_with_python():
    """What passes a C++ function by would be lost there: a tangent, a trace, a subclass, a function transform."""
    import torch.autograd.forward_ad as fwAD
    from flash_mi355 import attention, attention_varlen
    q, k, v = (torch.randn(1, 2, 64, 64, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    cu = torch.tensor([0, 20, 64], device="cuda", dtype=torch.int32)
    packed = [t[0].transpose(0, 1).contiguous() for t in (q, k, v)]
    want = attention(q, k, v, True)
    with fwAD.dual_level(), pytest.raises(RuntimeError, match="jvp|forward"):
        attention(fwAD.make_dual(q, torch.ones_like(q)), k, v, True)
    with fwAD.dual_level(), pytest.raises(RuntimeError, match="jvp|forward"):
        attention_varlen(fwAD.make_dual(packed[0], torch.ones_like(packed[0])), *packed[1:], cu, causal=True)
    for f in (lambda x: torch.func.vmap(lambda y: attention(y[None], k, v, True))(x), lambda x: torch.func.grad(lambda y: attention(y, k, v, True).sum())(x)):
        with pytest.raises(RuntimeError, match="setup_context|functorch"):
            f(q)

    class Sub(torch.Tensor):
        pass
    assert type(attention(q.as_subclass(Sub), k, v, True)) is Sub
    with pytest.raises(AssertionError):   # sizes are tensors there, and the feature size is no longer one of the known ones
        torch.jit.trace(lambda a, b, c: attention(a, b, c, True), (q, k, v), check_trace=False)
    assert torch.equal(attention(torch.nn.Parameter(q), k, v, True).detach(), want)


def test_saved_tensor_hooks_see_what_the_node_keeps():
    from flash_mi355 import attention
    q, k, v = (torch.randn(1, 2, 300, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    want = torch.autograd.grad(attention(q, k, v, True).sum(), (q, k, v))
    with torch.autograd.graph.save_on_cpu():
        out = attention(q, k, v, True)
    got = torch.autograd.grad(out.sum(), (q, k, v))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("native", [True, False])
def test_boundaries_may_be_refilled_before_the_backward(native):
    """One buffer of cumulative lengths for every micro-batch: it is read by the forward, not by the backward."""
    from flash_mi355 import attention_varlen
    scale = 0.125 if native else 2   # (a scale that is no float takes the Python path)
    q, k, v, do = (torch.randn(300, h, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True) for h in (4, 2, 2, 4))
    lens = torch.tensor([[0, 100, 164, 300], [0, 7, 70, 290]], device="cuda", dtype=torch.int32)
    def step(cu_q, cu_k):
        out = attention_varlen(q, k, v, cu_q, cu_k, causal=True, sm_scale=scale)
        assert (out.grad_fn.name() == "FlashAttentionBackward") == native
        return out
    want = [torch.autograd.grad(step(c, c.clone()), (q, k, v), do) for c in lens]
    cu_q, cu_k = lens[0].clone(), lens[0].clone()
    first = step(cu_q, cu_k)
    cu_q.copy_(lens[1]); cu_k.copy_(lens[1])
    second = step(cu_q, cu_k)
    cu_q.zero_(); cu_k.fill_(300)
    got = [torch.autograd.grad(o, (q, k, v), do) for o in (first, second)]
    for a, b in zip(got, want):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("shape", [(1, 1), (2, 1), (1, 4), (2, 4)])
def test_a_block_map_may_be_refilled_before_the_backward(shape):
    """One mask buffer for all layers: each call's backward belongs to the map its forward saw, and a map of any layout
    whose columns lie side by side gives the bits of a dense one."""
    from flash_mi355 import attention
    q, k, v, do = (torch.randn(2, h, 200, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True) for h in (4, 2, 2, 4))
    maps = [(torch.rand(*shape, 4, 4, device="cuda") < 0.5) | torch.eye(4, dtype=torch.bool, device="cuda") for _ in range(2)]
    run = lambda m: attention(q, k, v, True, block_mask=m)
    want = [torch.autograd.grad(run(m), (q, k, v), do) for m in maps]
    wide = torch.zeros(4, *shape, 9, dtype=torch.uint8, device="cuda")
    views = [maps[0].clone(), maps[0].to(torch.uint8) * 7, wide.permute(1, 2, 0, 3)[..., 2:6], wide.permute(1, 2, 0, 3)[..., 3:7]]
    for buf in views:
        buf.copy_(maps[0])
        first = run(buf)
        assert first.grad_fn.name() == "FlashAttentionBackward"
        buf.copy_(maps[1])
        second = run(buf)
        buf.zero_()
        got = [torch.autograd.grad(o, (q, k, v), do) for o in (first, second)]
        for a, b in zip(got, want):
            assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("kind", ["plain", "window", "doc", "pos", "block", "packed"])
def test_saved_tensor_hooks_with_every_mask(kind, native):
    """What the node keeps (operands, ids, the copy of a block map, positions, the plan) may be moved away and come back
    with other strides: ids that all heads share come back head by head."""
    from flash_mi355 import api, workloads as W
    B, H, Hk, L, D = 1, 4, 2, 300, 64
    q, k, v = (torch.randn(B, h, L, D, device="cuda", dtype=torch.bfloat16, requires_grad=True) for h in (H, Hk, Hk))
    ids = torch.from_numpy(W.doc_ids_uniform(np.random.default_rng(3), L, 8, 60, 0.1)).cuda()
    e = ids[None, None].expand(B, H, L)
    bm = (torch.rand(B, 1, 5, 5, device="cuda") < 0.5) | torch.eye(5, dtype=torch.bool, device="cuda")
    cu = torch.tensor([0, 100, 101, 290], device="cuda", dtype=torch.int32)

    def call():
        if kind == "packed":
            return api.attention_varlen(*(t[0].transpose(0, 1) for t in (q, k, v)), cu, causal=True, sm_scale=0.125 if native else 1)
        return _call(kind, q, k, v, e, bm, api.FlashAttentionWithLse, native)[0]
    want = torch.autograd.grad(call().square().sum(), (q, k, v))
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.dtype), t.cpu())[1], lambda t: t.cuda()):
        out = call()
    assert len(seen) >= (6 if kind in ("doc", "pos", "block", "packed") else 5)
    got = torch.autograd.grad(out.square().sum(), (q, k, v))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
