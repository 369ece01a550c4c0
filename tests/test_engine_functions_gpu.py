"""The differentiable entry points on plain tensors run as functions of the C++ engine
(host/ftc_host.cpp); calls that are watched or transformed run the Python functions.  Both give the
same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture()
def cp():
    from fast_transformers_amd import causal_product
    causal_product._host()   # (a process's first call goes through Python)
    return causal_product


def operator(cp, dtype, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.rand(2, 3, 70, w, device="cuda", generator=gen).to(dtype) for w in (64, 64, 32)]


def attention(seed=0, widths=(64, 64, 32), **kw):
    from fast_transformers_amd.attention import CausalLinearAttention
    from fast_transformers_amd.masking import LengthMask, TriangularCausalMask
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lengths = LengthMask(torch.tensor([70, 33], device="cuda"), max_len=70)
    module, mask = CausalLinearAttention(widths[0], **kw), TriangularCausalMask(70, device="cuda")
    inputs = [torch.randn(2, 70, 3, w, device="cuda", generator=gen) for w in widths]
    call = lambda *t: module(*t, mask, lengths, lengths)
    call.lengths = lengths.lengths
    return inputs, call


def in_engine(out):
    return "CppNode" in out.grad_fn.name()


@pytest.mark.parametrize("need", [(1, 1, 1), (1, 0, 0), (0, 1, 1), (0, 0, 0)], ids=str)
@pytest.mark.parametrize("way", ["fp32", "bf16", "attention"])
def test_same_bits_as_the_python_functions(cp, way, need):
    if way == "attention":
        inputs, call = attention()
        nhl = lambda t: t.permute(0, 2, 1, 3)
        lengths = torch.tensor([70, 33], device="cuda")
        python = lambda *t: nhl(cp.CausalLinearAttentionFunction.apply(*map(nhl, t), lengths, 1e-6))
    else:
        inputs, call = operator(cp, {"fp32": torch.float32, "bf16": torch.bfloat16}[way]), cp.causal_dot_product
        python = cp.CausalDotProduct.apply
    results = []
    for f in (call, python):
        t = [x.clone().requires_grad_(bool(n)) for x, n in zip(inputs, need)]
        out = f(*t)
        wanted = [x for x in t if x.requires_grad]
        if wanted:
            assert in_engine(out) == (f is call)
        grads = torch.autograd.grad(out.square().sum(), wanted) if wanted else ()
        results.append((out,) + grads)
        assert out.requires_grad == bool(wanted)
    for a, b in zip(*results):
        assert torch.equal(a, b) and a.dtype == b.dtype and a.stride() == b.stride()


def test_watched_calls_keep_the_python_functions(cp):
    class Mine(torch.Tensor):
        pass
    for inputs, call in ((operator(cp, torch.float32), cp.causal_dot_product), attention()):
        t = [x.clone().requires_grad_(True) for x in inputs]
        assert in_engine(call(*t))
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda x: (seen.append(1), x)[1], lambda x: x):
            out = call(*t)
        assert seen and not in_engine(out)
        assert not in_engine(call(t[0].as_subclass(Mine), *t[1:]).as_subclass(torch.Tensor))
        with pytest.raises(RuntimeError):
            torch.func.vmap(call)(*(x[None] for x in inputs))
    table = cp.CausalDotProduct.dot
    own = table["cuda"]
    table["cuda"] = lambda *a: (seen.append(2), own(*a))[1]
    try:
        cp.causal_dot_product(*operator(cp, torch.float32))
    finally:
        table["cuda"] = own
    assert seen[-1] == 2


def test_python_errors_in_the_engine_reach_the_caller(cp):
    host = cp._host()
    # (a few long chains: segment sums are exchanged through a workspace)
    q, k, v = (torch.rand(1, 2, 4096, 64, device="cuda").requires_grad_(True) for _ in range(3))
    out = cp.causal_dot_product(q, k, v)

    def broken(nbytes, key):
        raise ValueError("no workspace")
    host.setup({}, {}, broken, cp._watch, cp._probe, cp._check_if_possible)
    host.forget_sizes()
    try:
        with pytest.raises(ValueError, match="no workspace"):
            out.sum().backward()
    finally:
        host.setup(cp._workspaces, cp._probes, cp._make_workspace, cp._watch, cp._probe, cp._check_if_possible)
    again = cp.causal_dot_product(q, k, v)
    grads = torch.autograd.grad(again.sum(), (q, k, v))
    assert all(torch.isfinite(g).all() for g in grads)


def attention_at_128():
    inputs, call = attention(widths=(128, 128, 128))
    t = [x.clone().requires_grad_(True) for x in inputs]
    out = call(*t)
    assert in_engine(out)
    return t, call, torch.autograd.grad(out, t, torch.ones_like(out))


def test_lengths_may_change_between_forward_and_backward(cp):
    """... at rows of 128, as in the composition, whose mask is made in the forward."""
    t, call, want = attention_at_128()
    out = call(*t)
    call.lengths.fill_(5)
    for a, b in zip(torch.autograd.grad(out, t, torch.ones_like(out)), want):
        assert torch.equal(a, b)


def test_a_result_at_128_may_be_changed_in_place(cp):
    """... before the backward, as the composition's, which does not keep it."""
    t, call, _ = attention_at_128()
    want = torch.autograd.grad(call(*t) * 3, t, torch.ones_like(t[0]))
    out = call(*t).mul_(3)
    for a, b in zip(torch.autograd.grad(out, t, torch.ones_like(out)), want):
        assert torch.equal(a, b)


def test_inputs_at_128_without_a_gradient_may_change(cp):
    """Queries and keys that need no gradient are not watched for changes: the composition keeps their
    features."""
    (q, k, v), call, want = attention_at_128()
    q, k = q.detach().clone(), k.detach().clone()
    out = call(q, k, v)
    assert in_engine(out)
    q.zero_(), k.zero_()
    assert torch.equal(torch.autograd.grad(out, v, torch.ones_like(out))[0], want[2])


@pytest.mark.parametrize("need", [(1, 1, 1), (0, 1, 0)], ids=str)
def test_first_derivatives_at_128_are_differentiable_as_the_compositions(cp, need):
    """create_graph: the composition's element-wise parts can be differentiated again (its products
    cannot), and a gradient that takes part in them."""
    inputs, call, _ = attention_at_128()
    results = []
    for composed in (False, True):
        t = [x.detach().clone().requires_grad_(bool(n)) for x, n in zip(inputs, need)]
        wanted = [x for x in t if x.requires_grad]
        # (a call with hooks on its saved tensors is composed)
        same = (lambda x: x) if composed else None
        with torch.autograd.graph.saved_tensors_hooks(same, same) if composed else torch.enable_grad():
            out = call(*t)
            assert in_engine(out) != composed
            first = torch.autograd.grad(out.square().sum(), wanted, create_graph=True)
            second = torch.autograd.grad(sum(f.square().sum() for f in first), wanted, allow_unused=True)
        assert [f.requires_grad for f in first] == [x is not t[2] for x in wanted]
        results.append(first + second)
    for a, b in zip(*results):
        if a is None or b is None:
            assert a is b
            continue
        # (both sides fp32, the last operations the same: what the two forwards differ by)
        assert ((a - b).norm() / b.norm()).item() <= 5e-6


def test_an_eps_at_128_that_is_not_a_number(cp):
    """... makes every row one that is not, as in the composition; the fused kernels refuse it."""
    inputs, call = attention(widths=(128, 128, 128), eps=float("nan"))
    assert torch.isnan(call(*inputs)).all()


def test_a_profiler_sees_the_functions_by_name(cp):
    (inputs, call), operands = attention(), operator(cp, torch.float32)
    for f, t, name in ((call, inputs, "CausalLinearAttentionFunction"), (cp.causal_dot_product, operands, "CausalDotProduct")):
        t = [x.clone().requires_grad_(True) for x in t]
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            out = f(*t)
            out.sum().backward()
        names = [event.name for event in prof.events()]
        assert in_engine(out) and names.count(name) == 1 and names.count(name + "Backward") == 1
