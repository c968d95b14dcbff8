"""The low-rank kernels (csrc/gnf4_lora.hip) behind fused_grouped_lora: values
and gradients against the torch composition of the same delta, and the calls
that must keep taking that composition.

Tolerances: the fp32 sums run in another order (contractions of at most 2048
terms: relative error below 2048^0.5 * 2^-24 * a few, asserted at 1e-5); bf16
outputs of sums that close differ only where a rounding flips, by one bf16 step
(2^-8) in a small share of values: 1e-3 relative Frobenius error."""
import pytest
import torch

from _fixtures import rand_nf4_stack, rel_err

pytestmark = pytest.mark.gpu


def _case(sizes, ids, E, K, N, r, seed=0):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    T = sum(sizes)
    W, S = rand_nf4_stack(E, N, K, seed)
    x = rnd(T, K).to("cuda", torch.bfloat16)
    A = (rnd(E, r, K) / K ** 0.5).cuda()
    B = (rnd(E, N, r) * 0.3).cuda()
    go = (rnd(T, N) * 0.1).to("cuda", torch.bfloat16)
    return W, S, x, A, B, go


def _run(kernels, W, S, x, A, B, go, sizes, ids, monkeypatch):
    import nf4_qlora
    if not kernels:
        monkeypatch.setattr(nf4_qlora, "_kernels_take", lambda *a: False)
    x, A, B = (t.detach().clone().requires_grad_(True) for t in (x, A, B))
    out = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B, scaling=2.0)
    grads = torch.autograd.grad(out, (x, A, B), go)
    monkeypatch.undo()
    return [out.detach(), *grads]


@pytest.mark.parametrize("sizes,ids,E,K,N,r", [
    ([5, 0, 17, 33, 1], [3, 1, 0, 2, 4], 6, 64, 64, 4),
    ([16, 15, 31], [2, 0, 1], 3, 192, 72, 16),
    ([40, 3, 20], [1, 1, 0], 3, 2048, 264, 12),          # one expert in two groups
    ([64, 128], [0, 1], 2, 320, 520, 20),
    ([70, 7], [1, 0], 2, 128, 1032, 64),
    ([200] + [1] * 40, list(range(41)), 41, 64, 64, 8),  # far more padding than rows
    ([2] * 130, list(range(130)), 131, 64, 64, 32),      # groups past two lane passes
])
@pytest.mark.parametrize("dev_ids", [False, True])
def test_matches_the_torch_composition(sizes, ids, E, K, N, r, dev_ids, monkeypatch):
    case = _case(sizes, ids, E, K, N, r)
    arg = torch.tensor(ids, device="cuda") if dev_ids else ids
    got = _run(True, *case, sizes, arg, monkeypatch)
    want = _run(False, *case, sizes, ids, monkeypatch)
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert rel_err(a, b.double()) <= (1e-3 if i < 2 else 1e-5), i
    again = _run(True, *case, sizes, arg, monkeypatch)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_route_and_the_calls_that_keep_the_torch_composition(monkeypatch):
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, go = _case(sizes, ids, 2, 128, 64, 8)
    used = []
    orig = nf4_qlora._LoraAdd.apply
    monkeypatch.setattr(nf4_qlora._LoraAdd, "apply", lambda *a: used.append(1) or orig(*a))
    run = lambda **k: nf4_qlora.fused_grouped_lora(  # noqa: E731
        k.get("x", x), W, S, sizes, ids, k.get("A", A), k.get("B", B))
    ref = run()
    assert used == [1]
    torch.testing.assert_close(run(A=A.double().float()), ref)
    assert used == [1, 1]
    # bf16 adapters, strided adapters, autocast, forward mode: the composition
    run(A=A.bfloat16(), B=B.bfloat16())
    strided = A.transpose(1, 2).contiguous().transpose(1, 2)
    assert rel_err(run(A=strided), ref.double()) <= 1e-3
    with torch.autocast("cuda", dtype=torch.bfloat16):
        run()
    with torch.autograd.forward_ad.dual_level():
        d = run(A=torch.autograd.forward_ad.make_dual(A, torch.ones_like(A)))
        assert torch.autograd.forward_ad.unpack_dual(d).tangent is not None
    assert used == [1, 1]


def test_double_backward_and_saved_tensor_hooks(monkeypatch):
    """Gradients of gradients run through the torch composition; what is saved
    goes through saved-tensor hooks."""
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, go = _case(sizes, ids, 2, 128, 64, 8)
    res = []
    for kernels in (True, False):
        if not kernels:
            monkeypatch.setattr(nf4_qlora, "_kernels_take", lambda *a: False)
        a, b = A.clone().requires_grad_(True), B.clone().requires_grad_(True)
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t, lambda t: t):
            out = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, a, b, scaling=2.0)
        assert packed
        ga, = torch.autograd.grad(out, a, go, create_graph=True)
        res.append(torch.autograd.grad(ga.square().sum(), b)[0])
    assert rel_err(res[0], res[1].double()) <= 1e-4


@pytest.mark.parametrize("form,train_x", [
    (f, x) for f in ("broadcast", "padded", "odd_pad", "transposed") for x in (True, False)
] + [("offset", False)])
def test_gradients_of_every_layout(form, train_x, monkeypatch):
    """The incoming gradient in the layouts that autograd and callers produce:
    broadcast over the rows (``out.sum(0)``), rows of a wider buffer with
    aligned and odd strides, a transposed tensor, a dense one at an odd
    offset (the base half's dgrad refuses that one, so the activations are
    not trained there)."""
    import nf4_qlora
    sizes, ids, N = [9, 30, 1], [1, 0, 2], 64
    W, S, x, A, B, go = _case(sizes, ids, 3, 128, N, 8)
    T = sum(sizes)
    if form == "broadcast":
        g = go[0].expand(T, N)
    elif form in ("padded", "odd_pad"):
        g = torch.zeros(T, N + (16 if form == "padded" else 3), dtype=go.dtype, device="cuda")
        g[:, :N] = go
        g = g[:, :N]
    elif form == "transposed":
        g = go.t().contiguous().t()
    else:
        g = torch.empty(T * N + 1, dtype=go.dtype, device="cuda")[1:].view(T, N).copy_(go)
    res = []
    for kernels in (True, False):
        if not kernels:
            monkeypatch.setattr(nf4_qlora, "_kernels_take", lambda *a: False)
        ins = [A.clone().requires_grad_(True), B.clone().requires_grad_(True)]
        xt = x.clone().requires_grad_(train_x)
        out = nf4_qlora.fused_grouped_lora(xt, W, S, sizes, ids, *ins, scaling=2.0)
        res.append(torch.autograd.grad(out, ([xt] if train_x else []) + ins, g))
    for a, b in zip(*res):
        assert rel_err(a, b.double()) <= (1e-3 if a.dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("shape", [(), (64,)])
def test_tensor_scaling_is_multiplied_and_learned(shape):
    """A scaling that is a tensor (a learnable scalar, one factor per output
    column) enters the product and receives its gradient."""
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, go = _case(sizes, ids, 2, 128, 64, 8)
    s = torch.full(shape, 1.5, device="cuda", requires_grad=True)
    out = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B, scaling=s)
    grad, = torch.autograd.grad(out, s, go)
    base = nf4_qlora.gemm_4bit_grouped_train(x, W, S, sizes, ids)
    d = torch.cat([(x[r].float() @ A[e].t()) @ B[e].t()
                   for e, r in ((1, slice(0, 9)), (0, slice(9, 39)))])
    assert rel_err(out, base.double() + 1.5 * d.double()) <= 1e-2   # two bf16 roundings
    assert rel_err(grad, (go.double() * d.double()).sum_to_size(shape)) <= 1e-4
    plain = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B, scaling=1.5)
    assert rel_err(out.detach(), plain.double()) <= 1e-3


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64, None])
@pytest.mark.parametrize("twice", [False, True])
def test_routing_written_over_before_backward(dtype, twice, monkeypatch):
    """A caller may reuse its routing buffers (a device tensor of either width,
    host lists) for the next layer before this one's backward; ``twice``: also
    before a gradient of the gradient."""
    import nf4_qlora
    W, S, x, A, B, go = _case([9, 30, 5], [1, 0, 2], 3, 128, 64, 8)
    res = []
    for kernels in (True, False):
        if not kernels:
            monkeypatch.setattr(nf4_qlora, "_kernels_take", lambda *a: False)
        a, b = A.clone().requires_grad_(True), B.clone().requires_grad_(True)
        sizes, ids = [9, 30, 5], [1, 0, 2]
        if dtype is not None:
            ids = torch.tensor(ids, dtype=dtype, device="cuda")
        out = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, a, b, scaling=2.0)
        if kernels:
            sizes[:], ids[:] = [30, 5, 9], ([2, 2, 0] if dtype is None else 2)
        grads = torch.autograd.grad(out, (a, b), go, create_graph=twice)
        if twice:
            grads = torch.autograd.grad(grads[0].square().sum() + grads[1].square().sum(), (a, b))
        res.append(grads)
    for p, q in zip(*res):
        assert rel_err(p, q.double()) <= (1e-4 if twice else 1e-5)


@pytest.mark.parametrize("train_x", [True, False])
@pytest.mark.parametrize("twice", [False, True])
def test_inputs_updated_in_place_before_backward(train_x, twice):
    """An adapter update or a refilled activation buffer between forward and
    backward changes no gradient and raises nothing."""
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, go = _case(sizes, ids, 2, 128, 64, 8)
    res = []
    for update in (False, True):
        a, b = A.clone().requires_grad_(True), B.clone().requires_grad_(True)
        xt = x.clone().requires_grad_(train_x)
        ins = ([xt] if train_x else []) + [a, b]
        out = nf4_qlora.fused_grouped_lora(xt, W, S, sizes, ids, a, b, scaling=2.0)
        if update:
            with torch.no_grad():
                for t in (xt, a, b):
                    t.mul_(3).add_(1)
        grads = torch.autograd.grad(out, (a, b) if twice else ins, go, create_graph=twice)
        if twice:
            grads = torch.autograd.grad(sum(v.square().sum() for v in grads), (a, b))
        res.append(grads)
    assert all(torch.equal(p, q) for p, q in zip(*res))


def test_no_copies_without_a_graph(monkeypatch):
    """Evaluation with trainable adapters (no_grad) copies nothing."""
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, _ = _case(sizes, ids, 2, 128, 64, 8)
    A.requires_grad_(True)
    want = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B)
    rets = []
    orig = nf4_qlora._LoraAdd.apply
    monkeypatch.setattr(nf4_qlora._LoraAdd, "apply",
                        lambda *a: rets.append(orig(*a)) or rets[-1])
    with torch.no_grad():
        got = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B)
    assert torch.is_tensor(rets[0]) and torch.equal(got, want.detach())


def test_adapters_for_fewer_experts_than_the_stack(monkeypatch):
    """Adapters for the first 2 of 3 experts: ids within them give the delta
    (an empty group's id does not count), a host id past them raises, and
    device ids, which nothing on the host can vouch for, take the torch
    composition and its indexing."""
    import nf4_qlora
    sizes, ids = [9, 0, 30], [1, 2, 0]
    W, S, x, A, B, _ = _case(sizes, ids, 3, 128, 64, 8)
    want = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, A, B)
    used = []
    orig = nf4_qlora._LoraAdd.apply
    monkeypatch.setattr(nf4_qlora._LoraAdd, "apply", lambda *a: used.append(1) or orig(*a))
    run = lambda i: nf4_qlora.fused_grouped_lora(x, W, S, sizes, i, A[:2], B[:2])  # noqa: E731
    assert torch.equal(run(ids), want) and used == [1]
    with pytest.raises(IndexError):
        run([1, 0, 2])
    assert rel_err(run(torch.tensor(ids, device="cuda")), want.double()) <= 1e-3
    assert used == [1]


def test_batched_gradients_of_the_adapters():
    """Several gradients at once (``is_grads_batched``, as vectorised jacobians
    take them): the rows of one gradient at a time."""
    import nf4_qlora
    sizes, ids = [9, 30], [1, 0]
    W, S, x, A, B, go = _case(sizes, ids, 2, 128, 64, 8)
    a, b = A.clone().requires_grad_(True), B.clone().requires_grad_(True)
    out = nf4_qlora.fused_grouped_lora(x, W, S, sizes, ids, a, b, scaling=2.0)
    gs = torch.stack([go, go * 2, go.flip(0)])
    got = torch.autograd.grad(out, (a, b), gs, is_grads_batched=True, retain_graph=True)
    for i, g in enumerate(gs):
        for p, q in zip(got, torch.autograd.grad(out, (a, b), g, retain_graph=True)):
            assert rel_err(p[i], q.double()) <= 1e-5


@pytest.mark.parametrize("sizes,ids,E,K,N,r,split", [
    ([383, 64], [1, 0], 3, 128, 64, 16, False),           # the rule's line
    ([384, 64], [1, 0], 3, 128, 64, 16, True),
    ([384] * 33, list(range(33)), 33, 64, 64, 4, False),  # enough experts to fill the waves
    ([200, 0, 200, 7], [2, 0, 2, 1], 3, 576, 1032, 20, True),   # one expert in two groups
    ([255, 256, 257, 513], [3, 0, 2, 1], 70, 2048, 72, 64, True),
    ([1] * 70 + [769], list(range(71)), 72, 64, 520, 32, True),   # groups past a lane pass
])
@pytest.mark.parametrize("dev_ids", [False, True])
def test_adapter_gradients_of_long_groups(sizes, ids, E, K, N, r, split, dev_ids, monkeypatch):
    """The kernel that splits an expert's rows into 256-row chunks, at the
    chunks' edges and on both sides of the rule that takes it (device ids: by
    the largest group), against float64 (fp32 sums of at most 1000 terms,
    inputs and the two-step products rounded to fp32: 1e-5)."""
    import nf4_qlora
    W, S, x, A, B, go = _case(sizes, ids, E, K, N, r)
    arg = torch.tensor(ids, device="cuda") if dev_ids else ids
    if dev_ids and max(sizes) < 384:
        split = len(ids) > E
    names = []
    orig = nf4_qlora._Launches.__call__
    monkeypatch.setattr(nf4_qlora._Launches, "__call__",
                        lambda self, n, *a: names.append(n) or orig(self, n, *a))
    _out, _gx, gA, gB = _run(True, W, S, x, A, B, go, sizes, arg, monkeypatch)
    assert names.count("gnf4_hip_lora_wgrad_split") == (2 if split else 0)
    assert names.count("gnf4_hip_lora_wgrad") == (0 if split else 2)
    wA, wB, row = torch.zeros_like(A).double(), torch.zeros_like(B).double(), 0
    for m, e in zip(sizes, ids):
        xe, g = x[row:row + m].double(), go[row:row + m].double()
        wA[e] += 2 * (g @ B[e].double()).t() @ xe
        wB[e] += 2 * g.t() @ (xe @ A[e].double().t())
        row += m
    assert rel_err(gA, wA) <= 1e-5 and rel_err(gB, wB) <= 1e-5
    unused = [e for e in range(E) if e not in ids]
    assert not gA[unused].any() and not gB[unused].any()
