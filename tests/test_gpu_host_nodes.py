"""The C++ autograd nodes (csrc/host_torch.cpp) against the Python nodes they stand in for: the same calls of the library, so
the same bits, over the forms both accept; and what only the Python nodes take (transforms, forward mode) keeps going there."""
import pytest
import torch

from twinkle_amd import AdapterGroups, build_segments, multi_lora_delta, ops

pytestmark = pytest.mark.gpu


def _problem(dev, dtype=torch.bfloat16, weights=None, ranks=(8, 16, 0, 5), t=300, k=512, m=384, max_r=16, seed=0, wide=0):
    g = torch.Generator().manual_seed(seed)
    weights = weights or dtype
    a = [(torch.randn(max_r, k, generator=g) / k**0.5).to(dev, weights).requires_grad_(True) for _ in ranks]
    b = [(torch.randn(m, max_r, generator=g) * 0.1).to(dev, weights).requires_grad_(True) for _ in ranks]
    groups = AdapterGroups(a, b, list(ranks), [2.0] * len(ranks), act_dtype=dtype)
    ids = torch.randint(-1, len(ranks), (t,), generator=g, dtype=torch.int32).to(dev)
    x = torch.randn(t, k + wide, generator=g).to(dev, dtype)[:, :k]
    return groups, build_segments(ids, len(ranks)), x, torch.randn(t, m, generator=g).to(dev, dtype), a, b


def _grads(call, inputs, dy):
    y = call()
    return [y.detach().clone(), *torch.autograd.grad(y, inputs, dy, allow_unused=True)]


def _same(got, want):
    for i, (p, q) in enumerate(zip(got, want)):
        assert (p is None) == (q is None), i
        if p is not None:
            assert p.shape == q.shape and p.dtype == q.dtype and torch.equal(p, q), i


@pytest.mark.parametrize('dtype,weights,wide', [(torch.bfloat16, None, 0), (torch.float32, None, 0),
                                                (torch.bfloat16, torch.float32, 0), (torch.bfloat16, None, 24)])
@pytest.mark.parametrize('ranks', [(8, 16, 0, 5), (16, 16, 16), (16, 40, 8)])
@pytest.mark.parametrize('frozen', ['none', 'x', 'b'])
def test_delta_gives_the_bits_of_the_python_node(dev, dtype, weights, wide, ranks, frozen):
    max_r = max(16, max(ranks))
    groups, seg, x, base, a, b = _problem(dev, dtype, weights, ranks, max_r=max_r, wide=wide)
    x.requires_grad_(frozen != 'x')
    for w in b:
        w.requires_grad_(frozen != 'b')
    dy = torch.randn(base.shape, generator=torch.Generator().manual_seed(5)).to(dev, dtype)
    inputs = [v for v in [x, *a, *b] if v.requires_grad]
    got = _grads(lambda: multi_lora_delta(x, base.clone(), seg, groups), inputs, dy)
    want = _grads(lambda: ops._LoraDelta.apply(x, base.clone(), seg, groups, True, *groups.autograd_tensors()), inputs, dy)
    _same(got, want)


@pytest.mark.parametrize('n', [1, 2, 3])
@pytest.mark.parametrize('ranks', [(8, 16, 5), (32, 40, 8)])
@pytest.mark.parametrize('needs', ['x', 'weights', 'bias'])
def test_linear_gives_the_bits_of_the_python_node(dev, n, ranks, needs):
    gen = torch.Generator().manual_seed(n)
    parts = [_problem(dev, ranks=ranks, max_r=64, m=256 * (p + 1), seed=p) for p in range(n)]
    seg, x = parts[0][1], parts[0][2].requires_grad_(needs == 'x')
    groups = [p[0] for p in parts]
    ws = [(torch.randn(256 * (p + 1), 512, generator=gen) / 20).to(dev, torch.bfloat16).requires_grad_(needs == 'weights')
          for p in range(n)]
    bs = [torch.randn(256 * (p + 1), generator=gen).to(dev, torch.bfloat16).requires_grad_(needs == 'bias')
          if p != 1 else None for p in range(n)]
    dys = [torch.randn(x.shape[0], w.shape[0], generator=gen).to(dev, torch.bfloat16) for w in ws]
    inputs = [v for v in [x, *ws, *[b for b in bs if b is not None], *[w for p in parts for w in p[4] + p[5]]]
              if v.requires_grad]

    def run(call):
        ys = call()
        ys = [ys] if isinstance(ys, torch.Tensor) else list(ys)
        return [*[y.detach() for y in ys], *torch.autograd.grad(ys, inputs, dys)]

    if n == 1:
        got = run(lambda: ops.multi_lora_linear(x, ws[0], bs[0], seg, groups[0]))
        want = run(lambda: ops._LoraLinear.apply(x, ws[0], bs[0], seg, groups[0], True, *groups[0].autograd_tensors()))
    else:
        got = run(lambda: ops.multi_lora_linear_shared(x, ws, bs, seg, groups))
        has = tuple(b is not None for b in bs)
        lora = [w for g in groups for w in g.autograd_tensors()]
        want = run(lambda: ops._LoraLinearShared.apply(x, seg, tuple(groups), True, n, has, *ws,
                                                       *[b if b is not None else x.new_zeros(0) for b in bs], *lora))
    _same(got, want)


def test_autograd_bookkeeping(dev):
    groups, seg, x, base, a, b = _problem(dev)
    with torch.no_grad():
        y = base.clone()
        version = y._version
        assert multi_lora_delta(x, y, seg, groups) is y and y._version == version + 1 and not y.requires_grad
    with torch.inference_mode():
        z = base.clone()
        assert torch.equal(multi_lora_delta(x, z, seg, groups), y)
    leaf = base.clone().requires_grad_(True)
    with pytest.raises(RuntimeError):             # a leaf that needs a gradient is not updated in place
        multi_lora_delta(x, leaf, seg, groups)
    packed, x = [], x.requires_grad_(True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        y = multi_lora_delta(x, base.clone(), seg, groups)
    assert len(packed) == 2                       # x and h
    one = torch.autograd.grad(y.float().sum(), [x, a[0]], retain_graph=True)
    _same(torch.autograd.grad(y.float().sum(), [x, a[0]]), one)
    with pytest.raises(RuntimeError):             # the graph is gone
        torch.autograd.grad(y.float().sum(), [x])
    y = multi_lora_delta(x, base.clone(), seg, groups)
    with torch.no_grad():
        x.mul_(2)
    with pytest.raises(RuntimeError, match='modified by an inplace operation'):
        y.float().sum().backward()
    # gradients are tensors of their own: one changed in place leaves the others alone
    ga, gb = torch.autograd.grad(multi_lora_delta(x, base.clone(), seg, groups).float().sum(), [a[0], a[1]])
    kept = gb.clone()
    ga.add_(1)
    assert torch.equal(gb, kept)


def test_parameters_that_move_between_forward_and_backward(dev):
    groups, seg, x, base, a, b = _problem(dev)
    want = _grads(lambda: multi_lora_delta(x, base.clone(), seg, groups), [a[0], a[1], b[3]], base)
    y = multi_lora_delta(x, base.clone(), seg, groups)
    for w in a + b:
        w.data = w.data.clone()
    _same([y.detach(), *torch.autograd.grad(y, [a[0], a[1], b[3]], base)], want)
    _same(_grads(lambda: multi_lora_delta(x, base.clone(), seg, groups), [a[0], a[1], b[3]], base), want)


def test_what_only_the_python_node_takes_goes_there(dev):
    groups, seg, x, base, a, b = _problem(dev)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda v: multi_lora_delta(v, base.clone(), seg, groups))(x[None])
    with torch.autograd.forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        multi_lora_delta(dual, base.clone(), seg, groups)
    with pytest.raises(ValueError):
        multi_lora_delta(x.float(), base.clone(), seg, groups)
    with pytest.raises(ValueError):
        multi_lora_delta(x[:-1], base.clone(), seg, groups)
    with pytest.raises(RuntimeError):
        multi_lora_delta(x.cpu(), base.clone(), seg, groups)


def test_threads(dev):
    """Four threads, each with a stream of its own, on one AdapterGroups object."""
    import threading
    groups, seg, x, base, a, b = _problem(dev)
    want = _grads(lambda: multi_lora_delta(x, base.clone(), seg, groups), [*a, *b][:2], base)
    torch.cuda.synchronize()
    results = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                results[i] = _grads(lambda: multi_lora_delta(x, base.clone(), seg, groups), [*a, *b][:2], base)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for r in results:
        _same(r, want)


@pytest.mark.parametrize('n', [0, 1, 2])     # delta, linear, shared linear
def test_master_weights_take_the_python_node(dev, n):
    """fp32 masters of bf16 compute copies: the gradients are the masters', in their type, and the copies' values but for it."""
    parts = [_problem(dev, ranks=(16, 16, 5), seed=p) for p in range(max(n, 1))]
    seg, x, base = parts[0][1], parts[0][2].requires_grad_(True), parts[0][3]
    dy = torch.randn(base.shape, generator=torch.Generator().manual_seed(5)).to(dev, base.dtype)
    ws = [(torch.randn(384, 512, generator=torch.Generator().manual_seed(p)) / 20).to(dev, base.dtype) for p in range(n)]
    masters = [([w.detach().float().requires_grad_(True) for w in a], [w.detach().float().requires_grad_(True) for w in b])
               for *_, a, b in parts]
    groups = [AdapterGroups([w.detach() for w in p[4]], [w.detach() for w in p[5]], [16, 16, 5], [2.0] * 3, master_a=m[0],
                            master_b=m[1]) for p, m in zip(parts, masters)]

    def call(gs):
        if n == 0:
            return [multi_lora_delta(x, base.clone(), seg, gs[0])]
        if n == 1:
            return [ops.multi_lora_linear(x, ws[0], None, seg, gs[0])]
        return list(ops.multi_lora_linear_shared(x, ws, [None] * n, seg, gs))

    def run(gs, weights):
        ys = call(gs)
        return [*[y.detach() for y in ys], *torch.autograd.grad(ys, [x, *weights], [dy] * len(ys))]

    got = run(groups, [w for m in masters for side in m for w in side])
    want = run([p[0] for p in parts], [w for p in parts for side in p[4:] for w in side])
    k = len(want) - sum(len(p[4]) + len(p[5]) for p in parts)
    _same(got[:k], want[:k])
    for p, q in zip(got[k:], want[k:]):
        assert p.dtype == torch.float32 and torch.equal(p, q.float())


def test_calls_the_library_refuses_raise_the_same_errors(dev):
    """Rows on top of each other pass every check on shapes; the library refuses their stride."""
    groups, seg, x, base, a, b = _problem(dev)
    w = torch.zeros(384, 512, dtype=x.dtype, device=dev)
    flat, out = x[:1].expand(x.shape), base[:1].expand(base.shape)
    calls = [lambda: multi_lora_delta(flat, base.clone(), seg, groups), lambda: multi_lora_delta(x, out, seg, groups),
             lambda: ops.multi_lora_linear(flat, w, None, seg, groups),
             lambda: ops.multi_lora_linear_shared(flat, [w, w], [None, None], seg, [groups, groups]),
             lambda: ops._LoraDelta.apply(flat, base.clone(), seg, groups, True, *groups.autograd_tensors())]
    for call in calls:
        with pytest.raises(ValueError, match='invalid'):
            call()
    with torch.no_grad(), pytest.raises(ValueError, match='invalid'):
        calls[0]()


class _Tagged(torch.Tensor):
    """A subclass of the kind that has a ``__torch_function__`` and no dispatch key."""


@pytest.mark.parametrize('which', ['x', 'weight', 'bias', 'adapters', 'base'])
def test_tensor_subclasses_take_the_python_node(dev, which, monkeypatch):
    groups, seg, x, base, a, b = _problem(dev, ranks=(16, 16, 5))
    made = {'x': x, 'base': base, 'weight': (torch.randn(384, 512, generator=torch.Generator().manual_seed(1)) / 20),
            'bias': torch.zeros(384)}
    made = {k: v.to(dev, torch.bfloat16) for k, v in made.items()}
    if which == 'adapters':
        groups = AdapterGroups([w.detach().as_subclass(_Tagged).requires_grad_(True) for w in a], b, [16, 16, 5], [2.0] * 3)
    else:
        made[which] = made[which].as_subclass(_Tagged)
    x, base, w, bias = made['x'].requires_grad_(True), made['base'], made['weight'], made['bias']
    taken = []
    for name in ('_LoraDelta', '_LoraLinear', '_LoraLinearShared'):
        node = getattr(ops, name)
        monkeypatch.setattr(node, 'apply', lambda *args, node=node, apply=node.apply: taken.append(node) or apply(*args))
    ys = [multi_lora_delta(x, base.clone(), seg, groups), ops.multi_lora_linear(x, w, bias, seg, groups),
          ops.multi_lora_linear_shared(x, [w, w], [bias, None], seg, [groups, groups])[0]]
    want = {'x': (True, True, True), 'base': (True, False, False), 'adapters': (True, True, True)}.get(which, (False, True, True))
    assert [n in taken for n in (ops._LoraDelta, ops._LoraLinear, ops._LoraLinearShared)] == list(want)
    kept = {'x': (1, 2), 'weight': (1, 2), 'bias': (1, 2), 'base': (0,), 'adapters': ()}[which]
    assert [type(y) is _Tagged for y in ys] == [i in kept for i in range(3)]


def test_keys_of_a_subclass(dev):
    keys = torch.arange(40, dtype=torch.int32, device=dev) % 4
    assert torch.equal(build_segments(keys.as_subclass(_Tagged), 4).offsets, build_segments(keys, 4).offsets)


def test_linear_without_autograd_lays_nothing_out(dev):
    groups, seg, x, base, a, b = _problem(dev)
    w = torch.zeros(384, 512, dtype=x.dtype, device=dev)
    with torch.no_grad():
        ops.multi_lora_linear(x, w, None, seg, groups)
        ops.multi_lora_linear_shared(x, [w, w], [None, None], seg, [groups, groups])
    assert groups._host is None
    ops.multi_lora_linear(x, w, None, seg, groups)
    assert groups._host is not None


def test_inference_tensors_are_updated_in_their_mode_only(dev):
    groups, seg, x, base, a, b = _problem(dev)
    with torch.inference_mode():
        y = base.clone()
    for mode in (torch.no_grad, torch.enable_grad):
        with mode(), pytest.raises(RuntimeError, match='Inplace update to inference tensor'):
            multi_lora_delta(x, y, seg, groups)
    with torch.inference_mode():
        assert multi_lora_delta(x, y, seg, groups) is y
