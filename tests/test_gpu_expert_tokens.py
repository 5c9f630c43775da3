"""Packed experts on the tokens themselves (no permuted copy), and the backward whose GEMM takes the LoRA part of dx along:
against the same block put together from permute, experts and unpermute, and against float64."""
import pytest
import torch

from twinkle_amd import AdapterGroups, LoraConfig, build_segments, flat_keys_from_topk, ops, permute, unpermute
from twinkle_amd.expert_lora import ExpertLoraSlots, experts_forward, moe_experts_block
from twinkle_amd.ops import grouped_experts_linear
from twinkle_amd.segments import build_token_segments

pytestmark = pytest.mark.gpu


class _Experts(torch.nn.Module):

    def __init__(self, gate_up, down):
        super().__init__()
        self.gate_up_proj = torch.nn.Parameter(gate_up, requires_grad=False)
        self.down_proj = torch.nn.Parameter(down, requires_grad=False)
        self.act_fn = torch.nn.functional.silu


def _problem(dev, t, e, k, hidden, inter, ranks, max_r, seed=0):
    g = torch.Generator().manual_seed(seed)
    mod = _Experts((torch.randn(e, 2 * inter, hidden, generator=g) / hidden**0.5).bfloat16().to(dev),
                   (torch.randn(e, hidden, inter, generator=g) / inter**0.5).bfloat16().to(dev))
    slots = [ExpertLoraSlots(e, fin, fout, max_loras=len(ranks), max_r=max_r, dtype=torch.bfloat16, device=dev)
             for fin, fout in ((hidden, 2 * inter), (inter, hidden))]
    names = [f'lora_{j}' if r else None for j, r in enumerate(ranks)]
    params = []
    for s in slots:
        for name, r in zip(names, ranks):
            if name is None:
                continue
            s.configure_slot(name, LoraConfig(r=r, lora_alpha=2 * r))
            for p, std in ((s.lora_A[name], s.in_features**-0.5), (s.lora_B[name], 0.1)):
                with torch.no_grad():
                    p.copy_((torch.randn(p.shape, generator=g) * std).bfloat16())
                params.append(p)
    sel = torch.topk(torch.randn(t, e, generator=g), k).indices.to(dev)
    w = torch.rand(t, k, generator=g).bfloat16().to(dev).requires_grad_(True)
    tenant = torch.randint(0, len(ranks), (t,), generator=g, dtype=torch.int32).to(dev)
    x = torch.randn(t, hidden, generator=g).bfloat16().to(dev).requires_grad_(True)
    dy = torch.randn(t, hidden, generator=g).bfloat16().to(dev)
    return mod, slots, names, params, sel, w, tenant, x, dy


def _exact(mod, slots, names, sel, w, tenant, x, params):
    """float64, expert by expert and tenant by tenant, on merged weights (``params``: the adapters, as ``_problem`` lists them)."""
    live = [name for name in names if name is not None]
    out = torch.zeros_like(x)
    gate_up, down = mod.gate_up_proj.double(), mod.down_proj.double()
    for e in range(gate_up.shape[0]):
        for n, name in enumerate(names):
            hit = ((sel == e) & (tenant == n)[:, None]).nonzero()
            if not len(hit):
                continue
            t, k = hit.unbind(1)
            ws = [gate_up[e], down[e]]
            if name is not None:
                for i, s in enumerate(slots):
                    r, at = s.r[name], 2 * (i * len(live) + live.index(name))
                    ws[i] = ws[i] + s.scaling[name] * params[at + 1][e, :, :r] @ params[at][e, :r]
            gu = x[t] @ ws[0].t()
            gate, up = gu.chunk(2, -1)
            out = out.index_add(0, t, (torch.nn.functional.silu(gate) * up) @ ws[1].t() * w[t, k, None])
    return out


@pytest.mark.parametrize('t,e,k,hidden,inter,ranks,max_r', [
    (1, 4, 2, 128, 128, (8,), 8),                       # one token
    (37, 8, 3, 256, 128, (8, 8), 8),                    # widths that the 256-wide kernel takes in one direction only
    (300, 4, 4, 256, 256, (8, 5, 8), 8),                # rows of every expert, tenants of two and three tiles
    (700, 6, 2, 512, 256, (16, 0, 12), 16),             # a tenant without adapters
    (900, 3, 2, 256, 512, (64, 64), 64),                # a LoRA step per group
    (500, 4, 2, 256, 256, (8, 64), 64),                 # two rank classes: the LoRA part of dx in a pass of its own
    (2000, 2, 1, 256, 256, (32,) * 6, 32),              # several LoRA steps in a row block, top 1
])
def test_block_on_tokens(dev, t, e, k, hidden, inter, ranks, max_r):
    mod, slots, names, params, sel, w, tenant, x, dy = _problem(dev, t, e, k, hidden, inter, ranks, max_r)
    inputs = [x, w, *params]
    out = moe_experts_block(x, sel, w, tenant, mod, names, *slots)
    got = [out.detach(), *torch.autograd.grad(out, inputs, dy)]
    with torch.no_grad():
        assert torch.equal(moe_experts_block(x, sel, w, tenant, mod, names, *slots), got[0])
    # the same block put together from its parts: the same products, so the same bits forward
    nt = len(names)
    seg = build_segments(flat_keys_from_topk(sel, tenant if nt > 1 else None, nt), e * nt, num_tokens=t)
    rows, _ = permute(x, seg)
    ref = unpermute(experts_forward(mod, rows, seg, names, *slots), w, seg)
    assert torch.equal(ref, got[0])
    want = [ref.detach(), *torch.autograd.grad(ref, inputs, dy)]
    exact_in = [v.detach().double().requires_grad_(True) for v in inputs]
    exact_out = _exact(mod, slots, names, sel, exact_in[1], tenant, exact_in[0], exact_in[2:])
    exact = [exact_out, *torch.autograd.grad(exact_out, exact_in, dy.double())]
    for i, (p, q) in enumerate(zip(got, want)):
        # bf16 intermediates, four products in a row; the two paths share the backward's kernels, so that one is not enough
        scale = exact[i].abs().max().item()
        assert (p.double() - exact[i]).abs().max().item() <= 2e-2 * scale, i
        scale = q.double().abs().max().item()
        assert (p.double() - q.double()).abs().max().item() <= 2e-2 * scale, i


def test_strided_tokens_and_frozen_adapters(dev):
    mod, slots, names, params, sel, w, tenant, x, dy = _problem(dev, 200, 4, 2, 256, 256, (8, 8), 8)
    wide = torch.randn(200, 512, device=dev).bfloat16()
    wide[:, :256] = x.detach()
    view = wide[:, :256].requires_grad_(True)
    base = moe_experts_block(x, sel, w, tenant, mod, names, *slots)
    assert torch.equal(moe_experts_block(view, sel, w, tenant, mod, names, *slots), base)
    want, = torch.autograd.grad(base, [x], dy, retain_graph=True)
    for p in params:
        p.requires_grad_(False)
    only_x, = torch.autograd.grad(moe_experts_block(view, sel, w, tenant, mod, names, *slots), [view], dy)
    assert torch.equal(only_x, want)
    fixed, = torch.autograd.grad(moe_experts_block(view, sel, w.detach(), tenant, mod, names, *slots), [view], dy)
    assert torch.equal(fixed, want)              # routing weights that need no gradient
    # rows whose address no 16-byte load takes: the permuted copy
    off = torch.randn(200, 257, device=dev).bfloat16()
    off[:, 1:] = x.detach()
    assert torch.equal(moe_experts_block(off[:, 1:], sel, w, tenant, mod, names, *slots), base)


def test_weights_tables_and_adapters_that_do_not_fit_are_refused(dev):
    """Before anything is launched: with fewer experts than the table names the kernels would read past the weights."""
    e, nt, t, k, n = 4, 2, 60, 128, 256
    bf16 = torch.bfloat16
    sel = torch.randint(0, e, (t, 2), generator=torch.Generator().manual_seed(0)).to(dev)
    tenant = torch.zeros(t, dtype=torch.int32, device=dev)
    keys = flat_keys_from_topk(sel, tenant, nt)
    seg = build_token_segments(keys, e * nt, t)
    x, w = torch.zeros(t, k, dtype=bf16, device=dev), torch.zeros(e, n, k, dtype=bf16, device=dev)

    def adapters(kk=k, nn=n, g=e * nt, dtype=bf16):
        return AdapterGroups([torch.zeros(8, kk, dtype=dtype, device=dev)], [torch.zeros(nn, 8, dtype=dtype, device=dev)], [8] * g,
                             [1.0] * g, a_index=[0] * g, b_index=[0] * g)

    assert grouped_experts_linear(x, w, seg, nt, adapters(), tokens=True).shape == (2 * t, n)
    for args in ((x, w[:2], seg, nt), (x, w, seg, 1), (x, w.transpose(1, 2), seg, nt), (x, w.float(), seg, nt), (x, w[0], seg, nt),
                 (x, w, build_segments(keys, e * nt, num_tokens=t), nt), (x[:-1], w, seg, nt),
                 (x, w, seg, nt, adapters(dtype=torch.float32)), (x, w, seg, nt, adapters(kk=256)),
                 (x, w, seg, nt, adapters(nn=128)), (x, w, seg, nt, adapters(g=e))):
        with pytest.raises(ValueError):
            grouped_experts_linear(*args, tokens=True)
    for args in ((x, w.cpu(), seg, nt), (x.cpu(), w, seg, nt)):
        with pytest.raises(RuntimeError):
            grouped_experts_linear(*args, tokens=True)
    # slots of another type than the experts, through the block itself
    mod = _Experts(torch.zeros(e, 2 * k, k, dtype=bf16, device=dev), torch.zeros(e, k, k, dtype=bf16, device=dev))
    slots = [ExpertLoraSlots(e, k, out, max_loras=1, max_r=8, dtype=torch.float32, device=dev) for out in (2 * k, k)]
    for s in slots:
        s.configure_slot('lora_0', LoraConfig(r=8, lora_alpha=8))
    with pytest.raises(ValueError):
        moe_experts_block(x, sel, torch.ones(t, 2, dtype=bf16, device=dev), None, mod, ['lora_0'], *slots)
    wide = torch.zeros(2 * t, 3, dtype=torch.int32, device=dev)
    wide[:, 1] = keys
    assert torch.equal(build_token_segments(wide[:, 1], e * nt, t).workspace[:32], seg.workspace[:32])
    for bad in ((keys.float(), e * nt, t), (keys, 0, t), (keys, e * nt, 0), (keys, e * nt, t - 1), (keys[:0], e * nt, t)):
        with pytest.raises(ValueError):
            build_token_segments(*bad)
    with pytest.raises(RuntimeError):
        build_token_segments(keys.cpu(), e * nt, t)


def test_a_table_of_tokens_maps_no_rows(dev):
    """Its slots hold tokens: whatever updates rows through them is refused, rows in segment order are as with any table."""
    e, t, k, n = 4, 70, 128, 256
    g = torch.Generator().manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=g).to(dev, torch.bfloat16)  # noqa: E731
    keys = flat_keys_from_topk(torch.randint(0, e, (t, 2), generator=g).to(dev))
    seg, rows = build_token_segments(keys, e, t), build_segments(keys, e, num_tokens=t)
    groups = AdapterGroups([rand(8, k) for _ in range(e)], [rand(n, 8) for _ in range(e)], [8] * e, [1.0] * e)
    x, y, w = rand(2 * t, k), rand(2 * t, n), rand(n, k)
    for w_ in groups.a_tensors:
        w_.requires_grad_(True)
    h = torch.empty(ops.lora_h_bytes(seg, groups), dtype=torch.uint8, device=dev)
    for call in (lambda: ops.multi_lora_delta(x, y.clone(), seg, groups), lambda: ops.multi_lora_linear(x, w, None, seg, groups),
                 lambda: ops.multi_lora_delta_shared(x, [y.clone()], seg, [groups]),
                 lambda: ops.multi_lora_linear_shared(x, [w, w], [None, None], seg, [groups, groups]),
                 lambda: ops.lora_fwd_(x, y.clone(), seg, groups), lambda: ops.lora_shrink_(x, seg, groups, h),
                 lambda: ops.grouped_linear_(x, w.expand(e, n, k).contiguous(), seg, 1, map_rows=True), lambda: permute(x[:t], seg)):
        with pytest.raises(ValueError):
            call()
    got, want = (ops.multi_lora_delta(x, y.clone(), s, groups, map_rows=False) for s in (seg, rows))
    assert torch.equal(got, want)
    assert torch.equal(torch.autograd.grad(got, groups.a_tensors[0], y)[0], torch.autograd.grad(want, groups.a_tensors[0], y)[0])
