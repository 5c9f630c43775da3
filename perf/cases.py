"""Performance cases of the multi-LoRA path: what a serving or training program asks of it, from a decode step of a few
rows to a training batch of 32768.

A case is a dict of plain values.  ``prepare`` makes on the GPU what the program holds before the call (activations,
adapters, frozen weights), ``run`` is one pass through the public entry points and ``work`` the bytes and operations the
pass cannot do without.  Kinds:

``infer``   segment table + forward of one projection on the base layer's output, no gradients (serving)
``train``   segment table + forward + backward of one projection through autograd (``multi_lora_delta``: the base layer
            is not a plain ``nn.Linear``, as with quantised weights, or its GEMM is run by the model itself)
``inplace`` the same through ``lora_fwd_`` / ``lora_bwd_`` with kept buffers, dX added onto the base layer's dX
``block``   an attention block's q, k, v, o under ``MultiLora``: mixed batch, forward, backward, optimizer step
``moe``     packed experts from the router's outputs: permute, experts with LoRA, weighted unpermute (and back)
"""
import math

import torch

from twinkle_amd import (AdapterGroups, LoraConfig, MultiLora, MultiTenantAdamW, build_segments, lora_bwd_,
                         lora_bwd_workspace_bytes, lora_fwd_, lora_h_bytes, multi_lora_delta)
from twinkle_amd.expert_lora import ExpertLoraSlots, moe_experts_block

# how the rows of a batch are spread over the adapters: shuffled with Zipf(1.1) shares (independent requests), shuffled
# with uneven shares and two idle adapters, or one contiguous run per adapter (packed sequences)
ORDERS = ('zipf', 'uneven', 'packed')
MIXED = (8, 16, 32, 64)


def _projection(kind, tokens, k, m, adapters, rank, dtype='bf16', order='zipf', mixed=False, weights='same'):
    return {'kind': kind, 'tokens': tokens, 'in': k, 'out': m, 'adapters': adapters, 'rank': rank, 'mixed': mixed,
            'dtype': dtype, 'order': order, 'weights': weights}


def _moe(kind, tokens, experts, top_k, hidden, inter, tenants, rank=8):
    return {'kind': kind, 'tokens': tokens, 'experts': experts, 'top_k': top_k, 'hidden': hidden, 'inter': inter,
            'tenants': tenants, 'rank': rank}


def listed():
    return [
        # one decode step of 32 concurrent requests over 16 tenants: launches and latency count
        dict(_projection('infer', 32, 4096, 4096, 16, 16), name='decode'),
        # prompts of 16 tenants with ranks 8 to 64 packed one after the other, up-projection of an MLP
        dict(_projection('infer', 6000, 4096, 14336, 16, 64, order='packed', mixed=True), name='prefill'),
        # the small plumbing configuration: 512 rows in fp32, 4 adapters of rank 8
        dict(_projection('train', 512, 1024, 1024, 4, 8, dtype='fp32', order='packed'), name='train_small_fp32'),
        # fp32 activations and adapters (lora_compute_dtype=torch.float32: the reference's arithmetic)
        dict(_projection('train', 4096, 4096, 4096, 16, 16, dtype='fp32'), name='train_fp32'),
        # the headline workload: q projection, 16384 tokens, 16 adapters of rank 16, Zipf ids
        dict(_projection('train', 16384, 4096, 4096, 16, 16), name='train_q'),
        # up-projection of an MLP with 24 tenants of ranks 8 to 64, two of them idle
        dict(_projection('train', 32768, 4096, 14336, 24, 64, order='uneven', mixed=True), name='train_up'),
        # eight packed sequences, rank 64, buffers kept by the caller
        dict(_projection('inplace', 32768, 4096, 4096, 8, 64, order='packed'), name='train_packed'),
        # the largest rank the library takes
        dict(_projection('train', 8192, 4096, 4096, 4, 128, order='packed'), name='train_rank128'),
        # widths and a row count that are multiples of nothing the matrix cores like
        dict(_projection('train', 3001, 1000, 1500, 5, 24), name='train_ragged'),
        # one training step of an attention block: three tenants, fp32 adapters under a bf16 base
        {'kind': 'block', 'tokens': 2048, 'hidden': 4096, 'kv': 1024, 'tenants': 3, 'rank': 16, 'weights': 'fp32',
         'name': 'block_step'},
        # mixture of experts, training batch and decode batch
        dict(_moe('moe_train', 8192, 128, 8, 2048, 768, 4), name='moe_train'),
        dict(_moe('moe_infer', 32, 128, 8, 2048, 768, 4), name='moe_decode'),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choices(('infer', 'train', 'inplace', 'block', 'moe_infer', 'moe_train'), (28, 34, 12, 8, 8, 10))[0]
    if kind == 'block':
        return {'kind': kind, 'tokens': _log_int(rng, 16, 4096), 'hidden': rng.choice((1024, 2048, 4096)),
                'kv': rng.choice((512, 1024)), 'tenants': rng.randint(1, 3), 'rank': rng.choice((8, 16, 32, 64)),
                'weights': rng.choice(('fp32', 'fp32', 'same'))}
    if kind.startswith('moe'):
        tokens = _log_int(rng, 4, 256) if kind == 'moe_infer' else _log_int(rng, 256, 8192)
        return _moe(kind, tokens, rng.choice((8, 16, 32, 64, 128)), rng.choice((2, 4, 8)), rng.choice((1024, 2048)),
                    rng.choice((512, 768, 1024)), rng.randint(1, 4), rng.choice((8, 16, 32)))
    dtype = rng.choices(('bf16', 'fp32'), (76, 24))[0]
    tokens = _log_int(rng, 4, 32768)
    if rng.random() < 0.25:   # any width, also odd ones
        k, m = rng.randint(40, 4200), rng.randint(40, 4200)
    else:                     # model widths: hidden, key / value and MLP sizes
        k, m = rng.choice((1024, 1536, 2048, 4096, 14336)), rng.choice((512, 1024, 1536, 2048, 4096, 14336))
    mixed = rng.random() < 0.3
    rank = 64 if mixed else rng.choice((4, 8, 16, 16, 24, 32, 64, 64, 100, 128))
    weights = 'fp32' if dtype == 'bf16' and kind == 'train' and rng.random() < 0.3 else 'same'
    return _projection(kind, tokens, k, m, rng.randint(1, 28), rank, dtype, rng.choice(ORDERS), mixed, weights)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        if _cost(case) <= most:
            return case


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _ranks(case):
    n = case['adapters']
    return [MIXED[i % len(MIXED)] for i in range(n)] if case['mixed'] else [case['rank']] * n


def _row_ids(gen, case):
    """Adapter of every row, int32: see ORDERS."""
    t, n = case['tokens'], case['adapters']
    if case['order'] == 'packed':
        cuts = torch.sort(torch.randint(0, t + 1, (n - 1,), generator=gen)).values
        bounds = torch.cat([torch.zeros(1, dtype=torch.long), cuts, torch.tensor([t])])
        # sequences of about the same length: halfway between random cuts and an even split
        bounds = (bounds + torch.arange(n + 1) * t // n) // 2
        bounds[-1] = t
        return torch.repeat_interleave(torch.arange(n), bounds[1:] - bounds[:-1]).to(torch.int32)
    if case['order'] == 'zipf':
        share = torch.tensor([1.0 / (i + 1)**1.1 for i in range(n)])
    else:
        share = torch.rand(n, generator=gen) + 1e-3
        if n > 8:
            share[5] = share[n - 3] = 0.0
    return torch.multinomial(share, t, replacement=True, generator=gen).to(torch.int32)


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device=gen.device).mul_(std).to(dtype)


def _prepare_projection(case, seed):
    gen, cpu = torch.Generator('cuda').manual_seed(seed), torch.Generator().manual_seed(seed)
    dtype = torch.bfloat16 if case['dtype'] == 'bf16' else torch.float32
    wdtype = torch.float32 if case['weights'] == 'fp32' else dtype
    t, k, m, n, r = case['tokens'], case['in'], case['out'], case['adapters'], case['rank']
    ranks = _ranks(case)
    training = case['kind'] == 'train'
    a = [_randn(gen, r, k, std=1 / math.sqrt(3 * k), dtype=wdtype).requires_grad_(training) for _ in range(n)]
    b = [_randn(gen, m, r, std=0.02, dtype=wdtype).requires_grad_(training) for _ in range(n)]
    state = {'case': case, 'ids': _row_ids(cpu, case).cuda(), 'x': _randn(gen, t, k, dtype=dtype),
             'base': _randn(gen, t, m, std=0.5, dtype=dtype),
             'groups': AdapterGroups([w.detach() for w in a] if not training else a,
                                     [w.detach() for w in b] if not training else b, ranks, [2.0] * n,
                                     act_dtype=dtype), 'a': a, 'b': b}
    if training:
        state['x'].requires_grad_(True)
    if case['kind'] != 'infer':
        state['dy'] = _randn(gen, t, m, dtype=dtype)
    if case['kind'] == 'inplace':
        state['dx'] = _randn(gen, t, k, dtype=dtype)
        state['ga'], state['gb'] = [torch.zeros_like(w) for w in a], [torch.zeros_like(w) for w in b]
        state['pa'], state['pb'] = (torch.tensor([w.data_ptr() for w in g], dtype=torch.int64, device='cuda')
                                    for g in (state['ga'], state['gb']))
        seg = build_segments(state['ids'], n, want_perm=False, want_offsets=False)
        state['h'] = torch.empty(lora_h_bytes(seg, state['groups']), dtype=torch.uint8, device='cuda')
        state['ws'] = torch.empty(lora_bwd_workspace_bytes(seg, state['groups']), dtype=torch.uint8, device='cuda')
    return state


class _Attention(torch.nn.Module):
    """The four projections of an attention block; the attention core carries no adapter and is left out."""

    def __init__(self, hidden, kv):
        super().__init__()
        self.q_proj, self.o_proj = (torch.nn.Linear(hidden, hidden, bias=False) for _ in range(2))
        self.k_proj, self.v_proj = (torch.nn.Linear(hidden, kv, bias=False) for _ in range(2))

    def forward(self, x):
        q, k, v = self.q_proj(x), self.k_proj(x), self.v_proj(x)
        return self.o_proj(q), k, v


def _prepare_block(case, seed):
    gen, cpu = torch.Generator('cuda').manual_seed(seed), torch.Generator().manual_seed(seed)
    bf16, r, n = torch.bfloat16, case['rank'], case['tenants']
    with torch.device('cuda'):
        model = _Attention(case['hidden'], case['kv']).to(bf16)
    ml = MultiLora(max_loras=n + 1, max_r=r)
    model = ml.patch(model, target_modules='all-linear')
    with torch.no_grad():
        for name, p in model.named_parameters():
            if 'lora_' not in name:
                p.requires_grad_(False)
            elif case['weights'] == 'fp32':
                p.data = p.data.float()
            p.normal_(0, 0.02, generator=gen)
    ml.share_inputs([['model.q_proj', 'model.k_proj', 'model.v_proj']])
    names, optimizer = [f'tenant_{i}' for i in range(n)], MultiTenantAdamW()
    params = {}
    for name in names:
        slot = ml.acquire_lora(name, LoraConfig(r=r, lora_alpha=2 * r, target_modules='all-linear'))
        params[name] = [p for key, p in model.named_parameters() if f'.{slot}.' in key]
        optimizer.add_tenant(name, params[name], lr=1e-4)
    t, h, kv = case['tokens'], case['hidden'], case['kv']
    return {'case': case, 'ml': ml, 'model': model, 'names': names, 'optimizer': optimizer, 'params': params,
            'tenant': torch.randint(0, n, (t,), generator=cpu).cuda(), 'x': _randn(gen, t, h, dtype=bf16).requires_grad_(True),
            'dy': [_randn(gen, t, w, dtype=bf16) for w in (h, kv, kv)], 'tokens': {name: t // n + 1 for name in names}}


class _Experts(torch.nn.Module):
    """Packed frozen experts with a SiLU gate, the layout of the transformers library."""

    def __init__(self, gate_up, down):
        super().__init__()
        self.gate_up_proj = torch.nn.Parameter(gate_up, requires_grad=False)
        self.down_proj = torch.nn.Parameter(down, requires_grad=False)
        self.act_fn = torch.nn.functional.silu


def _prepare_moe(case, seed):
    gen = torch.Generator('cuda').manual_seed(seed)
    bf16, t, e, h, i, n = torch.bfloat16, case['tokens'], case['experts'], case['hidden'], case['inter'], case['tenants']
    training = case['kind'] == 'moe_train'
    experts = _Experts(_randn(gen, e, 2 * i, h, std=0.02, dtype=bf16), _randn(gen, e, h, i, std=0.02, dtype=bf16))
    slots = [ExpertLoraSlots(e, fin, fout, max_loras=n, max_r=case['rank'], dtype=bf16, device='cuda')
             for fin, fout in ((h, 2 * i), (i, h))]
    names = [f'lora_{j}' for j in range(n)]
    params = []
    for s in slots:
        for name in names:
            s.configure_slot(name, LoraConfig(r=case['rank'], lora_alpha=2 * case['rank']))
            for p, fan in ((s.lora_A[name], s.in_features), (s.lora_B[name], None)):
                with torch.no_grad():
                    p.normal_(0, 0.02 if fan is None else 1 / math.sqrt(3 * fan), generator=gen)
                params.append(p)
    probs = torch.softmax(_randn(gen, t, e), -1)
    weights, selected = torch.topk(probs, case['top_k'], dim=-1)
    weights = (weights / weights.sum(-1, keepdim=True)).to(bf16)
    return {'case': case, 'experts': experts, 'slots': slots, 'names': names, 'params': params,
            'selected': selected, 'weights': weights.requires_grad_(training),
            'tenant': torch.randint(0, n, (t,), generator=gen, device='cuda', dtype=torch.int32),
            'x': _randn(gen, t, h, dtype=bf16).requires_grad_(training),
            'dy': _randn(gen, t, h, dtype=bf16) if training else None}


def prepare(case, seed):
    if case['kind'] == 'block':
        return _prepare_block(case, seed)
    return (_prepare_moe if case['kind'].startswith('moe') else _prepare_projection)(case, seed)


# ---- one pass ----------------------------------------------------------------------------------------------------------

def _run_block(s):
    with s['ml'].batch(s['names'], s['tenant']):
        ys = s['model'](s['x'])
    s['x'].grad = None
    torch.autograd.backward(ys, s['dy'])
    s['optimizer'].clip_grad_and_step(s['tokens'])
    out = [*ys, s['x'].grad]
    for name in s['names']:
        out += [*s['params'][name], *s['optimizer'].state(name)['exp_avg']]
    return [t.detach() for t in out]


def _run_moe(s):
    args = (s['x'], s['selected'], s['weights'], s['tenant'], s['experts'], s['names'], *s['slots'])
    if s['case']['kind'] == 'moe_infer':
        with torch.no_grad():
            return moe_experts_block(*args)
    out = moe_experts_block(*args)
    return [out.detach(), *torch.autograd.grad(out, [s['x'], s['weights'], *s['params']], s['dy'])]


def run(state):
    s, kind = state, state['case']['kind']
    if kind == 'block':
        return _run_block(s)
    if kind.startswith('moe'):
        return _run_moe(s)
    seg = build_segments(s['ids'], s['case']['adapters'], want_perm=False, want_offsets=False)
    if kind == 'infer':
        with torch.no_grad():
            return multi_lora_delta(s['x'], s['base'], seg, s['groups'])
    if kind == 'train':
        y = multi_lora_delta(s['x'], s['base'].detach(), seg, s['groups'])
        live = [g for g, r in zip(range(len(s['a'])), s['groups'].ranks) if r > 0]
        grads = torch.autograd.grad(y, [s['x']] + [s['a'][g] for g in live] + [s['b'][g] for g in live], s['dy'])
        return [y.detach(), *grads]
    lora_fwd_(s['x'], s['base'], seg, s['groups'], h=s['h'])
    lora_bwd_(s['dy'], s['x'], s['h'], s['dx'], s['pa'], s['pb'], seg, s['groups'], workspace=s['ws'])
    return [s['base'], s['dx'], *s['ga'], *s['gb']]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case):
    """Every input read once and every output written once; operations of the products (a multiply-add is two)."""
    t = case['tokens']
    if case['kind'] == 'block':
        h, kv, n, r = case['hidden'], case['kv'], case['tenants'], case['rank']
        frozen, lora = 2 * h * h + 2 * h * kv, r * (6 * h + 2 * kv)        # elements: weights, adapters of one tenant
        wb = 4 if case['weights'] == 'fp32' else 2
        acts = t * 2 * (2 * h + 2 * (h + 2 * kv))                           # x, dx; y and dy of o, k, v
        return {'bytes': 2 * frozen + acts + n * lora * (2 * wb + 16),      # p and two fp32 moments, read and written
                'flops': 4 * t * frozen + 6 * t * lora}
    if case['kind'].startswith('moe'):
        e, h, i, n, r = case['experts'], case['hidden'], case['inter'], case['tenants'], case['rank']
        rows = t * case['top_k']
        touched = e * (1 - (1 - 1 / e)**rows)
        groups = e * n * (1 - (1 - 1 / (e * n))**rows)
        lora = r * (2 * h + 3 * i)
        train = case['kind'] == 'moe_train'
        size = touched * 3 * h * i + groups * lora + t * h * 2 + rows       # weights, adapters, tokens in and out
        if train:
            size += e * n * lora + t * h * 2 + rows                         # their gradients
        return {'bytes': 2 * size, 'flops': rows * (6 * h * i + 2 * lora) * (1 if not train else 2) +
                (2 * rows * lora if train else 0)}
    k, m, ranks = case['in'], case['out'], _ranks(case)
    elt = 2 if case['dtype'] == 'bf16' else 4
    wb = 4 if case['weights'] == 'fp32' else elt
    live = min(len(ranks), t)
    w = sum(ranks) * (k + m) * live / len(ranks)
    if case['kind'] == 'infer':
        return {'bytes': elt * t * (k + 2 * m) + wb * w, 'flops': 2 * t * (k + m) * sum(ranks) / len(ranks)}
    own = 1 if case['kind'] == 'inplace' else 0                             # dx is an input as well
    return {'bytes': elt * t * ((2 + own) * k + 3 * m) + wb * (w + sum(ranks) * (k + m)),
            'flops': 6 * t * (k + m) * sum(ranks) / len(ranks)}


def _cost(case):
    w = work(case)
    return max(w['bytes'], w['flops'] / 50)


def tolerance(case):
    """About four times the error against 64-bit sums.  fp32: 1e-6 for the gradients.  bf16: results, and the rank-sized
    intermediate before them, are rounded to eight bits once each: 2e-3 (outputs) to 2.4e-3 (gradients).  The block
    and the experts chain several such products: 4e-3 and 5e-3."""
    if case['kind'] == 'block' or case['kind'].startswith('moe'):
        return {'rel': 1.5e-2}
    return {'rel': 1e-5} if case['dtype'] == 'fp32' else {'rel': 1e-2}
