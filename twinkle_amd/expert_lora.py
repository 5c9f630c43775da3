"""LoRA on packed expert weights (3-D parameters), per (expert, tenant) segment.

The reference keeps, per slot, ``lora_A [E, max_r, in]`` and ``lora_B [E, out, max_r]``
and merges ``W + einsum(B, A) * scaling`` into the expert weights through a
parametrization for the one active tenant
(src/twinkle/model/multi_lora_target_parameters.py:97-114, :158-209); the
per-expert loop then runs on the merged weights
(src/twinkle/model/transformers/moe/expert_parallel.py:347-371).  Here the same
slot tensors are read in place by the segmented kernels: rows are grouped by
``expert * num_tenants + tenant`` and each group adds
``scale * (x A_e^T) B_e^T`` to the expert's output rows, so the ``[E, out, in]``
delta is never materialised and many tenants share one pass.
"""
from __future__ import annotations

import math
from contextlib import contextmanager
from types import MethodType
from typing import Dict, List, Optional, Sequence

import torch
from torch import nn

from .ops import AdapterGroups, multi_lora_delta
from .segments import SegmentTable


# what a tenant's config may not ask of packed-parameter LoRA (the reference refuses the same four,
# multi_lora_target_parameters.py:143-150)
_REFUSED_OPTIONS = (('lora_dropout', 'lora_dropout != 0'), ('fan_in_fan_out', 'fan_in_fan_out=True'),
                    ('use_dora', 'use_dora=True'), ('lora_bias', 'lora_bias=True'))


class ExpertLoraSlots(nn.Module):
    """Slot storage of one packed expert parameter: per slot ``lora_A [E, max_r, in]`` and ``lora_B [E, out, max_r]``
    (the tensors of the reference's ``TargetParameterLoraWrapper``, multi_lora_target_parameters.py:97-114), the
    rank and scaling of the tenant that holds the slot, and the group table the segmented kernels read them by."""

    def __init__(self, num_experts: int, in_features: int, out_features: int, max_loras: int, max_r: int,
                 dtype=torch.float32, device=None, key_prefix: str = ''):
        super().__init__()
        self.num_experts, self.in_features, self.out_features = num_experts, in_features, out_features
        self.max_loras, self.max_r = max_loras, max_r
        self.peft_key_prefix = key_prefix
        self.parameter_key = key_prefix       # name of the packed parameter inside the patched model
        self.out_in_layout = True             # the parameter is stored [E, out, in]
        names = [f'lora_{i}' for i in range(max_loras)]
        self.lora_A = nn.ParameterDict(
            {n: nn.Parameter(torch.empty(num_experts, max_r, in_features, device=device, dtype=dtype)) for n in names})
        self.lora_B = nn.ParameterDict(
            {n: nn.Parameter(torch.zeros(num_experts, out_features, max_r, device=device, dtype=dtype)) for n in names})
        self.r: Dict[str, int] = dict.fromkeys(names, max_r)
        self.scaling: Dict[str, float] = dict.fromkeys(names, 1.0)
        # the first initialisation of every slot's A (kaiming-uniform with a = sqrt(5), reference :119-123), kept on
        # the CPU: a released slot goes back to exactly these values
        self._first_A: Dict[str, torch.Tensor] = {}
        for n in names:
            nn.init.kaiming_uniform_(self.lora_A[n], a=math.sqrt(5))
            self._first_A[n] = self.lora_A[n].detach().to('cpu', copy=True)
        self._groups_cache: Dict[tuple, AdapterGroups] = {}

    def _slot(self, slot_name: str):
        if slot_name not in self.lora_A:
            raise ValueError(f'Unknown target-parameter LoRA slot: {slot_name}')
        return self.lora_A[slot_name], self.lora_B[slot_name]

    def reset_slot(self, slot_name: str) -> None:
        """What releasing a tenant does to its slot: A back to its first values, B to zero (reference :119-134)."""
        a, b = self._slot(slot_name)
        with torch.no_grad():
            a.copy_(self._first_A[slot_name])
            b.zero_()

    def configure_slot(self, slot_name: str, config) -> None:
        """Rank and scaling of the tenant that takes the slot.  ``ValueError`` for an unknown slot, a rank outside
        ``1 .. max_r`` and the options packed-parameter LoRA does not have (reference :136-156)."""
        self._slot(slot_name)
        r = config.r
        if r <= 0:
            raise ValueError(f'`r` should be a positive integer value but the value passed is {r}')
        if r > self.max_r:
            raise ValueError(f'LoRA rank {r} exceeds max_r={self.max_r}')
        for attr, what in _REFUSED_OPTIONS:
            if getattr(config, attr, None):
                raise ValueError(f'target_parameters LoRA does not support {what}')
        self.r[slot_name] = r
        self.scaling[slot_name] = config.lora_alpha / (math.sqrt(r) if getattr(config, 'use_rslora', False) else r)

    def live_blocks(self, slot_name: str):
        """``A[:, :r, :]`` and ``B[:, :, :r]`` of a slot: what its tenant trains and what a checkpoint holds."""
        a, b = self._slot(slot_name)
        r = self.r[slot_name]
        return a[:, :r, :], b[:, :, :r]

    def get_delta_weight(self, slot_name: str, out_in_layout: bool = True) -> torch.Tensor:
        """The merged delta ``B A * scaling`` per expert as the reference forms it (:158-179), ``[E, out, in]`` or
        ``[E, in, out]``.  The kernels never build it; it is there for export and for checks."""
        a, b = self.live_blocks(slot_name)
        delta = torch.bmm(b, a) * self.scaling[slot_name]
        return delta if out_in_layout else delta.transpose(1, 2)

    def _keys(self):
        return f'{self.peft_key_prefix}.lora_A.weight', f'{self.peft_key_prefix}.lora_B.weight'

    def get_state_dict(self, slot_name: str) -> Dict[str, torch.Tensor]:
        return {k: v.detach().clone() for k, v in zip(self._keys(), self.live_blocks(slot_name))}

    def set_state_dict(self, slot_name: str, state_dict: Dict[str, torch.Tensor]) -> set:
        """Load a tenant's ``[:r]`` blocks (the rest of the slot becomes zero); returns the keys it used.  Neither
        key present: nothing to do; one of the two: ``KeyError``; a wrong shape: ``ValueError``."""
        keys = self._keys()
        have = [k in state_dict for k in keys]
        if not any(have):
            return set()
        if not all(have):
            raise KeyError(f'Missing target-parameter LoRA pair for {self.peft_key_prefix}')
        blocks = self.live_blocks(slot_name)
        for side, key, block in zip(('lora_A', 'lora_B'), keys, blocks):
            if tuple(state_dict[key].shape) != tuple(block.shape):
                raise ValueError(f'Expected {side} shape {tuple(block.shape)}, got {tuple(state_dict[key].shape)}')
        with torch.no_grad():
            for full, key, block in zip(self._slot(slot_name), keys, blocks):
                full.zero_()
                block.copy_(state_dict[key].to(device=full.device, dtype=full.dtype))
        return set(keys)

    def groups(self, tenant_slots: Sequence[Optional[str]]) -> AdapterGroups:
        """Group table for keys ``expert * len(tenant_slots) + tenant``: one block of a slot tensor per group.
        A ``None`` entry is a tenant without LoRA on this parameter (its groups have rank 0)."""
        nt = len(tenant_slots)
        live = [s for s in tenant_slots if s is not None]
        if not live:
            raise ValueError('at least one tenant of the batch must hold a slot')
        # building the table costs a few host-to-device copies: kept until a slot's rank or scaling changes (moved
        # parameter storage is picked up by AdapterGroups.refresh at every call)
        key = (tuple(tenant_slots), tuple(self.r[s] for s in live), tuple(self.scaling[s] for s in live))
        hit = self._groups_cache.get(key)
        tensors = [self.lora_A[s] for s in live] + [self.lora_B[s] for s in live]
        if hit is not None and all(x is y for x, y in zip(hit.a_tensors + hit.b_tensors, tensors)):
            return hit
        which = {s: i for i, s in enumerate(live)}
        idx, a_off, b_off, ranks, scales = [], [], [], [], []
        for g in range(self.num_experts * nt):
            e, s = divmod(g, nt)[0], tenant_slots[g % nt]
            idx.append(which.get(s, 0))
            a_off.append(e * self.max_r * self.in_features)
            b_off.append(e * self.out_features * self.max_r)
            ranks.append(self.r[s] if s is not None else 0)
            scales.append(self.scaling[s] if s is not None else 0.0)
        if len(self._groups_cache) > 16:
            self._groups_cache.clear()
        table = AdapterGroups(tensors[:len(live)], tensors[len(live):], ranks, scales, a_index=idx, a_offset=a_off,
                              b_index=idx, b_offset=b_off)
        self._groups_cache[key] = table
        return table


def expert_lora_delta(x_sorted: torch.Tensor, y_sorted: torch.Tensor, seg: SegmentTable, slots: ExpertLoraSlots,
                      tenant_slots: Sequence[str], groups: Optional[AdapterGroups] = None) -> torch.Tensor:
    """Adds every (expert, tenant) group's LoRA term onto the expert outputs, in place and differentiably.

    ``x_sorted`` / ``y_sorted`` are the expert inputs / outputs in segment order (what
    :func:`twinkle_amd.permute` and the per-expert base GEMMs produce); ``seg`` was built from keys
    ``expert * len(tenant_slots) + tenant``.
    """
    if groups is None:
        groups = slots.groups(tenant_slots)
    return multi_lora_delta(x_sorted, y_sorted, seg, groups, map_rows=False)


class _ExpertPass:
    """What the patched expert modules apply while a context of the manager is open."""

    def __init__(self, slots: List[Optional[str]], token_tenant: Optional[torch.Tensor], disabled: bool):
        self.slots = slots                  # slot name per tenant index (None: that tenant has no expert LoRA)
        self.token_tenant = token_tenant    # [tokens] index into slots, or None: slots[0] for every token
        self.disabled = disabled


def _raw_module_path(root: nn.Module, module_name: str) -> str:
    """Path of a submodule inside the model PEFT wraps, whatever ``root`` is: the model itself, the holder that
    :func:`twinkle_amd.lora_layer.inject_adapter` returns (``model.`` in front) or a ``PeftModel``
    (``base_model.model.`` in front)."""
    from .lora_layer import LoraModel
    if isinstance(root, LoraModel):
        lead = 'model'
    elif hasattr(root, 'peft_config') and hasattr(root, 'base_model'):
        lead = 'base_model.model'
    else:
        return module_name
    if module_name == lead:
        return ''
    return module_name[len(lead) + 1:] if module_name.startswith(lead + '.') else module_name


class ExpertLoraManager:
    """Finds packed expert parameters in a model, gives each its slot storage, keeps the tenant -> slot map and
    makes the owning expert modules apply the active tenants' LoRA.

    Host-side counterpart of the reference's ``TargetParameterLoraManager``
    (src/twinkle/model/multi_lora_target_parameters.py:281-383): same method names, arguments and exception types.
    How a slot takes effect differs.  The reference registers a parametrization that merges ``W + B A * scaling``
    into the packed parameter while a tenant is active (:182-209), so the model's own expert forward sees merged
    weights.  Here :meth:`patch` rebinds the forward of every module that owns a patched ``gate_up_proj`` /
    ``down_proj`` pair (the packed-experts layout of transformers: ``forward(hidden_states, top_k_index,
    top_k_weights)``) to :func:`moe_experts_block`, which adds the low-rank term per (expert, tenant) segment:
    under :meth:`adapter` every token uses the one tenant's slot, under :meth:`batch` every token its own
    tenant's, with ``disable_lora`` or outside any context the module's original forward runs untouched.

    The slot tensors have the reference's shapes for both storage layouts.  The segmented kernels apply
    ``scale * (x A^T) B^T``, the reference's merged form for experts that compute ``F.linear(x, W[e])`` on
    ``[E, out, in]`` storage (its expert forward, moe/expert_parallel.py:360-371); a module that stores
    ``[E, in, out]`` keeps its own forward and can merge :meth:`ExpertLoraSlots.get_delta_weight` itself.
    """

    def __init__(self, max_loras: int, max_r: int):
        self.max_loras = max_loras
        self.max_r = max_r
        self.wrappers: List[ExpertLoraSlots] = []
        self.tenant_to_slot: Dict[str, str] = {}
        self.tenant_configs: Dict[str, object] = {}
        self.active_pass: Optional[_ExpertPass] = None
        self._target_parameters: Optional[tuple] = None

    # ---- installing -----------------------------------------------------------------------------------------------
    def patch(self, model: nn.Module, target_parameters) -> None:
        """Attach slot storage to every parameter whose dotted name equals an entry of ``target_parameters`` or ends
        in ``.entry`` (reference :291-319).  A 3-D parameter is ``[E, out, in]``, or ``[E, in, out]`` when its module
        says ``is_transposed``; a 2-D one is ``[out, in]`` with one expert (:47-52).  Patching again with the same
        list is a no-op, with another list a ``ValueError``; so is a list that matches nothing."""
        wanted = tuple(target_parameters)
        if not wanted:
            return
        if self._target_parameters is not None:
            if self._target_parameters != wanted:
                raise ValueError(f'target_parameters already patched as {self._target_parameters}, got {wanted}')
            return
        owners: Dict[str, list] = {}       # module name -> [(module, parameter name, slots)], in discovery order
        for module_name, module in model.named_modules():
            for param_name, parameter in module.named_parameters(recurse=False):
                dotted = f'{module_name}.{param_name}' if module_name else param_name
                if not any(dotted == t or dotted.endswith('.' + t) for t in wanted):
                    continue
                if parameter.ndim == 3:
                    experts, d1, d2 = parameter.shape
                    out_in = not getattr(module, 'is_transposed', False)
                    fout, fin = (d1, d2) if out_in else (d2, d1)
                elif parameter.ndim == 2:
                    experts, out_in = 1, True
                    fout, fin = parameter.shape
                else:
                    raise ValueError(f'target parameter {dotted} has {parameter.ndim} dimensions; only 2D and 3D '
                                     'are supported')
                device = 'cpu' if parameter.device.type == 'meta' else parameter.device
                slots = ExpertLoraSlots(experts, fin, fout, self.max_loras, self.max_r, dtype=parameter.dtype,
                                        device=device)
                slots.parameter_key, slots.out_in_layout = dotted, out_in
                owners.setdefault(module_name, []).append((module, param_name, slots))
        if not owners:
            raise ValueError(f'target_parameters={wanted} were set but no parameter was matched')
        for module_name, found in owners.items():
            # PEFT wraps a module once per target parameter, the first one found innermost: its keys carry one
            # `base_layer` per wrapper outside it (reference :321-330)
            raw = _raw_module_path(model, module_name)
            root = 'base_model.model' + ('.' + raw if raw else '')
            for depth, (module, param_name, slots) in enumerate(found):
                slots.peft_key_prefix = '.'.join([root] + ['base_layer'] * (len(found) - 1 - depth))
                module.add_module(f'_twinkle_lora_{param_name}', slots)
                self.wrappers.append(slots)
            self._bind_forward(found[0][0], {name: slots for _, name, slots in found})
        self._target_parameters = wanted

    def _bind_forward(self, module: nn.Module, by_param: Dict[str, ExpertLoraSlots]) -> None:
        """Route a packed-experts module through :func:`moe_experts_block` while a tenant is active."""
        gate_up, down = by_param.get('gate_up_proj'), by_param.get('down_proj')
        packed = (all(isinstance(getattr(module, n, None), torch.Tensor) and getattr(module, n).ndim == 3
                      for n in ('gate_up_proj', 'down_proj')) and not getattr(module, 'is_transposed', False)
                  and (hasattr(module, 'act_fn') or hasattr(module, '_apply_gate')))
        if not packed or (gate_up is None and down is None):
            return
        manager, original = self, module.forward

        def forward(mod, hidden_states, top_k_index, top_k_weights):
            now = manager.active_pass
            if now is None or now.disabled or all(s is None for s in now.slots):
                return original(hidden_states, top_k_index, top_k_weights)
            if not hidden_states.is_cuda:
                raise RuntimeError('expert LoRA needs the activations on the GPU: this path has no CPU implementation')
            tokens = hidden_states.reshape(-1, hidden_states.shape[-1])
            tenant = now.token_tenant
            if tenant is not None and tenant.numel() != tokens.shape[0]:
                raise ValueError(f'the batch has {tenant.numel()} rows but the experts see {tokens.shape[0]} tokens')
            out = moe_experts_block(tokens, top_k_index.reshape(tokens.shape[0], -1),
                                    top_k_weights.reshape(tokens.shape[0], -1), tenant, mod, now.slots, gate_up, down)
            return out.view(hidden_states.shape)

        module.forward = MethodType(forward, module)
        module._tk_original_forward = original

    # ---- tenants --------------------------------------------------------------------------------------------------
    def acquire(self, tenant_adapter_name: str, slot_name: str, config) -> None:
        if tenant_adapter_name in self.tenant_to_slot:
            raise ValueError(f'Lora {tenant_adapter_name} already exists')
        if getattr(config, 'target_parameters', None) and not self.wrappers:
            raise ValueError('target_parameters LoRA slots must be patched before acquire')
        for slots in self.wrappers:           # all checks pass before anything is recorded
            slots.configure_slot(slot_name, config)
        self.tenant_to_slot[tenant_adapter_name] = slot_name
        self.tenant_configs[tenant_adapter_name] = config

    def release(self, tenant_adapter_name: str) -> None:
        self.tenant_configs.pop(tenant_adapter_name, None)
        slot_name = self.tenant_to_slot.pop(tenant_adapter_name, None)
        if slot_name is not None:
            for slots in self.wrappers:
                slots.reset_slot(slot_name)

    @contextmanager
    def _during(self, expert_pass: _ExpertPass):
        previous, self.active_pass = self.active_pass, expert_pass
        try:
            yield expert_pass
        finally:
            self.active_pass = previous

    def adapter(self, tenant_adapter_name: str, disable_lora: bool = False):
        """One tenant for every token of the calls inside; a tenant without expert LoRA leaves the experts as they
        are, and so does ``disable_lora`` (reference :352-358)."""
        return self._during(_ExpertPass([self.tenant_to_slot.get(tenant_adapter_name)], None, disable_lora))

    def batch(self, tenant_adapter_names: Sequence[str], token_tenant: torch.Tensor):
        """Many tenants in one pass: token ``i`` uses ``tenant_adapter_names[token_tenant[i]]``; an index outside
        the list (``-1`` for padding) gives the token the frozen experts alone.  No counterpart in the reference,
        which activates one tenant per call."""
        slots = [self.tenant_to_slot.get(t) for t in tenant_adapter_names] + [None]
        index = token_tenant.reshape(-1).to(torch.int32)
        index = torch.where((index >= 0) & (index < len(slots) - 1), index, torch.full_like(index, len(slots) - 1))
        return self._during(_ExpertPass(slots, index, False))

    def slots_of(self, tenant_adapter_names: Sequence[str]) -> List[str]:
        """Slot names of the tenants of a mixed batch, in the order their ids appear in the group keys."""
        return [self.tenant_to_slot[t] for t in tenant_adapter_names]

    # ---- parameters and state ---------------------------------------------------------------------------------------
    def named_slot_parameters(self, tenant_adapter_name: str):
        slot_name = self.tenant_to_slot[tenant_adapter_name]
        for slots in self.wrappers:
            for side in ('lora_A', 'lora_B'):
                yield f'{slots.parameter_key}.{side}.{slot_name}.weight', getattr(slots, side)[slot_name]

    def parameters_for_tenant(self, tenant_adapter_name: str) -> List[nn.Parameter]:
        return [p for _, p in self.named_slot_parameters(tenant_adapter_name)]

    def get_state_dict(self, tenant_adapter_name: str) -> Dict[str, torch.Tensor]:
        slot_name = self.tenant_to_slot[tenant_adapter_name]
        return {k: v for slots in self.wrappers for k, v in slots.get_state_dict(slot_name).items()}

    def set_state_dict(self, tenant_adapter_name: str, state_dict: Dict[str, torch.Tensor]) -> set:
        slot_name = self.tenant_to_slot[tenant_adapter_name]
        return set().union(*[slots.set_state_dict(slot_name, state_dict) for slots in self.wrappers])


def _is_silu(fn) -> bool:
    return fn is torch.nn.functional.silu or isinstance(fn, nn.SiLU)


def _gated_activation(experts_mod: nn.Module, gate_up_out: torch.Tensor, fused: bool = True) -> torch.Tensor:
    """``_apply_gate`` if the module has one, else ``act_fn(gate) * up`` (moe/expert_parallel.py:363-366); with
    SiLU on the GPU the one-pass kernel does the same arithmetic in fp32 with one rounding."""
    from .ops import swiglu, swiglu_applies
    if hasattr(experts_mod, '_apply_gate'):
        return experts_mod._apply_gate(gate_up_out)
    if fused and _is_silu(experts_mod.act_fn) and swiglu_applies(gate_up_out):
        return swiglu(gate_up_out)
    gate, up = gate_up_out.chunk(2, dim=-1)
    return experts_mod.act_fn(gate) * up


def grouped_gemm_applies(weight: torch.Tensor, rows: torch.Tensor) -> bool:
    """Frozen bf16 packed weights whose two widths are multiples of 128: what ``tk_grouped_linear`` takes in the
    forward direction (``in`` a multiple of 64, ``out`` of 128) and, with the roles swapped, in the backward one."""
    return (weight.dtype == torch.bfloat16 and rows.dtype == torch.bfloat16 and weight.is_contiguous() and
            not weight.requires_grad and weight.shape[1] % 128 == 0 and weight.shape[2] % 128 == 0)


def experts_forward(experts_mod: nn.Module, rows: torch.Tensor, seg: SegmentTable, tenant_slots: Sequence[str],
                    gate_up_slots: Optional[ExpertLoraSlots] = None,
                    down_slots: Optional[ExpertLoraSlots] = None, grouped: Optional[bool] = None,
                    fused_activation: bool = True) -> torch.Tensor:
    """Packed experts on rows in (expert, tenant) segment order, every tenant's LoRA terms included.

    The per-expert loop of the reference's expert forward (moe/expert_parallel.py:333-378: ``F.linear`` with
    ``gate_up_proj[e]``, gate activation, ``F.linear`` with ``down_proj[e]`` on contiguous chunks), with two
    differences: the chunk boundaries come from the segment table in one device-to-host copy (the reference
    synchronises once per expert, :347-349), and the LoRA terms are added per (expert, tenant) segment by the
    segmented kernels instead of being merged into the weights.  ``seg`` was built from keys
    ``expert * len(tenant_slots) + tenant`` with ``want_offsets=True``; ``experts_mod`` holds
    ``gate_up_proj [E, 2 I, H]`` and ``down_proj [E, H, I]`` and either ``_apply_gate`` or ``act_fn``.

    ``grouped`` (default: whenever the shapes allow, i.e. frozen bf16 weights with widths that are multiples of
    64 / 128 in both directions) replaces the loop by one grouped GEMM per projection with the LoRA terms in its
    epilogue: no host copy of the boundaries at all, one launch instead of one per expert, and the expert outputs
    are written once.  Its backward runs the same kernel in its transposing form on the same weights.
    ``fused_activation`` lets a SiLU gate run as one kernel forward and one backward instead of torch's five.
    """
    if rows.shape[0] == 0:
        return rows                                                   # keeps the autograd edge (reference :340-344)
    nt = len(tenant_slots)
    gate_up, down = experts_mod.gate_up_proj, experts_mod.down_proj
    experts = gate_up.shape[0]
    if seg.num_groups != experts * nt:
        raise ValueError('the segment table must be built from expert * num_tenants + tenant keys')
    input_dtype = rows.dtype
    x = rows if rows.dtype == gate_up.dtype else rows.to(gate_up.dtype)
    can_group = x.is_cuda and grouped_gemm_applies(gate_up, x) and grouped_gemm_applies(down, x)
    if grouped and not can_group:
        raise ValueError('grouped=True needs frozen bf16 expert weights with widths that are multiples of 128')
    if grouped or (grouped is None and can_group):
        from .ops import grouped_experts_linear
        x = x.contiguous()
        gate_up_out = grouped_experts_linear(x, gate_up, seg, nt,
                                             gate_up_slots.groups(tenant_slots) if gate_up_slots is not None else None)
        hidden = _gated_activation(experts_mod, gate_up_out, fused_activation)
        out = grouped_experts_linear(hidden.contiguous(), down, seg, nt,
                                     down_slots.groups(tenant_slots) if down_slots is not None else None)
        return out if out.dtype == input_dtype else out.to(input_dtype)
    if seg.offsets is None:
        raise ValueError('the per-expert loop needs a segment table built with want_offsets=True')
    bounds = seg.offsets[::nt].tolist()                               # first sorted position of every expert

    def per_expert(inp, weight):
        chunks = [torch.nn.functional.linear(inp[bounds[e]:bounds[e + 1]], weight[e]) for e in range(experts)
                  if bounds[e + 1] > bounds[e]]
        # rows whose key named no expert come after the last expert's rows (offsets[num_groups] counts the rows that
        # have a group, not all rows): they get zero rows, so that the result has a row for every row of the input
        tail = inp.shape[0] - bounds[experts]
        if tail > 0 or not chunks:
            chunks.append(inp.new_zeros(max(tail, 0), weight.shape[1]))
        return torch.cat(chunks, dim=0)

    gate_up_out = per_expert(x, gate_up)
    if gate_up_slots is not None:
        gate_up_out = expert_lora_delta(x, gate_up_out, seg, gate_up_slots, tenant_slots)
    hidden = _gated_activation(experts_mod, gate_up_out, fused_activation).contiguous()
    out = per_expert(hidden, down)
    if down_slots is not None:
        out = expert_lora_delta(hidden, out, seg, down_slots, tenant_slots)
    return out if out.dtype == input_dtype else out.to(input_dtype)


def moe_experts_block(hidden_states: torch.Tensor, selected_experts: torch.Tensor, routing_weights: torch.Tensor,
                      tenant: Optional[torch.Tensor], experts_mod: nn.Module, tenant_slots: Sequence[str],
                      gate_up_slots: Optional[ExpertLoraSlots] = None,
                      down_slots: Optional[ExpertLoraSlots] = None) -> torch.Tensor:
    """Routed tokens through the packed experts and back: segment build, permute, :func:`experts_forward`,
    weighted unpermute (the single-rank part of the reference's patched block forward,
    moe/expert_parallel.py:253-255 and moe/ep_utils.py:99-149, :280-287).  ``tenant [T]`` gives every token's
    index into ``tenant_slots`` (``None``: one tenant)."""
    from .segments import build_segments, build_token_segments, flat_keys_from_topk, permute, unpermute
    nt = len(tenant_slots)
    experts = experts_mod.gate_up_proj.shape[0]
    tokens = hidden_states.shape[0]
    keys = flat_keys_from_topk(selected_experts, tenant if nt > 1 else None, nt)
    gate_up, down, x = experts_mod.gate_up_proj, experts_mod.down_proj, hidden_states
    if (x.is_cuda and keys.is_cuda and keys.numel() and grouped_gemm_applies(gate_up, x) and grouped_gemm_applies(down, x) and
            x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0):
        # the first GEMM reads the tokens where they are: their permuted copy would be written once and read three times
        from .ops import grouped_experts_linear
        seg = build_token_segments(keys, experts * nt, tokens)
        gate_up_out = grouped_experts_linear(x, gate_up, seg, nt,
                                             gate_up_slots.groups(tenant_slots) if gate_up_slots is not None else None,
                                             tokens=True)
        hidden = _gated_activation(experts_mod, gate_up_out).contiguous()
        out_rows = grouped_experts_linear(hidden, down, seg, nt,
                                          down_slots.groups(tenant_slots) if down_slots is not None else None)
        return unpermute(out_rows, routing_weights.to(x.dtype), seg)
    seg = build_segments(keys, experts * nt, num_tokens=tokens)
    rows, _ = permute(hidden_states, seg)
    out_rows = experts_forward(experts_mod, rows, seg, tenant_slots, gate_up_slots, down_slots)
    return unpermute(out_rows, routing_weights.to(hidden_states.dtype), seg)
