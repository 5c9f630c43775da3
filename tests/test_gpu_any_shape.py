"""The kernels for fp32 and for odd shapes (kernels_generic.hip) at the edges of their tiles, against the CPU oracle.

Bars as in test_gpu_lora.py: fp32 1e-5, bf16 2e-2 of the largest value.  fp32: products are exact; the longest sums are
dA and dB over an adapter's rows (about 2400 in the case of 4700 rows) of dh and h, which are themselves sums of at most 1100
terms.  In the worst case that is (2400 + 1100) * 2^-24 = 2e-4 of the sum of magnitudes; rounding errors of either sign add up
to about sqrt(3500) * 2^-24 = 4e-6 of it.
"""
import pytest
import torch

import oracle
from conftest import max_rel_err
from twinkle_amd import AdapterGroups, build_segments, lora_bwd_, lora_fwd_
from test_gpu_lora import TOL, _problem

pytestmark = pytest.mark.gpu


def _strided(t, dtype, dev, pad):
    """`t` as a view one element into rows that are `pad` elements longer: rows start at any element address."""
    wide = torch.zeros(t.shape[0], t.shape[1] + pad, dtype=dtype, device=dev)
    view = wide[:, 1:1 + t.shape[1]] if pad else wide
    view.copy_(t.to(dtype))
    return view


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('t,k,m,ranks,pad', [
    (5, 1, 1, [1, 1], 0),                            # a width inside one piece
    (64, 31, 33, [3, 5, 1], 0),                      # one element short of a step, one past it
    (130, 63, 127, [16, 7], 3),                      # the largest cut piece; rows at odd addresses
    (200, 65, 129, [17, 32], 2),
    (300, 257, 255, [33, 64, 2], 5),                 # four waves of steps and one element
    (300, 512, 256, [40, 64], 1),                    # whole widths at odd row starts
    (450, 513, 640, [128, 65, 100], 3),              # several slices of the source, the largest rank
    (1100, 1100, 72, [20, 128, 1, 0, 64], 0),        # ranks of every class in one call, one adapter not live
    (600, 1025, 65, [128, 128], 1),                  # few tiles, fp32 and bf16: three slices of a wide step
    (300, 1281, 64, [20], 1),                        # fp32: more than one slice
    (6100, 641, 33, [128], 0),                       # many tiles: one block walks all slices
    (4700, 72, 1031, [24, 8], 0),                    # groups of several chunks
])
def test_edges(dev, dtype, t, k, m, ranks, pad):
    max_r = max(ranks)
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, len(ranks), max_r, ranks, seed=t + k)
    ids[ids == 1] = 0 if t < 100 else 1              # the smallest ones leave an adapter without rows
    xd, dyd = _strided(x, dtype, dev, pad), _strided(dy, dtype, dev, pad)
    yd, dxd = _strided(base, dtype, dev, pad), _strided(torch.zeros(t, k), dtype, dev, pad)
    ad, bd = [w.to(dtype).to(dev) for w in a], [w.to(dtype).to(dev) for w in b]
    seg = build_segments(ids.to(torch.int32).to(dev), len(ranks), check=True)
    groups = AdapterGroups(ad, bd, ranks, scales)
    h = lora_fwd_(xd, yd, seg, groups)
    ga, gb = [torch.zeros_like(w) for w in ad], [torch.zeros_like(w) for w in bd]
    pa, pb = (torch.tensor([w.data_ptr() for w in g], dtype=torch.int64, device=dev) for g in (ga, gb))
    lora_bwd_(dyd, xd, h, dxd, pa, pb, seg, groups)
    f64 = lambda v: v.to(dtype).double()  # noqa: E731
    yo, dxo, dao, dbo = oracle.multi_lora_linear_grads(f64(x), f64(base), ids, [f64(w) for w in a], [f64(w) for w in b],
                                                        ranks, scales, f64(dy))
    tol = TOL[dtype]
    assert max_rel_err(yd, yo) < tol and max_rel_err(dxd, dxo) < tol
    for g, r in enumerate(ranks):
        if r:
            assert max_rel_err(ga[g], dao[g]) < tol, f'dA[{g}]'
            assert max_rel_err(gb[g], dbo[g]) < tol, f'dB[{g}]'
    for view in (yd, dxd):                            # what lies around the rows is untouched
        if pad:
            wide = view._base
            assert torch.count_nonzero(wide[:, 0]) == 0 and torch.count_nonzero(wide[:, 1 + view.shape[1]:]) == 0


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_an_infinite_row_stays_with_its_adapter(dev, dtype):
    """Row 0 is what the kernels read in place of a padding slot: an infinity in it reaches its own adapter only."""
    x, base, dy, a, b, _, ranks, scales = _problem(100, 40, 24, 3, 8, [8, 3, 5], seed=3)
    ids = torch.arange(100) % 3
    x[0, 5] = float('inf')
    dy[0, 7] = float('inf')
    ad, bd = [w.to(dtype).to(dev) for w in a], [w.to(dtype).to(dev) for w in b]
    seg = build_segments(ids.to(torch.int32).to(dev), 3)
    groups = AdapterGroups(ad, bd, ranks, scales)
    xd, yd, dyd = (v.to(dtype).to(dev) for v in (x, base, dy))
    dxd = torch.zeros_like(xd)
    h = lora_fwd_(xd, yd, seg, groups)
    ga, gb = [torch.zeros_like(w) for w in ad], [torch.zeros_like(w) for w in bd]
    pa, pb = (torch.tensor([w.data_ptr() for w in g], dtype=torch.int64, device=dev) for g in (ga, gb))
    lora_bwd_(dyd, xd, h, dxd, pa, pb, seg, groups)
    assert torch.isfinite(yd[1:]).all() and torch.isfinite(dxd[1:]).all()
    for g in (1, 2):
        assert torch.isfinite(ga[g]).all() and torch.isfinite(gb[g]).all()


@pytest.mark.parametrize('dtype,t,k,m,ranks', [
    (torch.bfloat16, 900, 256, 1024, [16, 3, 0, 9]),        # one pass over dy, flat expand
    (torch.bfloat16, 1500, 384, 640, [64, 20, 0, 33]),      # the expand above rank 16
    (torch.bfloat16, 1500, 384, 640, [64, 8, 0, 20]),       # three rank classes
    (torch.bfloat16, 333, 41, 24, [8, 0, 5, 3]),            # odd shapes
    (torch.float32, 333, 40, 24, [8, 0, 5, 3]),
    (torch.float32, 200, 40, 24, [0, 0, 0, 0]),             # no live adapter at all
])
def test_a_dx_that_is_written_equals_one_that_starts_at_zero(dev, dtype, t, k, m, ranks):
    """tk_lora_bwd_store into a buffer of NaN and tk_lora_bwd onto zeros: the same bits, zeros in the rows of dead
    adapters and of no adapter."""
    from twinkle_amd.ops import _lora_bwd
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, len(ranks), max(max(ranks), 1), ranks, seed=t)
    ids[::7] = -1
    ids[:70] = len(ranks)
    xd, yd, dyd = (v.to(dtype).to(dev) for v in (x, base, dy))
    seg = build_segments(ids.to(torch.int32).to(dev), len(ranks))
    groups = AdapterGroups([w.to(dtype).to(dev) for w in a], [w.to(dtype).to(dev) for w in b], ranks, scales)
    h = lora_fwd_(xd, yd, seg, groups)
    added, written = torch.zeros_like(xd), torch.full_like(xd, float('nan'))
    _lora_bwd('tk_lora_bwd', dyd, xd, h, added, None, None, seg, groups)
    _lora_bwd('tk_lora_bwd_store', dyd, xd, h, written, None, None, seg, groups)
    assert torch.equal(added, written)
    dead = (ids < 0) | (ids >= len(ranks)) | (torch.tensor(ranks + [0])[ids.clamp(0, len(ranks))] == 0)
    assert torch.count_nonzero(written[dead.to(dev)]) == 0


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('k,ranks', [(1, [8, 0]), (41, [8, 0]), (2053, [16, 0, 3]),        # one class: the expand clears
                                     (41, [8, 0, 20]), (2053, [40, 8, 0]), (2048, [0, 0])])  # several, none
def test_rows_of_no_adapter_are_cleared_up_to_their_ends(dev, dtype, k, ranks):
    """The written dx as rows at odd element addresses with three elements between them: zeros in every column of the rows
    of no live adapter (whole and cut pieces of 16 bytes, more than one block of columns) and nothing around them."""
    from twinkle_amd.ops import _lora_bwd
    t, m, n = 130, 24, len(ranks)
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, n, max(max(ranks), 1), ranks, seed=k)
    ids[::3] = -1
    xd, yd, dyd = (v.to(dtype).to(dev) for v in (x, base, dy))
    seg = build_segments(ids.to(torch.int32).to(dev), n)
    groups = AdapterGroups([w.to(dtype).to(dev) for w in a], [w.to(dtype).to(dev) for w in b], ranks, scales)
    h = lora_fwd_(xd, yd, seg, groups)
    added = torch.zeros_like(xd)
    written = _strided(torch.full((t, k), float('nan')), dtype, dev, 3)
    _lora_bwd('tk_lora_bwd', dyd, xd, h, added, None, None, seg, groups)
    _lora_bwd('tk_lora_bwd_store', dyd, xd, h, written, None, None, seg, groups)
    assert torch.equal(added, written)
    dead = (ids < 0) | (torch.tensor(ranks)[ids.clamp(0)] == 0)
    assert torch.count_nonzero(written[dead.to(dev)]) == 0
    assert torch.count_nonzero(written._base[:, 0]) == 0 and torch.count_nonzero(written._base[:, 1 + k:]) == 0


@pytest.mark.parametrize('max_r,ranks', [(8, [8, 8, 8]), (8, [8, 4, 8]), (8, [8, 0, 8]), (24, [24, 24, 24])])
def test_gradients_of_adapters_without_rows_are_zero(dev, max_r, ranks):
    """The gradient arena starts uninitialised where every live block is written: also the block of an adapter that no
    row of the batch uses, and never one past a smaller rank.  The freed block before it holds NaN."""
    from twinkle_amd import multi_lora_delta
    x, base, dy, a, b, _, _, scales = _problem(300, 128, 256, 3, max_r, ranks, seed=8)
    ids = torch.zeros(300, dtype=torch.int32)               # adapter 2 is live and has no row
    ad, bd = ([w.bfloat16().to(dev).requires_grad_(True) for w in ws] for ws in (a, b))
    groups = AdapterGroups(ad, bd, ranks, scales)
    xd, yd = x.bfloat16().to(dev).requires_grad_(True), base.bfloat16().to(dev)
    y = multi_lora_delta(xd, yd, build_segments(ids.to(dev), 3), groups)
    stale = [torch.full((n,), float('nan'), dtype=torch.bfloat16, device=dev)
             for n in (groups.a_arena_elems, groups.b_arena_elems, groups.a_arena_elems + groups.b_arena_elems) * 2]
    del stale
    y.backward(dy.bfloat16().to(dev))
    for g in range(3):
        for w in (ad[g], bd[g]):
            if ranks[g] == 0:
                assert w.grad is None
            else:
                assert torch.isfinite(w.grad).all()
                if g == 2:
                    assert torch.count_nonzero(w.grad) == 0


@pytest.mark.parametrize('ranks', [[8, 8, 8], [8, 4, 8]])    # one unbind per side, one view per tensor
def test_a_gradient_keeps_its_side_alive_and_no_more(dev, ranks):
    """The gradients of lora_A share one storage and those of lora_B another: a held gradient of one side does not keep the
    other side's memory."""
    from twinkle_amd import multi_lora_delta
    x, base, dy, a, b, ids, _, scales = _problem(200, 128, 256, 3, 8, ranks, seed=6)
    ad, bd = ([w.bfloat16().to(dev).requires_grad_(True) for w in ws] for ws in (a, b))
    y = multi_lora_delta(x.bfloat16().to(dev), base.bfloat16().to(dev), build_segments(ids.to(torch.int32).to(dev), 3),
                         AdapterGroups(ad, bd, ranks, scales))
    grads = torch.autograd.grad(y, ad + bd, dy.bfloat16().to(dev))
    for side, ws in ((grads[:3], ad), (grads[3:], bd)):
        assert all(g.untyped_storage().nbytes() <= sum(2 * w.numel() + 512 for w in ws) for g in side)
    assert grads[0].untyped_storage().data_ptr() != grads[3].untyped_storage().data_ptr()


@pytest.mark.parametrize('t,k,m,ranks', [
    (2304, 2048, 1024, [128, 65]),                  # long groups: weights shared in LDS, chunks in pairs
    (2304, 1024, 512, [100, 128]),                  # the narrowest source of that kernel
    (700, 256, 384, [128, 70, 128]),                # short groups: tile by tile
    (2600, 2048, 256, [128, 16, 40, 0]),            # rank classes next to rank 128
])
def test_rank_128(dev, t, k, m, ranks):
    from test_gpu_lora import _run
    _run(dev, torch.bfloat16, *_problem(t, k, m, len(ranks), 128, ranks, seed=t + m))


@pytest.mark.parametrize('t,k,m,ranks', [
    (1, 1024, 128, [16]),                           # one row, two slices
    (33, 1088, 256, [16, 5, 0]),                    # a last slice of one step, a dead adapter
    (300, 4096, 1024, [16, 8, 1]),                  # eight slices; dy in two
    (24, 4096, 1024, [16, 8, 1]),                   # eight rows an adapter: the eight slices summed in the expand
    (25, 4096, 1024, [16, 8, 1]),                   # ... and one more: before it
    (24, 4672, 256, [16, 8, 1]),                    # ten slices
    (2500, 2048, 1152, [16, 16]),                   # few blocks for the shrink, too many readings for the expand
    (7100, 4096, 128, [16]),                        # the most blocks of the few-tile shrink (224 tiles x 8 slices)
    (7105, 4096, 128, [16]),                        # one tile more: k_shrink_pair
    (8200, 4096, 128, [64, 40]),                    # more sets of eight tiles than CUs: four waves
    (6150, 4096, 128, [32, 20]),                    # ... at rank 32
    (2304, 2112, 384, [64, 40]),                    # rank 64, eight waves: slices that end in half a step
    (2400, 1024, 512, [32, 20, 32]),                # ... and rank 32, runs of several groups in eight tiles
])
def test_few_tiles_and_slices(dev, t, k, m, ranks):
    from test_gpu_lora import _run
    _run(dev, torch.bfloat16, *_problem(t, k, m, len(ranks), max(ranks), ranks, seed=t + m))


@pytest.mark.parametrize('k', [1001, 513, 1004])
@pytest.mark.parametrize('t,m,ranks', [
    (300, 256, [16, 5]),                            # padded rank 16: one class
    (300, 640, [32, 20]),
    (300, 384, [64, 33]),
    (300, 256, [128, 100]),
    (900, 640, [128, 64, 20, 8]),                   # every rank class
])
def test_dx_of_an_odd_width_behind_an_aligned_dy(dev, t, k, m, ranks):
    """dy suits the MFMA row contraction, which can carry the transposed weight copies in blocks of 8 x 8 features; the
    input width does not, so those copies have to reach its last columns some other way.  The workspace holds NaN."""
    from twinkle_amd import lora_bwd_workspace_bytes
    from twinkle_amd.ops import _lora_bwd
    bf16 = torch.bfloat16
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, len(ranks), max(ranks), ranks, seed=t + k)
    xd, yd, dyd = (v.to(bf16).to(dev) for v in (x, base, dy))
    ad, bd = [w.to(bf16).to(dev) for w in a], [w.to(bf16).to(dev) for w in b]
    seg = build_segments(ids.to(torch.int32).to(dev), len(ranks), check=True)
    groups = AdapterGroups(ad, bd, ranks, scales)
    h = lora_fwd_(xd, yd, seg, groups)
    f64 = lambda v: v.to(bf16).double()  # noqa: E731
    _, dxo, dao, dbo = oracle.multi_lora_linear_grads(f64(x), f64(base), ids, [f64(w) for w in a], [f64(w) for w in b],
                                                      ranks, scales, f64(dy))
    for entry, start in (('tk_lora_bwd', 0.0), ('tk_lora_bwd_store', float('nan'))):
        dxd = torch.full_like(xd, start)
        ws = torch.full((lora_bwd_workspace_bytes(seg, groups),), 255, dtype=torch.uint8, device=dev)
        ga, gb = [torch.zeros_like(w) for w in ad], [torch.zeros_like(w) for w in bd]
        pa, pb = (torch.tensor([w.data_ptr() for w in g], dtype=torch.int64, device=dev) for g in (ga, gb))
        _lora_bwd(entry, dyd, xd, h, dxd, pa, pb, seg, groups, workspace=ws)
        assert max_rel_err(dxd, dxo) < TOL[bf16], entry
        for g in range(len(ranks)):
            assert max_rel_err(ga[g], dao[g]) < TOL[bf16], f'dA[{g}]'
            assert max_rel_err(gb[g], dbo[g]) < TOL[bf16], f'dB[{g}]'


@pytest.mark.parametrize('r,r2', [(65, 64), (71, 3), (100, 99), (124, 17), (127, 8)])
def test_lora_b_as_columns_that_end_with_their_buffer(dev, r, r2):
    """Above rank 64 adapters may lie at any element address: B_g = the last r columns of a buffer whose row stride the
    MFMA kernels take.  The operand pieces of the last row then end with the buffer, also of a smaller rank."""
    t, k, m = 300, 128, 256
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, 2, r, [r, r2], seed=r)
    bf16, f64 = torch.bfloat16, lambda v: v.to(torch.bfloat16).double()  # noqa: E731
    ld = (r + 15) // 8 * 8
    bd = []
    for w in b:
        wide = torch.full((m, ld), float('nan'), dtype=bf16, device=dev)
        wide[:, ld - r:] = w.to(bf16).to(dev)
        bd.append(wide[:, ld - r:])
    groups = AdapterGroups([w.to(bf16).to(dev) for w in a], bd, [r, r2], scales)
    seg = build_segments(ids.to(torch.int32).to(dev), 2, check=True)
    yd = base.to(bf16).to(dev)
    lora_fwd_(x.to(bf16).to(dev), yd, seg, groups)
    yo, *_ = oracle.multi_lora_linear_grads(f64(x), f64(base), ids, [f64(w) for w in a], [f64(w) for w in b], [r, r2],
                                            scales, f64(dy))
    assert max_rel_err(yd, yo) < TOL[bf16]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_gradients_of_adapters_that_are_views_of_wider_buffers(dev, dtype):
    """Adapters with a row stride of their own through autograd: their gradients are written at that stride."""
    from twinkle_amd import multi_lora_delta
    t, k, m, ranks = 200, 72, 136, [8, 5]
    x, base, dy, a, b, ids, _, scales = _problem(t, k, m, 2, 8, ranks, seed=4)
    ad, bd = ([_strided(w, dtype, dev, 3).detach().requires_grad_(True) for w in ws] for ws in (a, b))
    y = multi_lora_delta(x.to(dtype).to(dev), base.to(dtype).to(dev), build_segments(ids.to(torch.int32).to(dev), 2),
                         AdapterGroups(ad, bd, ranks, scales))
    y.backward(dy.to(dtype).to(dev))
    f64 = lambda v: v.to(dtype).double()  # noqa: E731
    yo, _, dao, dbo = oracle.multi_lora_linear_grads(f64(x), f64(base), ids, [f64(w) for w in a], [f64(w) for w in b],
                                                     ranks, scales, f64(dy))
    assert max_rel_err(y.detach(), yo) < TOL[dtype]
    for g, r in enumerate(ranks):
        assert max_rel_err(ad[g].grad[:r], dao[g][:r]) < TOL[dtype]
        assert max_rel_err(bd[g].grad[:, :r], dbo[g][:, :r]) < TOL[dtype]
        assert torch.count_nonzero(ad[g].grad[r:]) == 0 and torch.count_nonzero(bd[g].grad[:, r:]) == 0


@pytest.mark.parametrize('t,r', [(6144, 32), (8192, 64)])
def test_eight_and_four_waves_give_the_same_bits(dev, t, r):
    """One row more than the most that k_shrink_oct takes goes through k_shrink_quad: the rows both have come out alike."""
    x, base, _, a, b, _, ranks, scales = _problem(t + 1, 4096, 128, 2, r, [r, r - 9], seed=r)
    ids = (torch.arange(t + 1) * 2 // t).clamp(max=1).to(torch.int32).to(dev)
    bf16 = torch.bfloat16
    groups = AdapterGroups([w.to(bf16).to(dev) for w in a], [w.to(bf16).to(dev) for w in b], ranks, scales)
    xd, out = x.to(bf16).to(dev), []
    for rows in (t, t + 1):
        yd = base[:rows].to(bf16).to(dev)
        lora_fwd_(xd[:rows], yd, build_segments(ids[:rows], 2), groups)
        out.append(yd)
    assert torch.equal(out[0], out[1][:t])
