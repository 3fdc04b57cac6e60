"""Norms and clipped sums of stored per-example gradients, at the edges of
their vector paths.

odp_sqnorm reads 16-byte pieces of each example's row and the elements before
and after them one by one, odp_scale_sum takes rows in 16-byte pieces, rows of
other lengths element by element, and transposed LoRA leaves through LDS
tiles of whole columns, and odp_clip_factors sums several groups side by side.

The clipped sum is defined to the bit (clip_pytree's scale.to(dtype) * leaf
rounded to the leaf's dtype, a float32 sum over the examples in order, a cast
and a division in the output dtype), so it is compared with those torch
operations exactly for 16-bit values.  For float32 ones the kernel adds
scale * value by fused multiply-adds, which leave out the product's rounding:
each term may differ by half a unit in its last place, and each partial sum
rounds differently in turn, within sqrt(n) 2^-23 of the sum of magnitudes.  Norms are fp64 sums of float32 squares in some order,
returned in float32: rel 1e-6.
"""

from __future__ import annotations

import math

import pytest
import torch

from opaque_amd import _native as N
from opaque_amd.engine import ClipSpec, GhostPlan, LeafOut, LoraSite, MaterializedLeaf, Segments
from opaque_amd.guard import guard_constants, leaf_guards

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _clip(leaves, dtype, thresholds):
    _, rnd = leaf_guards([lf.shape for lf in leaves], [dtype] * len(leaves))
    rel, ab = guard_constants(dtype, rnd)
    return ClipSpec(mode=N.CLIP_FIXED, thresholds=thresholds, effective=math.sqrt(sum(t * t for t in thresholds)),
                    normalize_by=3.0, guards=[(rel, ab, dtype)])


def _close(got, want, pe, c, power=1):
    if pe.dtype != torch.float32:
        return torch.equal(got, want)
    v = torch.where(torch.isfinite(pe), pe, torch.zeros_like(pe)).double()
    mag = (c.view(-1, *[1] * (pe.dim() - 1)) * v).abs().pow(power).sum(0)
    return bool(((got.double() - want.double()).abs() <= 2.0**-23 * pe.shape[0] ** 0.5 * mag).all())


def _sums(pe, c, out_dtype, nb=3.0):
    """Clipped sum and second moment of pe [n, ...] with scales c [n], torch operation by operation on the
    host (IEEE division)."""
    pe, c = pe.cpu(), c.cpu()
    acc = acc2 = torch.zeros(pe.shape[1:], dtype=torch.float32)
    v = torch.where(torch.isfinite(pe), pe, torch.zeros_like(pe))
    for i in range(pe.shape[0]):
        y = c[i].to(pe.dtype) * v[i]
        acc = acc + y.float()
        acc2 = acc2 + (y * y).float()
    return [(t.to(out_dtype) / torch.tensor(nb, dtype=out_dtype)).to(DEV) for t in (acc, acc2)]


# (elements per example, examples): below, at and past one piece, one workgroup's tile and one chunk of
# the norm kernel; odd rows; several groups of segments and a rest.
ROWS = [(1, 1), (3, 5), (8, 9), (1001, 17), (1024, 8), (2048, 4), (2052, 3), (8191, 2), (8192, 7), (24580, 13)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,n_ex", ROWS)
def test_materialised_rows(n, n_ex, dtype, second, offset):
    """offset: elements from the allocation's start to the leaf.  One past it no row of a length on the 16-byte grid
    lies on the grid itself: the sums then walk one element a thread over the tiles of 8 or 4, the norms read a
    head before each row's pieces."""
    print(f"stored sums: {n} x {n_ex} {dtype} second={second} offset={offset}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(n + n_ex)
    spread = torch.logspace(-1, 1, n_ex, device=DEV).view(-1, 1)
    pe = torch.empty(n_ex * n + offset, device=DEV, dtype=dtype)[offset:].view(n_ex, n)
    pe.copy_(torch.randn(n_ex, n, device=DEV, generator=g) * spread)
    assert (pe.data_ptr() % 16 != 0) == bool(offset)
    pe[0, 0] = float("nan")
    pe[n_ex - 1, n - 1] = float("-inf")
    leaves = [LeafOut((n,), dtype)]
    finite = torch.where(torch.isfinite(pe), pe, torch.zeros_like(pe)).float()
    norms = finite.square().double().sum(1).sqrt()
    C = float(norms.median())
    plan = GhostPlan(segments=Segments.padded(n_ex, 1), leaves=leaves, clip=_clip(leaves, dtype, [C]),
                     materialized=[MaterializedLeaf(pe, 0)], device=DEV, second_moment=second)
    res = plan.run()
    torch.cuda.synchronize()
    assert torch.allclose(res.norms.double(), norms, rtol=1e-6, atol=0)
    want = _sums(pe, res.scales[0, 0], dtype)
    assert _close(res.leaves[0], want[0], pe, res.scales[0, 0])
    if second:
        assert _close(res.second_moment[0], want[1], pe, res.scales[0, 0], 2)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype,second", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, True),
                                          (torch.float16, False)])
@pytest.mark.parametrize("n,n_ex", [(1 << 22, 1), ((1 << 22) + 8, 2), ((1 << 22) + 2056, 3), ((1 << 22) + 4104, 4),
                                    ((1 << 22) + 8, 5)])
def test_few_examples_of_large_rows(n, n_ex, dtype, second, offset):
    """Up to four examples of rows this long take several pieces a thread: whole and partial last workgroups, an odd
    example, and rows off the grid and five examples, which keep one piece."""
    test_materialised_rows(n, n_ex, dtype, second, offset)


@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r", [1, 4, 8, 12, 20, 64])
def test_transposed_leaves(r, dtype, second):
    """A leaf [d_in, r] and B leaf [d_out, r], both transposed from the [r][M]
    rows the plan stores; widths of less than one tile and of several with a
    rest."""
    print(f"stored sums: transposed rank {r} {dtype} second={second}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(r)
    n_ex, T, d_in, d_out = 9, 8, 24, 2072

    def rnd(*s):
        return torch.randn(*s, device=DEV, generator=g).to(dtype)

    x, gt, A, B = rnd(n_ex * T, d_in), rnd(n_ex * T, d_out), rnd(d_in, r), rnd(r, d_out)
    leaves = [LeafOut((d_in, r), dtype), LeafOut((d_out, r), dtype)]
    site = LoraSite(x, gt, A, B, 0.5, a_leaf=0, b_leaf=1, a_transposed=False, b_transposed=True, v=x @ A,
                    u=gt @ B.t().contiguous())
    plan = GhostPlan(segments=Segments.padded(n_ex, T), leaves=leaves, clip=_clip(leaves, dtype, [50.0]),
                     lora_sites=[site], device=DEV, second_moment=second)
    res = plan.run()
    torch.cuda.synchronize()
    for k, (pe, m) in enumerate(zip(plan.pe_views(), (d_in, d_out))):
        rows, c = pe.view(n_ex, r, m).transpose(1, 2), res.scales[0, 0]
        want = _sums(rows, c, dtype)
        assert _close(res.leaves[k], want[0], rows, c), k
        if second:
            assert _close(res.second_moment[k], want[1], rows, c, 2), k


@pytest.mark.parametrize("groups", [1, 2, 3, 8, 9, 16, 17, 40])
def test_groups_side_by_side(groups):
    """Groups share the clip kernel's 16 waves evenly, one wave each past 8 groups, in rounds past 16."""
    print(f"stored sums: {groups} clip groups", flush=True)
    g = torch.Generator(device=DEV).manual_seed(groups)
    n_ex = 3
    sizes = [1 + (7919 * k) % 30011 for k in range(groups + 2)]  # one to four partial slots each
    group = [k % groups for k in range(groups + 2)]
    pes = [torch.randn(n_ex, n, device=DEV, generator=g) for n in sizes]
    leaves = [LeafOut((n,), torch.float32, group=k) for n, k in zip(sizes, group)]
    want = torch.zeros(groups, n_ex, dtype=torch.float64, device=DEV)
    for pe, k in zip(pes, group):
        want[k] += pe.square().double().sum(1)
    C = (want.sqrt().mean(1) * 1.0).tolist()
    plan = GhostPlan(segments=Segments.padded(n_ex, 1), leaves=leaves, clip=_clip(leaves, torch.float32, C),
                     materialized=[MaterializedLeaf(pe, k) for k, pe in enumerate(pes)], device=DEV)
    res = plan.run()
    torch.cuda.synchronize()
    assert torch.allclose(res.group_norms.double(), want.sqrt(), rtol=1e-6)
    assert torch.allclose(res.norms.double(), want.sum(0).sqrt(), rtol=1e-6)
    thr = torch.tensor(C, device=DEV).view(-1, 1)
    assert torch.equal(res.clipped.bool(), res.group_norms > thr.float())


@pytest.mark.parametrize("r,frozen", [(8, False), (16, True), (24, False), (64, False)])
def test_f32_factor_rows(r, frozen):
    """float32 per-example factor rows (odp_seg_factor): ranks of one to four 16-row blocks, two sites on one
    activation (one with a frozen A: rows without a leaf), widths of less than a wave's 64 columns, of a
    workgroup's 256 and past it, segments of less than a step, of several pipelines and unaligned, rows outside
    the segments NaN.  Each entry is a float32 sum of L products: |error| <= (L + 2) 2^-24 sum |terms|."""
    print(f"stored sums: fp32 factor rows rank {r} frozen={frozen}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(r)
    starts, lengths, n_rows = [0, 5, 5, 22, 150], [5, 0, 17, 127, 1], 160
    seg = Segments(starts, lengths, list(range(5)), 5, n_rows)
    d_in, outs = 260, (60, 264)

    def rnd(*s):
        return torch.randn(*s, device=DEV, generator=g)

    inside = torch.zeros(n_rows, dtype=torch.bool, device=DEV)
    for s, n in zip(starts, lengths):
        inside[s : s + n] = True
    x = rnd(n_rows, d_in)
    x[~inside] = float("nan")
    sites, leaves = [], []
    for i, d_out in enumerate(outs):
        rr = r if i == 0 or r < 64 else 4
        gt, A, B = rnd(n_rows, d_out), rnd(d_in, rr), rnd(rr, d_out)
        gt[~inside] = float("nan")
        a = None
        if not (frozen and i == 0):
            a = len(leaves)
            leaves.append(LeafOut((d_in, rr), torch.float32))
        leaves.append(LeafOut((rr, d_out), torch.float32))
        sites.append(LoraSite(x, gt, A, B, 0.5, a_leaf=a, b_leaf=len(leaves) - 1, v=x @ A, u=gt @ B.t()))
    plan = GhostPlan(segments=seg, leaves=leaves, clip=_clip(leaves, torch.float32, [1e30]), lora_sites=sites,
                     device=DEV)
    plan.run()
    torch.cuda.synchronize()
    pes = plan.pe_views()
    for s in sites:
        for leaf, q, p in ((s.a_leaf, s.u, s.x), (s.b_leaf, s.v, s.g)):
            if leaf is None:
                continue
            got = pes[leaf].view(5, q.shape[1], p.shape[1])
            for k, (st, n) in enumerate(zip(starts, lengths)):
                a, b = q[st : st + n].double().t(), p[st : st + n].double()
                bound = (n + 2) * 2.0**-24 * 0.5 * (a.abs() @ b.abs())
                assert ((got[k].double() - 0.5 * (a @ b)).abs() <= bound).all(), (leaf, k)


# Partials per group: a group goes to the whole workgroup past 16384 partials a wave and four times its waves'
# even share (five to eight groups have two waves each, more have one).
LONG = {
    "one_of_sixteen": [64] * 7 + [40961] + [63] * 8,
    "at_the_limit": [1] * 9 + [16384],
    "past_the_limit": [1] * 9 + [16385],
    "two_waves": [3, 50001, 0, 7, 1],
    "three_long": [40000, 1, 2, 40001, 5, 6, 7, 39999, 9, 10],
    "last_of_forty": [17] * 39 + [100003],
    "even": [20000] * 10,
}


@pytest.mark.parametrize("name", sorted(LONG))
def test_one_long_group_among_short_ones(name):
    """odp_clip_factors called directly on partials of one group layout; fp64 sums in some order: rel 1e-6 of the
    float32 results, and the same bits from run to run."""
    print(f"stored sums: clip groups {name}", flush=True)
    lib, lens, n_ex = N.load(), LONG[name], 3
    g = torch.Generator(device=DEV).manual_seed(len(lens))
    part = torch.rand(n_ex, sum(lens), device=DEV, dtype=torch.float64, generator=g)
    bounds = [sum(lens[:k]) for k in range(len(lens) + 1)]
    want = torch.stack([part[:, a:b].sum(1) for a, b in zip(bounds, bounds[1:])])
    thr = want.sqrt().mean(1) + 0.5
    start = torch.tensor(bounds, device=DEV, dtype=torch.int64)
    guard, cls = torch.tensor([1.0, 0.0], device=DEV, dtype=torch.float64), torch.zeros(1, device=DEV, dtype=torch.int32)
    runs = []
    for _ in range(2):
        scales = torch.zeros(1, len(lens), n_ex, device=DEV, dtype=torch.float64)
        norms, gn = torch.zeros(n_ex, device=DEV), torch.zeros(len(lens), n_ex, device=DEV)
        clipped = torch.zeros(len(lens), n_ex, device=DEV, dtype=torch.uint8)
        total = torch.zeros(n_ex, device=DEV, dtype=torch.uint8)
        N.check(lib.odp_clip_factors(torch.cuda.current_stream().cuda_stream, part.data_ptr(), part.shape[1], n_ex,
                                     start.data_ptr(), len(lens), thr.data_ptr(), 1.0, N.CLIP_FIXED, 0.0, 1,
                                     guard.data_ptr(), cls.data_ptr(), scales.data_ptr(), norms.data_ptr(),
                                     gn.data_ptr(), clipped.data_ptr(), total.data_ptr()), name)
        runs.append((scales, norms, gn, clipped, total))
    torch.cuda.synchronize()
    scales, norms, gn, clipped, _ = runs[0]
    assert torch.allclose(gn.double(), want.sqrt(), rtol=1e-6)
    assert torch.allclose(norms.double(), want.sum(0).sqrt(), rtol=1e-6)
    assert torch.allclose(scales[0], (thr.view(-1, 1) / want.sqrt()).clamp(max=1.0), rtol=1e-6)
    assert torch.equal(clipped.bool(), gn > thr.float().view(-1, 1))
    assert all(torch.equal(a, b) for a, b in zip(*runs))


def test_more_tiles_than_one_launch_holds():
    """A leaf of 2^32 + 3 bfloat16 values, off the 16-byte grid: one element a thread would be 2^24 workgroups and
    more, 2^32 threads, which a launch does not hold; the workgroups walk over several tiles instead."""
    print("stored sums: 2^32 + 3 elements", flush=True)
    n, q = 2**32 + 3, 2**20 + 7
    m = n // q
    base = torch.randn(q, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)).to(torch.bfloat16)
    pe = torch.zeros(1, n, device=DEV, dtype=torch.bfloat16)
    pe[0, : m * q].view(m, q).copy_(base)
    pe[0, n - 1] = 2.0
    leaves = [LeafOut((n,), torch.bfloat16)]
    plan = GhostPlan(segments=Segments.padded(1, 1), leaves=leaves, clip=_clip(leaves, torch.bfloat16, [1e30]),
                     materialized=[MaterializedLeaf(pe, 0)], device=DEV)
    assert sum(t[5] for t in plan.tables if t[0] == "scale_sum") < 2**24
    res = plan.run()
    torch.cuda.synchronize()
    norm = (m * base.float().square().double().sum() + 4.0).sqrt()
    assert torch.allclose(res.norms.double(), norm, rtol=1e-6)
    want = _sums(base.view(1, q), res.scales[0, 0], torch.bfloat16)[0]
    got = res.leaves[0]
    assert bool((got[: m * q].view(m, q) == want).all())
    rest = torch.zeros(n - m * q, dtype=torch.bfloat16)
    rest[-1] = 2.0
    assert torch.equal(got[m * q :], _sums(rest.view(1, -1), res.scales[0, 0], torch.bfloat16)[0])
