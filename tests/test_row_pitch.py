"""Row views that the kernels take: a pitch of at least the row, within 32-bit offsets.

The factor kernels bound a segment's rows by rows x pitch bytes, so an
expanded activation (pitch 0: one row for every token, e.g. the output
gradient of a sum over tokens) or overlapping rows would read as zeros past
that bound, and rows 16 MiB or more apart could wrap a 32-bit offset back into
it.  Such inputs are copied; every plan over them equals, bit for bit, the
plan over contiguous copies, and the rows it stores equal the float64 product.
odp_seg_factor itself takes float32 rows of any pitch.
"""

from __future__ import annotations

import math

import pytest
import torch

from opaque_amd import _native as N
from opaque_amd.engine import MAX_ROW_PITCH, ClipSpec, GhostPlan, LeafOut, LoraSite, Segments, _rows
from opaque_amd.guard import guard_constants, leaf_guards

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _view(kind, rows, d, dt, dev, g):
    """[rows, d] of the kind's layout."""
    def rnd(*shape):
        return (torch.randn(*shape, generator=g) * 0.5).to(dt).to(dev)

    if kind == "expanded":
        return rnd(d).expand(rows, d)
    if kind == "expanded_batch":  # as a microbatch of one example brings it
        return rnd(d).expand(1, rows, d)
    if kind == "one_row":
        return rnd(d).as_strided((1, d), (0, 1))
    if kind == "overlapping":
        return rnd(d + 8 * (rows - 1)).as_strided((rows, d), (8, 1))
    if kind == "padded":
        return rnd(rows, d + 8)[:, :d]
    assert kind == "far"
    pitch = MAX_ROW_PITCH // dt.itemsize
    base = torch.zeros(pitch * (rows - 1) + d, dtype=dt, device=dev)
    far = base.as_strided((rows, d), (pitch, 1))
    far.copy_(rnd(rows, d))
    return far


COPIED = ["expanded", "expanded_batch", "one_row", "overlapping", "far"]


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("kind", COPIED + ["padded"])
def test_row_views(kind, dt):
    rows = 1 if kind == "one_row" else 3
    t = _view(kind, rows, 24, DTYPES[dt], "cpu", torch.Generator().manual_seed(1))
    v = _rows(t)
    assert torch.equal(v, t.reshape(-1, 24))
    assert v.stride(1) == 1 and v.stride(0) >= 24 and v.stride(0) * v.element_size() < MAX_ROW_PITCH
    if kind != "one_row":  # reshape() gives one row its own length as its pitch
        assert (v.data_ptr() == t.data_ptr()) == (kind == "padded")


@pytest.mark.gpu
@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("rank", [8, 20, 64])
@pytest.mark.parametrize("kind", COPIED + ["padded"])
def test_factor_rows_of_any_pitch(kind, rank, dt):
    print(f"row pitch: {kind} rank {rank} {dt}", flush=True)
    dtype, d_in, d_out, rows = DTYPES[dt], 136, 264, 1 if kind == "one_row" else 5
    gen = torch.Generator().manual_seed(rank)
    # One side in the layout under test, the other plain, both ways.
    for side in ("x", "g"):
        x = _view(kind if side == "x" else "padded", rows, d_in, dtype, "cuda", gen)
        g = _view(kind if side == "g" else "padded", rows, d_out, dtype, "cuda", gen)
        A = (torch.randn(d_in, rank, generator=gen) / math.sqrt(d_in)).to(dtype).cuda()
        B = (torch.randn(rank, d_out, generator=gen) * 0.05).to(dtype).cuda()
        x2, g2 = x.reshape(-1, d_in).clone(), g.reshape(-1, d_out).clone()
        v, u = x2 @ A, g2 @ B.t().contiguous()
        leaves = [LeafOut((d_in, rank), dtype), LeafOut((rank, d_out), dtype)]
        _, rnd = leaf_guards([lf.shape for lf in leaves], [dtype] * 2)
        rel, ab = guard_constants(dtype, rnd)
        outs = []
        for xx, gg in ((x, g), (x2, g2)):
            clip = ClipSpec(mode=N.CLIP_AUTOS, thresholds=[1.0], effective=1.0, gamma=0.01, normalize_by=1.0,
                            guards=[(rel, ab, dtype)])
            plan = GhostPlan(segments=Segments.padded(1, rows, [rows]), leaves=leaves, clip=clip,
                             lora_sites=[LoraSite(xx, gg, A, B, 2.0, a_leaf=0, b_leaf=1, v=v, u=u)], device="cuda")
            res = plan.run()
            torch.cuda.synchronize()
            outs.append([t.clone() for t in plan.pe_views()] + [t.clone() for t in res.leaves] + [res.norms.clone()])
        for a, b in zip(*outs):
            assert torch.equal(a, b), (side, kind)
        # Stored rows: [rank][M] products of at most 5 terms, one rounding to the dtype.
        want = [2.0 * u.double().t() @ x2.double(), 2.0 * v.double().t() @ g2.double()]
        eps = torch.finfo(dtype).eps
        for got, w in zip(outs[0], want):
            err = (got.double().view(w.shape) - w).norm() / w.norm()
            assert err < eps + 8 * torch.finfo(torch.float32).eps, (side, kind, float(err))


# Elements from one row to the next: one row for all, rows that overlap, the row itself, a padded row, and rows
# on both sides of the pitch whose offsets within a step pass 31 bits (128 MiB and 160 MiB).
F32_PITCHES = {"expanded": 0, "overlapping": 8, "contiguous": 264, "padded": 272, "128MiB": 1 << 25, "160MiB": 5 << 23}


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [3, 20, 64])
@pytest.mark.parametrize("kind", sorted(F32_PITCHES))
def test_f32_factor_entry_takes_any_pitch(kind, rank):
    """odp_seg_factor called directly.  Each entry is a float32 sum of at most 18 products: |error| <= (n + 2)
    2^-24 sum |terms|."""
    print(f"row pitch: odp_seg_factor f32, {kind} rank {rank}", flush=True)
    lib, M, pitch = N.load(), 264, F32_PITCHES[kind]
    # One row, an unaligned segment of two steps, and an empty one whose start lies past every row: it reads nothing.
    starts, lens, rows = [0, 2, 1 << 30], [1, 18, 0], 20
    if pitch > 1000:
        starts, lens, rows = [0, 1, 1 << 30], [1, 3, 0], 4
    g = torch.Generator(device="cuda").manual_seed(rank)
    base = torch.empty(pitch * (rows - 1) + M, device="cuda")
    P = base.as_strided((rows, M), (pitch, 1))
    if pitch < M:
        base.copy_(torch.randn(base.shape, device="cuda", generator=g))
    else:
        P.copy_(torch.randn(rows, M, device="cuda", generator=g))
    nkb, ldq = (rank + 15) // 16, (rows + 32 + 7) // 8 * 8
    Q = torch.randn(16 * nkb, ldq, device="cuda", generator=g)
    pe = torch.ones(3, rank, M, device="cuda")
    slots = N.FT_WAVE_SLOTS * int(lib.odp_seg_factor_tiles(N.DTYPE_F32, M, rank))
    part = torch.zeros(3, slots, device="cuda", dtype=torch.float64)
    row = [0] * N.FT_FIELDS
    row[N.FT_P], row[N.FT_LDP], row[N.FT_M] = P.data_ptr(), pitch, M
    row[N.FT_Q], row[N.FT_LDQ], row[N.FT_R] = Q.data_ptr(), ldq, rank
    row[N.FT_NSEG], row[N.FT_NLEAF] = 3, 1
    row[N.FT_SCALING] = int(torch.tensor([0.5], dtype=torch.float64).view(torch.int64).item())
    row[N.FT_LEAF0], row[N.FT_LEAF0 + 1] = pe.data_ptr(), rank << 16
    blocks = 3 * slots // N.FT_WAVE_SLOTS
    dev = [torch.tensor(v, device="cuda", dtype=dt) for v, dt in
           ((row, torch.int64), ([0, blocks], torch.int32), (starts, torch.int32), (lens, torch.int32),
            ([0, 1, 2], torch.int32))]
    probs, ws, sst, sln, sex = (t.data_ptr() for t in dev)
    N.check(lib.odp_seg_factor(torch.cuda.current_stream().cuda_stream, N.DTYPE_F32, probs, ws, 1, blocks, sst, sln,
                               sex, part.data_ptr(), slots, nkb), kind)
    torch.cuda.synchronize()
    for k, (st, n) in enumerate(zip(starts, lens)):
        if n == 0:
            assert not pe[k].any() and not part[k].any()
            continue
        a, b = Q[:rank, st : st + n].double(), P[st : st + n].double()
        bound = (n + 2) * 2.0**-24 * 0.5 * (a.abs() @ b.abs())
        assert ((pe[k].double() - 0.5 * (a @ b)).abs() <= bound).all(), (kind, k)
        # float32 squares in fp64: each rounds by at most 2^-24 of itself.
        assert torch.allclose(part[k].sum(), pe[k].double().square().sum(), rtol=2.0**-23)
