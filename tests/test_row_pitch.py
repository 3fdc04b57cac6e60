"""Row views that the kernels take: a pitch of at least the row, within 32-bit offsets.

The factor kernels bound a segment's rows by rows x pitch bytes, so an
expanded activation (pitch 0: one row for every token, e.g. the output
gradient of a sum over tokens) or overlapping rows would read as zeros past
that bound, and rows 16 MiB or more apart could wrap a 32-bit offset back into
it.  Such inputs are copied; every plan over them equals, bit for bit, the
plan over contiguous copies, and the rows it stores equal the float64 product.
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
