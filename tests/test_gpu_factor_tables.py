"""The streamed factor pass beyond one 16-row block and one fixed length.

odp_seg_factor_stream_tables takes segments of any length, leaves that span
several 16-row blocks of the rank plane (rank up to 64), chunks of several
sites whose ranks are packed on 16-column boundaries, and tables of several
rank block counts in one launch.  Its rows, partial slots and therefore every
output of a plan equal the tiled pass's (stream_factors=False) bit for bit:
both form the same 32-token MFMA blocks in the same order.  The tiled pass
is checked against the oracle elsewhere (test_gpu_kernels.py,
test_gpu_configs.py).
"""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from opaque_amd import _native as N
from opaque_amd.engine import ClipSpec, GhostPlan, LeafOut, LoraSite, Segments
from opaque_amd.guard import guard_constants, leaf_guards

DEV = "cuda"

# d_in, [(d_out, rank)] per activation; lengths of the examples
LIMIT = 1081  # odp_factor_project_max_len()
CASES = {
    # one step past the fixed-length kernels' bound, steps not a multiple of 64, an empty and a one-row segment
    "long": ([(264, [(520, 16)])], [LIMIT + 1, 0, 1, 2 * LIMIT + 9]),
    "rank20": ([(136, [(72, 20)])], [96, 33, 1, 70]),
    "rank32": ([(520, [(264, 32)])], [65, 0, 64, 63]),
    "rank64": ([(264, [(4360, 64)])], [129, 88, 5, 0]),  # 18 tiles in several groups, the last partial
    "rank64_long": ([(72, [(136, 64)])], [LIMIT + 70, 3, 700, 0]),
    "shared_r8": ([(256, [(256, 8), (64, 8), (64, 8)])], [128, 77, 0, 9]),  # three blocks of 8 of 16 rows
    "shared_r24": ([(128, [(264, 24), (72, 24)])], [96, 50, 3, 64]),  # two leaves of two blocks each
    "shared_four": ([(128, [(64, 4), (72, 16), (80, 12), (88, 1)])], [70, 64, 1, 0]),
    "shared_r20_tiled": ([(128, [(64, 20), (72, 20), (80, 20)])], [70, 64, 1, 0]),  # 96 columns: packed side by side
    "mixed": ([(256, [(256, 16), (64, 16), (64, 16)]), (72, [(200, 64)]), (512, [(128, 16)]),
               (136, [(264, 32)])], [200, 64, 31, 129]),  # tables of 1, 2, 3 and 4 blocks
}


def _case(name, scalings=(2.0,)):
    acts, lengths = CASES[name]
    g = torch.Generator(device=DEV).manual_seed(sum(map(ord, name)))
    T = max(lengths)
    n_rows = len(lengths) * T
    seg = Segments.padded(len(lengths), T, lengths)

    def rnd(*shape, scale=1.0):
        return (torch.randn(*shape, device=DEV, generator=g) * scale).to(torch.bfloat16)

    sites, leaves = [], []
    for d_in, outs in acts:
        x = rnd(n_rows, d_in)
        for k, (d_out, r) in enumerate(outs):
            gt, A, B = rnd(n_rows, d_out, scale=0.3), rnd(d_in, r, scale=1 / math.sqrt(d_in)), rnd(r, d_out, scale=0.05)
            n = len(leaves)
            leaves += [LeafOut((d_in, r), torch.bfloat16, group=n),
                       LeafOut((r, d_out), torch.bfloat16, group=n + 1)]
            sites.append(LoraSite(x, gt, A, B, scalings[k % len(scalings)], a_leaf=n, b_leaf=n + 1, v=x @ A,
                                  u=gt @ B.t().contiguous()))
    return seg, sites, leaves


def _plan(seg, sites, leaves, stream):
    _, rnd = leaf_guards([lf.shape for lf in leaves], [torch.bfloat16] * len(leaves))
    rel, ab = guard_constants(torch.bfloat16, rnd)
    clip = ClipSpec(mode=N.CLIP_AUTOS, thresholds=[1.0] * len(leaves), effective=math.sqrt(len(leaves)), gamma=0.01,
                    normalize_by=2.0, guards=[(rel, ab, torch.bfloat16)])
    return GhostPlan(segments=seg, leaves=leaves, clip=clip, lora_sites=sites, device=DEV, stream_factors=stream)


def _outputs(plan):
    res = plan.run()
    torch.cuda.synchronize()
    return [t.clone() for t in plan.pe_views()] + [t.clone() for t in res.leaves] + [
        res.norms.clone(), res.group_norms.clone(), plan.part.clone()]


def _check(name, scalings=(2.0,)):
    assert int(N.load().odp_factor_project_max_len()) == LIMIT
    seg, sites, leaves = _case(name, scalings)
    off, on = _plan(seg, sites, leaves, False), _plan(seg, sites, leaves, True)
    stages = {t[0] for t in on.tables if t[5] > 0}
    assert "factor_stream" in stages and ("factor" in stages) == name.endswith("tiled"), stages
    for k, (a, b) in enumerate(zip(_outputs(on), _outputs(off))):
        assert torch.isfinite(a.float()).all(), k
        assert torch.equal(a, b), k
    # Each leaf's group norm is that of its stored rows: fp64 sums of float32 squares, returned in float32.
    norms = on.run().group_norms.double()
    torch.cuda.synchronize()
    for k, pe in enumerate(on.pe_views()):
        want = pe.view(seg.n_ex, -1).float().square().double().sum(1).sqrt()
        assert torch.allclose(norms[k], want, rtol=1e-6), k
    return on


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_streamed_tables_equal_the_tiled_pass(name):
    print(f"streamed factor tables: {name}", flush=True)
    on = _check(name)
    if name == "mixed":
        assert {t[1] for t in on.tables if t[0] == "factor_stream" and t[5] > 0} == {1, 2, 3, 4}
        assert [i[1] for i in on.launch_info if i[0] == "factor_stream"] == [(1, 2, 3, 4)]


@pytest.mark.gpu
def test_sites_of_different_scalings_stream_their_own_rows():
    print("streamed factor tables: two scalings", flush=True)
    _check("shared_r24", (2.0, 0.5))


# Rank blocks: (first column, rank) of each leaf.  A block without a leaf, ranks below and at 16, and for the
# tables entry leaves that span blocks.
DIRECT = {1: [(0, 16)], 2: [(0, 9), (16, 16)], 3: [(0, 16), (32, 3)], 4: [(0, 40), (48, 16)]}


class _Direct:
    """One problem of nkb rank blocks for a direct call: segments of one step, none and several, unaligned, below
    odp_factor_project_max_len() rows; 18 column tiles, the last partial."""

    M, starts, lens = 4360, [0, 61, 61, 129], [61, 0, 67, 700]

    def __init__(self, nkb):
        g = torch.Generator(device=DEV).manual_seed(nkb)
        self.nkb, self.leaves, n_rows = nkb, DIRECT[nkb], 840
        self.r = self.leaves[-1][0] + self.leaves[-1][1]
        self.ldq = (n_rows + 32 + 7) // 8 * 8
        self.P = torch.randn(n_rows, self.M, device=DEV, generator=g).to(torch.bfloat16)
        self.Q = torch.randn(16 * nkb, self.ldq, device=DEV, generator=g).to(torch.bfloat16)
        self.tiles = int(N.load().odp_seg_factor_tiles(N.DTYPE_BF16, self.M, self.r))
        self.n_slots = len(self.leaves) * N.FT_WAVE_SLOTS * self.tiles
        self.seg = [torch.tensor(v, device=DEV, dtype=torch.int32) for v in (self.starts, self.lens, range(4))]

    def outputs(self):
        pes = [torch.full((4, rk, self.M), 7.0, device=DEV, dtype=torch.bfloat16) for _, rk in self.leaves]
        return pes, torch.full((4, self.n_slots), -1.0, device=DEV, dtype=torch.float64)

    def row(self, pes, groups=0):
        row = [0] * N.FT_FIELDS
        row[N.FT_P], row[N.FT_LDP], row[N.FT_M] = self.P.data_ptr(), self.M, self.M
        row[N.FT_Q], row[N.FT_LDQ], row[N.FT_R] = self.Q.data_ptr(), self.ldq, self.r
        row[N.FT_NSEG], row[N.FT_NLEAF], row[N.FT_GROUPS] = 4, len(self.leaves), groups
        row[N.FT_SCALING] = int(torch.tensor([2.0], dtype=torch.float64).view(torch.int64).item())
        for k, ((col, rk), pe) in enumerate(zip(self.leaves, pes)):
            row[N.FT_LEAF0 + 3 * k : N.FT_LEAF0 + 3 * k + 3] = [pe.data_ptr(), col | rk << 16 | 1 << 32,
                                                                k * N.FT_WAVE_SLOTS * self.tiles]
        return torch.tensor(row, dtype=torch.int64, device=DEV)

    def args(self, part):
        return (*(t.data_ptr() for t in self.seg), part.data_ptr(), self.n_slots)

    def tiled(self):
        pes, part = self.outputs()
        row, total = self.row(pes), 4 * self.tiles
        ws = torch.tensor([0, total], device=DEV, dtype=torch.int32)
        N.check(N.load().odp_seg_factor(torch.cuda.current_stream().cuda_stream, N.DTYPE_BF16, row.data_ptr(),
                                        ws.data_ptr(), 1, total, *self.args(part), self.nkb), "tiled")
        torch.cuda.synchronize()
        assert (part >= 0).all()  # every slot is written
        return pes, part


@pytest.mark.gpu
@pytest.mark.parametrize("groups", [1, 5, 18])
@pytest.mark.parametrize("nkb", [1, 2, 3])
def test_one_streamed_table_equals_the_tiled_pass(nkb, groups):
    """odp_seg_factor_stream (no plan launches it): rows and every partial slot, bit for bit."""
    print(f"streamed factor table: {nkb} rank blocks, {groups} groups", flush=True)
    d = _Direct(nkb)
    want, want_part = d.tiled()
    pes, part = d.outputs()
    row, total = d.row(pes, groups), 4 * groups
    ws = torch.tensor([0, total], device=DEV, dtype=torch.int32)
    N.check(N.load().odp_seg_factor_stream(torch.cuda.current_stream().cuda_stream, row.data_ptr(), ws.data_ptr(), 1,
                                           total, *d.args(part), nkb), "stream")
    torch.cuda.synchronize()
    assert torch.equal(part, want_part)
    assert all(torch.equal(a, b) for a, b in zip(pes, want))


@pytest.mark.gpu
@pytest.mark.parametrize("spare", [0, 9 << 20])
def test_streamed_tables_called_directly(spare):
    """Four tables at once; with spare workgroups (past a row's segments, which have nothing to do) two of them
    hold 2^23 and more, together more than one launch may have."""
    print(f"streamed factor tables: four at once, {spare} spare workgroups", flush=True)
    ds = [_Direct(k + 1) for k in range(4)]
    wants = [d.tiled() for d in ds]
    n_slots = max(d.n_slots for d in ds)
    outs = [d.outputs() for d in ds]
    # One partials buffer for the call: the tables' examples lie one after the other.
    part = torch.full((16, n_slots), -1.0, device=DEV, dtype=torch.float64)
    segs = [torch.cat([d.seg[j] for d in ds]) for j in range(2)] + [torch.arange(16, device=DEV, dtype=torch.int32)]
    groups, rows, maps = 5, [], []
    for k, (d, (pes, _)) in enumerate(zip(ds, outs)):
        row = d.row(pes, groups)
        row[N.FT_SEG_FIRST] = 4 * k
        work = torch.stack([torch.zeros(4 * groups, dtype=torch.int32), torch.arange(4 * groups, dtype=torch.int32)], 1)
        idle = torch.tensor([[0, 4 * groups]], dtype=torch.int32, device=DEV).expand(spare if k in (0, 2) else 0, 2)
        rows.append(row)
        maps.append(torch.cat([idle, work.to(DEV)]).contiguous())  # the work last
    call = N.load().odp_seg_factor_stream_tables
    N.check(call(torch.cuda.current_stream().cuda_stream, (ctypes.c_void_p * 4)(*[t.data_ptr() for t in rows]),
                 (ctypes.c_void_p * 4)(*[t.data_ptr() for t in maps]), (ctypes.c_int32 * 4)(1, 1, 1, 1),
                 (ctypes.c_int32 * 4)(*[t.shape[0] for t in maps]), *(t.data_ptr() for t in segs), part.data_ptr(),
                 n_slots), "tables")
    torch.cuda.synchronize()
    for k, (d, (pes, _), (want, want_part)) in enumerate(zip(ds, outs, wants)):
        assert torch.equal(part[4 * k : 4 * k + 4, : d.n_slots], want_part), k
        assert all(torch.equal(a, b) for a, b in zip(pes, want)), k


def test_argument_checks():
    lib = N.load()
    null, bad = (ctypes.c_void_p * 4)(), (ctypes.c_void_p * 4)(8, None, None, None)
    zero, one = (ctypes.c_int32 * 4)(), (ctypes.c_int32 * 4)(1, 0, 0, 0)
    call = lib.odp_seg_factor_stream_tables
    assert call(None, null, null, zero, zero, None, None, None, None, 1) == N.ODP_OK  # no work
    assert call(None, None, null, zero, zero, None, None, None, None, 1) == N.ERR_INVALID_ARGUMENT
    assert call(None, null, null, one, one, None, None, None, None, 1) == N.ERR_INVALID_ARGUMENT
    assert call(None, bad, bad, one, one, None, None, None, None, 1) == N.ERR_INVALID_ARGUMENT
    assert "null segment" in lib.odp_last_error().decode()
    assert call(None, bad, bad, zero, one, 8, 8, 8, 8, 1) == N.ERR_INVALID_ARGUMENT  # work without problems
    assert call(None, bad, bad, one, one, 8, 8, 8, 8, 0) == N.ERR_INVALID_ARGUMENT  # part_stride
