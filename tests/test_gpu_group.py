"""GPU: the programs run by dependency level (one launch per level, all programs and
columns of a group together) against the same programs run one instruction per launch
(set_option(fuse=False)): the operations and their order per element are the same, so F,
J, its fp32 columns and J^T w must agree bit for bit.

Sizes: smallest grids, odd and even line lengths, arrays of few outputs (a thread each)
and of many (a thread per line), element-wise regions of one and of several elements per
thread, both unknown orders, a system with a double unknown and integral equation, and
column ranges that start and end inside a program."""
import numpy as np
import pytest
import torch

from kadath_frontera_amd import programs
from kadath_frontera_amd.xcts import XctsSystem

pytestmark = pytest.mark.gpu

BOUNDS = [1.0, 2.0, 4.0, 8.0]


def _flat(sd, order, batch):
    nd = len(sd.bounds)
    radius = {d: sd.coloc(d)[0] for d in range(1, nd + 1)}
    s = sd.build(order=order, batch=batch)
    for d, r in radius.items():
        s.set_field("P", d, 1.0 + 1.0 / r)
        s.set_field("N", d, np.ones_like(r))
        for f in ("bet^x", "bet^y", "bet^z"):
            s.set_field(f, d, np.zeros_like(r))
    s.add_unknowns(s.perturbation(3))
    return s


@pytest.mark.parametrize("res,nd,order,spin", [((5, 5, 4), 2, 0, None), ((9, 7, 4), 3, 1, None),
                                               ((13, 6, 8), 2, 1, None), ((17, 9, 4), 2, 0, None),
                                               ((7, 7, 4), 2, 1, 0.1)])
def test_levels_give_the_instructions_results(ctx, res, nd, order, spin):
    s = _flat(programs.kerr(ctx, res, BOUNDS[:nd], n0=0.5, a=1.0, ome=0.05, spin=spin), order, 64)
    w = torch.tensor(np.random.default_rng(1).standard_normal(s.m), device="cuda")
    lo, cnt = s.n // 3 + 1, s.n // 2
    got = {}
    for fuse in (False, True):
        s.set_option(fuse=fuse)
        got[fuse] = [s.residual(), s.jacobian(), s.jvp_fill(lo, cnt, dtype=torch.float32), s.jvp_fill(s.n - 1, 1),
                     s.vjp(w)]
    for a, b in zip(got[False], got[True]):
        assert torch.equal(a, b)
    # J^T w against the columns' own products, in fp64 on the host
    J, v = got[True][1].cpu().numpy(), got[True][4].cpu().numpy()
    ref = J.T @ w.cpu().numpy()
    assert np.abs(v - ref).max() <= 1e-12 * np.abs(J).sum(axis=0).max() * np.abs(w.cpu().numpy()).max()
    s.close()


def test_traced_system_levels(ctx):
    s = XctsSystem(ctx, (8, 5, 8), BOUNDS[:3], n0=0.5, a=1.0, ome=0.05, batch=32, order=1)
    s.set_guess(s.perturbation(5))
    got = {}
    for fuse in (False, True):
        s.set_option(fuse=fuse)
        got[fuse] = (s.residual(), s.jacobian())
    assert torch.equal(got[False][0], got[True][0]) and torch.equal(got[False][1], got[True][1])
    s.close()


@pytest.mark.parametrize("nd,batch,spin", [(7, 3, None), (2, 16, None), (2, 1, None), (2, 7, 0.1)])
def test_columns_in_several_rounds(ctx, nd, batch, spin):
    """Few columns of a program at a time: programs split over many rounds that the arena's
    room ends (2 domains, 10 programs) or the 32 programs of a launch (7 domains, 35),
    column ranges that start and end inside a program and a split."""
    bounds = [2.0 ** q for q in range(nd)]
    got = {}
    for b in (512, batch):  # the reference: one instruction per launch, whole programs
        s = _flat(programs.kerr(ctx, (5, 5, 4), bounds, n0=0.5, a=1.0, ome=0.05, spin=spin), 1, b)
        s.set_option(fuse=b == batch)
        w = torch.tensor(np.random.default_rng(2).standard_normal(s.m), device="cuda")
        lo, cnt = s.n // 5 + 1, s.n // 2 + 1
        got[b] = [s.jvp_fill(0, s.n), s.jvp_fill(lo, cnt, dtype=torch.float32), s.vjp(w)]
        s.close()
    for a, b in zip(got[512], got[batch]):
        assert torch.equal(a, b)
    assert torch.equal(got[batch][0][:, lo:lo + cnt].float(), got[batch][1])


def _taken(f):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


def test_batch_bounds_the_arena(ctx):
    """J^T w forms no matrix: what it takes is the tangent arena, `batch` columns of every
    program at most."""
    taken = {}
    for batch in (4096, 8):  # (the first call also loads the kernels)
        s = _flat(programs.kerr(ctx, (9, 7, 4), BOUNDS[:3], n0=0.5, a=1.0, ome=0.05), 1, batch)
        w = torch.ones(s.m, dtype=torch.float64, device="cuda")
        s.residual()
        if batch == 4096:  # a few columns fit the set-up's arena
            s.set_option(fuse=False)
            s.jvp_fill(3, 5)
            s.set_option(fuse=True)
            assert _taken(lambda: s.jvp_fill(3, 5)) == 0
        taken[batch] = _taken(lambda: s.vjp(w))
        s.close()
    print(f"arena {taken}", flush=True)
    assert 0 < taken[8] < taken[4096] / 8  # programs of 130 to 230 columns: 16 times and more


def test_arena_leaves_room_on_the_card(ctx):
    """With some 2 GiB left on the card the arena takes at most half of them (all columns at
    once would take 6), and the columns go through it in more rounds with the same results."""
    s = _flat(programs.kerr(ctx, (13, 9, 8), BOUNDS, n0=0.5, a=1.0, ome=0.05), 1, 256)
    w = torch.tensor(np.random.default_rng(3).standard_normal(s.m), device="cuda")
    s.set_option(fuse=False)
    ref = s.vjp(w).clone()
    s.set_option(fuse=True)
    torch.cuda.empty_cache()
    hold = torch.empty(torch.cuda.mem_get_info()[0] - (2 << 30), dtype=torch.uint8, device="cuda")
    try:
        free = torch.cuda.mem_get_info()[0]
        taken = _taken(lambda: s.vjp(w))
        print(f"free {free} taken {taken}", flush=True)
        assert 0 < taken <= free // 2
        assert torch.equal(s.vjp(w), ref)
    finally:
        del hold
        s.close()
        torch.cuda.empty_cache()


def test_arrays_beyond_lds_build_and_refuse_to_run(ctx):
    """Domain arrays whose transforms need more LDS than a workgroup has: the system is built
    (its layout and coefficients are there), what would run a transform is refused."""
    s = XctsSystem(ctx, (33, 17, 16), BOUNDS[:2], n0=0.5, a=1.0, ome=0.05, batch=4, order=1)
    assert s.n == s.m and sum(q[3] for q in s.layout) == s.n
    cf = s.coef(0, 1)
    cf[0, 0, 0] = 1.25
    s.set_coef(0, 1, cf)
    assert s.coef(0, 1)[0, 0, 0] == 1.25
    for f in (s.residual, lambda: s.do_newton(1e-10, "f64-dd")):
        with pytest.raises(RuntimeError):
            f()
    s.close()
