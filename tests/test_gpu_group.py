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
