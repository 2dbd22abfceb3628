"""The far fill against m25x_far_block (one thread an entry, every kernel value of its own), bit for bit on and above the
diagonal: edges in the mesh's order (their tiles' triangles fit the LDS and are evaluated once) and in a random one
(they don't), at sizes with a partial last tile and below one tile."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', [torch.complex128, torch.complex64])
@pytest.mark.parametrize('order', ['mesh', 'random'])
def test_fill_far_is_far_block(gpu, order, dt):
    from mom25d_amd import boards
    from mom25d_amd.sim import Simulation
    dv, w = gpu, 2 * np.pi * 2.3e9
    st, shapes, ports, vias, kw = boards.seeded_board(dmax=3e-3, ncross=2)
    sim = Simulation(st, shapes, ports, vias, verbose=False, **kw)
    sim.fast.setup(2.3e9)
    rng = np.random.default_rng(4)
    for Ne in (1, 31, 64, 200, sim.Ne):
        pick = np.arange(Ne) if order == 'mesh' else rng.permutation(sim.Ne)[:Ne]
        g = {k: (v[pick] if k in ('ep', 'em', 'ap', 'am', 'vp', 'vm') else v) for k, v in sim.g.items()}
        if order == 'random' and Ne >= 64:                       # the case that the LDS cannot hold is there
            u = [len(np.unique(np.r_[g['ep'][a:a + 32], g['em'][a:a + 32]])) for a in (0, 32)]
            assert u[0] * u[1] > 1296
        mesh = dv.DevMesh(g)
        Z = torch.zeros((Ne, Ne), dtype=dt, device=dv.device())
        dv.fill_far(Z, mesh, sim.fast.tabs, w)
        idx = np.arange(Ne)
        want = dv.far_block(idx, idx, mesh, sim.fast.tabs, w).to(dt)
        m, n = torch.triu_indices(Ne, Ne, device=Z.device)
        assert torch.equal(Z[m, n], want[m, n]), Ne
        assert torch.equal(Z, Z.T), Ne


def test_near_moments_with_kept_parts(gpu):
    """The pairs' moments with the extracted parts kept (computed at the first call, read at the next) and without a
    store for them: the same bits, whichever way the parts come; and a store is filled again when they change."""
    from mom25d_amd import boards
    from mom25d_amd.sim import Simulation
    dv, w = gpu, 2 * np.pi * 2.3e9
    for board in (boards.microstrip, boards.seeded_board):
        st, shapes, ports, vias, kw = board(dmax=3e-3, ncross=2)
        sim = Simulation(st, shapes, ports, vias, verbose=False, **kw)
        fo = sim.fast
        fo.setup(2.3e9)
        want = dv.near_moments(fo.mesh, fo.tabs, fo.plan, w, stat=False)
        for kept in (False, True, True):
            assert fo.plan.stat_ready == kept
            for a, b in zip(dv.near_moments(fo.mesh, fo.tabs, fo.plan, w), want):
                assert torch.equal(torch.view_as_real(a), torch.view_as_real(b)), (board.__name__, kept)
        fo.plan.stat.fill_(float('nan'))
        fo.plan.stat_kind = None
        for a, b in zip(dv.near_moments(fo.mesh, fo.tabs, fo.plan, w), want):
            assert torch.equal(torch.view_as_real(a), torch.view_as_real(b)), board.__name__
