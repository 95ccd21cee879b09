"""Steps on boxes whose sides fall beside the tiles, rows and blocks of the kernels.

A tile is 64, 32 or 16 cells wide, a region spans the whole width, a chunk of cells is shared by three
blocks (one face direction each) and by the three edge or face types of the staggered scheme: sides one
above and below those sizes, and the thinnest boxes the step takes.  Two steps of the fused path, of both
sides of its choice where the cell records are written, and of the reference-shaped and staggered
paths, from the oracle's state and noise.  All of them keep the oracle's operation order, so there is no
tolerance: the valid cells are equal or the test fails.
"""
import numpy as np
import pytest

from fhdex_amd import params as P
from tests.helpers import perturbed_stag_state, perturbed_state, valid

pytestmark = pytest.mark.gpu

BOXES = [(2, (65, 17, 4)), (2, (4, 5, 6)), (3, (15, 33, 7)), (4, (33, 70, 5)), (5, (5, 4, 67)), (6, (9, 5, 7)),
         (7, (6, 9, 5)), (8, (17, 6, 9))]
STAG_BOXES = [(2, (65, 5, 4)), (3, (9, 6, 4)), (4, (4, 33, 5)), (5, (6, 9, 4)), (6, (5, 7, 6)),
              (7, (4, 6, 9)), (8, (17, 4, 6))]


def config(ns, shape):
    return P.argon_gas(0, shape=shape) if ns == 2 else P.species_prefix(ns, 0, 1, shape=shape)


@pytest.mark.parametrize("ns,shape", BOXES)
def test_collocated_steps(orc, ns, shape):
    import torch
    from fhdex_amd import compressible as fc
    from fhdex_amd import lib as L
    cfg = config(ns, shape)
    p = cfg.params
    print(f"case ragged step {ns} species {shape}", flush=True)
    st = perturbed_state(p, cfg, orc, seed=4, amp=0.02, vel=400.0)
    start, start_prim = (torch.from_numpy(a.copy()).cuda() for a in (st.cu, st.prim))
    ctx = L.Context(p)
    nz = fc.NoiseSets(p)
    for step in range(2):
        fc.fill_noise(ctx, nz, 9, step)
        for d in range(3):
            st.sA[d][...] = nz.A[d].t.cpu().numpy()
            st.sB[d][...] = nz.B[d].t.cpu().numpy()
        st.rA[...] = nz.rA.t.cpu().numpy()
        st.rB[...] = nz.rB.t.cpu().numpy()
        assert orc.rk3_step(p, st, cfg.dt) == 0
    default = ctx.get_tune()
    for rec in (0, 1):
        ctx.set_tune(default.tile_width, default.region_tiles, default.z_levels, default.noise_inline,
                     default.face_blocks_per_cu, rec)
        cu = fc.MultiFab(start.clone(), (-p.ngc,) * 3)
        prim = fc.MultiFab.cell(p, p.nprimvars)
        for step in range(2):
            fc.rk3_step(ctx, cu, prim, cfg.dt, 9, step)
        assert np.array_equal(valid(p, cu.t.cpu().numpy()), valid(p, st.cu)), f"fused cu, records {rec}"
        assert np.array_equal(valid(p, prim.t.cpu().numpy()), valid(p, st.prim)), f"fused prim, records {rec}"
    ds = fc.DeviceState(p)
    ds.cu.t.copy_(start)
    ds.prim.t.copy_(start_prim)
    for step in range(2):
        fc.RK3step(ctx, ds, cfg.dt, noise=None, seed=9, step=step)
    ctx.check()
    assert np.array_equal(valid(p, ds.cu.t.cpu().numpy()), valid(p, st.cu)), "reference-shaped cu"
    assert np.array_equal(valid(p, ds.prim.t.cpu().numpy()), valid(p, st.prim)), "reference-shaped prim"


@pytest.mark.parametrize("ns,shape", STAG_BOXES)
def test_staggered_steps(orc, ns, shape):
    import torch
    from fhdex_amd import lib as L
    from fhdex_amd import stag as S
    cfg = config(ns, shape)
    p = cfg.params
    print(f"case ragged staggered step {ns} species {shape}", flush=True)
    host = perturbed_stag_state(p, cfg, orc, seed=3, amp=0.03, vel=5e3)
    st = S.StagState(p)
    for dev, src in [(st.cu, host.cu), (st.prim, host.prim), *zip(st.cumom, host.mom), *zip(st.vel, host.vel)]:
        dev.t.copy_(torch.from_numpy(src))
    ctx = L.Context(p)
    for step in range(2):
        S.RK3stepStag(ctx, st, cfg.dt, 9, step)
    ctx.check()
    assert host.advance(2, cfg.dt, 9, 0) == 0
    for dev, src in [(st.cu, host.cu), (st.prim, host.prim), *zip(st.cumom, host.mom), *zip(st.vel, host.vel)]:
        assert np.array_equal(dev.t.cpu().numpy(), src)
