"""GPU: the trajectory from wind boxes staged in LDS, on tiles cut short in i, j and k: smooth
winds (one box for all iterations), winds that differ from point to point (a new box in every
iteration) and winds too ragged for any box (per-lane reads), against the oracle, bit for bit:
the arithmetic and its order do not depend on where the winds are read from."""
import numpy as np
import pytest

from gem_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = {
    # ni, nj, nk, halo, Courant number, ragged
    "odd_smooth": (71, 45, 13, 5, 2.0, 0.0), "odd_rough": (69, 51, 9, 4, 2.0, 1.0),
    "wide_wild": (130, 49, 12, 5, 20.0, 2.0), "short": (64, 47, 4, 4, 1.0, 0.3),
}


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("case", list(CASES))
def test_traject_boxes_bit_exact(cuda, case, storage):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    ni, nj, nk, halo, courant, ragged = CASES[case]
    cfg = S.Config("t", ni, nj, nk, halo, 300.0, jets=True, cmax_xy=courant, cmax_z=1.0, seed=ni + nk)
    g = S.grid_desc(cfg)
    G = O.Grid(g)
    rng = np.random.default_rng(nj)
    w = {k: v * torch.from_numpy(1.0 + ragged * rng.uniform(-1, 1, tuple(v.shape))).to(v.dtype)
         for k, v in S.winds(cfg, g).items()}
    wd = {k: v.cuda() for k, v in w.items()}
    ctx = A.AdzContext(g, L.ADZ_F32 if storage == "f32" else L.ADZ_F64)
    names = [("pxyzm", A.ADZ_A_PXYZM), ("uvw_dep", A.ADZ_A_UVW_DEP), ("pm", A.ADZ_A_PM), ("pmu", A.ADZ_A_PMU),
             ("pmv", A.ADZ_A_PMV), ("pt", A.ADZ_A_PT), ("pb", A.ADZ_A_PB)]
    ctx.adz_inittraj()
    state = None
    for step in range(2):
        print(f"[traj] {case} {storage} step {step}", flush=True)
        ctx.adz_traject(cfg.dt, wd["uu_ext"], wd["vv_ext"], wd["ww_ext"], wd["ut0"], wd["vt0"], wd["zdt0"])
        torch.cuda.synchronize()
        ref = G.traject({k: v.numpy() for k, v in w.items()}, cfg.dt, storage=storage, state=state, niter=cfg.niter)
        for name, which in names:
            got, exp = ctx.array(which).cpu().numpy(), ref[name]
            assert got.shape == exp.shape, name
            same = (got == exp) | (np.isnan(got) & np.isnan(exp))
            assert same.all(), (step, name, int((~same).sum()), got.size)
        state = dict(pxyzm=ref["pxyzm"], wpxyz=ref["wpxyz"])
    ctx.free()
