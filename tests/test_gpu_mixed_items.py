"""GPU: a plan with one item beyond 32-bit byte offsets among ordinary ones stages the ordinary
ones' boxes (the built-in stage is 7, not 2), and gives what per-lane loads give, bit for bit.
A plan of such items alone keeps per-lane loads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_one_large_item_leaves_the_others_staged(cuda):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A
    from gem_amd import tricublin as TC

    big, nk, ni, nj, nf = 2600, 84, 70, 21, 3  # a source of 2600 x 2600 x 84 FP32 values: 2.3 GB
    gen = torch.Generator(device="cuda").manual_seed(5)
    items, outs = [], []
    for n, m, at in ((ni + 8, nj + 8, 4.0), (big, big, 2300.0), (ni + 31, nj + 10, 4.0)):
        geom = TC.Ztab(np.arange(nk) + 1.0, n, m).set_bounds(1, n, 1, m)
        src = [torch.rand(n * m * nk, generator=gen, device="cuda")] * nf if n == big else [
            torch.rand(n * m * nk, generator=gen, device="cuda") for _ in range(nf)]
        pos = torch.rand(nk, nj, ni, 3, generator=gen, device="cuda") * 2 - 1
        pos[..., 0] += torch.arange(ni, device="cuda") + at
        pos[..., 1] += torch.arange(nj, device="cuda").view(1, nj, 1) + at
        pos[..., 2] += torch.arange(1, nk + 1, device="cuda").view(nk, 1, 1)
        pos[..., 2].clamp_(0.6, nk + 0.4)
        pos[0, 0, 0, 0] = float("nan")
        out = [torch.full((ni * nj * nk,), 7.0, device="cuda") for _ in range(nf)]
        items.append(dict(geom=geom.h, xyz=pos.reshape(-1), box=(1, ni, 1, nj, 1, nk), dlayout=(1, ni, 1, nj), ext=True,
                          fields=A.field_list([dict(src=s, dst=d) for s, d in zip(src, out)], 0, 0), keep=(geom, src)))
        outs.append(out)

    def run(stage, which):
        tune = stage and dict(fields_per_pass=nf, points_outer=0, blocks_per_cu=4, xcd_chunks=1, stage=stage, level_inner=3)
        p = A.Plan([items[q] for q in which], L.ADZ_F32, math=L.ADZ_MATH_F32, tune=tune)
        got = p.tune()["stage"]
        p.execute()
        torch.cuda.synchronize()
        p.free()
        return got, [o.clone() for q in which for o in outs[q]]

    print("[mixed] per-lane loads", flush=True)
    _, want = run(2, (0, 1, 2))
    print("[mixed] built-in", flush=True)
    stage, got = run(None, (0, 1, 2))
    assert stage == 7
    for q, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(torch.nan_to_num(a, nan=-1.0), torch.nan_to_num(b, nan=-1.0)), q
    print("[mixed] the large one alone", flush=True)
    assert run(None, (1,))[0] == 2
