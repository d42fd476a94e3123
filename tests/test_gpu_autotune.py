"""GPU: adz_plan_autotune leaves blocks_per_cu at its built-in 8 for the stagings that launch a block
per tile and do not use it (timing such candidates would find noise), and its tiles give what
per-lane loads give, bit for bit."""
import numpy as np
import pytest

from test_gpu_boxes import MH, _run, _setup

pytestmark = pytest.mark.gpu


def test_autotune_block_per_tile(cuda):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    ni, nj, nk, nf = 259, 150, 24, 6
    s = _setup(torch, A, L, ni, nj, nk, 5, torch.float32, torch.float32, nf, True, 3, 0.5, False)
    geom, box, xyz, src, soff = s
    n = (ni + 2 * MH) * (nj + 2 * MH) * nk
    stack = [dict(src=f, dst=torch.zeros(n, device="cuda")) for f in src]
    item = dict(geom=geom.h, xyz=xyz, box=box, dlayout=(1 - MH, ni + MH, 1 - MH, nj + MH), ext=True,
                fields=A.field_list(stack, soff, MH + (ni + 2 * MH) * MH))
    tune, ms = A.Plan.autotune([item], L.ADZ_F32, reps=2)
    print(f"[autotune] {tune} {ms:.3f} ms", flush=True)
    if tune["stage"] in (5, 6, 7):
        assert tune["blocks_per_cu"] == 8
    p = A.Plan([item], L.ADZ_F32, tune=tune)
    p.execute()
    torch.cuda.synchronize()
    p.free()
    want = _run(torch, A, L, s, torch.float32, L.ADZ_MATH_F32, 0, True, ni, nj, nk, 2)
    for e, w in zip(stack, want[::4]):
        got, inside = e["dst"].cpu().numpy(), w != 7.0
        assert np.array_equal(got[inside], w[inside])
