"""GPU: tiles whose source box does not fit in LDS (strong shear), which the staged kernels read
per lane: results bit for bit those of per-lane loads, over inputs where all tiles fit, none, or
some (counted here from the positions and the kernels' limits), and no slower than them.

Margin of the timing: the kernel of per-lane loads is 1.5 times as slow on this input as the
staged one with its waves in step, 0.85 times with its waves on their own; the line is 1.1."""
import numpy as np
import pytest

from test_gpu_boxes import MH, _run, _setup

pytestmark = pytest.mark.gpu
COLS = {4: 96, 8: 80, 2: 128}


def _rows(size, ref, post):
    return 62 if size == 8 else 85 if size == 2 or (ref and post) else 64


def _fits(xyz, ni, nj, nk, size, ref, post):
    """Tiles of 64 x 4 targets x 2 levels that surely fit, and that surely do not (planes of a
    stencil: four, two next to the first and last level; one column more for 2-byte elements)."""
    p = np.floor(xyz.double().cpu().numpy().reshape(nk, nj, ni, 3))
    yes = no = 0
    for k in range(0, nk, 2):
        for j in range(0, nj, 4):
            for i in range(0, ni, 64):
                t = p[k:k + 2, j:j + 4, i:i + 64].reshape(-1, 3)
                t = t[np.isfinite(t).all(1) & (np.abs(t) < 1e6).all(1)]
                if not len(t):
                    continue
                e = t.max(0) - t.min(0)
                rows, cols = _rows(size, ref, post), COLS[size]
                yes += e[0] + 4 + (size == 2) <= cols and (e[1] + 4) * (e[2] + 4) <= rows
                no += e[0] + 4 > cols or (e[1] + 4) * (e[2] + 2) > rows
    return yes, no


@pytest.mark.parametrize("kind", ["f32_f32", "f32_ref", "f64_ref", "bf16_f32"])
@pytest.mark.parametrize("post", [0, 1, 3])
@pytest.mark.parametrize("deform,special,share", [(0.3, False, "all"), (3.0, True, "some"), (12.0, True, "none")])
def test_unstaged_equals_per_lane(cuda, deform, special, share, post, kind):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    field, arith = kind.split("_")
    fdt = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}[field]
    ref = arith == "ref"
    ni, nj, nk, nf = 131, 42, 9, 3
    print(f"[unstaged] {kind} post={post} deform={deform}", flush=True)
    s = _setup(torch, A, L, ni, nj, nk, 5, fdt, torch.float32, nf, True, 77, deform, special)
    yes, no = _fits(s[2], ni, nj, nk, src_size(fdt, torch), ref, post)
    assert (no == 0 and yes > 0, yes > 0 and no > 0, no > 0 and yes == 0)[("all", "some", "none").index(share)], (yes, no)
    math = L.ADZ_MATH_REF if ref else L.ADZ_MATH_F32
    want = _run(torch, A, L, s, fdt, math, post, True, ni, nj, nk, 2)
    for stage in ("call", None, 7):
        got = _run(torch, A, L, s, fdt, math, post, True, ni, nj, nk, stage)
        for q, (a, b) in enumerate(zip(got, want)):
            same = (a == b) | (np.isnan(a) & np.isnan(b))  # (NaN, and zeros of either sign, compare as equal)
            assert same.all(), (stage, q, int((~same).sum()))


def src_size(fdt, torch):
    return torch.empty(0, dtype=fdt).element_size()


def test_sheared_call_no_slower_than_per_lane_loads(cuda):
    import math

    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A
    from gem_amd import tricublin as TC

    ni, nj, nk, nf = 512, 384, 60, 4
    nx, ny = ni + 2 * MH, nj + 2 * MH
    geom = TC.Ztab(np.arange(nk) + 1.0, nx, ny).set_bounds(1 - MH, ni + MH, 1 - MH, nj + MH)
    k, j, i = torch.meshgrid(*(torch.arange(1, n + 1, device="cuda", dtype=torch.float64) for n in (nk, nj, ni)), indexing="ij")
    pos = torch.stack([(i + 6 * torch.sin(2 * math.pi * j / 64)).clamp(1.01, ni - 0.01),
                       (j + 6 * torch.sin(2 * math.pi * i / 64)).clamp(1.01, nj - 0.01),
                       (k + 1.5 * torch.sin(2 * math.pi * (i + j) / 48)).clamp(0.6, nk + 0.4)], -1).float().reshape(-1)
    gen = torch.Generator(device="cuda").manual_seed(3)
    n = nx * ny * nk
    stack = [dict(src=torch.rand(n, generator=gen, device="cuda"), dst=torch.zeros(n, device="cuda")) for _ in range(nf)]
    box, lay, off = (1, ni, 1, nj, 1, nk), (1 - MH, ni + MH, 1 - MH, nj + MH), MH + nx * MH
    item = dict(geom=geom.h, xyz=pos, box=box, dlayout=lay, ext=False, fields=A.field_list(stack, off, off))
    plan = A.Plan([item], L.ADZ_F32, tune=dict(fields_per_pass=nf, points_outer=0, blocks_per_cu=4, xcd_chunks=1, stage=2,
                                               level_inner=3))

    def call():
        A.adz_tricub_hlt(stack, pos, geom.h, *box[:5], box[5], lay, ext=False, post=0, math=L.ADZ_MATH_F32, src_off=off)

    def ms(fn):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = 1e9
        for _ in range(5):
            a.record()
            for _ in range(5):
                fn()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best / 5

    t = ms(call), ms(plan.execute)
    plan.free()
    print(f"[unstaged] sheared call {t[0]:.3f} ms, per-lane loads {t[1]:.3f} ms", flush=True)
    assert t[0] < 1.1 * t[1], t
