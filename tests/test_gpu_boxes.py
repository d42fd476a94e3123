"""GPU: the LDS-staged interpolation kernels against per-lane loads, bit for bit, where the
staged box can go wrong: rows of every length modulo 4 elements, tiles cut short in i, j and k,
one to three fields (the double buffer's ends), boxes too large to stage (strong
deformation), stencils at the first and last element of the source, positions out of range,
and infinities and NaN in the sources.

Both forms run the same operations in the same order, so the comparison is exact (NaN where
NaN).  The per-lane form is pinned to the oracle in test_gpu_hlt.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MH = 2


def _setup(torch, A, L, ni, nj, nk, halo, fdt, pdt, nf, ext, seed, deform, special, lead=0):
    from gem_amd import tricublin as TC

    H = halo if ext else MH
    nx, ny = ni + 2 * H, nj + 2 * H
    rng = np.random.default_rng(seed)
    geom = TC.Ztab(np.cumsum(rng.uniform(0.5, 1.5, nk)), nx, ny).set_bounds(1 - H, ni + H, 1 - H, nj + H)
    box = (1, ni, 1, nj, 1, nk)
    i, j, k = np.meshgrid(np.arange(1, ni + 1), np.arange(1, nj + 1), np.arange(1, nk + 1), indexing="ij")
    pos = np.stack([i, j, k], -1).astype(np.float64).transpose(2, 1, 0, 3)  # (k, j, i, 3)
    ph = rng.uniform(0, 6, 3)
    pos[..., 0] += deform * np.sin(pos[..., 1] * 0.7 + ph[0]) + rng.uniform(-0.4, 0.4, pos.shape[:3])
    pos[..., 1] += deform * np.sin(pos[..., 0] * 0.9 + ph[1]) + rng.uniform(-0.4, 0.4, pos.shape[:3])
    pos[..., 2] += 1.5 * np.sin(pos[..., 0] * 0.3 + ph[2]) + rng.uniform(-0.4, 0.4, pos.shape[:3])
    lo, hix, hiy = 2.0 - H, ni + H - 2.0 + 0.999, nj + H - 2.0 + 0.999  # first and last stencil of the source
    pos[..., 0] = np.clip(pos[..., 0], lo, hix)
    pos[..., 1] = np.clip(pos[..., 1], lo, hiy)
    if special:
        pos[0, 0, 0] = (1.0e12, 1.0, 1.0)
        pos[-1, -1, -1] = (np.nan, 2.0, 2.0)
        pos[0, -1, 0] = (lo - 1.5, 2.0, 2.0)
    xyz = torch.from_numpy(np.ascontiguousarray(pos)).to(pdt).cuda().reshape(-1)
    src = []
    for _ in range(nf):
        f = rng.lognormal(0.0, 1.0, nx * ny * nk)
        if special:
            f[rng.integers(0, f.size, 5)] = np.inf
            f[rng.integers(0, f.size, 5)] = np.nan
            f[rng.integers(0, f.size, 200)] = -0.0
        first = lead * (len(src) % 2)  # element its first value is at, in an allocation of its own
        src.append(torch.cat([torch.zeros(first, dtype=fdt), torch.from_numpy(f).to(fdt)]).cuda()[first:])
    return geom, box, xyz, src, H + nx * H


def _run(torch, A, L, s, fdt, math, post, ext, ni, nj, nk, stage):
    geom, box, xyz, src, soff = s
    n = (ni + 2 * MH) * (nj + 2 * MH) * nk
    doff = MH + (ni + 2 * MH) * MH
    out = [{m: torch.full((n,), 7.0, dtype=fdt, device="cuda") for m in ("dst", "lin", "min", "max")} for _ in src]
    stack = [dict(src=f, **o) for f, o in zip(src, out)]
    lay = (1 - MH, ni + MH, 1 - MH, nj + MH)
    if stage == "call":
        A.adz_tricub_hlt(stack, xyz, geom.h, *box[:5], box[5], lay, ext=ext, post=post, math=math, src_off=soff)
    else:
        item = dict(geom=geom.h, xyz=xyz, box=box, dlayout=lay, ext=ext, fields=A.field_list(stack, soff, doff))
        tune = None if stage is None else dict(fields_per_pass=2, points_outer=1, blocks_per_cu=2, xcd_chunks=1,
                                               stage=stage, level_inner=2)
        p = A.Plan([item], {torch.float32: L.ADZ_F32, torch.float64: L.ADZ_F64, torch.bfloat16: L.ADZ_BF16}[fdt],
                   math=math, post=post, tune=tune)
        p.execute()
        torch.cuda.synchronize()
        p.free()
    torch.cuda.synchronize()
    return [t.float().cpu().numpy() if fdt == torch.bfloat16 else t.cpu().numpy() for o in out for t in o.values()]


CASES = [
    # ni, nj, nk, halo, nf, ext, deform, special
    (64, 20, 9, 4, 1, True, 1.0, False), (65, 33, 7, 5, 2, True, 2.0, True), (127, 26, 5, 4, 3, False, 1.5, False),
    (130, 28, 8, 5, 3, True, 0.5, True), (63, 24, 6, 5, 1, False, 9.0, False), (70, 40, 11, 4, 2, False, 4.0, True),
]


@pytest.mark.parametrize("math_ref", [True, False])
@pytest.mark.parametrize("post", [0, 1, 3])
@pytest.mark.parametrize("ni,nj,nk,halo,nf,ext,deform,special", CASES)
def test_staged_f32_equals_per_lane(cuda, ni, nj, nk, halo, nf, ext, deform, special, post, math_ref):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    math = L.ADZ_MATH_REF if math_ref else L.ADZ_MATH_F32
    pdt = torch.float32 if ni % 2 else torch.float64
    s = _setup(torch, A, L, ni, nj, nk, halo, torch.float32, pdt, nf, ext, ni + nk, deform, special)
    print(f"[boxes] {ni}x{nj}x{nk} nf={nf} ext={ext} deform={deform} post={post} ref={math_ref}", flush=True)
    want = _run(torch, A, L, s, torch.float32, math, post, ext, ni, nj, nk, 2)
    for stage in (5, 6, 7, None, "call") + (() if math_ref else (8,)):
        got = _run(torch, A, L, s, torch.float32, math, post, ext, ni, nj, nk, stage)
        for q, (a, b) in enumerate(zip(got, want)):
            same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))
            if not math_ref:  # minNum / maxNum do not tell +0 from -0
                same |= (a == 0) & (b == 0)
            assert same.all(), (stage, q, int((~same).sum()))


@pytest.mark.parametrize("post", [0, 1, 3])
@pytest.mark.parametrize("ni,nj,nk,halo,nf,ext,deform,special", CASES)
def test_staged_f64_equals_per_lane(cuda, ni, nj, nk, halo, nf, ext, deform, special, post):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    pdt = torch.float64 if ni % 2 else torch.float32
    s = _setup(torch, A, L, ni, nj, nk, halo, torch.float64, pdt, nf, ext, ni + nk, deform, special, lead=1)
    print(f"[boxes] f64 {ni}x{nj}x{nk} nf={nf} ext={ext} deform={deform} post={post}", flush=True)
    want = _run(torch, A, L, s, torch.float64, L.ADZ_MATH_REF, post, ext, ni, nj, nk, 2)
    for stage in (3, 4, 5, 6, 7, 8, None, "call"):
        got = _run(torch, A, L, s, torch.float64, L.ADZ_MATH_REF, post, ext, ni, nj, nk, stage)
        for q, (a, b) in enumerate(zip(got, want)):
            same = (a.view(np.uint64) == b.view(np.uint64)) | (np.isnan(a) & np.isnan(b))
            assert same.all(), (stage, q, int((~same).sum()))


@pytest.mark.parametrize("post", [0, 1, 3])
@pytest.mark.parametrize("lead", [0, 1])  # 1: every other field begins in the middle of a word
@pytest.mark.parametrize("ni,nj,nk,halo,nf,ext,deform,special", CASES)
def test_staged_bf16_equals_per_lane(cuda, ni, nj, nk, halo, nf, ext, deform, special, lead, post):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    pdt = torch.float32 if ni % 2 else torch.float64
    s = _setup(torch, A, L, ni, nj, nk, halo, torch.bfloat16, pdt, nf, ext, ni + nk, deform, special, lead=lead)
    print(f"[boxes] bf16 {ni}x{nj}x{nk} nf={nf} ext={ext} lead={lead} deform={deform} post={post}", flush=True)
    want = _run(torch, A, L, s, torch.bfloat16, L.ADZ_MATH_F32, post, ext, ni, nj, nk, 2)
    for stage in (3, 4, 5, 6, 7, 8, None, "call"):
        got = _run(torch, A, L, s, torch.bfloat16, L.ADZ_MATH_F32, post, ext, ni, nj, nk, stage)
        for q, (a, b) in enumerate(zip(got, want)):
            # minNum / maxNum do not tell +0 from -0
            same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b)) | ((a == 0) & (b == 0))
            assert same.all(), (stage, q, int((~same).sum()))


def test_more_blocks_than_a_row_of_the_grid(cuda):
    """One column of 4099 x 4101 targets: 2.1 M tiles, whose blocks take a second row of the
    grid; the call and the plan against per-lane loads."""
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A
    from gem_amd import tricublin as TC

    ni, nj, nk = 1, 4099, 4101
    nx, ny = ni + 2 * MH, nj + 2 * MH
    gen = torch.Generator(device="cuda").manual_seed(7)
    geom = TC.Ztab(np.arange(nk) + 1.0, nx, ny).set_bounds(1 - MH, ni + MH, 1 - MH, nj + MH)
    pos = torch.rand(nk, nj, ni, 3, generator=gen, device="cuda") * 0.9
    pos[..., 0] += 1.0
    pos[..., 1] += torch.arange(1, nj + 1, device="cuda").view(1, nj, 1)
    pos[..., 2] += torch.arange(1, nk + 1, device="cuda").view(nk, 1, 1)
    src = [torch.rand(nx * ny * nk, generator=gen, device="cuda") for _ in range(2)]
    s = (geom, (1, ni, 1, nj, 1, nk), pos.reshape(-1), src, MH + nx * MH)
    want = _run(torch, A, L, s, torch.float32, L.ADZ_MATH_F32, 0, False, ni, nj, nk, 2)
    for stage in ("call", None, 7):
        got = _run(torch, A, L, s, torch.float32, L.ADZ_MATH_F32, 0, False, ni, nj, nk, stage)
        for q, (a, b) in enumerate(zip(got, want)):
            same = (a.view(np.uint32) == b.view(np.uint32)) | ((a == 0) & (b == 0))
            assert same.all(), (stage, q, int((~same).sum()))
