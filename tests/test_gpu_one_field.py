"""GPU: one field alone is read per lane or from staged boxes by its type, arithmetic and outputs and
the number of targets; the built-in tile parameters of a plan say which, and where one field is
staged it gives what per-lane loads give, bit for bit (row lengths on either side of a tile)."""
import numpy as np
import pytest

from test_gpu_boxes import _run, _setup

pytestmark = pytest.mark.gpu
MANY, FEW = (520, 400, 84), (300, 200, 60)  # 17.5 and 3.6 million targets


@pytest.mark.parametrize("field,arith,post,size,stage", [
    ("f32", "f32", 0, MANY, 2), ("f32", "f32", 2, MANY, 2), ("f32", "f32", 1, MANY, 7), ("f32", "f32", 3, FEW, 2),
    ("f32", "ref", 0, MANY, 2), ("f32", "ref", 1, MANY, 2), ("f64", "ref", 0, MANY, 7), ("f64", "ref", 0, FEW, 2),
    ("f64", "ref", 1, FEW, 7), ("f64", "ref", 2, MANY, 2), ("bf16", "f32", 0, FEW, 7), ("bf16", "f32", 2, FEW, 7),
])
def test_built_in_stage(cuda, field, arith, post, size, stage):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A
    from gem_amd import tricublin as TC

    ni, nj, nk = size
    fdt = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}[field]
    geom = TC.Ztab(np.arange(nk) + 1.0, ni, nj).set_bounds(1, ni, 1, nj)
    x = torch.zeros(8, dtype=fdt, device="cuda")  # the plan is made, not executed
    pos = torch.zeros(24, device="cuda")
    item = dict(geom=geom.h, xyz=pos, box=(1, ni, 1, nj, 1, nk), dlayout=(1, ni, 1, nj), ext=False,
                fields=A.field_list([dict(src=x, dst=x, lin=x, min=x, max=x)], 0, 0))
    p = A.Plan([item], {"f32": L.ADZ_F32, "f64": L.ADZ_F64, "bf16": L.ADZ_BF16}[field],
               math=L.ADZ_MATH_REF if arith == "ref" else L.ADZ_MATH_F32, post=post)
    got = p.tune()["stage"]
    p.free()
    assert got == stage


@pytest.mark.parametrize("arith,post", [("f32", 1), ("f32", 3), ("ref", 0)])
def test_one_staged_field_equals_per_lane(cuda, arith, post):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    ni, nj, nk = 449, 410, 46  # 8.47 million targets, a little over 2^23
    math = L.ADZ_MATH_REF if arith == "ref" else L.ADZ_MATH_F32
    print(f"[one field] {arith} post={post}", flush=True)
    s = _setup(torch, A, L, ni, nj, nk, 5, torch.float32, torch.float32, 1, True, 9, 1.0, True)
    want = _run(torch, A, L, s, torch.float32, math, post, True, ni, nj, nk, 2)
    got = _run(torch, A, L, s, torch.float32, math, post, True, ni, nj, nk, "call")
    for q, (a, b) in enumerate(zip(got, want)):
        same = (a == b) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (q, int((~same).sum()))
