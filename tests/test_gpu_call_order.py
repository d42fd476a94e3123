"""GPU: adz_tricub_hlt on boxes on either side of the size from which the staged kernel walks
super-columns of three tile rows (planes of 16 MB): bit for bit what per-lane loads give, with a
number of tile rows that three does not divide."""
import numpy as np
import pytest

from test_gpu_boxes import _run, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nf", [("f32_f32", 3), ("f32_ref", 3), ("f64_ref", 2), ("bf16_f32", 7)])
@pytest.mark.parametrize("post", [0, 2])
@pytest.mark.parametrize("ni,nj", [(449, 434), (449, 280)])
def test_call_equals_per_lane(cuda, ni, nj, post, kind, nf):
    import torch

    from gem_amd import _lib as L
    from gem_amd import adz as A

    field, arith = kind.split("_")
    fdt = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}[field]
    size = torch.empty(0, dtype=fdt).element_size()
    assert (ni * nj * 8 * nf * size > 16 << 20) == (nj == 434) and -(-nj // 4) % 3
    math = L.ADZ_MATH_REF if arith == "ref" else L.ADZ_MATH_F32
    nk = 7
    print(f"[call order] {kind} {ni}x{nj}x{nk} nf={nf} post={post}", flush=True)
    s = _setup(torch, A, L, ni, nj, nk, 5, fdt, torch.float32, nf, True, nj, 1.0, True)
    want = _run(torch, A, L, s, fdt, math, post, True, ni, nj, nk, 2)
    got = _run(torch, A, L, s, fdt, math, post, True, ni, nj, nk, "call")
    for q, (a, b) in enumerate(zip(got, want)):
        same = (a == b) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (q, int((~same).sum()))
