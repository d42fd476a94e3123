"""GPU: ILMC where many windows can be visited at a time: the number of waves follows from the
windows found, not from the number of tracers.  Bit for bit against the oracle's sequential loop
where the rule gives the fewest waves, some and all of them, and the time of one tracer with
violations everywhere against that of four.

Margin of the timing: with waves by the number of tracers one took 0.67 of the time of four; now a
third.  The line is 0.5."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_ilmc_order import MH, _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk,S,autobar,dense", [
    (40, 30, 12, 2, False, 0.1),   # fewest
    (96, 64, 24, 2, False, 1.0),   # 3 x 90 windows
    (128, 48, 16, 1, True, 1.0), (100, 90, 20, 1, False, 1.0),  # all
])
def test_dense_bit_exact(cuda, ni, nj, nk, S, autobar, dense):
    import torch

    from gem_amd import adz as A

    print(f"[ilmc dense] {ni}x{nj}x{nk} S={S} autobar={autobar} dense={dense}", flush=True)
    layout, trs, air, off = _case(ni, nj, nk, 1, ni + S, dense)
    box = (1, ni, 1, nj, 1)
    f, mn, mx = trs[0]
    dev = dict(f=torch.from_numpy(f.copy()).cuda(), min=torch.from_numpy(mn).cuda(), max=torch.from_numpy(mx).cuda())
    il = A.IlmcLam([dev], layout, box, off, sweep_max=S, min_max=True, autobar=autobar)
    counts = torch.zeros(3, dtype=torch.int64, device="cuda")
    il(torch.from_numpy(air).cuda(), counts)
    torch.cuda.synchronize()
    il.free()
    exp = f.copy()
    c = O.ilmc(exp, mn, mx, air, layout, box, sweep_max=S, min_max=True, autobar=autobar)
    got = dev["f"].cpu().numpy()
    assert np.array_equal(got.view(np.uint32), exp.view(np.uint32)), int(np.count_nonzero(got != exp))
    assert counts.cpu().tolist() == c.tolist()


def test_one_dense_tracer_takes_a_share_of_four(cuda):
    import torch

    from gem_amd import adz as A

    ni, nj, nk = 256, 192, 40
    n = (ni + 2 * MH) * (nj + 2 * MH) * nk
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda: torch.rand(n, generator=gen, device="cuda")  # noqa: E731
    trs = []
    for _ in range(4):
        src = torch.exp(rand() * 2 - 1)
        f = torch.where(rand() < 0.3, src * (0.4 + 1.2 * rand()), src)
        trs.append(dict(f=f.clone(), min=src * (0.7 + 0.3 * rand()), max=src * (1 + 0.3 * rand()), start=f))
    air = 0.5 + 1.5 * rand()

    def ms(m):
        il = A.IlmcLam([{k: t[k] for k in ("f", "min", "max")} for t in trs[:m]],
                       (1 - MH, ni + MH, 1 - MH, nj + MH, nk), (1, ni, 1, nj, 1), MH + (ni + 2 * MH) * MH, sweep_max=2,
                       min_max=True)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = 1e9
        for _ in range(4):
            for t in trs[:m]:
                t["f"].copy_(t["start"])
            a.record()
            il(air)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        il.free()
        return best

    t = ms(1), ms(4)
    print(f"[ilmc dense] one tracer {t[0]:.2f} ms, four {t[1]:.2f} ms", flush=True)
    assert t[0] < 0.5 * t[1], t
