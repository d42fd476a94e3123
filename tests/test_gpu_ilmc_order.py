"""The order of ILMC's visits (adz_ilmc.hip): windows of 4 cells of a row, listed by
t = wi + a dj + b dk with d = ceil(2S / 4), a = d + 1, b = d + 2S a + 1 (b = 0 with
Schm_autobar_L), each waiting for the earlier ones within reach.

CPU: a cell that the sequential (k, j, i) loop visits earlier and that lies within distance 2S
is in the same window or in one with smaller t, over every offset and place in a window.
GPU: bit for bit against the oracle's sequential loop, with the counts, for rows that end on
either side of a window or of a 64-cell word, with waits that give up at once (the remaining
windows are then visited by one wave) and with the default bound.
"""
import numpy as np
import pytest

from oracle import oracle as O

MH = 2
WIN = 4


@pytest.mark.parametrize("S", [1, 2, 3, 4])
@pytest.mark.parametrize("autobar", [False, True])
def test_earlier_neighbours_have_smaller_t(S, autobar):
    D = 2 * S
    d = -(-D // WIN)
    a, b = d + 1, 0 if autobar else d + D * (d + 1) + 1
    di, dj, dk = 30 * WIN, 100, 50
    for place in range(WIN):
        for ek in range(-D if not autobar else 0, 1):
            for ej in range(-D, D + 1 if ek < 0 else 1):
                for ei in range(-D, D + 1):
                    if (ek, ej, ei) >= (0, 0, 0):
                        continue
                    here = ((di + place) // WIN, dj, dk)
                    there = ((di + place + ei) // WIN, dj + ej, dk + ek)
                    t = [w[0] + a * w[1] + b * w[2] for w in (here, there)]
                    assert there == here or t[1] < t[0], (place, ek, ej, ei)


def _case(ni, nj, nk, ntr, seed, dense):
    layout = (1 - MH, ni + MH, 1 - MH, nj + MH, nk)
    n = (ni + 2 * MH) * (nj + 2 * MH) * nk
    rng = np.random.default_rng(seed)
    trs = []
    for _ in range(ntr):
        src = rng.lognormal(0.0, 1.0, n).astype(np.float32)
        mn = (src * rng.uniform(0.7, 1.0, n)).astype(np.float32)
        mx = (src * rng.uniform(1.0, 1.3, n)).astype(np.float32)
        f = (src * rng.uniform(0.4, 1.6, n)).astype(np.float32)
        f = np.where(rng.uniform(size=n) < dense, f, src).astype(np.float32)
        trs.append((f, mn, mx))
    return layout, trs, rng.uniform(0.5, 2.0, n).astype(np.float32), MH + (ni + 2 * MH) * MH


@pytest.mark.gpu
@pytest.mark.parametrize("spin", [None, 0, 40])
@pytest.mark.parametrize("ni,nj,nk,S,autobar,dense", [
    (15, 9, 7, 2, False, 1.0), (16, 20, 9, 2, False, 1.0), (17, 12, 8, 4, False, 0.5), (33, 6, 6, 3, False, 1.0),
    (3, 7, 5, 2, False, 1.0), (4, 5, 4, 1, False, 1.0),
    (64, 10, 7, 1, False, 0.2), (65, 10, 7, 2, True, 1.0), (130, 21, 9, 2, False, 0.05), (8, 8, 4, 4, True, 1.0),
])
def test_windows_bit_exact(cuda, ni, nj, nk, S, autobar, dense, spin):
    import torch

    from gem_amd import adz as A

    print(f"[ilmc order] {ni}x{nj}x{nk} S={S} autobar={autobar} dense={dense} spin={spin}", flush=True)
    layout, trs, air, off = _case(ni, nj, nk, 2, ni * 7 + S, dense)
    box = (1, ni, 1, nj, 1)
    dev = [dict(f=torch.from_numpy(f.copy()).cuda(), min=torch.from_numpy(mn).cuda(), max=torch.from_numpy(mx).cuda())
           for f, mn, mx in trs]
    il = A.IlmcLam(dev, layout, box, off, sweep_max=S, min_max=True, autobar=autobar)
    if spin is not None:
        il.set_spin_limit(spin)
    counts = torch.full((3 * len(trs),), -1, dtype=torch.int64, device="cuda")
    il(torch.from_numpy(air).cuda(), counts)
    torch.cuda.synchronize()
    il.free()
    for q, (f, mn, mx) in enumerate(trs):
        exp = f.copy()
        c = O.ilmc(exp, mn, mx, air, layout, box, sweep_max=S, min_max=True, autobar=autobar)
        got = dev[q]["f"].cpu().numpy()
        assert np.array_equal(got.view(np.uint32), exp.view(np.uint32)), (q, int(np.count_nonzero(got != exp)))
        assert counts[3 * q:3 * q + 3].cpu().tolist() == c.tolist(), q
