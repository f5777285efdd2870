"""The boundary kernels at the sizes where their thread shapes can go wrong:
one point, a ragged last group of 32 points, velocity counts around the rows
and the unrolled sweeps, a velocity batch in the middle of the grid.  Against
the same sums in numpy (FP64, 1e-13 of the largest value)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf,nvars,vidx,vsize", [(1, 27, 0, 27), (33, 64, 0, 64), (36, 1000, 24, 1030),
                                                 (70, 4100, 0, 4100), (5, 9000, 0, 9000)])
def test_diffuse_wall_edges(nf, nvars, vidx, vsize, device):
    import torch
    from dgfs_hip import fr
    rng = np.random.default_rng(nf + nvars)
    nblk = -(-nf // 32)
    ld = nblk * nvars * 32
    L = rng.uniform(0.1, 1.0, size=ld)
    off = np.array([(i // 32) * nvars * 32 + i % 32 for i in range(nf)], dtype=np.int64)
    ang = rng.uniform(0, 2 * np.pi, nf)
    nl, mag = np.stack([np.cos(ang), np.sin(ang)]), rng.uniform(0.5, 2.0, nf)
    cv = rng.uniform(-5, 5, size=(3, vsize))
    f0 = rng.uniform(0.1, 1.0, vsize)
    bc0 = rng.uniform(0.1, 1.0, 2 * nf)
    U, cw = (0.3, -0.1, 0.0), 0.7
    t = lambda a, d=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=d, device=device)
    Lt, ot, nt, mt, ct, ft, bt = t(L), t(off, torch.int64), t(nl), t(mag), t(cv), t(f0), t(bc0)
    st = torch.cuda.current_stream().cuda_stream
    print("wall", nf, nvars, vidx, flush=True)
    fr.bccupdate(fr.BC_DIFFUSE, 2, nf, nvars, vidx, Lt, ot, nt, ft, bt, U, cw, ct, vsize, st)
    c = cv[:, vidx:vidx + nvars]
    ul = L[off[:, None] + 32 * np.arange(nvars)[None]]
    fac = nl[0][:, None] * (c[0] - U[0]) + nl[1][:, None] * (c[1] - U[1])
    f0b = f0[vidx:vidx + nvars]
    b0 = np.where(fac >= 0, fac * ul * cw, 0).sum(1)
    b1 = np.where(fac < 0, fac * f0b * cw, 0).sum(1)
    if vidx:
        b0, b1 = b0 + bc0[:nf], b1 + bc0[nf:]
    got = bt.cpu().numpy()
    assert np.abs(got - np.concatenate([b0, b1])).max() < 1e-13 * max(np.abs(b0).max(), np.abs(b1).max())
    fr.bccflux(fr.BC_DIFFUSE, 2, nf, nvars, vidx, Lt, ot, nt, mt, ft, bt, None, U, ct, vsize, st)
    torch.cuda.synchronize()
    nc = nl[0][:, None] * c[0] + nl[1][:, None] * c[1]
    ur = np.where(fac < 0, f0b * (-got[:nf] / got[nf:])[:, None], ul)
    fn = (0.5 * nc * (ul + ur) + 0.5 * np.abs(nc) * (ul - ur)) * mag[:, None]
    out = Lt.cpu().numpy()
    ref = L.copy()
    ref[off[:, None] + 32 * np.arange(nvars)[None]] = fn
    assert np.abs(out - ref).max() < 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("nf,nvars", [(4096, 1024), (4097, 1024), (4096, 1023), ((1 << 22) + 3, 2)])
def test_diffuse_balance_of_many_points(nf, nvars, device):
    """Both sides of the limits of the wide block (1024 velocities, 4096
    points), and more points than a grid of 1024-thread blocks takes (2^32
    threads): every point against the same sums in torch, FP64 sums of up to
    1024 terms, so 1e-13 of the largest value."""
    import torch
    from dgfs_hip import fr
    g = torch.Generator(device=device).manual_seed(nf)
    r = lambda *s: torch.rand(s, dtype=torch.float64, device=device, generator=g)
    rows = min(nf, 4097)  # the points share these rows of states
    L = r(-(-rows // 32) * nvars * 32)
    i = torch.arange(nf, device=device) % rows
    off = (i // 32) * nvars * 32 + i % 32
    ang = 6.283 * r(nf)
    nl = torch.stack([torch.cos(ang), torch.sin(ang)]).contiguous()
    cv = 10 * r(3, nvars) - 5
    f0 = r(nvars)
    bc = torch.full((2, nf), float("nan"), dtype=torch.float64, device=device)
    U, cw = (0.3, -0.1, 0.0), 0.7
    print("wall balance", nf, nvars, flush=True)
    fr.bccupdate(fr.BC_DIFFUSE, 2, nf, nvars, 0, L, off, nl, f0, bc, U, cw, cv, nvars,
                 torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    b0, b1 = torch.zeros(nf, dtype=torch.float64, device=device), torch.zeros(nf, dtype=torch.float64, device=device)
    for v in range(nvars):
        fac = nl[0] * (cv[0, v] - U[0]) + nl[1] * (cv[1, v] - U[1])
        b0 += torch.where(fac >= 0, fac * L[off + 32 * v] * cw, 0.0)
        b1 += torch.where(fac < 0, fac * f0[v] * cw, 0.0)
    assert float((bc[0] - b0).abs().max()) < 1e-13 * float(b0.abs().max())
    assert float((bc[1] - b1).abs().max()) < 1e-13 * float(b1.abs().max())


@pytest.mark.parametrize("nf", [32 * 511, 32 * 513, 32 * 4097 - 5])
def test_flux_of_many_points(nf, device):
    """Point counts on both sides of where a thread takes more than 4
    velocities (64 workgroups per CU: 512 groups of 32 points at 1024
    velocities on 256 CUs) and where it takes 32, a ragged last row: a wall
    that lets through, ul = 0.5 n.c (ul + ur) + 0.5 |n.c| (ul - ur)."""
    import torch
    from dgfs_hip import fr
    nvars = 1021
    g = torch.Generator(device=device).manual_seed(nf)
    r = lambda *s: torch.rand(s, dtype=torch.float64, device=device, generator=g)
    L = r(-(-nf // 32) * nvars * 32)
    i = torch.arange(nf, device=device)
    off = (i // 32) * nvars * 32 + i % 32
    ang = 6.283 * r(nf)
    nl, mag = torch.stack([torch.cos(ang), torch.sin(ang)]).contiguous(), 0.5 + r(nf)
    cv, f0 = 10 * r(3, nvars) - 5, r(nvars)
    before = L.clone()
    print("boundary flux", nf, flush=True)
    fr.bccflux(fr.BC_INLET, 2, nf, nvars, 0, L, off, nl, mag, f0, None, None, (0.3, -0.1, 0.0), cv, nvars,
               torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    worst = 0.0
    for v in range(nvars):
        ul = before[off + 32 * v]
        nc = nl[0] * cv[0, v] + nl[1] * cv[1, v]
        fac = nl[0] * (cv[0, v] - 0.3) + nl[1] * (cv[1, v] + 0.1)
        # at fac = 0 up to rounding either side is the state: leave those points out
        ur = torch.where(fac < 0, f0[v], ul)
        want = mag * (0.5 * nc * (ul + ur) + 0.5 * nc.abs() * (ul - ur))
        worst = max(worst, float(((L[off + 32 * v] - want) * (fac.abs() > 1e-12)).abs().max()))
    assert worst < 1e-13 * float(L.abs().max())
