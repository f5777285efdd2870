"""The HIP moments kernel at the sizes where it can go wrong: element counts at
the edges of the 32-element blocks, every workgroup width, velocity counts
that are no multiple of a sweep, and padding that must not be read.  Against
direct sums in numpy; FP64 sums of up to 4096 terms of size <= 1e3, so 1e-12
of each output's largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # nupts, neles, vsize: the three widths are taken at >= 256, >= 128 and
    # fewer 32-element blocks (times nupts)
    (1, 1, 27), (1, 31, 64), (3, 33, 125), (9, 64, 216), (4, 32 * 33 - 1, 64), (4, 32 * 64 + 5, 27), (1, 2, 4096),
    # short and long velocity grids (256) at every width
    (3, 33, 256), (3, 33, 257), (4, 32 * 33 - 1, 260), (4, 32 * 64 + 5, 256), (4, 32 * 64 + 5, 300),
    # many solution points (the grid's second dimension)
    (65537, 1, 8),
]


@pytest.mark.parametrize("nupts,neles,vsize", CASES)
def test_moments_edges(nupts, neles, vsize, device):
    import torch
    from dgfs_hip import fr
    rng = np.random.default_rng(vsize + neles)
    cv = rng.uniform(-7.0, 7.0, size=(3, vsize))
    f = rng.uniform(0.1, 1.0, size=(nupts, vsize, neles))
    nparr = -(-neles // 32) * 32
    reg = np.full((nupts, nparr // 32, vsize, 32), np.nan)   # the padding is never read
    for e in range(neles):
        reg[:, e // 32, :, e % 32] = f[:, :, e]
    rt = torch.as_tensor(reg.reshape(nupts, -1), device=device)
    ct = torch.as_tensor(cv, device=device)
    out = torch.full((nupts, 15, neles), float("nan"), dtype=torch.float64, device=device)
    print("moments", nupts, neles, vsize, flush=True)
    fr.moments(nupts, neles, vsize, rt, nparr * vsize, ct, 0.3, out, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    cw = 0.3
    rho = f.sum(1) * cw
    U = np.einsum("uve,dv->due", f, cv) * cw / rho
    c = cv[:, None, :, None] - U[:, :, None, :]
    c2 = (c * c).sum(0)
    T = (f * c2).sum(1) * cw * (2.0 / 3.0) / rho
    q = [(f * c[d] * c2).sum(1) * cw for d in range(3)]
    P = [2 * (f * c[a] * c[b]).sum(1) * cw for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))]
    ref = np.stack([rho, *U, T, *q, *P, rho * T], axis=1)
    scale = np.abs(ref).max(axis=(0, 2), keepdims=True)
    # cancelling sums (odd moments) are held to the size of their terms
    scale = np.maximum(scale, np.abs(f).sum(1).max() * cw)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= 1e-12 * scale).all()
