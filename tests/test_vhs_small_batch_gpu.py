"""FP64 at Nv = 16 on a design without planar directions: prep and finalize in
the one-pencil kernels, and the x-forward pass on both sides of the batch size
where its sum over the radial nodes is spread over waves (2 Nv^2 columns per
point against one wave per SIMD: 128 points on 256 CUs), against the oracle and
between batch sizes."""
import sys

import numpy as np
import pytest

from oracle import vhs as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("project", [False, True])
@pytest.mark.parametrize("Nrho", [1, 8, 11])
def test_fp64_16_batches(Nrho, project, device):
    import torch
    from dgfs_hip.solvers.dgfs.scattering import VHSOperator
    from dgfs_hip.solvers.dgfs.velocitymesh import DGFSVelocityMesh
    N, M, npts = 16, 6, 600
    vm = DGFSVelocityMesh.from_params(None, N, 6.0, Nrho, M)
    op = VHSOperator(N, Nrho, M, vm.L(), 0.38, 1.0, vm.qz(), vm.qw(), vm.sz(), vm.sw(), vm.cw(), precision=64,
                     project=project)
    ov = O.VelocityMesh(N, 6.0, Nrho, M)
    rng = np.random.default_rng(Nrho)
    base = np.stack([0.5 * O.maxwellian(ov, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) +
                     0.5 * O.maxwellian(ov, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) for _ in range(6)])
    want = O.VHSOracle(ov, 0.38, 1.0).q(base)
    if project:
        want = O.project_invariants(ov, want)
    f = torch.as_tensor(np.tile(base, (npts // 6, 1)), device=device)
    for n in (1, 5, 128, 129, npts):
        print("fp64 16^3", Nrho, project, n, flush=True)
        sys.stdout.flush()
        Q = torch.full_like(f[:n], float("nan"))
        op.eval_contig(f.data_ptr(), Q.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = Q.cpu().numpy()
        # the bound of the oracle comparisons at these sizes: roundoff of both
        # transforms, amplified by the cancellation of gain and loss
        assert rel(got[:6], want[:n]) < 1e-10
        for i in range(6, n):
            assert np.array_equal(got[i], got[i % 6])
