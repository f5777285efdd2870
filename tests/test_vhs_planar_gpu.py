"""The planar-direction gain (csrc/vhs_planar.hpp), the automatic choice at Nv
16, 24 and 32 when every direction of the half-sphere design has exactly one
zero component and comes with its mirror image, against the multi-pass kernel
(algorithm 1), which transforms every direction on its own.

FP64: the two are the same sum in another order, so roundoff (1e-12 relative
L2).  The rough states are white noise: the unpaired Nyquist modes, which the
planar form carries as separate terms, are then as large as any other.
FP32: the distance of Q from the FP64 operator is within a factor of 1.5 of
the multi-pass kernel's on the same states."""
import sys

import numpy as np
import pytest

from oracle import vhs as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def designs():
    twelve = O.half_sphere_design(12)
    rng = np.random.default_rng(5)
    signs = rng.choice([-1.0, 1.0], size=(12, 1))
    cubo = np.array([[1, 1, 0], [1, -1, 0], [1, 0, 1], [1, 0, -1], [0, 1, 1], [0, 1, -1]]) / np.sqrt(2.0)
    # one axis pair only, unequal components
    flat = np.array([[0.6, 0.8, 0.0], [0.6, -0.8, 0.0], [0.28, 0.96, 0.0], [-0.28, 0.96, 0.0]])
    return {"m12": twelve, "m12_shuffled": (twelve * signs)[rng.permutation(12)], "m6_cuboctahedron": cubo,
            "m4_one_pair": flat}


def make(N, sz, precision, project=False, Nrho=4, algorithm=0):
    from dgfs_hip.solvers.dgfs.scattering import VHSOperator
    from dgfs_hip.solvers.dgfs.velocitymesh import DGFSVelocityMesh
    vm = DGFSVelocityMesh.from_params(None, N, 6.0, Nrho, 6)
    op = VHSOperator(N, Nrho, len(sz), vm.L(), 0.38, 1.0, vm.qz(), vm.qw(), sz, 2 * np.pi / len(sz), vm.cw(),
                     precision=precision, project=project)
    op.set_algorithm(algorithm)
    return op


def run(op, f, device):
    import torch
    ft = torch.as_tensor(f, device=device)
    Qt = torch.full_like(ft, float("nan"))
    op.eval_contig(ft.data_ptr(), Qt.data_ptr(), f.shape[0], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return Qt.cpu().numpy()


@pytest.mark.parametrize("name", list(designs()))
@pytest.mark.parametrize("N", [16, 24, 32])
def test_planar_matches_multipass_on_rough_states(N, name, device):
    rng = np.random.default_rng(N)
    sz = designs()[name]
    f = rng.uniform(0.0, 1.0, size=(3, N ** 3))
    say("planar", N, name)
    ref = run(make(N, sz, 64, algorithm=1), f, device)
    op = make(N, sz, 64)
    for groups in (0, 1, 3):
        op.set_groups(groups)
        e = rel(run(op, f, device), ref)
        say("  fp64 groups", groups, e)
        assert e < 1e-12
    e_mp = rel(run(make(N, sz, 32, algorithm=1), f, device), ref)
    e_pl = rel(run(make(N, sz, 32), f, device), ref)
    say("  fp32 multi-pass", e_mp, "planar", e_pl)
    assert e_pl < 1.5 * e_mp


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("N,npts", [(16, 1), (16, 300), (24, 5), (32, 1), (32, 37)])
def test_planar_batches_and_registers(N, npts, precision, device):
    """Small batches, contiguous and as AoSoA registers of a ragged element
    count, with the projection; FP32 within the module's factor of 1.5 of the
    multi-pass kernel's distance from FP64."""
    import torch
    sz = designs()["m12"]
    vm = O.VelocityMesh(N, 6.0, 4, 12)
    rng = np.random.default_rng(npts)
    f = np.stack([0.5 * O.maxwellian(vm, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) +
                  0.5 * O.maxwellian(vm, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) for _ in range(npts)])
    say("planar batch", N, npts, precision)
    op = make(N, sz, precision, project=True)
    Q = run(op, f, device)
    sub = np.unique(np.linspace(0, npts - 1, 6).astype(int))
    ref = run(make(N, sz, 64, project=True, algorithm=1), f[sub], device)
    e = rel(Q[sub], ref)
    say("  vs FP64 multi-pass", e)
    if precision == 64:
        assert e < 1e-11
    else:
        assert e < 1.5 * rel(run(make(N, sz, 32, project=True, algorithm=1), f[sub], device), ref)
    # elements [1, neles) of a register of one point per element
    neles, n = npts + 1, N ** 3
    nparr = -(-neles // 32) * 32
    reg = np.zeros((1, nparr // 32, n, 32))
    for e in range(npts):
        reg[0, (e + 1) // 32, :, (e + 1) % 32] = f[e]
    rt = torch.as_tensor(reg.reshape(1, -1), device=device)
    qt = torch.zeros_like(rt)
    op.eval_aosoa(rt.data_ptr(), qt.data_ptr(), 1, nparr * n, n, neles, 1, npts,
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    qr = qt.cpu().numpy().reshape(nparr // 32, n, 32)
    got = np.stack([qr[(e + 1) // 32, :, (e + 1) % 32] for e in range(npts)])
    assert np.array_equal(got, Q)
    assert not qr[0, :, 0].any()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("N", [16, 24, 32])
def test_planar_large_batches(N, precision, device):
    """Batches on both sides of where the x pass takes a wave per pencil block
    (its pencils are a wave per SIMD) and of where the operand kernel takes 256
    threads (more points than CUs), with more items than are resident at once.
    Against the FP64 oracle (1e-10; FP32 within 1.5 of the multi-pass kernel's
    distance), and every point bitwise that of its state wherever it lies."""
    import torch
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    limit = 64 * 4 * cus // ((N // 2 + 1) * N * (precision // 32))
    vm = O.VelocityMesh(N, 6.0, 4, 12)
    rng = np.random.default_rng(N)
    base = np.stack([0.5 * O.maxwellian(vm, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) +
                     0.5 * O.maxwellian(vm, 1, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.5, 1.5)) for _ in range(3)])
    want = O.project_invariants(vm, O.VHSOracle(vm, 0.38, 1.0).q(base))
    sz = designs()["m12"]
    bound = 1e-10
    if precision == 32:
        bound = 1.5 * rel(run(make(N, sz, 32, project=True, algorithm=1), base, device), want)
    op = make(N, sz, precision, project=True)
    for npts in (limit, limit + 1, max(limit, 2 * cus) + 3):
        say("planar large batch", N, precision, npts)
        ft = torch.as_tensor(base, device=device)[torch.arange(npts, device=device) % 3].contiguous()
        Qt = torch.full_like(ft, float("nan"))
        op.eval_contig(ft.data_ptr(), Qt.data_ptr(), npts, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert op.ran_planar()
        e = rel(Qt[:3].cpu().numpy(), want)
        say("  vs oracle", e)
        assert e < bound
        for i in range(3):
            assert bool((Qt[i::3] == Qt[i]).all())


def test_other_designs_keep_the_general_gain(device):
    """A direction with no zero component, or a missing mirror image, takes
    the general kernels: same Q as with the algorithm named."""
    N = 16
    f = np.random.default_rng(3).uniform(0.0, 1.0, size=(2, N ** 3))
    for sz in (O.half_sphere_design(6), designs()["m12"][:11]):
        say("general design", len(sz))
        auto, named = run(make(N, sz, 64), f, device), run(make(N, sz, 64, algorithm=6), f, device)
        assert np.array_equal(auto, named)


def test_operator_tells_which_gain_ran(device):
    """`planar` is the library's own rule (mirror images included), and
    ran_planar tells the planar gain from the kernel that it stands in for."""
    N = 16
    f = np.random.default_rng(3).uniform(0.0, 1.0, size=(2, N ** 3))
    say("which gain ran")
    for precision, general in ((64, 6), (32, 4)):
        op = make(N, designs()["m12"], precision)
        assert op.planar and not op.ran_planar()
        run(op, f, device)
        assert op.ran_planar() and op.get_algorithm() == general
        for algorithm in (general, 1):
            op.set_algorithm(algorithm)
            run(op, f, device)
            assert op.planar and not op.ran_planar() and op.get_algorithm() == algorithm
        op.set_algorithm(0)
        run(op, f, device)
        assert op.ran_planar()
        # each direction has one zero component, but one lacks its mirror image
        op = make(N, designs()["m12"][:11], precision)
        run(op, f, device)
        assert not op.planar and not op.ran_planar() and op.get_algorithm() == general
    assert not make(12, designs()["m12"], 64).planar


# groups (pairs of mirrored directions), radial nodes, whether the automatic
# choice is planar: both sides of each line
LINES = {(16, 64): [(1, 2, False), (1, 3, True), (2, 2, True)], (16, 32): [(1, 5, False), (1, 6, True), (2, 2, False), (2, 3, True), (6, 1, True)],
         (24, 64): [(2, 8, False), (3, 1, True)], (24, 32): [(2, 8, False), (3, 4, False), (3, 5, True), (6, 1, True)],
         (32, 64): [(1, 8, False), (2, 1, True)], (32, 32): [(2, 1, False), (1, 3, True), (6, 1, True)]}


@pytest.mark.parametrize("N,precision", list(LINES))
def test_designs_of_few_groups(N, precision, device):
    """Designs of few directions take the planar gain from where their groups
    and radial nodes are enough work; on both sides of the line Q is the
    multi-pass kernel's (the module's bounds)."""
    flat = designs()["m4_one_pair"]
    by_groups = {1: flat[:2], 2: flat, 3: designs()["m6_cuboctahedron"], 6: designs()["m12"]}
    f = np.random.default_rng(N).uniform(0.0, 1.0, size=(2, N ** 3))
    for groups, Nrho, planar in LINES[N, precision]:
        sz = by_groups[groups]
        say("few groups", N, precision, groups, Nrho)
        op = make(N, sz, precision, Nrho=Nrho)
        assert op.planar == planar
        Q = run(op, f, device)
        assert op.ran_planar() == planar
        ref = run(make(N, sz, 64, Nrho=Nrho, algorithm=1), f, device)
        if precision == 64:
            assert rel(Q, ref) < 1e-12
        else:
            assert rel(Q, ref) < 1.5 * rel(run(make(N, sz, 32, Nrho=Nrho, algorithm=1), f, device), ref)


# Nrho 4 and 13: up to six parts and up to two of the groups
@pytest.mark.parametrize("N,npts,Nrho", [(16, 400, 4), (24, 60, 4), (16, 100, 13), (24, 20, 13)])
def test_small_batch_captured_after_a_larger_one(N, npts, Nrho, device):
    """A batch small enough to split its groups over work items finds room for
    the parts' transforms in the workspace of a larger batch: captured without
    an allocation, every replay equal to the eager result."""
    import torch
    rng = np.random.default_rng(N)
    f = rng.uniform(0.0, 1.0, size=(npts, N ** 3))
    say("planar capture", N, npts, Nrho)
    op = make(N, designs()["m12"], 64, Nrho=Nrho)
    big = run(op, f, device)
    for n in (1, 3, 11):
        ft = torch.as_tensor(f[:n], device=device)
        Qt = torch.zeros_like(ft)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            op.eval_contig(ft.data_ptr(), Qt.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
        eager = run(op, f[:n], device)
        assert rel(eager, big[:n]) < 1e-12
        for _ in range(3):
            Qt.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(Qt.cpu().numpy(), eager)
