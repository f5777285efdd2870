"""The surrogate's large-tile FP32 GEMM and fused layer kernels at the sizes
where they can go wrong: edges of the 128 x 64 x 32 tiles, short and split
reductions, every transposition, unaligned leading dimensions (which take the
general kernel), and batches of one and odd sizes through a whole layer stack.
FP32 sums of K products: |error| <= sqrt(K) 2^-22 |A| |B| entrywise bound of a
random-sign sum with a margin of 4."""
import numpy as np
import pytest

from oracle import surrogate as S

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("M,N,K", [(128, 64, 32), (129, 65, 33), (200, 100, 7), (512, 96, 512), (131, 67, 4100),
                                   (128, 64, 1), (300, 64, 1030)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f32_edges(M, N, K, ta, tb, device):
    import torch
    from dgfs_hip import surrogate as D
    rng = np.random.default_rng(M + K)
    A, B = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    C0 = rng.normal(size=(M, N)).astype(np.float32)
    for pad in (0, 3):  # leading dimensions rounded up to 4, or odd
        def store(X):
            ld = -(-X.shape[1] // 4) * 4 + pad
            out = np.full((X.shape[0], ld), np.nan, dtype=np.float32)
            out[:, :X.shape[1]] = X
            return torch.as_tensor(out, device=device), ld
        At, lda = store(A.T if ta else A)
        Bt, ldb = store(B.T if tb else B)
        Ct = torch.as_tensor(C0, device=device)
        say("gemm", M, N, K, ta, tb, pad)
        D.gemm(ta, tb, M, N, K, 0.5, At, lda, Bt, ldb, 2.0, Ct, N, bf16=False,
               stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        ref = 0.5 * (A.astype(np.float64) @ B.astype(np.float64)) + 2.0 * C0
        err = np.abs(Ct.cpu().numpy() - ref)
        assert err.max() <= 4 * np.sqrt(K) * 2.0 ** -22 * np.abs(A).max() * np.abs(B).max() + 4 * 2.0 ** -23 * np.abs(ref).max()


@pytest.mark.parametrize("P", [1, 3, 17])
def test_layers_small_batches(P, device):
    """Forward and every gradient at small and odd batches against the FP64
    oracle: 1e-5 of each output's norm (FP32 sums of up to 512 P terms)."""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    sur = SpectralSurrogate(8, 5.0, (10.0 / 8) ** 3, 0.38, 1.0, max_batch=32, device=device, seed=3)
    rng = np.random.default_rng(P)
    x, lt = rng.normal(size=(P, 512)), rng.normal(size=P) * 0.2
    dout = rng.normal(size=(P, 512))
    f32 = lambda a: torch.as_tensor(a, dtype=torch.float32, device=device).contiguous()
    xt, ltt, dt = f32(x), f32(lt), f32(dout)
    out = torch.empty((P, 512), dtype=torch.float32, device=device)
    say("layers", P)
    sur.forward(xt, ltt, P, out)
    sur.backward(dt)
    torch.cuda.synchronize()
    th = sur.params_bf16.cpu().numpy().astype(np.float64)
    ref, cache = S.forward(th, xt.cpu().numpy(), ltt.cpu().numpy())
    g = S.backward(th, cache, dt.cpu().numpy().astype(np.float64))
    e = np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)
    eg = np.linalg.norm(sur.grad.cpu().numpy() - g) / np.linalg.norm(g)
    say("  forward", e, "gradient", eg)
    assert e < 1e-5 and eg < 1e-5


@pytest.mark.parametrize("P", [129, 300])
def test_layers_of_several_tiles_per_wave(P, device):
    """Batches beyond 128 points, where a wave of the backward layer takes more
    than one tile and the last round is uneven, and the layer products are not
    split: every parameter block's gradient on its own (a norm over the whole
    vector is K's), against the FP64 oracle.  Output gradients of one sign, so
    that no block is the small difference of large sums: FP32 sums of up to 512
    P terms, 1e-5 of the block's norm."""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    sur = SpectralSurrogate(8, 5.0, (10.0 / 8) ** 3, 0.38, 1.0, max_batch=P, device=device, seed=3)
    rng = np.random.default_rng(P)
    f32 = lambda a: torch.as_tensor(a, dtype=torch.float32, device=device).contiguous()
    xt, ltt = f32(rng.normal(size=(P, 512)) * 0.3), f32(rng.normal(size=P) * 0.2)
    dt = f32(rng.uniform(0.5, 1.5, size=(P, 512)))
    out = torch.empty((P, 512), dtype=torch.float32, device=device)
    print("layers", P, flush=True)
    sur.forward(xt, ltt, P, out)
    sur.backward(dt)
    torch.cuda.synchronize()
    th = sur.params_bf16.cpu().numpy().astype(np.float64)
    ref, cache = S.forward(th, xt.cpu().numpy().astype(np.float64), ltt.cpu().numpy().astype(np.float64))
    assert np.linalg.norm(out.cpu().numpy() - ref) < 1e-5 * np.linalg.norm(ref)
    g, got = S.backward(th, cache, dt.cpu().numpy().astype(np.float64)), sur.grad.cpu().numpy()
    sizes = [("P0", S.WIDTH), ("P1", S.WIDTH), ("E", S.MODES * S.WIDTH)]
    for l in range(S.LAYERS):
        sizes += [(f"K{l}", S.MODES ** 2), (f"W{l}", S.WIDTH ** 2), (f"R{l}", S.WIDTH ** 2), (f"b{l}", S.WIDTH)]
    sizes += [("Pout", S.WIDTH), ("bout", S.MODES)]
    assert sum(n for _, n in sizes) == g.size
    at = 0
    for name, n in sizes:
        e = np.linalg.norm(got[at:at + n] - g[at:at + n]) / np.linalg.norm(g[at:at + n])
        say(" ", name, e)
        assert e < 1e-5, name
        at += n


@pytest.mark.parametrize("N", [12, 16, 24, 32])
def test_encode_decode_grids(N, device):
    """Encoder and projecting decoder on every built grid, one point and more
    points than fit one sweep of workgroups' columns, against the FP64
    oracle: FP32 rounding on the modes, 1e-10 on the FP64 outputs plus the
    forward error of the per-axis factorisations, at most about eps times the
    condition number of their Gram matrices, three axes, with a margin of 4.
    (At N = 8 the eight functions fill the eight points: the Gram matrix is
    numerically singular and its modes mean nothing.)"""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    L = 6.0 if N >= 16 else 5.0
    rng = np.random.default_rng(N)
    P = 3
    c = S.grid(N, L)
    I, J, K = np.meshgrid(c, c, c, indexing="ij")
    f = []
    for _ in range(P):
        u, T = rng.uniform(-0.4, 0.4, 3), rng.uniform(0.9, 1.6)
        g = np.exp(-((I - u[0]) ** 2 + (J - u[1]) ** 2 + (K - u[2]) ** 2) / T) / (np.pi * T) ** 1.5
        f.append((g * (1 + 0.05 * (I - u[0]) * (J - u[1]))).ravel())
    f = np.array(f)
    sur = SpectralSurrogate(N, L, (2 * L / N) ** 3, 0.38, 1.0, max_batch=8, device=device, seed=1)
    ft = torch.as_tensor(f, device=device)
    mom = torch.empty((P, 8), dtype=torch.float64, device=device)
    x = torch.empty((P, 512), dtype=torch.float32, device=device)
    lt = torch.empty((P,), dtype=torch.float32, device=device)
    say("encode / decode", N)
    sur.encode(ft, P, mom, x, lt)
    y = rng.normal(size=(P, 512)).astype(np.float32)
    yt = torch.as_tensor(y, device=device)
    Q = torch.full_like(ft, float("nan"))
    Q0 = torch.full_like(ft, float("nan"))
    sur.decode(yt, mom, P, Q, project=True)
    sur.decode(yt, mom, P, Q0, project=False)
    torch.cuda.synchronize()
    mh = mom.cpu().numpy()
    for i in range(P):
        mref, a, _ = S.encode(f[i], N, L)
        cond = max(np.linalg.cond(v.T @ v) for v in S._vander(N, L, mref[1:4], mref[4]))
        tol = 1e-10 + 12 * 2.0 ** -52 * cond
        say("  largest condition number", cond, "errors", np.abs(mh[i, :7] - mref).max())
        assert np.abs(mh[i, :6] - mref[:6]).max() < 1e-10
        assert np.abs(mh[i, 6] - mref[6]) < tol
        assert np.abs(x.cpu().numpy()[i] - a).max() < (1e-6 + tol) * max(1.0, np.abs(a).max())
        q0 = S.decode(y[i], mref, N, L, 0.38, 1.0)
        sc = np.abs(q0).max()
        assert np.abs(Q0.cpu().numpy()[i] - q0).max() < tol * sc
        assert np.abs(Q.cpu().numpy()[i] - S.project(q0, N, L)).max() < tol * sc


def _stream_products(n, device, seed):
    """n products of the split form (512 x 512, K split in two; 64 x 64 from a
    long K through the general kernel) on each of two streams."""
    import torch
    g = torch.Generator(device="cpu").manual_seed(seed)
    shapes = [(512, 512, 512), (64, 60, 9001), (512, 512, 1500)]
    jobs = []
    for s in range(2):
        ops = []
        for i in range(n):
            M, N, K = shapes[(i + s) % 3]
            ops.append((M, N, K, torch.randn((M, K), generator=g).to(device), torch.randn((K, N), generator=g).to(device),
                        torch.full((M, N), float("nan"), device=device)))
        jobs.append(ops)
    return jobs


def _launch(ops, stream):
    from dgfs_hip import surrogate as D
    for M, N, K, A, B, Cm in ops:
        D.gemm(0, 0, M, N, K, 1.0, A, K, B, N, 0.0, Cm, N, bf16=False, stream=stream.cuda_stream)


@pytest.mark.parametrize("threads", [False, True])
def test_split_products_on_two_streams(threads, device):
    """Products whose reduction is split, on two streams at once (from one
    thread in turn, and from two threads): each equals, bitwise, the same
    product with nothing else in flight, whose order of sums is the same."""
    import threading
    import torch
    jobs = _stream_products(12, device, 11)
    print("split products on two streams", threads, flush=True)
    quiet = torch.cuda.Stream()
    want = []
    for ops in jobs:
        _launch(ops, quiet)
        torch.cuda.synchronize()
        want.append([o[-1].clone() for o in ops])
    for ops in jobs:
        for o in ops:
            o[-1].fill_(float("nan"))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    if threads:
        ts = [threading.Thread(target=_launch, args=(ops, s)) for ops, s in zip(jobs, streams)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    else:
        for a, b in zip(*jobs):
            _launch([a], streams[0])
            _launch([b], streams[1])
    torch.cuda.synchronize()
    for ops, ws in zip(jobs, want):
        for o, w in zip(ops, ws):
            assert torch.equal(o[-1], w)


def test_captured_product_takes_no_shared_workspace(device):
    """Under capture the product runs unsplit: replays with eager split
    products on another stream in between stay equal to the first one, and to
    the eager product within the order of the sums (bound of the module)."""
    import torch
    (job, other) = _stream_products(3, device, 5)
    M, N, K, A, B, Cm = job[0]
    s = torch.cuda.Stream()
    _launch([job[0]], s)
    torch.cuda.synchronize()
    eager = Cm.clone()
    g = torch.cuda.CUDAGraph()
    print("captured product", flush=True)
    with torch.cuda.graph(g):
        _launch([job[0]], torch.cuda.current_stream())
    first = None
    for _ in range(4):
        Cm.fill_(float("nan"))
        torch.cuda.synchronize()
        _launch(other, s)
        g.replay()
        torch.cuda.synchronize()
        first = Cm.clone() if first is None else first
        assert torch.equal(Cm, first)
    bound = 8 * np.sqrt(K) * 2.0 ** -22 * float(A.abs().max()) * float(B.abs().max())
    assert float((first - eager).abs().max()) <= bound


@pytest.mark.parametrize("P", [5, 130])
def test_first_forward_and_backward_captured(P, device):
    """A handle's first forward and backward may be under capture: nothing is
    allocated after its creation, and every replay equals the eager result."""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    rng = np.random.default_rng(P)
    f32 = lambda a: torch.as_tensor(a, dtype=torch.float32, device=device).contiguous()
    x, lt, dout = f32(rng.normal(size=(P, 512))), f32(rng.normal(size=P) * 0.2), f32(rng.normal(size=(P, 512)))
    out = torch.empty((P, 512), dtype=torch.float32, device=device)
    sur = SpectralSurrogate(8, 5.0, (10.0 / 8) ** 3, 0.38, 1.0, max_batch=P, device=device, seed=3)
    torch.cuda.synchronize()
    print("captured first forward", P, flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        sur.forward(x, lt, P, out)
        sur.backward(dout)
    sur.forward(x, lt, P, out)
    sur.backward(dout)
    torch.cuda.synchronize()
    eager, grad = out.clone(), sur.grad.clone()
    for _ in range(3):
        out.zero_()
        sur.grad.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and torch.equal(sur.grad, grad)


@pytest.mark.parametrize("P", [3, 130])
def test_layer_sums_of_its_two_products_apart(P, device):
    """A layer adds U W and Z R as whole sums: with U W = 2^24 everywhere and
    Z R = 2 from 32 products of 1/16, the result is 2^24 + 2 exactly, where a
    chain that added the small products to the large sum one after another
    would lose every one of them.  The other layers pass it on (K = W = 0, R
    the identity; GELU is the identity at this size)."""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    th = np.zeros_like(S.init_params(0))
    D, Wd = S.MODES, S.WIDTH
    th[S.OFF_E:S.OFF_E + D * Wd] = 1.0
    for l in range(S.LAYERS):
        o = S.OFF_LAYERS + l * S.LAYER_SIZE
        K, W, R = (th[a:a + n] for a, n in ((o, D * D), (o + D * D, Wd * Wd), (o + D * D + Wd * Wd, Wd * Wd)))
        if l == 0:
            K[:] = np.eye(D).ravel()
            W[:] = 2.0 ** 19
            R[:] = 2.0 ** -4
        else:
            R[:] = np.eye(Wd).ravel()
    th[S.OFF_POUT] = 1.0
    sur = SpectralSurrogate(8, 5.0, (10.0 / 8) ** 3, 0.38, 1.0, max_batch=P, device=device, seed=0)
    f32 = lambda a: torch.as_tensor(a, dtype=torch.float32, device=device).contiguous()
    out = torch.empty((P, D), dtype=torch.float32, device=device)
    print("layer sums", P, flush=True)
    sur.forward(f32(np.zeros((P, D))), f32(np.zeros(P)), P, out, params=f32(th))
    torch.cuda.synchronize()
    assert (out == 2.0 ** 24 + 2.0).all()


@pytest.mark.parametrize("N", [8, 12, 16, 24, 32])
@pytest.mark.parametrize("P", [1, 1030])
def test_encode_without_modes(N, P, device):
    """Moments and indicator alone (no x), one point and more points than a
    sweep of workgroups, for drifting two-stream states: bitwise those of the
    call that encodes the modes too, and those of the FP64 oracle (1e-10)."""
    import torch
    from dgfs_hip.surrogate import SpectralSurrogate
    L = 6.0 if N >= 16 else 5.0
    rng = np.random.default_rng(N)
    c = S.grid(N, L)
    I, J, K = np.meshgrid(c, c, c, indexing="ij")
    base = []
    for _ in range(3):
        f = 0.0
        for w in (0.7, 0.3):
            u, T = rng.uniform(-0.5, 0.5, 3), rng.uniform(0.9, 1.6)
            f = f + w * np.exp(-((I - u[0]) ** 2 + (J - u[1]) ** 2 + (K - u[2]) ** 2) / T) / (np.pi * T) ** 1.5
        base.append(f.ravel())
    ft = torch.as_tensor(np.array(base), device=device)[torch.arange(P, device=device) % 3].contiguous()
    sur = SpectralSurrogate(N, L, (2 * L / N) ** 3, 0.38, 1.0, max_batch=8, device=device, seed=1)
    mom, alone = (torch.full((P, 8), float("nan"), dtype=torch.float64, device=device) for _ in range(2))
    x = torch.empty((P, 512), dtype=torch.float32, device=device)
    lt, lt1 = (torch.full((P,), float("nan"), dtype=torch.float32, device=device) for _ in range(2))
    print("moments alone", N, P, flush=True)
    sur.encode(ft, P, mom, x, lt)
    sur.encode(ft, P, alone, None, lt1)
    torch.cuda.synchronize()
    assert torch.equal(mom[:, :6], alone[:, :6]) and torch.equal(lt, lt1)
    assert not alone[:, 6:].any()
    for i in range(min(P, 3)):
        assert np.abs(alone[i, :6].cpu().numpy() - S.encode(base[i], N, L)[0][:6]).max() < 1e-10
