"""GPU parity of parallel_scan_fn (forward and adjoint) against the float64 oracle."""
import numpy as np
import pytest
import torch

from mamba_windows_cuda import parallel_scan_fn, parallel_scan_ref, workloads
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

TOL = {torch.float32: dict(rtol=1e-3, atol=1e-4), torch.float16: dict(rtol=1e-2, atol=1e-2),
       torch.bfloat16: dict(rtol=2e-2, atol=2e-2)}


def _np(t):
    return t.detach().cpu().double().numpy()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 32, 128, 16), (1, 16, 64, 8), (3, 5, 1000, 3), (2, 1, 1, 7),
                                   (2, 777, 40), (1, 300, 1024), (2, 129, 64)])
def test_pscan_forward_backward(dev, shape, dtype):
    print(f"case pscan shape={shape} dtype={dtype}", flush=True)
    g = torch.Generator().manual_seed(len(shape) * 100 + shape[-2])
    A = (0.5 + 0.5 * torch.rand(shape, generator=g)).to(dtype)
    X = torch.randn(shape, generator=g).to(dtype)
    dH = torch.randn(shape, generator=g).to(dtype)
    Ad = A.to(dev).requires_grad_(True)
    Xd = X.to(dev).requires_grad_(True)
    H = parallel_scan_fn(Ad, Xd)
    H.backward(dH.to(dev))
    torch.cuda.synchronize()
    ref = orc.pscan_fwd(A, X)
    np.testing.assert_allclose(_np(H), ref, **TOL[dtype])
    # adjoint with the oracle's own H (the kernel's H differs only by rounding)
    rdA, rdX = orc.pscan_bwd(A, torch.from_numpy(ref), dH)
    np.testing.assert_allclose(_np(Xd.grad), rdX, **TOL[dtype])
    np.testing.assert_allclose(_np(Ad.grad), rdA, **TOL[dtype])


# Narrow sequences run in tiles of 8 or 16 columns by 256 steps and 32 columns by 128, the columns of one lane each;
# a single tile along L has no look-back. Lengths around a run, a tile and two.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(768, 1, 8), (769, 7, 3), (768, 9, 1), (768, 65, 8), (768, 129, 5), (770, 257, 8),
                                   (768, 31, 16), (768, 33, 9), (767, 33, 16), (771, 64, 11), (768, 200, 16),
                                   (2048, 17, 32), (2049, 33, 17), (2047, 33, 32), (2048, 100, 25),
                                   (5, 513, 8), (3, 256, 16), (9, 1025, 10), (4, 129, 32)])
def test_pscan_narrow_sequences(dev, shape, dtype):
    print(f"case pscan narrow shape={shape} dtype={dtype}", flush=True)
    g = torch.Generator().manual_seed(shape[0] + shape[1])
    A = (0.5 + 0.5 * torch.rand(shape, generator=g)).to(dtype)
    A[:, 0] = float("inf")  # A_0 is not used
    X = torch.randn(shape, generator=g).to(dtype)
    dH = torch.randn(shape, generator=g).to(dtype)
    Ad, Xd = A.to(dev).requires_grad_(True), X.to(dev).requires_grad_(True)
    H = parallel_scan_fn(Ad, Xd)
    H.backward(dH.to(dev))
    torch.cuda.synchronize()
    A[:, 0] = 0
    ref = orc.pscan_fwd(A, X)
    rdA, rdX = orc.pscan_bwd(A, torch.from_numpy(ref), dH)
    np.testing.assert_allclose(_np(H), ref, **TOL[dtype])
    np.testing.assert_allclose(_np(Xd.grad), rdX, **TOL[dtype])
    np.testing.assert_allclose(_np(Ad.grad), rdA, **TOL[dtype])


# Pairs of 16-bit columns: 33 to 64 and more, whole and ragged column blocks, and the odd widths, fewer tiles and
# misaligned tensors that stay with single columns. Tickets are shared from 1024 tiles on: (7, 2100, 1282) in 16 bits
# has 77 pair blocks of 17 tiles in groups of 39 and 38, in fp32 147 blocks in groups of 49; (4, 2100, 1050) shares them
# in fp32 only (68 blocks in groups of 34), (65, 2100, 64) in every type, with single columns (33 and 32). (1101, 33, .)
# have one tile along L and more than 1024 in all.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,offset", [((128, 5, 34), 0), ((130, 128, 64), 0), ((64, 130, 66), 0),
                                          ((64, 257, 62), 1), ((3, 2049, 382), 0), ((3, 2049, 382), 1), ((3, 2049, 381), 0),
                                          ((2, 300, 1050), 0), ((4, 2100, 1050), 0), ((7, 2100, 1282), 0),
                                          ((65, 2100, 64), 1), ((1, 129, 130), 0),
                                          ((1101, 33, 64), 0), ((1101, 33, 128), 0)])
def test_pscan_column_pairs(dev, shape, offset, dtype):
    print(f"case pscan pairs shape={shape} offset={offset} dtype={dtype}", flush=True)
    g = torch.Generator().manual_seed(shape[0] + shape[1])
    A = (0.5 + 0.5 * torch.rand(shape, generator=g)).to(dtype)
    X, dH = (torch.randn(shape, generator=g).to(dtype) for _ in range(2))

    def put(t):  # contiguous, `offset` elements into its storage
        s = torch.empty(t.numel() + offset, dtype=dtype, device=dev)[offset:].view(shape)
        return s.copy_(t.to(dev)).requires_grad_(True)

    Ad, Xd = put(A), put(X)
    H = parallel_scan_fn(Ad, Xd)
    H.backward(dH.to(dev))
    torch.cuda.synchronize()
    ref = orc.pscan_fwd(A, X)
    rdA, rdX = orc.pscan_bwd(A, torch.from_numpy(ref), dH)
    np.testing.assert_allclose(_np(H), ref, **TOL[dtype])
    np.testing.assert_allclose(_np(Xd.grad), rdX, **TOL[dtype])
    np.testing.assert_allclose(_np(Ad.grad), rdA, **TOL[dtype])


def _range_inputs(kind, a, shape, dtype):
    """Sequences whose coefficients multiply out of fp32's range over a run, a tile or two while the scan itself stays
    in it. zero: nothing enters before the scan's last 20 steps (the adjoint's: before its first 20). tiny: 1e-30
    enters first, and grows. inf: an infinity enters early and stays, whatever the decay."""
    L = shape[1]
    g = torch.Generator().manual_seed(L + shape[2])
    A = torch.full(shape, a)
    X, dH = torch.zeros(shape), torch.zeros(shape)
    if kind == "zero":
        A[:, :24] = A[:, -24:] = 0.5
        X[:, -20:] = torch.randn(shape[0], 20, shape[2], generator=g)
        dH[:, :20] = torch.randn(shape[0], 20, shape[2], generator=g)
    elif kind == "tiny":  # up to 1e-30 * a^n <= 1e15, from the start of a run on
        n = int(np.log(1e45) / np.log(abs(a)))
        lo = L // 64 * 32
        A[:, :lo] = 1.0
        A[:, lo + n:] = 1.0
        X[:, 0] = dH[:, -1] = 1e-30
    else:
        X[:, 10, ::2] = float("inf")
        X[:, 10, 1::2] = -float("inf")
        dH[:, -10] = X[:, 10]
        X[:, 3] = 1.0
    return A.to(dtype), X.to(dtype), dH.to(dtype)


# Narrow and wide tiles, pairs (128 columns in 16 bits), several tiles along L and one; mean coefficients that leave
# fp32 over 2 tiles (1.3), one (1.5, 3), a run of 16 or 32 steps (300; 0.01 downwards).
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(3, 1024, 8), (2, 1100, 16), (3, 1024, 32), (2, 1024, 64), (40, 1024, 128),
                                   (3, 250, 16)])
@pytest.mark.parametrize("kind,a", [("zero", 1.3), ("zero", 1.5), ("zero", -3.0), ("zero", 300.0), ("tiny", 1.5),
                                    ("tiny", 300.0), ("inf", 0.5), ("inf", 0.01)])
def test_pscan_coefficient_range(dev, kind, a, shape, dtype):
    print(f"case pscan range kind={kind} a={a} shape={shape} dtype={dtype}", flush=True)
    if kind == "tiny" and dtype == torch.float16:
        dtype = torch.float32  # 1e-30 is not an fp16 value
    A, X, dH = _range_inputs(kind, a, shape, dtype)
    Ad, Xd = A.to(dev).requires_grad_(True), X.to(dev).requires_grad_(True)
    H = parallel_scan_fn(Ad, Xd)
    H.backward(dH.to(dev))
    torch.cuda.synchronize()
    ref = orc.pscan_fwd(A, X)
    rdA, rdX = orc.pscan_bwd(A, H.detach().cpu(), dH)  # dA = G * H: from the H that the backward is given
    if kind == "zero":
        assert np.isfinite(ref).all() and np.isfinite(rdX).all()
    np.testing.assert_allclose(_np(H), ref, **TOL[dtype])
    np.testing.assert_allclose(_np(Xd.grad), rdX, **TOL[dtype])
    np.testing.assert_allclose(_np(Ad.grad), rdA, **TOL[dtype])


def test_pscan_matches_reference_loop_and_ignores_A0(dev):
    """parallel_scan_ref semantics (pscan.py:153-171): H_0 = X_0 whatever A_0 is."""
    g = torch.Generator().manual_seed(2)
    A = torch.rand(2, 3, 50, 4, generator=g)
    X = torch.randn(2, 3, 50, 4, generator=g)
    H = parallel_scan_fn(A.to(dev), X.to(dev)).cpu()
    torch.testing.assert_close(H, parallel_scan_ref(A, X), rtol=1e-5, atol=1e-5)
    A2 = A.clone()
    A2[:, :, 0] = 77.0
    assert torch.equal(parallel_scan_fn(A2.to(dev), X.to(dev)).cpu(), H)


def test_pscan_config4b(dev):
    """(4, 65536, 1024) fp32 with a ~ U(0.9, 1), b ~ N(0, 1), against the float64 scan."""
    a, b = workloads.pscan_inputs()
    H = parallel_scan_fn(a.to(dev), b.to(dev))
    torch.cuda.synchronize()
    ref = orc.pscan_fwd(a, b)
    np.testing.assert_allclose(_np(H), ref, rtol=1e-3, atol=1e-4)


def test_scan_beyond_2_31_elements(dev):
    """(4, 2^20, 1024) fp32, 2^32 elements per tensor (the last sequence starts 3*2^30 elements in, its
    look-back chains are 8192 tiles long): the forward and the adjoint address with 64-bit offsets.
    Checked by restarting the scan: the last 4096 steps of the last sequence equal a scan of those
    steps whose first input folds in the state before them, and the adjoint's last steps equal the
    adjoint of that shorter scan (it depends only on later steps)."""
    from mamba_windows_cuda.pscan import pscan_check

    S, L, C, T = 4, 1 << 20, 1024, 4096
    print(f"case scan beyond 2^31 elements ({S}, {L}, {C})", flush=True)
    g = torch.Generator(device=dev).manual_seed(5)
    A = torch.rand(S, L, C, generator=g, device=dev).mul_(0.1).add_(0.9).requires_grad_(True)
    X = torch.randn(S, L, C, generator=g, device=dev).requires_grad_(True)
    H = parallel_scan_fn(A, X)
    dH = torch.randn(S, L, C, generator=g, device=dev)
    H.backward(dH)
    t0 = L - T
    with torch.no_grad():
        At = A[S - 1:, t0:].clone()
        Xt = X[S - 1:, t0:].clone()
        Xt[:, 0] += At[:, 0] * H[S - 1:, t0 - 1]
    At.requires_grad_(True)
    Xt.requires_grad_(True)
    Ht = parallel_scan_fn(At, Xt)
    Ht.backward(dH[S - 1:, t0:])
    pscan_check()
    torch.cuda.synchronize()
    torch.testing.assert_close(H[S - 1:, t0:], Ht, rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(X.grad[S - 1:, t0:], Xt.grad, rtol=1e-4, atol=1e-4)
    # dA_t = g_t * H_{t-1}: the restarted scan's first step has no H_{t-1} of its own
    torch.testing.assert_close(A.grad[S - 1:, t0 + 1:], At.grad[:, 1:], rtol=1e-4, atol=1e-4)
    del A, X, H, dH
    torch.cuda.empty_cache()  # hand the ~100 GB back before the next test
