"""GPU parity of tg_csr_spmm (the HIP SpMV/SpMM behind MatrixCSR::Dot) against the oracle.

Bars: FP64 within 1e-12 normwise relative error (max|Y-Y_ref|/max|Y_ref|, the reference's
metric) and inside the per-entry rounding bound gamma_{L+3}(|alpha||A||X| + |beta||Y|);
FP32 inside the same bound with u = 2^-24 and within sqrt(eps_f32) normwise (the
reference's own rule, Unit_Test_SpMM/main.cpp:144).  Structure-free cases with small
integers are compared bit for bit.
"""
import itertools

import numpy as np
import pytest
import torch

import oracle
from helpers import dense_of, random_csr_np, rel_err, spmm_bound
from tensors_amd import _capi as capi
from tensors_amd import generators as gen
from tensors_amd.sparse import MatrixCSR, spmm_raw

pytestmark = pytest.mark.gpu

ALPHAS = [-1.0, 0.0, 1.0, 2.0, np.pi]
BETAS = [-1.0, 0.0, 1.0, np.pi]


def to_dev(a, dev, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    return t if dtype is None else t.to(dtype)


def run_gpu(dev, rp, ci, val, m, n, alpha, X, beta, Y0, k, rp_dtype=torch.int64, NRHS=0, use_jp=False,
            ldX=None, ldY=None):
    dt = torch.float64 if X.dtype == np.float64 else torch.float32
    rpd = to_dev(rp, dev).to(rp_dtype)
    cid = to_dev(ci, dev)
    vd = None if val is None else to_dev(val, dev, dt)
    Xd = to_dev(X, dev, dt)
    Yd = to_dev(Y0, dev, dt)
    jp, blocks = None, 0
    if use_jp:
        blocks = capi.lib().tg_csr_default_blocks(m, int(rp[m]), k)
        jp = torch.empty(blocks + 1, dtype=torch.int32, device=dev)
        capi.call("tg_csr_job_pointers", m, rpd.data_ptr(), capi.I64 if rp_dtype == torch.int64 else capi.I32,
                  blocks, jp.data_ptr(), 0)
    st = spmm_raw(m, n, int(rp[m]), rpd, cid, vd, alpha, Xd, ldX or X.shape[1], beta, Yd, ldY or Y0.shape[1], k,
                  NRHS, jp, blocks, None)
    torch.cuda.synchronize()
    return st, Yd.cpu().numpy()


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 16, 32, 64, 100, 130])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_spmm_alpha_beta_grid(cuda, k, dtype):
    m, n = 300, 257
    rp, ci, val = random_csr_np(m, n, 0.06, seed=k, empty_rows=0.1, dtype=dtype)
    rng = np.random.default_rng(k)
    X = rng.uniform(-1, 1, (n, k)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (m, k)).astype(dtype)
    u = 2.0 ** -53 if dtype == np.float64 else 2.0 ** -24
    for alpha, beta in itertools.product(ALPHAS, BETAS):
        st, Y = run_gpu(cuda, rp, ci, val, m, n, alpha, X, beta, Y0, k)
        assert st == 0
        Yo = Y0.copy()
        assert oracle.spmm(rp, ci, val, m, n, alpha, X, k, beta, Yo, k, k) == 0
        bound = spmm_bound(m, n, rp, ci, val.astype(np.float64), alpha, X.astype(np.float64), beta,
                           Y0.astype(np.float64), u)
        exact = alpha * (dense_of(m, n, rp, ci, val.astype(np.float64)) @ X.astype(np.float64)) \
            + (beta * Y0.astype(np.float64) if beta != 0 else 0)
        if alpha == 0.0:
            exact = beta * Y0.astype(np.float64)
        assert np.all(np.abs(Y.astype(np.float64) - exact) <= bound), (alpha, beta)
        tol = 1e-12 if dtype == np.float64 else np.sqrt(np.finfo(np.float32).eps)
        assert rel_err(Y, Yo) <= tol, (alpha, beta, rel_err(Y, Yo))


@pytest.mark.parametrize("rp_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("use_jp", [False, True])
@pytest.mark.parametrize("k", [1, 4, 16])
def test_index_types_and_partition(cuda, rp_dtype, use_jp, k):
    m, n = 2000, 1500
    rp, ci, val = random_csr_np(m, n, 0.01, seed=3, empty_rows=0.05)
    rng = np.random.default_rng(0)
    X = rng.integers(-6, 7, (n, k)).astype(np.float64)
    Y0 = rng.integers(-6, 7, (m, k)).astype(np.float64)
    vi = rng.integers(-3, 4, len(ci)).astype(np.float64)
    st, Y = run_gpu(cuda, rp, ci, vi, m, n, 2.0, X, -1.0, Y0, k, rp_dtype=rp_dtype, use_jp=use_jp)
    assert st == 0
    Yo = Y0.copy()
    oracle.spmm(rp, ci, vi, m, n, 2.0, X, k, -1.0, Yo, k, k)
    assert np.array_equal(Y, Yo)  # exact integer arithmetic: bit-exact


def test_binary_matrix(cuda):
    m, n, k = 500, 400, 8
    rp, ci, _ = random_csr_np(m, n, 0.02, seed=4, empty_rows=0.1)
    X = np.random.default_rng(1).integers(-9, 10, (n, k)).astype(np.float64)
    Y0 = np.full((m, k), np.nan)
    st, Y = run_gpu(cuda, rp, ci, None, m, n, 1.0, X, 0.0, Y0, k)
    assert st == 0
    assert np.array_equal(Y, dense_of(m, n, rp, ci, None) @ X)


def test_beta_zero_nan_and_empty_rows(cuda):
    m, n = 400, 300
    rp, ci, val = random_csr_np(m, n, 0.02, seed=5, empty_rows=0.3)
    empty = np.diff(rp) == 0
    for k in (1, 4, 16):
        X = np.ones((n, k))
        st, Y = run_gpu(cuda, rp, ci, val, m, n, 1.0, X, 0.0, np.full((m, k), np.nan), k)
        assert st == 0 and np.all(np.isfinite(Y)) and np.all(Y[empty] == 0.0)
        st, Y = run_gpu(cuda, rp, ci, val, m, n, 1.0, X, 1.0, np.full((m, k), np.inf), k)
        assert np.all(np.isinf(Y[empty]))


def test_strided_and_misaligned(cuda):
    m, n, k, ld = 333, 222, 6, 11
    rp, ci, val = random_csr_np(m, n, 0.05, seed=6)
    rng = np.random.default_rng(2)
    Xf = rng.uniform(-1, 1, (n, ld))
    Yf = rng.uniform(-1, 1, (m, ld))
    st, Y = run_gpu(cuda, rp, ci, val, m, n, 1.5, Xf, -0.5, Yf, k, ldX=ld, ldY=ld)
    assert st == 0
    Yo = Yf.copy()
    oracle.spmm(rp, ci, val, m, n, 1.5, Xf, ld, -0.5, Yo, ld, k)
    assert rel_err(Y[:, :k], Yo[:, :k]) <= 1e-12
    assert np.array_equal(Y[:, k:], Yf[:, k:])
    # X starting one element off a 16-byte boundary forces the scalar-load path
    dev = cuda
    Xbuf = torch.zeros(n * 4 + 1, dtype=torch.float64, device=dev)
    Xv = Xbuf[1:].view(n, 4)
    Xv.copy_(torch.from_numpy(Xf[:, :4]))
    Yd = torch.zeros(m, 4, dtype=torch.float64, device=dev)
    st = spmm_raw(m, n, int(rp[m]), to_dev(rp, dev), to_dev(ci, dev), to_dev(val, dev), 1.0, Xv, 4, 0.0, Yd,
                  4, 4)
    Yo = np.zeros((m, 4))
    oracle.spmm(rp, ci, val, m, n, 1.0, np.ascontiguousarray(Xf[:, :4]), 4, 0.0, Yo, 4, 4)
    assert st == 0 and rel_err(Yd.cpu().numpy(), Yo) <= 1e-12


def test_noop_error_cases(cuda):
    m = n = 64
    rp, ci, val = random_csr_np(m, n, 0.1, seed=7)
    dev = cuda
    Xd = torch.ones(n, 2, dtype=torch.float64, device=dev)
    snap = Xd.clone()
    st = spmm_raw(m, n, int(rp[m]), to_dev(rp, dev), to_dev(ci, dev), to_dev(val, dev), 1.0, Xd, 2, 0.0, Xd, 2,
                  2)
    assert st == capi.ERR_ALIAS and torch.equal(Xd, snap)
    Yd = torch.full((m, 2), 7.0, dtype=torch.float64, device=dev)
    st = spmm_raw(m, n, int(rp[m]), to_dev(rp, dev), to_dev(ci, dev), to_dev(val, dev), 1.0, Xd, 2, 0.0, Yd, 2,
                  2, NRHS=4)
    assert st == capi.ERR_NRHS and torch.all(Yd == 7.0)
    # empty matrix (nnz == 0): every row empty
    rp0 = np.zeros(m + 1, np.int64)
    st, Y = run_gpu(dev, rp0, np.zeros(0, np.int32), np.zeros(0), m, n, 1.0, np.ones((n, 3)), 0.0,
                    np.full((m, 3), np.nan), 3)
    assert st == 0 and np.all(Y == 0.0)
    # m == 0 and nrhs == 0 are no-ops
    assert capi.lib().tg_csr_spmm(0, n, 0, to_dev(rp0, dev).data_ptr(), capi.I64, None, None, capi.F64, 1.0,
                                  Xd.data_ptr(), 2, 0.0, Yd.data_ptr(), 2, 2, 0, None, 0, None) == 0


def test_grid_laplacian_256_config(cuda):
    """GridLaplacian(256), FP64, nrhs 1 and 16, alpha = 1, beta = 0 (configs[0] shape)."""
    rp, ci, val = oracle.grid_laplacian(256, 1.0)
    m = n = 256 * 256
    assert len(ci) == 326656
    for k in (1, 16):
        X = gen.uniform(1001, n * k).reshape(n, k)
        st, Y = run_gpu(cuda, rp, ci, val, m, n, 1.0, X, 0.0, np.zeros((m, k)), k)
        Yo = np.zeros((m, k))
        oracle.spmm(rp, ci, val, m, n, 1.0, X, k, 0.0, Yo, k, k)
        assert st == 0 and rel_err(Y, Yo) <= 1e-12


@pytest.mark.parametrize("k", [1, 4, 16, 64])
def test_random_csr_1e5(cuda, k):
    """configs[1] generator at n = 1e5 (oracle-sized): FP64 and FP32."""
    m = n = 100_000
    rp, ci, v64, v32 = gen.random_csr(m, n, seed=2002, want32=True)
    X = gen.uniform(2002, n * k).reshape(n, k)
    Yo = np.zeros((m, k))
    oracle.spmm(rp, ci, v64, m, n, 1.0, X, k, 0.0, Yo, k, k, threads=8)
    st, Y = run_gpu(cuda, rp, ci, v64, m, n, 1.0, X, 0.0, np.zeros((m, k)), k)
    assert st == 0 and rel_err(Y, Yo) <= 1e-12
    X32 = X.astype(np.float32)
    st, Y32 = run_gpu(cuda, rp, ci, v32, m, n, 1.0, X32, 0.0, np.zeros((m, k), np.float32), k)
    Yo32 = np.zeros((m, k), np.float32)
    oracle.spmm(rp, ci, v32, m, n, 1.0, X32, k, 0.0, Yo32, k, k, threads=8)
    assert st == 0 and rel_err(Y32, Yo32) <= 1e-5


@pytest.mark.parametrize("k", [1, 16, 64])
def test_random_csr_full_size_properties(cuda, k):
    """n = 1e6 (full configs[1] size): linearity A(X1 + X2) = A X1 + A X2 and a sampled
    set of rows checked against the oracle on the corresponding sub-matrix."""
    m = n = 1_000_000
    rp, ci, v64, _ = gen.random_csr(m, n, seed=2002)
    dev = cuda
    rpd, cid, vd = to_dev(rp, dev), to_dev(ci, dev), to_dev(v64, dev)
    X1 = torch.from_numpy(gen.uniform(7, n * k).reshape(n, k)).to(dev)
    X2 = torch.from_numpy(gen.uniform(8, n * k).reshape(n, k)).to(dev)
    Y1 = torch.empty(m, k, dtype=torch.float64, device=dev)
    Y2 = torch.empty_like(Y1)
    Y3 = torch.empty_like(Y1)
    nnz = int(rp[m])
    for X, Y in ((X1, Y1), (X2, Y2), (X1 + X2, Y3)):
        assert spmm_raw(m, n, nnz, rpd, cid, vd, 1.0, X, k, 0.0, Y, k, k) == 0
    torch.cuda.synchronize()
    lin = (Y3 - Y1 - Y2).abs().max().item() / Y3.abs().max().item()
    assert lin < 1e-13
    rows = np.sort(np.random.default_rng(0).choice(m, 2000, replace=False))
    srp = np.r_[0, np.cumsum(rp[rows + 1] - rp[rows])].astype(np.int64)
    idx = np.concatenate([np.arange(rp[r], rp[r + 1]) for r in rows])
    Yo = np.zeros((len(rows), k))
    X1h = X1.cpu().numpy()
    oracle.spmm(srp, ci[idx], v64[idx], len(rows), n, 1.0, X1h, k, 0.0, Yo, k, k)
    assert rel_err(Y1.cpu().numpy()[rows], Yo) <= 1e-12


def test_matrixcsr_dot_overloads(cuda):
    """Python mirror of MatrixCSR::Dot: Tensor1 / Tensor2 overloads and the shape check."""
    m, n = 120, 90
    rp, ci, val = random_csr_np(m, n, 0.1, seed=10)
    A = MatrixCSR(rp, ci, val, m, n)
    x = torch.from_numpy(np.random.default_rng(0).uniform(-1, 1, n)).to(cuda)
    y = torch.zeros(m, dtype=torch.float64, device=cuda)
    assert A.Dot(1.0, x, 0.0, y) == 0
    assert rel_err(y.cpu().numpy(), dense_of(m, n, rp, ci, val) @ x.cpu().numpy()) <= 1e-12
    X = torch.from_numpy(np.random.default_rng(1).uniform(-1, 1, (n, 5))).to(cuda)
    Y = torch.zeros(m, 5, dtype=torch.float64, device=cuda)
    assert A.Dot(2.0, X, 0.0, Y, use_job_ptr=True) == 0
    assert rel_err(Y.cpu().numpy(), 2.0 * dense_of(m, n, rp, ci, val) @ X.cpu().numpy()) <= 1e-12
    Ybad = torch.full((m + 1, 5), 3.0, dtype=torch.float64, device=cuda)
    assert A.Dot(1.0, X, 0.0, Ybad) == capi.ERR_SHAPE and torch.all(Ybad == 3.0)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_spmv_kernel_variants(cuda, variant, dtype):
    """Both nrhs == 1 kernels (streaming and team-per-row) against the oracle, including
    rows longer than one streaming chunk and blocks of more than 1024 rows."""
    L = capi.lib()
    old = L.tg_tune_get(b"spmv_kernel")
    try:
        assert L.tg_tune_set(b"spmv_kernel", variant) == 0
        # long rows (up to 5000 nonzeros) next to many empty / short rows
        rng = np.random.default_rng(11)
        m, n = 6000, 7000
        lens = rng.integers(0, 4, m)
        lens[rng.choice(m, 5, replace=False)] = rng.integers(2500, 5000, 5)
        rp = np.r_[0, np.cumsum(lens)].astype(np.int64)
        ci = np.concatenate([np.sort(rng.choice(n, L_, replace=False)) for L_ in lens]).astype(np.int32)
        val = rng.normal(size=len(ci)).astype(dtype)
        X = rng.uniform(-1, 1, (n, 1)).astype(dtype)
        Y0 = rng.uniform(-1, 1, (m, 1)).astype(dtype)
        for alpha, beta in ((1.0, 0.0), (-2.0, 1.0), (0.5, np.pi)):
            st, Y = run_gpu(cuda, rp, ci, val, m, n, alpha, X, beta, Y0, 1)
            Yo = Y0.copy()
            oracle.spmm(rp, ci, val, m, n, alpha, X, 1, beta, Yo, 1, 1)
            tol = 1e-12 if dtype == np.float64 else 1e-5
            assert st == 0 and rel_err(Y, Yo) <= tol
    finally:
        L.tg_tune_set(b"spmv_kernel", old)


def skewed_csr(m, n, mean, seed, longest):
    """Rows of 0 to about 2 mean nonzeros (every ninth empty) and one of `longest`."""
    rng = np.random.default_rng(seed)
    lens = np.minimum(rng.integers(0, 2 * mean + 1, m), n)
    lens[::9] = 0
    lens[m // 2] = min(longest, n)
    rp = np.zeros(m + 1, np.int64)
    np.cumsum(lens, out=rp[1:])
    ci = np.concatenate([np.sort(rng.choice(n, L, replace=False)) for L in lens]).astype(np.int32)
    return rp, ci, rng.integers(-4, 5, int(rp[-1])).astype(np.float64)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 11, 33, 37])
@pytest.mark.parametrize("mean,longest", [(3, 40), (20, 3000)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("plan", [False, True], ids=["call", "plan"])
def test_spmm_kernel_choices_are_exact(cuda, k, mean, longest, dtype, plan):
    """The streaming kernel (up to 4 columns; a row spans its chunks) and the row per lane
    group (a last vector moved back where its width does not divide k, groups of every
    width), with leading dimensions that leave no row aligned, pointers offset by one
    element, int32 / int64 row pointers, binary matrices, empty rows and every beta rule.
    Small integers: every sum is exact, so the bits are the oracle's; the columns beyond k
    and the element before Y stay as they were."""
    m, n = 700, 3100
    rp, ci, val = skewed_csr(m, n, mean, 5 * k + mean, longest)
    if plan and mean == 20:  # no long row: the plan's middling rule
        rp, ci, val = skewed_csr(m, n, mean, 5 * k + mean, 2 * mean)
    rng = np.random.default_rng(k)
    ldx, ldy = k + 3, k + 1
    X = rng.integers(-3, 4, (n, ldx)).astype(dtype)
    Y0 = rng.integers(-3, 4, (m, ldy)).astype(dtype)
    dt = torch.float64 if dtype == np.float64 else torch.float32

    def shifted(a):  # one element past the allocation's alignment
        flat = torch.zeros(a.size + 1, dtype=dt, device=cuda)
        flat[0] = 99.0
        flat[1:] = to_dev(a.reshape(-1), cuda, dt)
        return flat, flat[1:].view(*a.shape)

    rpd = to_dev(rp if k % 2 else rp.astype(np.int32), cuda)
    cid, vd = to_dev(ci, cuda), to_dev(val, cuda, dt)
    for a, alpha, beta in ((vd, 1.0, 0.0), (vd, -2.0, 1.0), (None, 2.0, 2.0), (vd, 1.0, -1.0)):
        _, Xd = shifted(X)
        whole, Yd = shifted(Y0)
        if plan:
            from tensors_amd.sparse import SlicePlan
            P = SlicePlan(m, n, len(ci), rpd, cid)
            assert P.spmm(a, alpha, Xd, ldx, beta, Yd, ldy, k) == 0
        else:
            assert spmm_raw(m, n, len(ci), rpd, cid, a, alpha, Xd, ldx, beta, Yd, ldy, k) == 0
        Yo = Y0.astype(np.float64).copy()
        oracle.spmm(rp, ci, None if a is None else val, m, n, alpha, X.astype(np.float64), ldx, beta, Yo, ldy, k)
        assert np.array_equal(Yd.cpu().numpy().astype(np.float64), Yo), (alpha, beta)
        assert whole[0].item() == 99.0


def test_narrow_bands_take_no_slices(cuda):
    """A banded matrix whose window of X fits an L2 is not sliced and keeps no re-laid copy;
    the same sizes with scattered columns do and are."""
    n = 600_000
    i = np.arange(n)
    rp = np.arange(0, 3 * n + 1, 3, dtype=np.int64)
    band = np.stack([(i - 40) % n, i, (i + 40) % n], 1)
    band[:40, 0], band[-40:, 2] = 80, n - 120  # no wrap-around
    band = np.sort(band, 1)
    far = np.sort(np.stack([i, (i * 7919 + 11) % n, (i * 104729 + 5) % n], 1), 1)
    X = torch.ones(n, 2, dtype=torch.float64, device=cuda)
    for cols, sliced in ((band, False), (far, True)):
        A = MatrixCSR(rp, cols.reshape(-1).astype(np.int32), np.arange(3 * n) % 5 - 2.0, n, n)
        Y = torch.zeros_like(X)
        assert A.Dot(1.0, X, 0.0, Y) == 0
        v = A.device_arrays(torch.float64)[2]
        assert A.Plan().uses_split(v, 2) == sliced and (A.Plan().slices(torch.float64, 2) > 0) == sliced
        want = (np.arange(3 * n) % 5 - 2.0).reshape(n, 3).sum(1)
        assert np.array_equal(Y.cpu().numpy(), np.stack([want, want], 1))


def test_stream_handle_is_the_current_stream(cuda):
    """Products go to torch's current stream: the default one, a `with torch.cuda.stream` block's
    (nested, and of each thread), or the one passed."""
    import threading

    from tensors_amd.sparse import stream_handle

    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    default = torch.cuda.current_stream().cuda_stream
    assert stream_handle() == default and stream_handle(a) == a.cuda_stream
    seen = []
    with torch.cuda.stream(a):
        t = threading.Thread(target=lambda: seen.append(stream_handle()))
        t.start()
        t.join()
        with torch.cuda.stream(b):
            assert stream_handle() == b.cuda_stream and stream_handle(a) == a.cuda_stream
        assert stream_handle() == a.cuda_stream
    assert stream_handle() == default and seen == [default]


@pytest.mark.parametrize("m,nrhs,dtype", [(1 << 20, 1, torch.float64), (1 << 20, 3, torch.float64),
                                          (1 << 20, 8, torch.float32), ((1 << 27) + 3, 2, torch.float32)])
def test_int32_row_pointers_up_to_the_last_entry(cuda, m, nrhs, dtype):
    """2^31 - 1 nonzeros under int32 row pointers: the loops over nonzeros step past 2^31 at the
    end of the last rows unless they count what is left (rows streamed, a row per wave, short
    rows).  A binary matrix, columns 0 but for the last 3000 entries, integer X: every sum is
    exact."""
    nnz = (1 << 31) - 1
    if torch.cuda.mem_get_info()[0] < (48 << 30):
        pytest.skip("needs 48 GB of free device memory")
    rp = torch.arange(m + 1, dtype=torch.int64, device=cuda) * nnz // m
    ci = torch.zeros(nnz, dtype=torch.int32, device=cuda)
    ci[nnz - 3000:] = 1
    X = torch.arange(1, 2 * nrhs + 1, dtype=dtype, device=cuda).reshape(2, nrhs)
    Y = torch.full((m, nrhs), -1.0, dtype=dtype, device=cuda)
    print(f"2^31 - 1 nonzeros, {m} rows, {nrhs} columns", flush=True)
    assert spmm_raw(m, 2, nnz, rp.to(torch.int32), ci, None, 1.0, X, nrhs, 0.0, Y, nrhs, nrhs) == 0
    ones = (rp[1:] - rp[:-1].clamp(min=nnz - 3000)).clamp_(min=0)  # entries of a row in column 1
    want = (rp[1:] - rp[:-1] - ones).to(dtype)[:, None] * X[0] + ones.to(dtype)[:, None] * X[1]
    assert torch.equal(Y, want)


@pytest.mark.parametrize("dtype,k", [(torch.float64, 15), (torch.float64, 16), (torch.float32, 30), (torch.float32, 32)])
def test_short_rows_with_vectors_that_fill_the_cache(cuda, dtype, k):
    """X and Y of 240-256 MB with a matrix of 44-64 MB beside them: the short-row form that
    streams A.  Five diagonals and X of small integers, so every sum is exact; an update of Y,
    rows cut off at both ends, a last lane that shares columns with the one before (k = 15, 30)."""
    n = 1000003
    i = torch.arange(n, device=cuda)
    off = (-1000, -1, 0, 1, 1000)
    cols = torch.stack([i + d for d in off], 1)
    keep = (cols >= 0) & (cols < n)
    vals = torch.stack([(i * 7 + 3 * j) % 11 - 5 for j in range(5)], 1).to(dtype)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=cuda)
    torch.cumsum(keep.sum(1), 0, out=rp[1:])
    A = MatrixCSR.from_device(rp.to(torch.int32), cols[keep].to(torch.int32), vals[keep], n, n)
    X = ((i[:, None] * 5 + torch.arange(k, device=cuda) * 3) % 13 - 6).to(dtype)
    Y = ((i[:, None] + torch.arange(k, device=cuda)) % 9).to(dtype)
    want = -Y
    for j, d in enumerate(off):
        lo, hi = max(0, -d), min(n, n - d)
        want[lo:hi] += 2 * vals[lo:hi, j, None] * X[lo + d:hi + d]
    A.Dot(2.0, X, -1.0, Y)
    assert torch.equal(Y, want)


@pytest.mark.parametrize("longest", [9, 64, 65, 66, 700])
@pytest.mark.parametrize("dtype,k", [(torch.float64, 5), (torch.float64, 11), (torch.float64, 32), (torch.float32, 7),
                                     (torch.float32, 18), (torch.float32, 60)])
def test_short_rows_with_one_long_row(cuda, dtype, k, longest):
    """Rows of about five nonzeros and one of up to / more than 64, which sends the product to the
    form that fetches a chunk of pairs ahead: chunks of 8, 16 and 32 pairs and their
    remainders, empty rows beside the long one.  Integers: every sum is exact."""
    import scipy.sparse as sp

    m, n = 3001, 2003
    rng = np.random.default_rng(longest * 100 + k)
    S = sp.random(m, n, density=5 / n, format="csr", random_state=3)
    S.data = rng.integers(-4, 5, S.nnz).astype(np.float64)
    S = S.tolil()
    S[1000:1040] = 0
    S[1017, rng.choice(n, longest, replace=False)] = 3
    S = S.tocsr()
    S.sort_indices()
    assert np.diff(S.indptr).max() >= longest
    X = rng.integers(-3, 4, (n, k)).astype(np.float64)
    A = MatrixCSR(S.indptr.astype(np.int32), S.indices, S.data.astype(np.float64 if dtype == torch.float64 else np.float32),
                  m, n)
    Y = torch.full((m, k), 7.0, dtype=dtype, device=cuda)
    A.Dot(1.0, torch.from_numpy(X).to(cuda).to(dtype), 0.0, Y)
    assert np.array_equal(Y.double().cpu().numpy(), S @ X)
