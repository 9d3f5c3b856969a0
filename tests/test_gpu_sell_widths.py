"""The column-slice kernel where its launch changes form: 9 to 15 columns, widths
that are no whole 16-byte piece (staged a float per lane, or through the Gemm
form's padded transpose), 4 to 16 waves per workgroup, one chunk and several,
and int8 weights, whose copy holds the dequantised values.

Bar: strict mode bit for bit the oracle's sparse_matmul on the (dequantised)
weight; fast mode within the forward error bound of any summation order."""
import numpy as np
import pytest

from oracle import oracle as O
from pyflamert_amd import rocm, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = rocm.Context(0)
    yield c
    c.close()


def build_copies(W, K):
    """Products until the weight holds both sliced-ELL copies, which an int8 weight
    builds after some (fast products would do with the strict one for long)."""
    X = np.ones((K, 64), np.float32)
    for mode in ("fast", "strict"):
        b = W.device_bytes()
        for _ in range(60):
            W.spmm(X, mode=mode)
            if W.device_bytes() > b:
                break
        assert W.device_bytes() > b, mode


@pytest.mark.parametrize("M,K,widths", [
    (700, 768, (9, 11, 12, 15, 1023)),  # one chunk
    (768, 1500, (13, 1024)),            # two chunks, 12 waves at 1024
    (3001, 2049, (9, 37, 99, 130, 255)),
    (3070, 250, (1024,)),               # one chunk, 8 waves in the Gemm form for its many rounds
    (40, 3000, (10, 33))])
def test_widths(ctx, M, K, widths):
    import torch

    for values in ("f32", "i8"):
        if values == "f32":
            ip, ix, v = workloads.csr_uniform(M, K, 0.08, 0.02, seed=M + K)
            W, dense = ctx.csr_upload(M, K, ip, ix, v), v
        else:
            ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.08, 0.5, 0.02, seed=M + K)
            W, dense = ctx.csr_upload(M, K, ip, ix, q, row_scales=sc), workloads.dequant_rows(ip, q, sc)
        build_copies(W, K)
        Wd = workloads.csr_to_dense(M, K, ip, ix, dense)
        for N in widths:
            print(f"column slices {values} M={M} K={K} N={N}", flush=True)
            X = workloads.dense_normal((K, N), 1.0, seed=N)
            R = O.orc_csr_spmm(M, K, ip, ix, dense, X)
            assert np.array_equal(W.spmm(X, mode="strict").view(np.uint32), R.view(np.uint32))
            # columns inside wider, unaligned rows
            dX = torch.full((K, N + 3), float("nan"), device="cuda")
            dX[:, :N] = torch.from_numpy(X).cuda()
            dY = torch.full((M, N + 1), 3.0, device="cuda")
            torch.cuda.synchronize()
            W.spmm_dev(dX.data_ptr(), N, dY.data_ptr(), ldx=N + 3, ldy=N + 1, mode="strict")
            ctx.synchronize()
            Y = dY.cpu().numpy()
            assert np.array_equal(Y[:, :N].view(np.uint32), R.view(np.uint32)) and (Y[:, N:] == 3.0).all()
            # the Gemm form: bias of one row, of another length, alpha
            A = np.ascontiguousarray(X.T)
            for alpha, csz in ((1.0, M), (-0.5, 7)):
                b = workloads.dense_normal((csz,), 0.1, seed=csz)
                G = O.orc_gemm(A, np.ascontiguousarray(Wd.T), b, alpha, 1.5, 0, 0)
                assert np.array_equal(ctx.gemm_csr(A, W, alpha=alpha, beta=1.5, C_=b).view(np.uint32),
                                      G.view(np.uint32)), (alpha, csz)
            F = W.spmm(X, mode="fast").astype(np.float64)
            exact = Wd.astype(np.float64) @ X.astype(np.float64)
            mag = np.abs(Wd).astype(np.float64) @ np.abs(X).astype(np.float64)
            terms = np.diff(ip)[:, None] + 2
            g = terms * 2.0 ** -24
            assert (np.abs(F - exact) <= g / (1 - g) * mag + 1e-30).all()
        W.free()


@pytest.mark.parametrize("M,K,N,alpha,act", [
    (16, 64, 9, 1.0, None),       # one slab, one chunk
    (500, 784, 32, 1.0, "relu"),  # one chunk, a staging wave
    (515, 1020, 33, -2.0, None),  # alpha applied before the test for infinities
    (515, 2052, 47, 1.0, "gelu"),
    (3100, 1500, 200, 1.0, None),  # two chunks, 12 waves
    (4096, 2000, 256, 1.0, None)])  # two chunks, 16 waves
def test_nonfinite_rule_in_kernel(ctx, M, K, N, alpha, act):
    """A handle with the dense kernels' semantics, Gemm form: the launch that
    stages the activation itself makes exactly the outputs NaN that cpu_gemm
    on the zero-filled weight does, as do the launches after a transpose."""
    import torch

    rng = np.random.default_rng(M + K + N)
    ip, ix, v = workloads.csr_uniform(M, K, 0.06, 0.05, seed=M + N)
    W = ctx.csr_upload(M, K, ip, ix, v)
    W.dense_semantics()
    build_copies(W, K)
    Wt = np.ascontiguousarray(workloads.csr_to_dense(M, K, ip, ix, v).T)
    b = workloads.dense_normal((M,), 0.1, seed=M)
    A = workloads.dense_normal((N, K), 1.0, seed=N)
    A[0, K - 1], A[N // 2, 0], A[N - 1, K // 2] = np.inf, np.nan, -np.inf
    if alpha != 1.0:
        A[2, 3] = 3e38  # infinite once scaled
    db, dA = torch.from_numpy(b).cuda(), torch.from_numpy(A).cuda()
    dY = torch.empty((N, M), device="cuda")
    for bad in (True, False):
        if not bad:  # and finite activations leave every bit alone
            A = np.where(np.abs(A) < 100, A, 0).astype(np.float32)
            dA = torch.from_numpy(A).cuda()
        print(f"non-finite rule M={M} K={K} N={N} bad={bad}", flush=True)
        torch.cuda.synchronize()
        W_args = dict(relu=act == "relu", gelu=act == "gelu")
        ctx.gemm_csr_dev(dA.data_ptr(), N, K, W, dY.data_ptr(), alpha, 1.0, db.data_ptr(), M, mode="strict", **W_args)
        ctx.synchronize()
        Y = dY.cpu().numpy()
        with np.errstate(all="ignore"):
            R = O.orc_gemm(A, Wt, b, alpha, 1.0, 0, 0)
        if act == "relu":
            R = np.where(0 < R, R, 0).astype(np.float32)
        if act == "gelu":  # the fused epilogue has a separate Gelu's bits
            R = ctx.gelu(R)
        assert np.array_equal(np.isnan(Y), np.isnan(R))
        ok = ~np.isnan(R)
        assert np.array_equal(Y[ok].view(np.uint32), R[ok].view(np.uint32))
    W.free()


@pytest.mark.parametrize("values", ["f32", "i8"])
def test_rows_that_repeat_columns(ctx, values):
    """Rows that list a column several times: where one has more entries in a
    chunk than the chunk has columns, the fast copy keeps storage order."""
    M, K, N = 40, 2100, 17
    rng = np.random.default_rng(90)
    cols = []
    for r in range(M):
        n = 1500 if r in (3, 20) else int(rng.integers(0, 300))
        c = rng.integers(0, 1000 if n == 1500 else K, n)  # more than 1024 entries in columns 0 .. 999
        cols.append(np.sort(c))
    ip = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    ix = np.concatenate(cols)
    q = rng.integers(1, 100, len(ix)).astype(np.int8)
    sc = rng.uniform(0.001, 0.002, M).astype(np.float32)
    vals = workloads.dequant_rows(ip, q, sc)
    X = workloads.dense_normal((K, N), 1.0, seed=91)
    W = ctx.csr_upload(M, K, ip, ix, vals) if values == "f32" else ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
    build_copies(W, K)
    print(f"rows that repeat columns: {values}", flush=True)
    R = O.orc_csr_spmm(M, K, ip, ix, vals, X)
    assert np.array_equal(W.spmm(X, mode="strict").view(np.uint32), R.view(np.uint32))
    F = W.spmm(X, mode="fast").astype(np.float64)
    exact, mag = np.zeros((M, N)), np.zeros((M, N))
    for r in range(M):
        v, x = vals[ip[r]:ip[r + 1], None].astype(np.float64), X[ix[ip[r]:ip[r + 1]]].astype(np.float64)
        exact[r], mag[r] = (v * x).sum(0), np.abs(v * x).sum(0)
    g = (np.diff(ip)[:, None] + 2) * 2.0 ** -24
    assert (np.abs(F - exact) <= g / (1 - g) * mag + 1e-30).all()
    W.free()
