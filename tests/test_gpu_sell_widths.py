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


@pytest.mark.parametrize("M,K,widths", [
    (700, 768, (9, 11, 12, 15, 1023)),  # one chunk
    (768, 1500, (13, 1024)),            # two chunks, 12 waves at 1024
    (3001, 2049, (9, 37, 99, 130, 255)),
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
