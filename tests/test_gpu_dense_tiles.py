"""The dense strict product over its four workgroup tiles (32 x 32, 64 x 32,
64 x 64 and 128 x 64 outputs), at the edges of the tiles and of the k chunks
(32 or 64): one chunk and several, whole and not, with the operands' rows
aligned and not, padded leading dimensions and both orientations of A.
test_dispatch_coverage.py checks that the shapes reach every tile so.

Bar: bit for bit the oracle's cpu_gemm (math.cpp:377-438), denormal products
included; NaN where it has NaN."""
import numpy as np
import pytest

from oracle import oracle as O
from pyflamert_amd import rocm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = rocm.Context(0)
    yield c
    c.close()


SHAPES = [
    # 32 x 32 tiles: K around its chunk of 64 and down to 1, and of several chunks
    (1, 1, 33), (31, 3, 1), (33, 63, 65), (32, 64, 32), (65, 65, 31), (5, 129, 200), (40, 68, 7), (70, 132, 90),
    (33, 192, 100),
    # 64 x 32, 64 x 64 and 128 x 64 tiles (chunk 32), one row and column past them
    (513, 33, 3072), (512, 32, 3041), (1024, 31, 3073), (1025, 36, 3072), (4096, 65, 2047), (4097, 4, 2048),
    (512, 96, 3041), (500, 101, 3072), (513, 100, 3000), (500, 29, 3072),
    (1000, 96, 4096), (1001, 100, 4095), (1000, 97, 4000), (1000, 30, 4096),
    (1920, 256, 2048), (1921, 260, 2047), (1919, 257, 2048)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_dense_tiles_bit_exact(ctx, M, K, N):
    import torch

    rng = np.random.default_rng(M + 7 * K + 13 * N)
    B = rng.standard_normal((K, N)).astype(np.float32)
    Cb = rng.standard_normal(N).astype(np.float32)
    for ta in (0, 1):
        A = rng.standard_normal((K, M) if ta else (M, K)).astype(np.float32)
        A.flat[::5] *= np.float32(1e-30)  # products down among the denormals
        A.flat[1::97] = np.float32(1e-41)
        A.flat[::1013] = np.inf
        print(f"dense tiles M={M} K={K} N={N} transA={ta}", flush=True)
        for alpha, C_ in ((1.0, Cb), (-0.75, Cb[:min(N, 7)])):
            if M * K * N > 3e8 and (alpha == 1.0) == bool(ta):
                continue  # (the oracle takes seconds)
            R = O.orc_gemm(A, B * np.float32(1e-9), C_, alpha, 1.5, ta, 0)
            ldb, ldy = N + 3, N + 1
            dB = torch.full((K, ldb), float("nan"), device="cuda")
            dB[:, :N] = torch.from_numpy(B * np.float32(1e-9)).cuda()
            dC = torch.from_numpy(np.ascontiguousarray(C_)).cuda()
            for off in (0, 1):  # A on a 16-byte boundary and past one
                dA = torch.empty(A.size + off, device="cuda")
                dA[off:] = torch.from_numpy(A).cuda().reshape(-1)
                dY = torch.full((M, ldy), 7.0, device="cuda")
                torch.cuda.synchronize()
                ctx.gemm_dense_dev(dA.data_ptr() + 4 * off, M, K, dB.data_ptr(), N, dY.data_ptr(), transA=ta,
                                   alpha=alpha, beta=1.5, C_ptr=dC.data_ptr(), c_size=C_.size, ldb=ldb, ldy=ldy)
                ctx.synchronize()
                Y = dY.cpu().numpy()
                assert (Y[:, N:] == 7.0).all()
                nan = np.isnan(R)
                assert np.array_equal(np.isnan(Y[:, :N]), nan)
                assert np.array_equal(Y[:, :N].view(np.uint32)[~nan], R.view(np.uint32)[~nan]), (ta, alpha, off)


def test_more_columns_than_32_wide_tiles_reach(ctx):
    """A launch takes fewer than 2^32 threads along a row of outputs: from 2^29
    columns on only the 64-column tiles serve, also a single row."""
    import torch

    N = (1 << 29) + 5
    B = torch.arange(N, dtype=torch.int32, device="cuda").remainder_(1 << 20).to(torch.float32)
    Y = torch.full((N,), 7.0, device="cuda")
    A = torch.tensor([0.75], device="cuda")
    torch.cuda.synchronize()
    print(f"dense 1 x 1 x {N}", flush=True)
    ctx.gemm_dense_dev(A.data_ptr(), 1, 1, B.data_ptr(), N, Y.data_ptr())
    ctx.synchronize()
    assert torch.equal(Y, 0.75 * B)  # exact: 20-bit integers
