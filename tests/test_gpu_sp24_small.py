"""The small-tile 2:4 kernel (few columns or few tiles): every tile it has, from
the activation's transpose and reading it in place, the remainders of its
rows, columns and k steps, waves without a step, and each form that runs on
it: int8 W.X with the three outputs, uint8 with a zero point (host value and
device scalar), the x.W form from aligned rows and through the padded copy,
and bf16, with non-finite values in the last k row too.
test_dispatch_coverage.py checks that the shapes reach every tile in each form.

Bar: int32 and requantised int8 exact, float outputs exact to the bit (the
exact accumulator times RN(w_scale * x_scale), quant_ops.cpp:435); bf16 within
the forward error bound of a float32 sum of K / 2 terms in any order."""
import numpy as np
import pytest

from pyflamert_amd import _lib, rocm, workloads

pytestmark = pytest.mark.gpu

# tiles of 16 x 16, 32 x 16, 32 x 32, 64 x 32 and 64 x 64 outputs; K of one
# step or less, of fewer steps than waves, and of no whole step
SHAPES = [(1, 4, 1), (17, 100, 3), (100, 500, 17), (300, 1156, 16), (4100, 608, 9), (4096, 1024, 64),
          (3985, 900, 49), (4096, 1040, 128), (4000, 512, 121), (4096, 1028, 200), (4033, 640, 195), (1088, 640, 512),
          (17000, 100, 16), (500, 272, 32), (12000, 100, 16), (3001, 640, 65)]


@pytest.fixture(scope="module")
def ctx():
    c = rocm.Context(0)
    yield c
    c.close()


def weight(rng, M, K):
    w = workloads.keep_top2_of_4(rng.standard_normal((M, K), dtype=np.float32))
    return workloads.symmetric_int8_rows(w)


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_int8(ctx, M, K, N):
    import torch

    rng = np.random.default_rng(M + K + N)
    q, s = weight(rng, M, K)
    W = ctx.sp24_pack(q, s)
    print(f"small 2:4 int8 M={M} K={K} N={N}", flush=True)
    X = rng.integers(-128, 128, (K, N)).astype(np.int8)
    acc = (q.astype(np.float64) @ X.astype(np.float64)).astype(np.int64)
    assert np.array_equal(W.gemm_i8(X, out="i32"), acc.astype(np.int32))
    f = acc.astype(np.float32) * (s * np.float32(0.05))[:, None]
    assert np.array_equal(W.gemm_i8(X, x_scale=0.05, out="f32").view(np.uint32), f.view(np.uint32))
    for out_scale, zp in ((2.0, 0), (0.7, -5)):
        p = workloads.round_half_away(f * (np.float32(1.0) / np.float32(out_scale)))
        r = np.clip(p.astype(np.int64) + zp, -128, 127).astype(np.int8)
        assert np.array_equal(W.gemm_i8(X, x_scale=0.05, out="i8", out_scale=out_scale, out_zp=zp), r)
    # a uint8 activation with a zero point, columns inside wider rows and not
    for ldx, ldy in ((N + 5, N + 3), (N, N)):
        U = rng.integers(0, 256, (K, ldx)).astype(np.uint8)
        accu = (q.astype(np.float64) @ (U[:, :N].astype(np.float64) - 77)).astype(np.int64)
        dU = torch.from_numpy(U).cuda()
        dY = torch.full((M, ldy), -1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        W.gemm_q_dev(dU.data_ptr(), True, N, dY.data_ptr(), x_zp=77, out="i32", ldx=ldx, ldy=ldy)
        ctx.synchronize()
        Y = dY.cpu().numpy()
        assert np.array_equal(Y[:, :N], accu.astype(np.int32)) and (Y[:, N:] == -1).all()


@pytest.mark.parametrize("M,K,T", SHAPES)
def test_x_w_form(ctx, M, K, T):
    import torch

    rng = np.random.default_rng(M + 3 * K + T)
    q, s = weight(rng, M, K)
    W = ctx.sp24_pack(q, s)
    L = _lib.load()
    for u8, ldx in ((True, K), (False, K + 16 - K % 16), (True, K + 1)):
        print(f"small 2:4 x.W M={M} K={K} T={T} u8={u8} ldx={ldx}", flush=True)
        X = rng.integers(0, 256, (T, ldx)).astype(np.uint8)
        x, zp = X[:, :K].astype(np.int64), 131
        if not u8:
            x, zp = X[:, :K].view(np.int8).astype(np.int64), -9
        acc = ((x - zp).astype(np.float64) @ q.T.astype(np.float64)).astype(np.int64)
        R = acc.astype(np.float32) * (s * np.float32(0.03))[None, :]
        dX = torch.from_numpy(X).cuda()
        dS = torch.tensor([0.03], dtype=torch.float32, device="cuda")
        dZ = torch.tensor([zp & 255], dtype=torch.uint8, device="cuda")
        dY = torch.full((T, M + 2), 5.0, device="cuda")
        torch.cuda.synchronize()
        _lib.check(L.pfr_sp24_gemm_qt_dev(ctx.handle, W.handle, dX.data_ptr(), _lib.PFR_U8 if u8 else _lib.PFR_I8, T,
                                          ldx, 0.03, 0 if u8 else zp, dS.data_ptr() if u8 else None,
                                          dZ.data_ptr() if u8 else None, dY.data_ptr(), M + 2))
        ctx.synchronize()
        Y = dY.cpu().numpy()
        assert np.array_equal(Y[:, :M].view(np.uint32), R.view(np.uint32)) and (Y[:, M:] == 5.0).all()


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_bf16(ctx, M, K, N):
    rng = np.random.default_rng(M + 5 * K + N)
    wb = workloads.bf16_bits_rne(workloads.keep_top2_of_4(rng.standard_normal((M, K), dtype=np.float32)))
    xb = workloads.bf16_bits_rne(rng.standard_normal((K, N), dtype=np.float32))
    W = ctx.sp24_pack(wb)
    print(f"small 2:4 bf16 M={M} K={K} N={N}", flush=True)
    Y = W.gemm_bf16(xb).astype(np.float64)
    w = (wb.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x = (xb.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    n = K // 2 + 8  # terms, and the sums across waves
    bound = n * 2.0 ** -24 / (1 - n * 2.0 ** -24) * (np.abs(w) @ np.abs(x))
    assert (np.abs(Y - w @ x) <= bound + 1e-30).all()
    # inf and NaN in the last k row: the rows read past it (K is no whole step)
    # must not repeat it against the packing's zeros
    xi = xb.copy()
    xi[K - 1, 0], xi[K - 1, N // 2] = 0x7F80, 0x7FC0
    odd = np.zeros(N, bool)
    odd[[0, N // 2]] = True
    Z = W.gemm_bf16(xi).astype(np.float64)
    assert np.array_equal(Z[:, ~odd], Y[:, ~odd])
    assert np.array_equal(~np.isfinite(Z[:, odd]), np.repeat(w[:, K - 1:] != 0, odd.sum(), axis=1))
