"""Products whose output lies over their activation: calls whose activation is
not a whole 16-byte-aligned operand of the large tiles, or is one row, used to
be served from a copy of it, so Y could be A or X, and still can: the routes
that read the activation in place leave such calls to the copy.

Bar: the bits of the same call with an output of its own; bf16, whose float
sums take another order on another route, twice the forward error bound.  The weights have far
more rows than the GPU's workgroups hold at once, so the last ones start when
the first have written."""
import numpy as np
import pytest

from pyflamert_amd import _lib, rocm, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = rocm.Context(0)
    yield c
    c.close()


def both(ctx, buf, x, y_at, y_elems, dtype, call):
    """call(x_ptr, y_ptr) with an output apart and with one y_at bytes into buf,
    where x lies at the start: the two outputs."""
    import torch

    n = x.numel() * x.element_size()
    buf[:n] = x.reshape(-1).view(torch.uint8)
    apart = torch.empty(y_elems, dtype=dtype, device="cuda")
    torch.cuda.synchronize()
    call(buf.data_ptr(), apart.data_ptr())
    call(buf.data_ptr(), buf.data_ptr() + y_at)
    ctx.synchronize()
    size = y_elems * apart.element_size()
    return apart.view(torch.uint8).cpu().numpy(), buf[y_at:y_at + size].cpu().numpy()


@pytest.mark.parametrize("Mb,values", [(1, "f32"), (1, "i8"), (2, "f32"), (12, "f32"), (16, "i8"), (33, "f32")])
def test_gemm_over_its_activation(ctx, Mb, values):
    import torch

    M, K = 60000, 1024
    ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.02, 0.5, 0.02, seed=70)
    W = ctx.csr_upload(M, K, ip, ix, q, row_scales=sc) if values == "i8" else \
        ctx.csr_upload(M, K, ip, ix, workloads.dequant_rows(ip, q, sc))
    A = torch.from_numpy(workloads.dense_normal((Mb, K), 1.0, seed=71)).cuda()
    buf = torch.empty(4 * Mb * (M + K), dtype=torch.uint8, device="cuda")
    # once for the copies the products build
    ctx.gemm_csr_dev(A.data_ptr(), Mb, K, W, buf.data_ptr(), mode="strict")
    for y_at in (0, 2 * K):
        print(f"Gemm over its activation: {values} Mb={Mb} offset {y_at}", flush=True)
        want, got = both(ctx, buf, A, y_at, Mb * M, torch.float32,
                         lambda a, y: ctx.gemm_csr_dev(a, Mb, K, W, y, mode="strict"))
        assert np.array_equal(want, got)
    W.free()


@pytest.mark.parametrize("N", [16, 48])
def test_sp24_over_its_activation(ctx, N):
    import torch

    M, K = 40000, 256
    rng = np.random.default_rng(N)
    w = workloads.keep_top2_of_4(rng.standard_normal((M, K), dtype=np.float32))
    q, s = workloads.symmetric_int8_rows(w)
    Wi, Wb = ctx.sp24_pack(q, s), ctx.sp24_pack(workloads.bf16_bits_rne(w))
    x8 = torch.from_numpy(rng.integers(0, 256, (K, N)).astype(np.uint8)).cuda()
    xb = torch.from_numpy(workloads.bf16_bits_rne(rng.standard_normal((K, N), dtype=np.float32)).view(np.int16)).cuda()
    buf = torch.empty(4 * M * N, dtype=torch.uint8, device="cuda")
    L = _lib.load()
    calls = {
        "int8 requantised": (x8, torch.int8, lambda x, y: Wi.gemm_i8_dev(x, N, y, x_scale=0.05, out="i8", out_scale=2.0)),
        "int8 accumulators": (x8, torch.int32, lambda x, y: Wi.gemm_i8_dev(x, N, y, out="i32")),
        "uint8": (x8, torch.float32, lambda x, y: Wi.gemm_q_dev(x, True, N, y, x_scale=0.05, x_zp=77, out="f32")),
        "bf16": (xb, torch.float32, lambda x, y: Wb.gemm_bf16_dev(x, N, y)),
        # x . W: N rows of K bytes
        "x.W": (x8, torch.float32, lambda x, y: _lib.check(L.pfr_sp24_gemm_qt_dev(
            ctx.handle, Wi.handle, x, _lib.PFR_U8, N, K, 0.05, 77, None, None, y, M))),
    }
    for name, (x, dtype, call) in calls.items():
        print(f"2:4 over its activation: {name} N={N}", flush=True)
        want, got = both(ctx, buf, x, 0, M * N, dtype, call)
        if name == "bf16":
            n = K // 2 + 8  # terms, and the sums across waves
            w64, x64 = ((b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
                        for b in (workloads.bf16_bits_rne(w), xb.cpu().numpy().view(np.uint16)))
            bound = 2 * n * 2.0 ** -24 / (1 - n * 2.0 ** -24) * (np.abs(w64) @ np.abs(x64))
            d = want.view(np.float32).astype(np.float64) - got.view(np.float32)
            assert (np.abs(d).reshape(M, N) <= bound).all()
        else:
            assert np.array_equal(want, got), name
