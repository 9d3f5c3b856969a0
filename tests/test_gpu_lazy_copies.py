"""Derived copies built on first use, through pfr_csr_device_bytes: a handle
starts with the CSR itself (uint16 columns when K <= 65536, values, row
pointers, row scales), the row-block table and the merge-path partition;
the first product that runs on the nnz-balanced copy (fast, 2 <= N <= 8),
the row-chain copy (strict, N <= 8) or the sliced-ELL copy (float32,
N >= 16) builds it, and later products reuse it; int8 weights and 9 to 15
columns build theirs after some products in place.  Products match the oracle
as everywhere else (strict bit for bit, fast within 1e-5 normwise).  A
product captured into a HIP graph while its copy is still pending builds
nothing and reads the CSR in place: in strict mode the same bits as the
copy's kernel, on every replay, before and after the copy exists."""
import sys

import numpy as np
import pytest

from oracle import oracle as O
from pyflamert_amd import workloads

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def close_normwise(Y, R, tol=1e-5):
    Y = np.asarray(Y, np.float64)
    R = np.asarray(R, np.float64)
    scale = max(float(np.abs(R).max()), 1e-30)
    return bool(np.abs(Y - R).max() <= tol * scale)


@pytest.fixture(scope="module")
def ctx():
    from pyflamert_amd import rocm

    c = rocm.Context(0)
    yield c
    c.close()


def test_int8_decode_weight_footprint(ctx):
    """4096 x 4096 int8 decode weight at 30 % (lognormal rows): about 3 bytes
    per nonzero after upload, unchanged by batch-1 fast products (the
    merge-path kernel reads the CSR in place); the first batch-8 fast product
    adds the balanced copy (int8 value + uint16 offset per padded entry), the
    first strict product the row-chain copy, each once."""
    M, K = 4096, 4096
    ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.3, 0.5, 0.02, seed=41)
    nnz = len(ix)
    vals = workloads.dequant_rows(ip, q, sc)
    W = ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
    rng = np.random.default_rng(42)
    x1 = rng.standard_normal(K).astype(np.float32)
    x8 = rng.standard_normal((K, 8)).astype(np.float32)
    b0 = W.device_bytes()
    say(f"int8 {M}x{K} nnz={nnz}: {b0 / nnz:.4f} B/nnz after upload")
    assert 3 * nnz <= b0 <= 3.1 * nnz
    Y = W.spmm(x1, mode="fast")
    assert W.device_bytes() == b0
    assert close_normwise(Y, O.orc_csr_spmm(M, K, ip, ix, vals, x1))
    Y8 = W.spmm(x8, mode="fast")
    b1 = W.device_bytes()
    say(f"after the first batch-8 fast product: {b1 / nnz:.4f} B/nnz")
    assert 3 * nnz <= b1 - b0 <= 3.2 * nnz
    assert close_normwise(Y8, O.orc_csr_spmm(M, K, ip, ix, vals, x8))
    assert np.array_equal(bits(W.spmm(x8, mode="fast")), bits(Y8))
    assert W.device_bytes() == b1
    Ys = W.spmm(x1, mode="strict")
    b2 = W.device_bytes()
    say(f"after the first strict product: {b2 / nnz:.4f} B/nnz")
    assert 3 * nnz <= b2 - b1 <= 3.3 * nnz
    assert np.array_equal(bits(Ys), bits(O.orc_csr_spmm(M, K, ip, ix, vals, x1)))
    Ys8 = W.spmm(x8, mode="strict")
    assert W.device_bytes() == b2
    assert np.array_equal(bits(Ys8), bits(O.orc_csr_spmm(M, K, ip, ix, vals, x8)))
    W.free()


@pytest.mark.parametrize("K", [3000, 70000])
def test_float_weight_copies_on_first_use(ctx, K):
    """Float32 weights, uint16 columns (K = 3000) and int32 ones (K =
    70000, past uint16): 6 and 8 bytes per nonzero after upload; N = 64
    builds the sliced-ELL copy, strict N = 3 the row-chain copy, fast N = 4
    the balanced copy (where K allows it); every product against the
    oracle."""
    M = 1500
    ip, ix, v = workloads.csr_uniform(M, K, 0.05 if K < 10000 else 0.004, 0.02, seed=K)
    nnz = len(ix)
    W = ctx.csr_upload(M, K, ip, ix, v)
    per = 6 if K <= 65536 else 8
    b = W.device_bytes()
    say(f"float32 {M}x{K} nnz={nnz}: {b / nnz:.4f} B/nnz after upload")
    assert per * nnz <= b <= per * nnz + 64 * M + (1 << 20)
    rng = np.random.default_rng(K + 1)
    for N, mode in ((64, "strict"), (64, "fast"), (3, "strict"), (4, "fast"), (1, "strict"), (8, "fast")):
        X = rng.standard_normal((K, N)).astype(np.float32)
        Y = W.spmm(X, mode=mode)
        R = O.orc_csr_spmm(M, K, ip, ix, v, X)
        nb = W.device_bytes()
        say(f"  N={N} {mode}: {nb / nnz:.4f} B/nnz")
        assert nb >= b
        b = nb
        if mode == "strict":
            assert np.array_equal(bits(Y), bits(R)), (N, mode)
        else:
            assert close_normwise(Y, R), (N, mode)
    W.free()


def test_capture_before_copy_reads_in_place(ctx):
    """Strict batch-1 and batch-4 products and a fast batch-8 one captured
    on a fresh int8 handle: the capture allocates nothing (device bytes
    unchanged), and each replay -- before the eager products build the
    copies and after -- gives the strict copies' bits and the fast result
    within 1e-5 normwise of the oracle."""
    import torch

    M, K = 2048, 3000
    ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.3, 0.5, 0.02, seed=43)
    vals = workloads.dequant_rows(ip, q, sc)
    W = ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
    g = torch.Generator(device="cuda").manual_seed(44)
    x1 = torch.randn((K, 1), device="cuda", generator=g)
    x4 = torch.randn((K, 4), device="cuda", generator=g)
    x8 = torch.randn((K, 8), device="cuda", generator=g)
    out = {k: torch.empty((M, n), device="cuda") for k, n in (("s1", 1), ("s4", 4), ("f8", 8))}

    def run(o):
        W.spmm_dev(x1.data_ptr(), 1, o["s1"].data_ptr(), mode="strict")
        W.spmm_dev(x4.data_ptr(), 4, o["s4"].data_ptr(), mode="strict")
        W.spmm_dev(x8.data_ptr(), 8, o["f8"].data_ptr(), mode="fast")

    main = torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()
    b0 = W.device_bytes()
    graph = torch.cuda.CUDAGraph()
    say(f"capture on a fresh {M}x{K} int8 handle")
    with torch.cuda.graph(graph):
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        run(out)
    ctx.set_stream(main)
    assert W.device_bytes() == b0
    R = {"s1": O.orc_csr_spmm(M, K, ip, ix, vals, x1.cpu().numpy()),
         "s4": O.orc_csr_spmm(M, K, ip, ix, vals, x4.cpu().numpy()),
         "f8": O.orc_csr_spmm(M, K, ip, ix, vals, x8.cpu().numpy())}
    eager = {k: torch.empty_like(v) for k, v in out.items()}
    for rep in range(3):
        for v in out.values():
            v.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        if rep == 1:
            run(eager)  # builds the row-chain and balanced copies
            torch.cuda.synchronize()
            assert W.device_bytes() > b0
            for k in ("s1", "s4"):
                assert np.array_equal(bits(eager[k].cpu().numpy()), bits(R[k])), k
            assert close_normwise(eager["f8"].cpu().numpy(), R["f8"])
        say(f"replay {rep}")
        for k in ("s1", "s4"):
            assert np.array_equal(bits(out[k].cpu().numpy()), bits(R[k])), (rep, k)
        assert close_normwise(out["f8"].cpu().numpy(), R["f8"]), rep
    del graph
    W.free()


@pytest.mark.parametrize("values", ["f32", "i8"])
@pytest.mark.parametrize("Mb", [4, 32])
def test_allocation_free_products_beside_a_build(ctx, values, Mb):
    """One thread's allocation-free products on its own stream, which wait for
    no build, while another thread's first products through the same handle
    build the row-chain, balanced and both sliced-ELL copies: each result is
    the oracle's, bit for bit, whether it read the CSR in place or a copy that
    was complete."""
    import threading

    import torch

    from pyflamert_amd import rocm

    M, K = 4096, 1536
    ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.2, 0.5, 0.02, seed=45)
    vals = workloads.dequant_rows(ip, q, sc)
    A = workloads.dense_normal((Mb, K), 1.0, seed=46)
    X = np.ascontiguousarray(A.T)
    R = O.orc_csr_spmm(M, K, ip, ix, vals, X).T
    other = rocm.Context(0)
    dA = torch.from_numpy(A).cuda()
    dY = torch.empty((Mb, M), device="cuda")
    torch.cuda.synchronize()
    for rep in range(4):
        W = ctx.csr_upload(M, K, ip, ix, vals) if values == "f32" else ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
        failed, done = [], threading.Event()

        def build():
            try:
                # (fast products would do with the strict copy for long)
                for mode in ("fast", "strict"):
                    b = W.device_bytes()
                    for _ in range(60):
                        Y = W.spmm(X, mode=mode)
                        if mode == "strict" and not np.array_equal(bits(Y), bits(R.T)):
                            failed.append("the building product")
                        if W.device_bytes() > b:
                            break
                    else:
                        failed.append(f"no copy: {mode}")
            except Exception as e:
                failed.append(repr(e))
            finally:
                done.set()

        t = threading.Thread(target=build)
        t.start()
        n, last = 0, False
        while not last:  # once more after the build
            last = done.is_set()
            other.gemm_csr_dev(dA.data_ptr(), Mb, K, W, dY.data_ptr(), mode="strict", noalloc=True)
            other.synchronize()
            n += 1
            if not np.array_equal(bits(dY.cpu().numpy()), bits(R)):
                failed.append(f"allocation-free product {n}")
                break
        t.join()
        say(f"{values} Mb={Mb} build {rep}: {n} allocation-free products beside it")
        assert not failed, failed
        W.free()
    other.close()


def test_two_threads_build_on_one_context(ctx):
    """Two threads building handles, from a host CSR and from a dense device
    weight, and their sliced-ELL copies on one context at once: one of them has
    the context's page-locked and counting buffers, the other memory of its
    own; every product is the oracle's."""
    import threading

    import torch

    N = 16
    work = []
    for i, (M, K) in enumerate(((2048, 1500), (3000, 700))):
        ip, ix, v = workloads.csr_uniform(M, K, 0.1, 0.02, seed=50 + i)
        X = workloads.dense_normal((K, N), 1.0, seed=60 + i)
        work.append((M, K, ip, ix, v, torch.from_numpy(workloads.csr_to_dense(M, K, ip, ix, v)).cuda(),
                     torch.from_numpy(X).cuda(), torch.empty((12, M, N), device="cuda"), O.orc_csr_spmm(M, K, ip, ix, v, X)))
    torch.cuda.synchronize()
    failed, start, handles = [], threading.Barrier(2), []

    def builds(i):
        M, K, ip, ix, v, D, dX, dY, _ = work[i]
        try:
            start.wait()
            for j in range(dY.shape[0]):
                W = ctx.csr_from_dense_dev(D.data_ptr(), M, K) if j % 2 else ctx.csr_upload(M, K, ip, ix, v)
                handles.append(W)
                W.spmm_dev(dX.data_ptr(), N, dY[j].data_ptr(), mode="strict")
        except Exception as e:
            failed.append(repr(e))

    say("two threads build on one context")
    threads = [threading.Thread(target=builds, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ctx.synchronize()
    assert not failed, failed
    for *_, dY, R in work:
        for Y in dY.cpu().numpy():
            assert np.array_equal(bits(Y), bits(R))
    for W in handles:
        W.free()


@pytest.mark.parametrize("values,M,K,N", [("i8", 4096, 1500, 12), ("i8", 512, 512, 64), ("f32", 3000, 768, 9),
                                          ("f32", 700, 2100, 15), ("i8", 2000, 4000, 200)])
def test_sliced_copy_built_once_it_pays(ctx, values, M, K, N):
    """An int8 weight, and a float32 one on 9 to 15 columns: the first product
    reads the CSR in place (nothing is allocated), a later one builds the
    sliced-ELL copy, once, and strict products have the oracle's bits on both
    sides; 16 columns of the float32 weight build theirs at once."""
    ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.1, 0.5, 0.02, seed=M + N)
    vals = workloads.dequant_rows(ip, q, sc)
    X = workloads.dense_normal((K, N), 1.0, seed=N)
    R = O.orc_csr_spmm(M, K, ip, ix, vals, X)
    for mode in ("strict", "fast"):
        W = ctx.csr_upload(M, K, ip, ix, vals) if values == "f32" else ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
        b, grew = W.device_bytes(), []
        for i in range(60):
            Y = W.spmm(X, mode=mode)
            assert np.array_equal(bits(Y), bits(R)) if mode == "strict" else close_normwise(Y, R), (mode, i)
            if W.device_bytes() != b:
                grew.append(i)
                b = W.device_bytes()
        say(f"{values} {M}x{K} N={N} {mode}: copy built by product {grew}")
        assert len(grew) == 1 and grew[0] > 0
        W.free()
    if values == "f32":
        W = ctx.csr_upload(M, K, ip, ix, vals)
        b = W.device_bytes()
        X = workloads.dense_normal((K, 16), 1.0, seed=1)
        assert np.array_equal(bits(W.spmm(X)), bits(O.orc_csr_spmm(M, K, ip, ix, vals, X)))
        assert W.device_bytes() > b
        W.free()


# hipMalloc that fails with hipErrorOutOfMemory above `limit` bytes.
NO_MEMORY_C = """
#include <stddef.h>
static int (*real)(void**, size_t);
static size_t limit = (size_t)-1;
static int refused;
void set_real(void* f) { real = (int (*)(void**, size_t))f; }
void set_limit(size_t n) { limit = n; }
int times_refused(void) { return refused; }
int hipMalloc(void** p, size_t n) {
    if (!real) return 3; /* hipErrorNotInitialized */
    if (n <= limit) return real(p, n);
    ++refused;
    *p = 0;
    return 2; /* hipErrorOutOfMemory */
}
"""

NO_MEMORY_PY = """
import ctypes, re, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # ahead of the HIP runtime, for this process
shim.set_limit.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import numpy as np, torch
from oracle import oracle as O
from pyflamert_amd import rocm, workloads
hip = re.search(r"(/\\S*libamdhip64\\S*)", open("/proc/self/maps").read()).group(1)
shim.set_real(ctypes.cast(ctypes.CDLL(hip).hipMalloc, ctypes.c_void_p))
ctx = rocm.Context(0)
M, K = 4096, 2000
ip, ix, q, sc = workloads.csr_int8_lognormal(M, K, 0.2, 0.5, 0.02, seed=47)
vals = workloads.dequant_rows(ip, q, sc)
for values, N in (("i8", 64), ("f32", 12)):
    X = workloads.dense_normal((K, N), 1.0, seed=N)
    R = O.orc_csr_spmm(M, K, ip, ix, vals, X)
    W = ctx.csr_upload(M, K, ip, ix, vals) if values == "f32" else ctx.csr_upload(M, K, ip, ix, q, row_scales=sc)
    b = W.device_bytes()
    W.spmm(X)  # the context's staging buffers
    assert W.device_bytes() == b
    shim.set_limit(1 << 20)
    before = shim.times_refused()
    for i in range(40):
        assert np.array_equal(W.spmm(X).view(np.uint32), R.view(np.uint32)), (values, i)
        assert np.abs(W.spmm(X, mode="fast") - R).max() <= 1e-5 * np.abs(R).max(), (values, i)
    assert W.device_bytes() == b
    refused = shim.times_refused() - before
    assert 2 <= refused < 60, refused  # tried, in both modes, and not by every product
    shim.set_limit(ctypes.c_size_t(-1).value)
    for i in range(40):
        assert np.array_equal(W.spmm(X).view(np.uint32), R.view(np.uint32)), (values, i)
    assert W.device_bytes() > b
    print(values, "copies refused", refused, "times, built when there was memory", flush=True)
"""


def test_no_memory_for_a_copy(ctx, tmp_path):
    """Where the sliced-ELL copy cannot be allocated, the products that did
    without it before stay in place, with the same bits, and build it once
    there is memory.  (A process of its own, whose hipMalloc refuses large
    requests from the host's side; the GPU's memory stays as it is.)"""
    import os
    import subprocess

    (tmp_path / "no_memory.c").write_text(NO_MEMORY_C)
    shim = str(tmp_path / "no_memory.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", shim, str(tmp_path / "no_memory.c")], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    say("products without memory for a copy, in a child process")
    r = subprocess.run([sys.executable, "-c", NO_MEMORY_PY, shim, root], capture_output=True, text=True, timeout=100)
    say(r.stdout, r.stderr[-2000:])
    assert r.returncode == 0 and r.stdout.count("built when there was memory") == 2
