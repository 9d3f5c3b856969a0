// Dense float32 products for weights above the sparse path's density gate:
// the arithmetic of the reference's dense kernels, cpu_gemm and cpu_matmul
// (src/backends/cpu/ops/math.cpp:268-438), bit for bit.  Each output is
// summed in ascending k from +0 with a separate multiply and add per term,
// the term being (alpha * a[i, k]) * b[k, j] as the reference evaluates it,
// then beta * c[(i * N + j) % c_size] is added; the fused activation is the
// same function of that value as the separate Relu / Gelu kernels.  So
// non-finite inputs propagate exactly as there: an inf or NaN activation
// meets every weight, zeros included.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace {

typedef float v32f __attribute__((ext_vector_type(32)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

// One k of a wave's tile as an outer product on the matrix unit: the f32 MFMA
// with a single k and C = 0 rounds each a * b once, to nearest, denormals
// kept (compared with the host's products over random bit patterns, denormal
// inputs and results among them: no difference in 13.6 million), so it is the
// reference's RN(a * b).  A wave's tile is WM x WN outputs, NV per lane, made
// by NA instructions one below the other: lane l supplies op(A) of tile row
// arow(l) + i * AR to instruction i and B of tile column bcol(l) to each, and
// its register v holds tile row crow(l, v) + i * AR, column ccol(l, v).
template <int NV>
struct Outer;
template <>
struct Outer<32> {  // two 32 x 32 blocks, one below the other
    static constexpr int WM = 64, WN = 32, KT = 32, NA = 1, AR = 64, OCC = 2;
    typedef v32f V;
    static __device__ __forceinline__ V mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, V(0.0f), 0, 0, 0);
    }
    static __device__ __forceinline__ int arow(int l) { return l; }
    static __device__ __forceinline__ int bcol(int l) { return l & 31; }
    static __device__ __forceinline__ int crow(int l, int v) {
        return 32 * (v >> 4) + 8 * ((v & 15) >> 2) + 4 * (l >> 5) + (v & 3);
    }
    static __device__ __forceinline__ int ccol(int l, int) { return l & 31; }
};
template <>
struct Outer<16> {  // 2 x 2 blocks of 16 x 16
    static constexpr int WM = 32, WN = 32, KT = 32, NA = 1, AR = 32, OCC = 3;
    typedef v16f V;
    static __device__ __forceinline__ V mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, V(0.0f), 0, 0, 0);
    }
    static __device__ __forceinline__ int arow(int l) { return 16 * (l >> 5) + (l & 15); }
    static __device__ __forceinline__ int bcol(int l) { return 16 * ((l >> 4) & 1) + (l & 15); }
    static __device__ __forceinline__ int crow(int l, int v) { return 16 * (v >> 3) + 4 * (l >> 4) + (v & 3); }
    static __device__ __forceinline__ int ccol(int l, int v) { return 16 * ((v >> 2) & 1) + (l & 15); }
};
struct Outer4x4 {  // 4 x 4 blocks of 4 x 4
    typedef v4f V;
    static __device__ __forceinline__ V mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, V(0.0f), 0, 0, 0);
    }
    static __device__ __forceinline__ int arow(int l) { return 4 * (l >> 4) + (l & 3); }
    static __device__ __forceinline__ int bcol(int l) { return l & 15; }
    static __device__ __forceinline__ int crow(int l, int v) { return 4 * (l >> 4) + v; }
    static __device__ __forceinline__ int ccol(int l, int) { return l & 15; }
};
template <>
struct Outer<8> : Outer4x4 {
    static constexpr int WM = 32, WN = 16, KT = 32, NA = 2, AR = 16, OCC = 4;
};
template <>
struct Outer<4> : Outer4x4 {
    static constexpr int WM = 16, WN = 16, KT = 64, NA = 1, AR = 16, OCC = 4;
};

// 256 threads: 2 x 2 waves, each a tile of Outer<NV>.  op(A) (scaled by alpha
// on the way: the reference's alpha * a) and B go through LDS in chunks of KT
// k, both with k contiguous (row pitch KT + 4 floats: a 16-byte read of 16
// rows covers all banks), so one 16-byte read per operand serves four k; two
// LDS buffers, and two register sets that hold the next two chunks' elements
// while the current one is multiplied.  Per k the wave issues one MFMA (the
// products) and NV v_add_f32 (the sums, in k order): the multiplies, which
// the strict result needs rounded apart from the adds, run on the matrix unit
// beside the adds instead of taking turns with them on the vector unit, so
// the bound is one add per term: 78.6 TFLOP/s instead of 39.3.
// The last chunk of a K that is no multiple of KT ends at K and holds +0
// where it repeats the chunk before (a K below KT: +0 from K on).  A term +0
// * +0 leaves every sum unchanged: a sum of products that starts at +0 is
// never -0 in round-to-nearest, and inf or NaN plus +0 is itself.  Tile rows
// and columns past M and N repeat the last one and are not written.
// AVEC: op(A) = A with 16-byte aligned rows.
// PART: K has a chunk of its own that is not whole, or no more than two chunks: the
// last chunk's padding is stepped over and no chunk loaded that no one reads.
// (A product of whole chunks that carries those two branches takes 2 % longer.)
template <int NV, bool TA, bool AVEC, bool PART>
__global__ __launch_bounds__(256, Outer<NV>::OCC) void k_gemm_dense(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb, int64_t M, int64_t N,
    int64_t K, float alpha, const float* __restrict__ C, int64_t c_size, float beta, int act,
    float* __restrict__ Y, int64_t ldy) {
    using O = Outer<NV>;
    constexpr int TM = 2 * O::WM, TN = 2 * O::WN, KT = O::KT, P = KT + 4;
    constexpr int QA = TM * KT / 1024, QB = TN * KT / 1024;  // four-k pieces per thread
    __shared__ __align__(16) float As[2][TM * P];            // As[.][i * P + k]
    __shared__ __align__(16) float Bs[2][TN * P];            // Bs[.][j * P + k]
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int64_t i0 = (int64_t)blockIdx.y * TM, j0 = (int64_t)blockIdx.x * TN;
    // piece i of this thread: tile row (op(A)) or column (B) x, k 4q .. 4q +
    // 3 of the chunk; consecutive threads read consecutive addresses
    auto a_x = [&](int i) { const int e = t + 256 * i; return TA ? e % TM : e / (KT / 4); };
    auto a_q = [&](int i) { const int e = t + 256 * i; return TA ? e / TM : e % (KT / 4); };
    auto b_x = [&](int i) { return (t + 256 * i) % TN; };
    auto b_q = [&](int i) { return (t + 256 * i) / TN; };
    const bool tiny = K < KT;
    const int nk = tiny ? 1 : (int)((K + KT - 1) / KT);
    const int tail = tiny ? 0 : (int)(nk * (int64_t)KT - K);  // k of the last chunk that the one before holds
    const int64_t ak = TA ? lda : 1;  // floats between k and k + 1 of op(A)
    // the chunk to load next; a K below KT has one chunk, loaded by clamped
    // addresses, and then reads its first element (never used)
    const float* pa[QA];
    const float* pb[QB];
#pragma unroll
    for (int i = 0; i < QA; ++i) {
        const int64_t r = min(i0 + a_x(i), M - 1);
        pa[i] = A + (TA ? r : r * lda) + (tiny ? 0 : 4 * a_q(i)) * ak;
    }
#pragma unroll
    for (int i = 0; i < QB; ++i) pb[i] = B + min(j0 + b_x(i), N - 1) + (tiny ? 0 : 4 * b_q(i)) * ldb;
    const int64_t au = tiny ? 0 : ak, bu = tiny ? 0 : ldb;
    struct Set {
        float a[QA][4], b[QB][4];
    };
    auto load = [&](Set& s, int c) {  // chunk min(c, nk - 1), and on to the one after it
#pragma unroll
        for (int i = 0; i < QA; ++i) {
            if constexpr (AVEC) {
                const v4f v = *reinterpret_cast<const v4f*>(pa[i]);
#pragma unroll
                for (int u = 0; u < 4; ++u) s.a[i][u] = v[u];
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) s.a[i][u] = pa[i][u * au];
            }
        }
#pragma unroll
        for (int i = 0; i < QB; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) s.b[i][u] = pb[i][u * bu];
        const int d = c + 2 < nk ? KT : (c + 2 == nk ? KT - tail : 0);
#pragma unroll
        for (int i = 0; i < QA; ++i) pa[i] += d * ak;
#pragma unroll
        for (int i = 0; i < QB; ++i) pb[i] += d * ldb;
    };
    auto load_tiny = [&](Set& s) {
#pragma unroll
        for (int i = 0; i < QA; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) s.a[i][u] = pa[i][min((int64_t)4 * a_q(i) + u, K - 1) * ak];
#pragma unroll
        for (int i = 0; i < QB; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) s.b[i][u] = pb[i][min((int64_t)4 * b_q(i) + u, K - 1) * ldb];
    };
    auto put = [&](const Set& s, int h, auto whole, int lo, int hi) {
#pragma unroll
        for (int i = 0; i < QA; ++i) {
            v4f v;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v[u] = alpha * s.a[i][u];  // (1.0f * a is a)
                if constexpr (!decltype(whole)::value) {
                    const int k = 4 * a_q(i) + u;
                    v[u] = k >= lo && k < hi ? v[u] : 0.0f;
                }
            }
            *reinterpret_cast<v4f*>(&As[h][a_x(i) * P + 4 * a_q(i)]) = v;
        }
#pragma unroll
        for (int i = 0; i < QB; ++i) {
            v4f v;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v[u] = s.b[i][u];
                if constexpr (!decltype(whole)::value) {
                    const int k = 4 * b_q(i) + u;
                    v[u] = k >= lo && k < hi ? v[u] : 0.0f;
                }
            }
            *reinterpret_cast<v4f*>(&Bs[h][b_x(i) * P + 4 * b_q(i)]) = v;
        }
    };
    auto store = [&](const Set& s, int c, int h) {
        // the chunk's own k: positions lo .. hi - 1
        const int lo = c + 1 == nk ? tail : 0, hi = tiny ? (int)K : KT;
        if (lo == 0 && hi == KT) put(s, h, std::true_type{}, lo, hi);
        else put(s, h, std::false_type{}, lo, hi);
    };
    const int wm = (w >> 1) * O::WM, wn = (w & 1) * O::WN;
    const int ao = (wm + O::arow(l)) * P, bo = (wn + O::bcol(l)) * P;
    constexpr int NA = O::NA;
    using V = typename O::V;
    V acc[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[i] = V(0.0f);
    struct Op {
        v4f a[NA], b;  // four k
    };
    auto fetch = [&](Op& o, int h, int k) {
#pragma unroll
        for (int i = 0; i < NA; ++i) o.a[i] = *reinterpret_cast<const v4f*>(&As[h][ao + i * O::AR * P + k]);
        o.b = *reinterpret_cast<const v4f*>(&Bs[h][bo + k]);
    };
    // four k: the products of k + 1 are under way while k's are added
    auto group = [&](const Op& cur, const Op& nxt, V (&p)[NA], bool more) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            V n[NA];
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                n[i] = p[i];
                if (u < 3) n[i] = O::mul(cur.a[i][u + 1], cur.b[u + 1]);
                else if (more) n[i] = O::mul(nxt.a[i][0], nxt.b[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                acc[i] = acc[i] + p[i];
                asm volatile("" : "+v"(acc[i]));  // here, not after all the products
                p[i] = n[i];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto multiply = [&](int h) {
        Op cur;
        fetch(cur, h, 0);
        V p[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i) p[i] = O::mul(cur.a[i][0], cur.b[0]);
#pragma unroll
        for (int k = 0; k < KT; k += 4) {
            Op nxt = cur;
            if (k + 4 < KT) fetch(nxt, h, k + 4);
            group(cur, nxt, p, k + 4 < KT);
            cur = nxt;
        }
    };
    // the k positions k0 .. k1 - 1 of a chunk that is not all its own, both
    // multiples of 4 (walking the padding too, 4096 x 4096 outputs took 62 us
    // at K = 33 and 40 at K = 1 in 64 x 64 tiles; now 44 and 28)
    auto multiply_part = [&](int h, int k0, int k1) {
        Op cur;
        fetch(cur, h, k0);
        V p[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i) p[i] = O::mul(cur.a[i][0], cur.b[0]);
#pragma unroll 1
        for (int k = k0; k < k1; k += 4) {
            Op nxt;
            fetch(nxt, h, min(k + 4, KT - 4));  // (the last one's product is not used)
            group(cur, nxt, p, true);
            cur = nxt;
        }
    };
    // chunk c: its buffer is read while `cur` (already in LDS) takes chunk c +
    // 2, then chunk c + 1 goes from `nxt` into the other buffer, which was
    // last read before the previous barrier
    auto step = [&](Set& cur, const Set& nxt, int c) {
        if (!PART || c + 2 < nk) load(cur, c + 2);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (PART) {
            const int lo = c + 1 == nk ? tail : 0, hi = tiny ? (int)K : KT;
            if (lo < 4 && hi > KT - 4) multiply(c & 1);
            else multiply_part(c & 1, lo & ~3, (hi + 3) & ~3);
        } else {
            multiply(c & 1);
        }
        if (c + 1 < nk) store(nxt, c + 1, (c + 1) & 1);
        __syncthreads();
    };
    if (K > 0) {
        Set s0, s1;
        if (tiny) load_tiny(s0);
        else load(s0, 0);
        if (!PART || nk > 1) load(s1, 1);
        store(s0, 0, 0);
        __syncthreads();
        for (int c = 0; c < nk; c += 2) {
            step(s0, s1, c);
            if (c + 1 < nk) step(s1, s0, c + 1);
        }
    }
    // a bias of one row (c_size == N, the usual one) is indexed by the column
    const bool brow = C != nullptr && c_size == N;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int i = v / (NV / NA), u = v % (NV / NA);
        const int64_t r = i0 + wm + i * O::AR + O::crow(l, u), c = j0 + wn + O::ccol(l, u);
        if (r >= M || c >= N) continue;
        if (brow) Y[r * ldy + c] = pfr::bias_add_at(acc[i][u], C + c, beta, act);
        else Y[r * ldy + c] = pfr::bias_add(acc[i][u], r * N + c, C, c_size, beta, act);
    }
}

struct DenseArgs {
    const float* A;
    int64_t lda;
    const float* B;
    int64_t ldb, M, N, K;
    float alpha;
    const float* C;
    int64_t c_size;
    float beta;
    int act;
    float* Y;
    int64_t ldy;
};

template <int NV>
void launch_dense(pfr_ctx* ctx, const DenseArgs& a, bool transA) {
    constexpr int TM = 2 * Outer<NV>::WM, TN = 2 * Outer<NV>::WN;
    const dim3 grid((unsigned)((a.N + TN - 1) / TN), (unsigned)((a.M + TM - 1) / TM));
    const bool avec = !transA && a.lda % 4 == 0 && a.K >= 4 && (reinterpret_cast<uintptr_t>(a.A) & 15) == 0;
#define PFR_DENSE(T, V, P)                                                                                            \
    hipLaunchKernelGGL((k_gemm_dense<NV, T, V, P>), grid, dim3(256), 0, ctx->stream, a.A, a.lda, a.B, a.ldb, a.M, a.N, \
                       a.K, a.alpha, a.C, a.c_size, a.beta, a.act, a.Y, a.ldy)
    const bool part = a.K % Outer<NV>::KT != 0 || a.K <= 2 * Outer<NV>::KT;
    if (transA && part) PFR_DENSE(true, false, true);
    else if (transA) PFR_DENSE(true, false, false);
    else if (avec && part) PFR_DENSE(false, true, true);
    else if (avec) PFR_DENSE(false, true, false);
    else if (part) PFR_DENSE(false, false, true);
    else PFR_DENSE(false, false, false);
#undef PFR_DENSE
}

void gemm_dense_dev(pfr_ctx* ctx, const float* A, int64_t M, int64_t K, int transA, const float* B, int64_t N,
                    int64_t ldb, float alpha, float beta, const float* C, int64_t c_size, float* Y, int64_t ldy,
                    int act) {
    pfr::require(M >= 0 && K >= 0 && N >= 0, "negative dimension");
    pfr::require(ldb >= N && ldy >= N, "leading dimension smaller than N");
    pfr::require(act == PFR_ACT_NONE || act == PFR_ACT_RELU || act == PFR_ACT_GELU, "unknown activation");
    if (M == 0 || N == 0) return;
    pfr::require(Y != nullptr && ((A != nullptr && B != nullptr) || K == 0), "null A/B/Y");
    pfr::require((M + 63) / 64 < 65536, "too many rows for the dense product's grid");
    pfr::require((N + 63) / 64 < (int64_t(1) << 31), "too many columns for the dense product's grid");
    if (C == nullptr || c_size <= 0) {
        C = nullptr;
        c_size = 0;
    }
    const DenseArgs a{A, transA ? M : K, B, ldb, M, N, K, alpha, C, c_size, beta, act, Y, ldy};
    // The tile with the least estimated time.  Small tiles give a small product
    // more waves (a sum is a chain over all of K, so K cannot be split) and let
    // the MFMAs of one wave run beside the adds of another: within one wave
    // they take turns (205 clocks per k at NV = 32 against 134 with two waves
    // per SIMD).  Large ones read their operands less often.  A k takes k1[n - 1]
    // ns on a CU that holds n workgroups, up to four, and four at a time where
    // there are more (an odd one on NV = 32 runs half alone); a workgroup
    // takes `each` ns besides, for its start and its outputs.  Measured over 64 x
    // 768 to 4096 x 4096 outputs and K from 1 to 2048; with K = 768 (us; NV = 4 /
    // 8 / 16 / 32): 64 x 768 outputs 19.4 / 31.0 / 48.0 / 83.8, 512 x 3072 56.1 /
    // 55.0 / 59.2 / 84.7, 1000 x 4096 138 / 122 / 115 / 110, 2048 x 3072 204 / 181 /
    // 168 / 188, and 2048 cubed 357 / 320 / 292 / 277; with K = 16: 4096 x 4096 53 /
    // 38 / 33 / 39.  (With the multiplies and adds both on the vector unit and one
    // 64 x 64 tile: 117, 118, 162, 234, 448 and 31.)
    auto cost = [&](int64_t tm, int64_t tn, int64_t each, const int (&k1)[4]) {
        const int64_t wgs = (M + tm - 1) / tm * ((N + tn - 1) / tn), n = (wgs + ctx->num_cu - 1) / ctx->num_cu;
        return n * each + K * (n / 4 * k1[3] + (n % 4 ? k1[n % 4 - 1] : 0));
    };
    // (A launch has fewer than 2^16 grid rows here and takes fewer than 2^32
    // threads along x: 2^24 workgroups, N up to 2^29 in 32 columns each.)
    const bool n32 = (N + 31) / 32 < (int64_t(1) << 24);
    const int64_t c4 = n32 && M < (int64_t(1) << 20) ? cost(32, 32, 600, {19, 23, 35, 42}) : INT64_MAX;
    const int64_t c8 = n32 ? cost(64, 32, 750, {34, 40, 63, 75}) : INT64_MAX;
    const int64_t c16 = cost(64, 64, 1450, {55, 68, 110, 136}), c32 = cost(128, 64, 3500, {100, 129, 226, 257});
    const int64_t best = std::min(std::min(c4, c8), std::min(c16, c32));
    if (best == c32) launch_dense<32>(ctx, a, transA != 0);
    else if (best == c16) launch_dense<16>(ctx, a, transA != 0);
    else if (best == c8) launch_dense<8>(ctx, a, transA != 0);
    else launch_dense<4>(ctx, a, transA != 0);
    PFR_HIP(hipGetLastError());
}

}  // namespace

extern "C" {

int pfr_gemm_dense_dev(pfr_ctx* ctx, const float* A, int64_t M, int64_t K, int transA, const float* B, int64_t N,
                       int64_t ldb, float alpha, float beta, const float* C, int64_t c_size, float* Y, int64_t ldy,
                       int act) {
    return pfr::guarded([&] {
        pfr::bind(ctx);
        gemm_dense_dev(ctx, A, M, K, transA, B, N, ldb, alpha, beta, C, c_size, Y, ldy, act);
    });
}

}  // extern "C"
