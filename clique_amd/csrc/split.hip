// FP32 updates of the factorization on the half-precision matrix cores (gfx950),
// for callers that ask for them (CLIQG_GEMM_TILE=11).
#include "device.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace cliqg {

namespace {

typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

// 32x32x16 MFMA: lane l supplies A(l % 32, 8 (l / 32) .. + 7) and B the same
// way; result register r of lane l is C(8 (r / 4) + 4 (l / 32) + r % 4, l % 32).
__device__ __forceinline__ f16v mfma_f16(u4v a, u4v b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, a),
                                                  __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}

template <class T> struct SplitLayout {
    static constexpr bool CPX = Scalar<T>::complex;
    static constexpr int NPL = CPX ? 4 : 2;   // re high, re low (, im high, im low)
    static constexpr int KS = 2;              // 16-deep K steps of a chunk
    static constexpr int KC = 16 * KS;
    static constexpr int THREADS = KS * NPL * 64;   // one run each of 32 rows of a chunk
    // K steps of a slab of kc columns, whole chunks (the tail is zero)
    static __host__ __device__ int steps(int kc) { return (kc + KC - 1) / KC * KS; }
};

// binary exponent e of a value, 2^(e-1) <= |x| < 2^e; NO_EXP for zero
constexpr int NO_EXP = -4000;
__device__ __forceinline__ int exponent(float x) {
    return x == 0.0f ? NO_EXP : __builtin_amdgcn_frexp_expf(x);
}
__device__ __forceinline__ int exponent(cfloat x) { return max(exponent(x.x), exponent(x.y)); }
__device__ __forceinline__ int exponent(double x) { return __builtin_amdgcn_frexp_exp(x); }
__device__ __forceinline__ int exponent(cdouble x) {
    return exponent(fabs(x.x) > fabs(x.y) ? x.x : x.y);
}

// Operands of one K slab as MFMA operands: every entry times a power of two is
// the sum of two half-precision numbers (high part rounded to 11 bits, low part
// the remainder rounded to 11 bits), 32 rows x 16 k of one part a block of
// 1 KB whose 16 bytes per lane are that lane's eight k. The powers of two bring
// the largest entry of a row (of its slab) to 2^15, and the two operands of a
// product, W = L D and L, to the same size in every column (|D|^(1/2) each),
// so that what falls below half precision's range is 2^-40 of the largest
// products of its row pair. Sums are therefore accurate against their rows'
// largest products and not term by term: an entry 2^p below its row's largest is
// kept to 2^-23 up to p = 16, to 2^-21 at 18, 2^-17 at 22, 2^-13 at 26, where
// FP32 keeps 24 bits of each. No launch takes these products by itself. One
// workgroup per 32 rows: a pass for the rows' largest exponents, then one that
// splits and writes.
// HBM-bound (eight bytes read twice, the second time from L2, and written once
// per complex entry): 8192 rows of two operands x 1024 complex columns 75 us,
// 3.6 TB/s; packing once leaves the product kernel no conversions (splitting
// while staging reached 180 TFLOP/s complex where this pair reaches 264).
template <class T>
__global__ __launch_bounds__(256) void k_split_pack(const GemmDesc<T>* __restrict__ descs,
                                                    const SplitDesc* __restrict__ split,
                                                    const int* __restrict__ pack_start, int ndesc,
                                                    int k0, u4v* __restrict__ parts,
                                                    int* __restrict__ exps) {
    using V = typename Scalar<T>::wide;
    using SL = SplitLayout<T>;
    __shared__ short bal[SPLIT_SLAB];
    __shared__ int top[32];
    const int w = blockIdx.x;
    const int di = find_segment(pack_start, ndesc, w);
    const GemmDesc<T> d = descs[di];
    const SplitDesc sd = split[di];
    const int kc = min(SPLIT_SLAB, d.K - k0);
    if (kc <= 0) return;
    int rb = w - pack_start[di];
    const int na = (d.M + 127) / 128 * 4;
    const bool isB = rb >= na;
    if (isB) rb -= na;
    const T* src = isB ? d.B : d.A;
    const int64_t ld = isB ? d.ldb : d.lda;
    const int rows = isB ? d.N : d.M;
    const int tid = threadIdx.x, lr = tid & 31, kg = tid >> 5;
    const int row = 32 * rb + lr;
    const bool in = row < rows;
    src += min(row, rows - 1) + (int64_t)k0 * ld;
    for (int k = tid; k < kc; k += 256) {
        const int e = exponent(gload(static_cast<const V*>(sd.D) + k0 + k)) >> 1;
        bal[k] = (short)(isB ? e : -e);
    }
    if (tid < 32) top[tid] = NO_EXP;
    __syncthreads();
    int e = NO_EXP;
    for (int k = kg; k < kc; k += 64) {
        T x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = gload(src + (int64_t)min(k + 8 * j, kc - 1) * ld);
#pragma unroll
        for (int j = 0; j < 8; ++j) e = max(e, exponent(x[j]) + bal[min(k + 8 * j, kc - 1)]);
    }
    atomicMax(&top[lr], e);
    __syncthreads();
    e = top[lr];
    if (kg == 0) exps[(isB ? sd.eB : sd.eA) + row] = e;
    const int nks = SL::steps(kc);
    u4v* out = parts + (isB ? sd.B : sd.A) + (int64_t)rb * nks * (SL::NPL * 64);
    const float sg = isB && (d.flags & G_CONJB) ? -1.0f : 1.0f;
    for (int q = kg; q < 2 * nks; q += 8) {
        float y[8][2];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * q + j, kk = min(k, kc - 1);
            const T x = pick(in && k < kc, gload(src + (int64_t)kk * ld), zero<T>());
            const int s = bal[kk] - e + 15;
            y[j][0] = __builtin_amdgcn_ldexpf(re(x), s);
            y[j][1] = SL::CPX ? __builtin_amdgcn_ldexpf(sg * im(x), s) : 0.0f;
        }
#pragma unroll
        for (int c = 0; c < (SL::CPX ? 2 : 1); ++c) {
            u4v hi, lo;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float a = y[2 * j][c], b = y[2 * j + 1][c];
                const h2v h{(_Float16)a, (_Float16)b};
                const h2v l{(_Float16)(a - (float)h[0]), (_Float16)(b - (float)h[1])};
                hi[j] = __builtin_bit_cast(unsigned, h);
                lo[j] = __builtin_bit_cast(unsigned, l);
            }
            u4v* p = out + ((q >> 1) * SL::NPL + 2 * c) * 64 + (q & 1) * 32 + lr;
            p[0] = hi;
            p[64] = lo;
        }
    }
}

// Updates C -= W op(L)^T (lower part) of a K slab from the packed operands:
// three products of parts (high high, high low, low high) per real product,
// summed in FP32. The low low product, 2^-24 of the whole on average, has
// either sign off the diagonal; on it, where it has one, diagonal tiles add
// it.
// Bound by the matrix cores: three MFMAs (twelve for complex) at sixteen times
// the FP32 rate per product. Lower 8192 x 8192, K = 4096, with the packing:
// complex 4.1 ms (264 TFLOP/s counting four real products) against 6.8 of the
// 64x64 FP32 kernel, which multiplies with three; real 1.7 ms (164) against
// 3.1. At K = 256, 4096 x 4096: complex 0.108 ms against 0.153, real 0.066
// against 0.076.
// Error of one update relative to sum |w l| (4096 x 4096): off the diagonal
// 5e-9 at K = 2048 and 1e-8 at 256, FP32 kernel 3e-8 and 4e-8; on it (one
// sign) 7e-8 against 5e-7 and 2.5e-7. The MFMA truncates small products
// against the largest of its sixteen, which leaves a bias of some 5e-8 in sums
// of one sign. First FP32 solves against FP64 factors with the sums of K >= 384
// split and not, geometric means of 12 systems of 40^3 to 80^3: shifted
// Laplacians 3.0e-7 and 3.1e-7, Helmholtz 1.42e-5 and 1.45e-5, with PML 2.4e-6 and
// 2.5e-6, diffusion 1.1e-6 and 1.8e-6: in norm no worse. Entry by entry it is: of
// the solution for a point source in a screened 64^3 Laplacian (10^-30 across the
// grid), the worst is off by 7e-2 where FP32 updates leave 2e-5.
// A workgroup owns a 128 x 128 tile; its waves own 64 x 32 of it (complex,
// eight waves) or 64 x 64 (real, four waves, two workgroups per CU). Chunks of
// 32 K pass through two LDS buffers, each thread holding its share of the next
// one in registers. Blocks are stored in lane order, so LDS accesses are linear
// and free of conflicts.
template <class T>
__global__ __launch_bounds__(SplitLayout<T>::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_gemm_split(
    const GemmDesc<T>* __restrict__ descs, const SplitDesc* __restrict__ split,
    const int* __restrict__ tile_start, int ndesc, int k0, const u4v* __restrict__ parts,
    const int* __restrict__ exps) {
    using SL = SplitLayout<T>;
    constexpr bool CPX = SL::CPX;
    constexpr int NPL = SL::NPL, KS = SL::KS, NP = CPX ? 2 : 1;
    constexpr int BLK = SL::THREADS;             // 16-byte runs of 32 rows of a chunk
    constexpr int NW = CPX ? 1 : 2;              // 32-column blocks of a wave
    __shared__ u4v lds[2][8][BLK];

    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int di = find_segment(tile_start, ndesc, tile);
    const GemmDesc<T> d = descs[di];
    const SplitDesc sd = split[di];
    const int kc = min(SPLIT_SLAB, d.K - k0);
    if (kc <= 0 && k0 > 0) return;
    const bool lower = d.flags & G_LOWER, accum = (d.flags & G_ACCUM) || k0 > 0;
    const bool neg = d.flags & G_NEG;
    int ti, tj;
    group_tile(tile - tile_start[di], (d.M + 127) / 128, (d.N + 127) / 128, lower, ti, tj);
    const int row0 = ti * 128, col0 = tj * 128;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave & 1, wj = wave >> 1;     // 64 x 32 NW of the tile
    const int nks = SL::steps(max(kc, 0)), nk = nks / KS;
    const int64_t rstride = (int64_t)nks * (NPL * 64);   // runs of 32 rows of the slab
    const u4v* pa = parts + sd.A + 4 * ti * rstride + tid;
    const u4v* pb = parts + sd.B + 4 * tj * rstride + tid;

    u4v x[8];
    auto fetch = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = pa[i * rstride];
            x[4 + i] = pb[i * rstride];
        }
        pa += BLK;
        pb += BLK;
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 8; ++i) lds[buf][i][tid] = x[i];
    };
    // A chunk's products start from zero and are added to the running sum in
    // one rounding: the MFMA's own accumulation loses a little more than a
    // rounding per step, which over a long K (one sign, as on the diagonal)
    // adds up.
    f16v acc[NW][2][NP];
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int q = 0; q < NP; ++q)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][a][q][r] = 0.0f;
    // products of parts (i of W, j of L), smallest first
    constexpr int PI[4] = {1, 1, 0, 0}, PJ[4] = {1, 0, 1, 0};
    auto multiply = [&](int buf, auto diag) {
        constexpr int M0 = decltype(diag)::value ? 0 : 1;
        f16v part[NW][2][NP];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u4v b[NW][NPL];
#pragma unroll
            for (int n = 0; n < NW; ++n)
#pragma unroll
                for (int p = 0; p < NPL; ++p)
                    b[n][p] = lds[buf][4 + NW * wj + n][(s * NPL + p) * 64 + lane];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                u4v w[NPL];
#pragma unroll
                for (int p = 0; p < NPL; ++p)
                    w[p] = lds[buf][2 * wi + a][(s * NPL + p) * 64 + lane];
                // (the operand that indexes the result's lanes is W's: lane =
                // row of C, registers = columns)
#pragma unroll
                for (int m = M0; m < 4; ++m)
#pragma unroll
                    for (int n = 0; n < NW; ++n) {
                        f16v* c = part[n][a];
                        const f16v z{};
                        const bool first = s == 0 && m == M0;
                        c[0] = mfma_f16(b[n][PJ[m]], w[PI[m]], first ? z : c[0]);
                        if constexpr (CPX) {
                            c[1] = mfma_f16(b[n][2 + PJ[m]], w[PI[m]], first ? z : c[1]);
                            c[0] = mfma_f16(b[n][2 + PJ[m]] ^ 0x80008000u, w[2 + PI[m]], c[0]);
                            c[1] = mfma_f16(b[n][PJ[m]], w[2 + PI[m]], c[1]);
                        }
                    }
            }
        }
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int q = 0; q < NP; ++q) acc[n][a][q] += part[n][a][q];
    };
    if (nk > 0) {
        fetch();
        stage(0);
        __syncthreads();
    }
    auto step = [&](int c, int buf, auto diag) {
        if (c + 1 < nk) fetch();
        multiply(buf, diag);
        if (c + 1 < nk) stage(buf ^ 1);
        lds_barrier();
    };
    auto sum = [&](auto diag) {
        for (int c = 0; c < nk; c += 2) {
            step(c, 0, diag);
            if (c + 1 < nk) step(c + 1, 1, diag);
        }
    };
    if (ti == tj)
        sum(std::true_type{});
    else
        sum(std::false_type{});
    const int hi = lane >> 5;
    const int* ea = exps + sd.eA + row0 + 64 * wi + (lane & 31);
    const int* eb = exps + sd.eB + col0 + 32 * NW * wj + 4 * hi;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int gi = row0 + 64 * wi + 32 * a + (lane & 31);
        const int e0 = nk > 0 ? ea[32 * a] - 30 : 0;
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int jr = 32 * n + 8 * (r / 4) + r % 4;
                const int gj = col0 + 32 * NW * wj + 4 * hi + jr;
                if (gi >= d.M || gj >= d.N || (lower && gi < gj)) continue;
                const int e = e0 + (nk > 0 ? eb[jr] : 0);
                T v = make_t<T>(__builtin_amdgcn_ldexpf(acc[n][a][0][r], e),
                                CPX ? __builtin_amdgcn_ldexpf(acc[n][a][NP - 1][r], e) : 0.0f);
                if (neg) v = -v;
                T* pc = d.C + gi + (int64_t)gj * d.ldc;
                if (accum) v = gload(pc) + v;
                gstore(pc, v);
            }
    }
}

}  // namespace

template <class T>
int64_t split_runs(int rows, int K) {
    return (int64_t)((rows + 127) / 128 * 4) * SplitLayout<T>::steps(std::min(K, SPLIT_SLAB)) *
           (SplitLayout<T>::NPL * 64);
}

template <class T>
void launch_gemm_split(const GemmDesc<T>* d_descs, const SplitDesc* d_split,
                       const int* d_tile_start, const int* d_pack_start, int ndesc, int ntiles,
                       int npack, int maxK, void* ws, int64_t runs, hipStream_t s) {
    if (ntiles <= 0 || ndesc <= 0) return;
    u4v* parts = static_cast<u4v*>(ws);
    int* exps = reinterpret_cast<int*>(parts + runs);
    for (int k0 = 0; k0 < std::max(maxK, 1); k0 += SPLIT_SLAB) {
        hipLaunchKernelGGL(k_split_pack<T>, dim3(npack), dim3(256), 0, s, d_descs, d_split,
                           d_pack_start, ndesc, k0, parts, exps);
        hipLaunchKernelGGL(k_gemm_split<T>, dim3(ntiles), dim3(SplitLayout<T>::THREADS), 0, s, d_descs, d_split,
                           d_tile_start, ndesc, k0, parts, exps);
    }
}

#define CLIQG_SPLIT_INST(T)                                                                      \
    template int64_t split_runs<T>(int, int);                                                    \
    template void launch_gemm_split<T>(const GemmDesc<T>*, const SplitDesc*, const int*,         \
                                       const int*, int, int, int, int, void*, int64_t,           \
                                       hipStream_t);
CLIQG_SPLIT_INST(float)
CLIQG_SPLIT_INST(cfloat)
#undef CLIQG_SPLIT_INST

}  // namespace cliqg
