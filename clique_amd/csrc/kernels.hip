// Device kernels of libcliqg for gfx950 (CDNA4). See kernels.hpp.
#include "device.hpp"
#include "kernels.hpp"

#include <cstdlib>
#include <type_traits>

namespace cliqg {

namespace {

constexpr int LPAD = 16;

// number of column-major lower-trapezoid tiles before tile column tj
__host__ __device__ __forceinline__ long long lower_prefix(long long tj, long long tilesM) {
    return tj * tilesM - tj * (tj - 1) / 2;
}

}  // namespace

int gemm_tile_m(int variant) {
    if (variant == TILE_STREAM || variant == TILE_STREAM_16) return 16;
    return (variant == TILE_32 || variant == TILE_32_K64 || variant == TILE_STREAM_32)
               ? 32
               : ((variant == TILE_128 || variant == TILE_128_8W || variant == TILE_SPLIT) ? 128 : 64);
}
// a streaming tile takes all N <= 64 columns
int gemm_tile_n(int variant) { return gemm_tile_streams(variant) ? 64 : gemm_tile_m(variant); }

int gemm_tiles(int M, int N, int flags, int variant) {
    if (M <= 0 || N <= 0) return 0;
    const int TM = gemm_tile_m(variant), TN = gemm_tile_n(variant);
    const int tm = (M + TM - 1) / TM, tn = (N + TN - 1) / TN;
    if ((flags & G_LOWER) && TM != TN)
        throw Error(1, "lower-masked GEMM launches need square tiles");
    if (flags & G_LOWER) {
        const int c = tn < tm ? tn : tm;
        return (int)lower_prefix(c, tm);
    }
    return tm * tn;
}

// ---------------------------------------------------------------------------
// Grouped GEMM: one TM x TN output tile per workgroup of WM x WN waves;
// each wave owns a (TM/WM) x (TN/WN) part of 16x16 MFMA blocks. K is
// consumed in chunks of 16 through two LDS buffers (one barrier per chunk);
// the next chunk is prefetched into registers while the current one feeds
// the MFMAs. Complex products run on planar (re, im) tiles: three real MFMAs
// per block for complex FP32 (below), four for complex FP64.
// ---------------------------------------------------------------------------
template <class T, int TM, int TN, int ROLE, int TK, int WM = 2, int WN = 2>
__global__ __launch_bounds__(64 * WM * WN)
__attribute__((amdgpu_waves_per_eu((TM * TN / (WM * WN) >= 2048) ? 2
                                   : (sizeof(T) <= 8 ? 4 : 2), 8))) void k_gemm(const GemmDesc<T>* __restrict__ descs,
                                                       const int* __restrict__ tile_start,
                                                       int ndesc) {
    using R = typename Scalar<T>::real;
    using W = typename Scalar<T>::wide;
    using A4 = typename Acc4<R>::type;
    constexpr bool CPX = Scalar<T>::complex;
    constexpr int NP = CPX ? 2 : 1;
    constexpr int NT = 64 * WM * WN;                       // threads
    constexpr int WTM = TM / WM, WTN = TN / WN;            // wave tile
    constexpr int BM = WTM / 16, BN = WTN / 16;            // 16x16 blocks per wave
    constexpr int LA = TM * TK / NT, LB = TN * TK / NT;
    constexpr bool F64 = sizeof(R) == 8;
    constexpr bool SCALED = ROLE == 2;   // every descriptor of the launch has scaleK
    constexpr bool PRIO = !(ROLE == 3 && !F64);   // raised priority over the MFMA loop

    __shared__ R As[2][NP][TK][TM + LPAD];
    __shared__ R Bs[2][NP][TK][TN + LPAD];
    // The pivots of a chunk (scaleK) live in column TM of As, which is padding
    // the fragments never read: a separate array would push the complex tiles
    // past a quarter (complex float) or half (complex double) of the 160 KB
    // LDS and cost one resident block per CU.

    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int di = find_segment(tile_start, ndesc, tile);
    const GemmDesc<T> d = descs[di];
    const int t = tile - tile_start[di];
    int ti, tj;
    group_tile(t, (d.M + TM - 1) / TM, (d.N + TN - 1) / TN, d.flags & G_LOWER, ti, tj);
    const int row0 = ti * TM, col0 = tj * TN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = wave % WM, wj = wave / WM;
    const bool transA = d.flags & G_TRANSA, transB = d.flags & G_TRANSB;
    const bool conjA = d.flags & G_CONJA, conjB = d.flags & G_CONJB;
    const W* scaleK = reinterpret_cast<const W*>(d.scaleK);

    // Complex FP32 products use three real MFMAs per block (Gauss):
    // P1 = sum aR bR, P2 = sum aI bI, P3 = sum (aR + aI)(bR + bI);
    // Re = P1 - P2, Im = P3 - P1 - P2. Complex FP64 keeps four.
    constexpr bool M3 = CPX && !F64 && GEMM_3M && BM * BN <= 8;   // registers: 64x32 wave tiles at most
    A4 accR[BM][BN], accI[BM][BN], accS[M3 ? BM : 1][M3 ? BN : 1];
#pragma unroll
    for (int a = 0; a < BM; ++a)
#pragma unroll
        for (int b = 0; b < BN; ++b) {
            accR[a][b] = A4{0, 0, 0, 0};
            accI[a][b] = A4{0, 0, 0, 0};
            if constexpr (M3) accS[a][b] = A4{0, 0, 0, 0};
        }

    // Fixed per-thread load geometry: element r of the A chunk is
    // (iA + r*dIA, kA + r*dKA) of the TM x TK tile, element r of the B chunk
    // (kB + r*dKB, jB + r*dJB) of the TK x TN tile; the global addresses of a
    // thread's elements differ by multiples of lda (ldb), and a chunk advances
    // them by a fixed stride.
    static_assert(NT % TM == 0 && NT % TN == 0 && NT % TK == 0, "load geometry");
    int iA, kA, dIA, dKA, jB, kB, dJB, dKB;
    if (!transA) { iA = tid % TM; kA = tid / TM; dIA = 0; dKA = NT / TM; }
    else { kA = tid % TK; iA = tid / TK; dIA = NT / TK; dKA = 0; }
    if (transB) { jB = tid % TN; kB = tid / TN; dJB = 0; dKB = NT / TN; }
    else { kB = tid % TK; jB = tid / TK; dJB = NT / TK; dKB = 0; }
    const int64_t stepA = transA ? TK : (int64_t)TK * d.lda;
    const int64_t stepB = transB ? (int64_t)TK * d.ldb : TK;
    unsigned rowOK = 0, colOK = 0;   // bit r: element r's row (column) is inside the matrix
#pragma unroll
    for (int r = 0; r < LA; ++r) rowOK |= (row0 + iA + r * dIA < d.M) ? 1u << r : 0u;
#pragma unroll
    for (int r = 0; r < LB; ++r) colOK |= (col0 + jB + r * dJB < d.N) ? 1u << r : 0u;
    const int ldsA = kA * (TM + LPAD) + iA, ldsAStep = dKA * (TM + LPAD) + dIA;
    const int ldsB = kB * (TN + LPAD) + jB, ldsBStep = dKB * (TN + LPAD) + dJB;

    T ra[LA], rb[LB];
    // element r of a thread sits r*offA elements after its first one (one of
    // dIA, dKA is zero); pA is the lane's pointer at the current chunk
    const int64_t offA = (int64_t)(transA ? dIA : dKA) * d.lda;
    const int64_t offB = (int64_t)(transB ? dKB : dJB) * d.ldb;
    const T* pA = nullptr;
    const T* pB = nullptr;
    auto start_at = [&](int k0) {
        pA = transA ? d.A + (k0 + kA) + (int64_t)(row0 + iA) * d.lda
                    : d.A + (row0 + iA) + (int64_t)(k0 + kA) * d.lda;
        pB = transB ? d.B + (col0 + jB) + (int64_t)(k0 + kB) * d.ldb
                    : d.B + (k0 + kB) + (int64_t)(col0 + jB) * d.ldb;
    };
    // Loads never branch per element: an element outside the matrix reads the
    // operand's first entry and is replaced by zero when it is stored to LDS,
    // so all of a chunk's loads are in flight together and the only wait is
    // before the store (a divergent load would wait inside its branch). Tiles
    // inside the matrix take a uniform fast path with no masks at all: every
    // VALU instruction here is issue time the MFMAs do not get.
    W rdw = one<W>();
    unsigned okA = 0, okB = 0;
    bool okD = false, fastA = false, fastB = false;
    const bool innerA = row0 + TM <= d.M, innerB = col0 + TN <= d.N;
    auto load = [&](int k0) {
        const bool fullK = k0 + TK <= d.K;
        if constexpr (SCALED) {
            okD = tid < TK && k0 + tid < d.K;
            rdw = gload(scaleK + (okD ? k0 + tid : 0));
        }
        fastA = innerA && fullK;
        fastB = innerB && fullK;
        if (fastA) {
#pragma unroll
            for (int r = 0; r < LA; ++r) ra[r] = gload(pA + r * offA);
        } else {
            okA = 0;
#pragma unroll
            for (int r = 0; r < LA; ++r) {
                const bool ok = ((rowOK >> r) & 1u) && (fullK || k0 + kA + r * dKA < d.K);
                okA |= ok ? 1u << r : 0u;
                ra[r] = gload(ok ? pA + r * offA : d.A);
            }
        }
        if (fastB) {
#pragma unroll
            for (int r = 0; r < LB; ++r) rb[r] = gload(pB + r * offB);
        } else {
            okB = 0;
#pragma unroll
            for (int r = 0; r < LB; ++r) {
                const bool ok = ((colOK >> r) & 1u) && (fullK || k0 + kB + r * dKB < d.K);
                okB |= ok ? 1u << r : 0u;
                rb[r] = gload(ok ? pB + r * offB : d.B);
            }
        }
        pA += stepA;
        pB += stepB;
    };
    // stage n elements v[] at p0[off + r*step] (re) and p1[...] (im), with the
    // mask and conjugation decided once per chunk (uniform branches)
    auto stage = [&](const T* v, int n, unsigned ok, bool fast, bool conj, R* p0, R* p1, int off,
                     int step) {
        if (fast && !conj) {
#pragma unroll
            for (int r = 0; r < (LA > LB ? LA : LB); ++r)
                if (r < n) {
                    p0[off + r * step] = re(v[r]);
                    if constexpr (CPX) p1[off + r * step] = im(v[r]);
                }
        } else {
#pragma unroll
            for (int r = 0; r < (LA > LB ? LA : LB); ++r)
                if (r < n) {
                    T x = (fast || ((ok >> r) & 1u)) ? v[r] : zero<T>();
                    if (conj) x = conj_(x);
                    p0[off + r * step] = re(x);
                    if constexpr (CPX) p1[off + r * step] = im(x);
                }
        }
    };
    auto store = [&](auto bufc) {
        constexpr int buf = decltype(bufc)::value;
        if constexpr (SCALED)
            if (tid < TK) {
                T dv = zero<T>();
                if (okD) dv = (d.flags & G_INVK) ? cvt<T>(one<W>() / rdw) : cvt<T>(rdw);
                As[buf][0][tid][TM] = re(dv);
                if constexpr (CPX) As[buf][NP - 1][tid][TM] = im(dv);
            }
        stage(ra, LA, okA, fastA, conjA, &As[buf][0][0][0], &As[buf][NP - 1][0][0], ldsA, ldsAStep);
        stage(rb, LB, okB, fastB, conjB, &Bs[buf][0][0][0], &Bs[buf][NP - 1][0][0], ldsB, ldsBStep);
    };

    // K range of this row tile: triangular op(A) bounds it by the tile's rows
    int kbeg = 0, kend = d.K;
    if (d.flags & G_KLO) kbeg = min((row0 / TK) * TK, d.K);
    if (d.flags & G_KHI) kend = min(d.K, row0 + TM);
    const int nk = kend > kbeg ? (kend - kbeg + TK - 1) / TK : 0;
    start_at(kbeg);
    if (nk > 0) {
        load(kbeg);
        store(std::integral_constant<int, 0>{});
        __syncthreads();
    }
    // One K chunk from LDS buffer BUF (a compile-time constant: the loop below
    // runs chunks in pairs, so LDS addresses fold into instruction offsets).
    auto chunk = [&](int c, auto bufc) {
        constexpr int buf = decltype(bufc)::value;
        if (c + 1 < nk) load(kbeg + (c + 1) * TK);
        // raised wave priority while feeding the MFMAs (measured on the
        // 120^3 complex factorizations: FP64 updates 1.5 % faster with it,
        // FP32 updates 1 % faster without); the TRSMs, on the factorization's
        // critical path beside the lookahead updates, one level higher
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(ROLE == 0 ? 2 : 1);
#pragma unroll
        for (int kk = 0; kk < TK / 4; ++kk) {
            const int kr = kk * 4 + (lane >> 4);
            R aR[BM], aI[BM], bR[BN], bI[BN];
#pragma unroll
            for (int q = 0; q < BM; ++q) {
                aR[q] = As[buf][0][kr][wi * WTM + q * 16 + (lane & 15)];
                if constexpr (CPX) aI[q] = As[buf][NP - 1][kr][wi * WTM + q * 16 + (lane & 15)];
            }
            if constexpr (SCALED) {
                // op(A)(i,k) * D(k): the lane's k is kr for all of its A fragments
                const R dR = As[buf][0][kr][TM];
                const R dI = CPX ? As[buf][NP - 1][kr][TM] : R(0);
#pragma unroll
                for (int q = 0; q < BM; ++q) {
                    if constexpr (CPX) {
                        const R xr = aR[q] * dR - aI[q] * dI;
                        const R xi = aR[q] * dI + aI[q] * dR;
                        aR[q] = xr;
                        aI[q] = xi;
                    } else {
                        aR[q] = aR[q] * dR;
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < BN; ++q) {
                bR[q] = Bs[buf][0][kr][wj * WTN + q * 16 + (lane & 15)];
                if constexpr (CPX) bI[q] = Bs[buf][NP - 1][kr][wj * WTN + q * 16 + (lane & 15)];
            }
            if constexpr (M3) {
                R sA[BM], sB[BN];
#pragma unroll
                for (int a = 0; a < BM; ++a) sA[a] = aR[a] + aI[a];
#pragma unroll
                for (int b = 0; b < BN; ++b) sB[b] = bR[b] + bI[b];
#pragma unroll
                for (int a = 0; a < BM; ++a)
#pragma unroll
                    for (int b = 0; b < BN; ++b) {
                        accR[a][b] = mfma16(aR[a], bR[b], accR[a][b]);   // P1
                        accI[a][b] = mfma16(aI[a], bI[b], accI[a][b]);   // P2
                        accS[a][b] = mfma16(sA[a], sB[b], accS[a][b]);   // P3
                    }
            } else {
#pragma unroll
                for (int a = 0; a < BM; ++a)
#pragma unroll
                    for (int b = 0; b < BN; ++b) {
                        accR[a][b] = mfma16(aR[a], bR[b], accR[a][b]);
                        if constexpr (CPX) {
                            accR[a][b] = mfma16(-aI[a], bI[b], accR[a][b]);
                            accI[a][b] = mfma16(aR[a], bI[b], accI[a][b]);
                            accI[a][b] = mfma16(aI[a], bR[b], accI[a][b]);
                        }
                    }
            }
        }
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(ROLE == 0 ? 1 : 0);
        if (c + 1 < nk) store(std::integral_constant<int, buf ^ 1>{});
        __syncthreads();
    };
    for (int c = 0; c < nk; c += 2) {
        chunk(c, std::integral_constant<int, 0>{});
        if (c + 1 < nk) chunk(c + 1, std::integral_constant<int, 1>{});
    }

    const bool lower = d.flags & G_LOWER, accum = d.flags & G_ACCUM, neg = d.flags & G_NEG;
    const bool symm = lower && (d.flags & G_SYMM);
#pragma unroll
    for (int a = 0; a < BM; ++a)
#pragma unroll
        for (int b = 0; b < BN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int rin = F64 ? (lane >> 4) + 4 * r : 4 * (lane >> 4) + r;
                const int gi = row0 + wi * WTM + a * 16 + rin;
                const int gj = col0 + wj * WTN + b * 16 + (lane & 15);
                if (gi >= d.M || gj >= d.N || (lower && gi < gj)) continue;
                T v;
                if constexpr (M3)
                    v = make_t<T>(accR[a][b][r] - accI[a][b][r],
                                  accS[a][b][r] - accR[a][b][r] - accI[a][b][r]);
                else
                    v = make_t<T>(accR[a][b][r], CPX ? accI[a][b][r] : R(0));
                if (neg) v = -v;
                T* p = d.C + gi + (int64_t)gj * d.ldc;
                if (accum) v = gload(p) + v;
                if (symm) {
                    // Hermitian output (conj mirror) has a real diagonal
                    if (conjA && gi == gj) v = make_t<T>(re(v), R(0));
                    if (gi > gj) gstore(d.C + gj + (int64_t)gi * d.ldc, conjA ? conj_(v) : v);
                }
                gstore(p, v);
            }
}

template <class T, int TM, int TN, int KT = 16, int WM = 2, int WN = 2>
static void launch_gemm_shape(const GemmDesc<T>* d, const int* ts, int nd, int nt, int role,
                              hipStream_t s) {
    const dim3 block(64 * WM * WN);
    if (role == 0)
        hipLaunchKernelGGL((k_gemm<T, TM, TN, 0, KT, WM, WN>), dim3(nt), block, 0, s, d, ts, nd);
    else if (role == 2)
        hipLaunchKernelGGL((k_gemm<T, TM, TN, 2, KT, WM, WN>), dim3(nt), block, 0, s, d, ts, nd);
    else if (role == 3)
        hipLaunchKernelGGL((k_gemm<T, TM, TN, 3, KT, WM, WN>), dim3(nt), block, 0, s, d, ts, nd);
    else
        hipLaunchKernelGGL((k_gemm<T, TM, TN, 1, KT, WM, WN>), dim3(nt), block, 0, s, d, ts, nd);
}

template <class T>
void launch_gemm(const GemmDesc<T>* d_descs, const int* d_tile_start, int ndesc, int ntiles,
                 int variant, int role, int cols, hipStream_t s) {
    if (ntiles <= 0 || ndesc <= 0) return;
    if (variant == TILE_128) {
        if constexpr (gemm_variant_allowed<T>(TILE_128))
            launch_gemm_shape<T, 128, 128, 16, 2, 2>(d_descs, d_tile_start, ndesc, ntiles, role, s);
        else
            throw Error(1, "128x128 GEMM tiles are built for real types only");
    } else if (variant == TILE_128_8W) {
        if constexpr (gemm_variant_allowed<T>(TILE_128_8W))
            launch_gemm_shape<T, 128, 128, 16, 2, 4>(d_descs, d_tile_start, ndesc, ntiles, role, s);
        else
            throw Error(1, "eight-wave 128x128 GEMM tiles are built for complex FP32 only");
    } else if (gemm_tile_streams(variant)) {
        launch_gemm_stream<T>(d_descs, d_tile_start, ndesc, ntiles, variant, cols, s);
    } else if (variant == TILE_32) {
        launch_gemm_shape<T, 32, 32>(d_descs, d_tile_start, ndesc, ntiles, role, s);
    } else if (variant == TILE_32_K64) {
        if constexpr (gemm_variant_allowed<T>(TILE_32_K64))
            launch_gemm_shape<T, 32, 32, 64>(d_descs, d_tile_start, ndesc, ntiles, role, s);
        else
            throw Error(1, "64-deep 32x32 GEMM tiles are not built for complex FP64");
    } else {
        launch_gemm_shape<T, 64, 64>(d_descs, d_tile_start, ndesc, ntiles, role, s);
    }
}

// ---------------------------------------------------------------------------
// Clearing of update matrices (one ZERO_CHUNK-entry chunk per workgroup)
// ---------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(256) void k_zero_segments(const ZeroSeg<T>* __restrict__ segs,
                                                       const int* __restrict__ chunk_start,
                                                       int nseg) {
    const int g = blockIdx.x;
    const int si = find_segment(chunk_start, nseg, g);
    const ZeroSeg<T> sg = segs[si];
    const int64_t base = (int64_t)(g - chunk_start[si]) * ZERO_CHUNK;
    const int64_t end = min((int64_t)ZERO_CHUNK, sg.n - base);
    T* p = sg.p + base;
    for (int64_t i = threadIdx.x; i < end; i += blockDim.x) gstore(p + i, zero<T>());
}

// one wave per column, four per workgroup
template <class T>
__global__ __launch_bounds__(256) void k_zero_lower(const ZeroLowerDesc<T>* __restrict__ descs,
                                                    const int* __restrict__ col_start, int nd,
                                                    int ncols) {
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (g >= ncols) return;
    const int c = find_segment(col_start, nd, g);
    const ZeroLowerDesc<T> d = descs[c];
    const int j = g - col_start[c];
    T* col = d.p + (int64_t)j * d.ld;
    for (int i = j + (threadIdx.x & 63); i < d.rows; i += 64) gstore(col + i, zero<T>());
}

template <class T>
void launch_zero_lower(const ZeroLowerDesc<T>* d_descs, const int* d_col_start, int ndesc,
                       int ncols, hipStream_t s) {
    if (ncols <= 0 || ndesc <= 0) return;
    hipLaunchKernelGGL(k_zero_lower<T>, dim3((ncols + 3) / 4), dim3(256), 0, s, d_descs,
                       d_col_start, ndesc, ncols);
}

template <class T>
void launch_zero_segments(const ZeroSeg<T>* d_segs, const int* d_chunk_start, int nseg,
                          int nchunks, hipStream_t s) {
    if (nchunks <= 0) return;
    hipLaunchKernelGGL(k_zero_segments<T>, dim3(nchunks), dim3(256), 0, s, d_segs, d_chunk_start,
                       nseg);
}

template <class T>
__global__ __launch_bounds__(256) void k_copy2d(const CopyDesc<T>* __restrict__ descs,
                                                const int* __restrict__ chunk_start, int ndesc) {
    const int g = blockIdx.x;
    const int di = find_segment(chunk_start, ndesc, g);
    const CopyDesc<T> d = descs[di];
    const int64_t total = (int64_t)d.rows * d.cols;
    const int64_t base = (int64_t)(g - chunk_start[di]) * 1024;
    // all four loads before the stores (source and destination may share a
    // pool, so the compiler would otherwise wait a round trip per entry)
    T v[4];
    int64_t at[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t e = base + threadIdx.x + 256 * q;
        const bool ok = e < total;
        const int64_t r = ok ? e % d.rows : 0, c = ok ? e / d.rows : 0;
        at[q] = ok ? r + c * d.ldd : -1;
        v[q] = d.src[r + c * d.lds];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (at[q] >= 0) d.dst[at[q]] = v[q];
}

template <class T>
void launch_copy2d(const CopyDesc<T>* d_descs, const int* d_chunk_start, int ndesc, int nchunks,
                   hipStream_t s) {
    if (nchunks <= 0 || ndesc <= 0) return;
    hipLaunchKernelGGL(k_copy2d<T>, dim3(nchunks), dim3(256), 0, s, d_descs, d_chunk_start, ndesc);
}

// One 1024-element chunk of one split product per workgroup; each element
// sums its slices in order, so results do not depend on scheduling.
template <class T>
__global__ __launch_bounds__(256) void k_reduce_slices(const ReduceDesc<T>* __restrict__ descs,
                                                       const int* __restrict__ chunk_start,
                                                       int ndesc) {
    const int g = blockIdx.x;
    const int di = find_segment(chunk_start, ndesc, g);
    const ReduceDesc<T> d = descs[di];
    const int64_t total = (int64_t)d.rows * d.cols;
    const int64_t base = (int64_t)(g - chunk_start[di]) * 1024;
    for (int i = threadIdx.x; i < 1024; i += blockDim.x) {
        const int64_t e = base + i;
        if (e >= total) break;
        T v = gload(d.ws + e);
        for (int sl = 1; sl < d.slices; ++sl) v = v + gload(d.ws + sl * total + e);
        if (d.flags & G_NEG) v = -v;
        T* p = d.C + e % d.rows + (e / d.rows) * d.ldc;
        if (d.flags & G_ACCUM) v = gload(p) + v;
        gstore(p, v);
    }
}

template <class T>
void launch_reduce_slices(const ReduceDesc<T>* d_descs, const int* d_chunk_start, int ndesc,
                          int nchunks, hipStream_t s) {
    if (nchunks <= 0 || ndesc <= 0) return;
    hipLaunchKernelGGL(k_reduce_slices<T>, dim3(nchunks), dim3(256), 0, s, d_descs, d_chunk_start,
                       ndesc);
}

// ---------------------------------------------------------------------------
// Assembly of A into the fronts (scatter through a precomputed map)
// ---------------------------------------------------------------------------
template <class T, class V>
__global__ void k_assemble(const V* __restrict__ vals, const int64_t* __restrict__ dst,
                           int64_t nnz, T* __restrict__ pool, bool conj) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = dst[e];
        if (t >= 0) pool[t] = cvt<T>(cj(vals[e], conj));
    }
}

template <class T, class V>
void launch_assemble(const V* vals, const int64_t* dst, int64_t nnz, T* pool, bool conj,
                     hipStream_t s) {
    if (nnz <= 0) return;
    int64_t blocks = (nnz + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL((k_assemble<T, V>), dim3((unsigned)blocks), dim3(256), 0, s, vals, dst,
                       nnz, pool, conj);
}

// ---------------------------------------------------------------------------
// One inverted diagonal block of n <= 2 NB columns (the solves' wide blocks,
// the block fronts' diagonal) per workgroup: LW(0:n0, 0:n0) = X0, LW(0:n0,
// n0:n) = 0, LW(n0:n, n0:n) = X1 and LW(n0:n, 0:n0) = -X1 (L10 X0), the two 64
// x 64 products with both operands in LDS and a 4 x 4 register tile per
// thread. Bound by one workgroup's chain (12 us FP64, 35 complex); all blocks
// of a level in one launch, in place of its clearing, copies and two grouped
// products per 64 columns.
// ---------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(256) void k_wide_inverse(const WideInvDesc<T>* __restrict__ descs) {
    // rows padded to a multiple of four entries: a thread's four consecutive
    // entries are one 16-byte aligned LDS read (or two, complex)
    __shared__ __attribute__((aligned(16))) T Sa[NB][NB + 4];   // Sa[k][i] = A(i, k)
    __shared__ __attribute__((aligned(16))) T Sb[NB][NB + 4];   // Sb[k][j] = B(k, j)
    constexpr int PT = NB * NB / 256;   // entries of a 64 x 64 block per thread
    const WideInvDesc<T> d = descs[blockIdx.x];
    const int n = d.n, tid = threadIdx.x;
    const int n0 = min(n, NB), b1 = n - n0;
    // Every copy issues all of a thread's loads before its first store (a
    // load followed by its store per iteration would wait a global round
    // trip per entry). Element t of a thread is (i, j) = (e % 64, e / 64)
    // with e = tid + 256 t: lanes run down a column.
    T v[PT], w[PT];
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
        v[t] = gload(d.X0 + i + j * NB);
    }
    if (b1 > 0) {
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
            w[t] = gload(d.X1 + i + j * NB);
        }
    }
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
        if (i < n0 && j < n0) d.LW[i + j * d.ldw] = v[t];
    }
    if (b1 <= 0) return;
    T l[PT];
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
        const bool ok = i < b1;
        l[t] = gload(d.L10 + (ok ? i + (int64_t)j * d.ldl : 0));
    }
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
        // zero block above X1, X1 itself
        if (j < b1) d.LW[i + (NB + j) * d.ldw] = zero<T>();
        if (i < b1 && j < b1) d.LW[(NB + i) + (NB + j) * d.ldw] = w[t];
        // T1 = L10 X0: Sa[k][i] = L10(i, k) (rows >= b1 read as zero), Sb[k][j] = X0(k, j)
        Sa[j][i] = (i < b1) ? l[t] : zero<T>();
        Sb[i][j] = v[t];
    }
    __syncthreads();
    const int ti = 4 * (tid & 15), tj = 4 * (tid >> 4);
    T acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = zero<T>();
    for (int k2 = 0; k2 < NB; ++k2) {
        T av[4], bv[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) av[a] = Sa[k2][ti + a];
#pragma unroll
        for (int b = 0; b < 4; ++b) bv[b] = Sb[k2][tj + b];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] += av[a] * bv[b];
    }
    __syncthreads();
    // X10 = -X1 T1: Sa[k][i] = X1(i, k), Sb[k][j] = T1(k, j)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) Sb[ti + a][tj + b] = acc[a][b];
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int e = tid + 256 * t, i = e & (NB - 1), j = e / NB;
        Sa[j][i] = w[t];
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = zero<T>();
    for (int k2 = 0; k2 < NB; ++k2) {
        T av[4], bv[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) av[a] = Sa[k2][ti + a];
#pragma unroll
        for (int b = 0; b < 4; ++b) bv[b] = Sb[k2][tj + b];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] += av[a] * bv[b];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (ti + a < b1) d.LW[(NB + ti + a) + (tj + b) * d.ldw] = -acc[a][b];
}

template <class T>
void launch_wide_inverse(const WideInvDesc<T>* d_descs, int ndesc, hipStream_t s) {
    if (ndesc <= 0) return;
    hipLaunchKernelGGL(k_wide_inverse<T>, dim3(ndesc), dim3(256), 0, s, d_descs);
}

// ---------------------------------------------------------------------------
// Extend-add: one workgroup per EXT_ROWS rows x cw columns of the parent's
// trapezoid (tiles above the diagonal return at once), one row per thread,
// the columns in groups of C. A parent row's entries in the children come from
// the inverse of their relative indices; child rows follow each other, so
// loads stay coalesced. Both children in one pass: the parent is read and
// written once. Bound by memory on large fronts and by one chain of three
// loads on small ones: a thread issues the loads of a group before its stores
// (the pools may alias, so the compiler would not). Per factorization against a
// pass per child (twice the launches): real 30^3 136 us from 191, 96 2D
// problems 0.65 ms from 0.77, complex 64^3 3.7 ms (5.1 TB/s) from 4.0, complex
// 120^3 in FP32 28 ms from 31; real 80^3 in FP32 3.5 ms from 3.25.
// ---------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(EXT_ROWS) void k_extend_add(const ExtendDesc<T>* __restrict__ descs,
                                                         const int* __restrict__ tile_start, int nd) {
    constexpr int C = sizeof(T) > 8 ? 4 : 8;
    const int c = find_segment(tile_start, nd, blockIdx.x);
    const ExtendDesc<T> d = descs[c];
    const int t = blockIdx.x - tile_start[c], chunks = (d.mp - d.j0 + EXT_ROWS - 1) / EXT_ROWS;
    const int i0 = d.j0 + t % chunks * EXT_ROWS, i = i0 + threadIdx.x;
    int J0 = d.j0 + t / chunks * d.cw;
    const int J1 = min(min(J0 + d.cw, d.j0 + d.nc), i0 + EXT_ROWS);
    if (J0 >= J1) return;
    const int2 r = i < d.mp ? d.inv[i] : int2{-1, -1};
    const bool in0 = r.x >= 0, in1 = r.y >= 0;
    for (; J0 < J1; J0 += C) {
        T v0[C], v1[C], w[C];
        bool a0[C], a1[C];
        T* dst[C];
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int J = min(J0 + q, J1 - 1);
            const bool low = J == J0 + q && i >= J;
            const int2 jc = d.inv[J];
            a0[q] = low && in0 && jc.x >= 0;
            a1[q] = low && in1 && jc.y >= 0;
            dst[q] = (J < d.np ? d.Lp + (int64_t)J * d.mp
                               : d.Up + (int64_t)(J - d.np) * d.up - d.np) + i;
            if (a0[q]) v0[q] = d.Uc[0][r.x + (int64_t)jc.x * d.uc[0]];
            if (a1[q]) v1[q] = d.Uc[1][r.y + (int64_t)jc.y * d.uc[1]];
            if (a0[q] || a1[q]) w[q] = *dst[q];
        }
#pragma unroll
        for (int q = 0; q < C; ++q) {
            if (a0[q]) w[q] += v0[q];
            if (a1[q]) w[q] += v1[q];
            if (a0[q] || a1[q]) *dst[q] = w[q];
        }
    }
}

template <class T>
void launch_extend_add(const ExtendDesc<T>* d_descs, const int* d_tile_start, int ndesc,
                       int ntiles, hipStream_t s) {
    if (ntiles <= 0) return;
    hipLaunchKernelGGL(k_extend_add<T>, dim3(ntiles), dim3(EXT_ROWS), 0, s, d_descs, d_tile_start,
                       ndesc);
}

// ---------------------------------------------------------------------------
// Fused panel step of the LDL solves' triangular sweeps over the inverted
// SB-wide diagonal blocks (FrontLowerForwardSolve / FrontLowerBackwardSolve,
// lower_solve/local_front.hpp:35-82): one launch per panel of a level instead
// of two dependent products. Every workgroup forms, for 16 right-hand sides,
//     forward:  Y = Linv_pp X(p),         backward: Y = op(Linv_pp)^T X2(p)
// (Linv_pp lower triangular: only the triangle's K range is read); the
// panel's own workgroups write Y as the panel's rows of the output, the band
// workgroups apply to 64 rows r of the band
//     forward:  X(r) -= L(r, p) Y,        backward: X2(r) -= op(L(p, r))^T Y.
// Y is recomputed by each workgroup (no dependency inside the launch); the
// host keeps the band to the panels of one super-panel and updates the rows
// past it with one grouped product per super-panel.
// 512 threads: in the Y product wave w owns rows 16w..16w+15; in the band
// product wave w owns rows 16(w & 3).. of the 64 and half (w >> 2) of K, the
// two halves summed through LDS. Complex FP32 uses three real MFMAs per
// block as the grouped GEMM does.
// ---------------------------------------------------------------------------
template <class T, bool BWD, bool CONJ>
__global__ __launch_bounds__(512) void k_panel_step(const PanelStepDesc<T>* __restrict__ descs,
                                                    const int* __restrict__ task_start, int nd) {
    using R = typename Scalar<T>::real;
    using A4 = typename Acc4<R>::type;
    constexpr bool CPX = Scalar<T>::complex;
    constexpr bool F64 = sizeof(R) == 8;
    constexpr bool M3 = CPX && !F64 && GEMM_3M;
    constexpr int NP = CPX ? 2 : 1;
    constexpr int NA = M3 ? 3 : (CPX ? 2 : 1);   // accumulators per block
    constexpr int PB = PANEL_MAX;
    constexpr int K2 = PB / 8;                   // 4-deep steps of one K half of the band product
    __shared__ R Bs[NP][PB][16];     // the panel's rows of the input
    __shared__ R Ys[NP][PB][16];     // Y
    __shared__ R Red[4][NA][64][4];  // K-half partial sums of the band product

    const int t = blockIdx.x;
    const int di = find_segment(task_start, nd, t);
    const PanelStepDesc<T> d = descs[di];
    const int cg = (d.k + 15) / 16;
    const int loc = t - task_start[di];
    const bool owner = loc < cg;
    const int c16 = owner ? loc : (loc - cg) % cg;
    const int rb = owner ? 0 : (loc - cg) / cg;
    const int c0 = 16 * c16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sbw = d.sbw;
    auto opc = [](T v) { return CONJ ? conj_(v) : v; };
    // fragment layout of the 16x16x4 MFMAs: lane holds A(l % 16, k0 + l / 16),
    // B(k0 + l / 16, l % 16) and, of the 16x16 result, rows rin(r), column l % 16
    const int fr = lane & 15, fk = lane >> 4;
    auto rin = [&](int r) { return F64 ? fk + 4 * r : 4 * fk + r; };

    // Loads that do not depend on Y are all issued first, none behind a
    // branch (a value merged after a branch waits for its load there; an
    // out-of-range element reads the block's first entry and is replaced by
    // zero when used): the panel's rows of the input, the band fragments
    // op(L)(r, k) of this wave, and the band rows of X this wave updates.
    T xb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int idx = tid + 512 * e, kr = idx >> 4, j = idx & 15;
        const bool ok = kr < sbw && c0 + j < d.k;
        xb[e] = gload(d.Xin + (ok ? (d.w0 + kr) + (int64_t)(c0 + j) * d.ldx : 0));
    }
    const int r0 = d.b0 + 64 * rb;
    const int half = wave >> 2, blk = wave & 3;
    const int r2 = r0 + 16 * blk + fr;
    const int kb2 = 64 * half, ke2 = min(sbw, kb2 + 64);
    T a2[K2];
    unsigned ok2 = 0;
#pragma unroll
    for (int q = 0; q < K2; ++q) {
        const int kA = kb2 + 4 * q + fk;
        const bool ok = !owner && r2 < d.b1 && kA < ke2;
        const int64_t off = BWD ? kA + (int64_t)r2 * d.ldl : r2 + (int64_t)kA * d.ldl;
        a2[q] = gload(d.Lp + (ok ? off : 0));
        ok2 |= ok ? 1u << q : 0u;
    }
    T xo[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = r0 + 16 * blk + rin(q);
        const bool ok = !owner && half == 0 && row < d.b1 && c0 + fr < d.k;
        xo[q] = gload(d.Xin + (ok ? row + (int64_t)(c0 + fr) * d.ldx : 0));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int idx = tid + 512 * e, kr = idx >> 4, j = idx & 15;
        const T x = pick(kr < sbw && c0 + j < d.k, xb[e], zero<T>());
        Bs[0][kr][j] = re(x);
        if constexpr (CPX) Bs[NP - 1][kr][j] = im(x);
    }
    __syncthreads();

    auto mac = [&](A4 (&acc)[3], T a, int kr, R (*B)[PB][16]) {
        const R aR = re(a), aI = CPX ? im(a) : R(0);
        const R bR = B[0][kr][fr], bI = CPX ? B[NP - 1][kr][fr] : R(0);
        if constexpr (M3) {
            acc[0] = mfma16(aR, bR, acc[0]);
            acc[1] = mfma16(aI, bI, acc[1]);
            acc[2] = mfma16(aR + aI, bR + bI, acc[2]);
        } else {
            acc[0] = mfma16(aR, bR, acc[0]);
            if constexpr (CPX) {
                acc[0] = mfma16(-aI, bI, acc[0]);
                acc[1] = mfma16(aR, bI, acc[1]);
                acc[1] = mfma16(aI, bR, acc[1]);
            }
        }
    };
    auto value = [&](const A4 (&acc)[3], int r) -> T {
        if constexpr (M3) return make_t<T>(acc[0][r] - acc[1][r], acc[2][r] - acc[0][r] - acc[1][r]);
        else return make_t<T>(acc[0][r], CPX ? acc[1][r] : R(0));
    };

    // Y: wave w, rows 16w..16w+15, K over the triangle in 16-deep chunks,
    // the next chunk's fragments loaded while the current one is multiplied
    {
        A4 acc[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[a] = A4{0, 0, 0, 0};
        const int i1 = 16 * wave + fr;
        const int kb = BWD ? 16 * wave : 0;
        const int ke = 16 * wave < sbw ? (BWD ? sbw : min(sbw, 16 * wave + 16)) : kb;
        auto fetch = [&](T (&av)[4], int k0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kA = k0 + 4 * q + fk;
                const bool ok = i1 < sbw && kA < ke;
                const int64_t off = BWD ? kA + (int64_t)i1 * sbw : i1 + (int64_t)kA * sbw;
                const T v = gload(d.LW + (ok ? off : 0));
                av[q] = pick(ok, BWD ? opc(v) : v, zero<T>());
            }
        };
        T cur[4], nxt[4];
        if (kb < ke) fetch(cur, kb);
        for (int k0 = kb; k0 < ke; k0 += 16) {
            if (k0 + 16 < ke) fetch(nxt, k0 + 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) mac(acc, cur[q], k0 + 4 * q + fk, Bs);
#pragma unroll
            for (int q = 0; q < 4; ++q) cur[q] = nxt[q];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * wave + rin(r);
            const T y = value(acc, r);
            Ys[0][row][fr] = re(y);
            if constexpr (CPX) Ys[NP - 1][row][fr] = im(y);
            if (owner && row < sbw && c0 + fr < d.k)
                gstore(d.Xout + (d.w0 + row) + (int64_t)(c0 + fr) * d.ldx, y);
        }
    }
    if (owner) return;
    __syncthreads();

    // band rows r0 .. r0 + 63 (clipped to b1): X(r) -= op(L) Y
    A4 acc[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) acc[a] = A4{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < K2; ++q) {
        const int k4 = kb2 + 4 * q;
        if (k4 < ke2) {   // uniform across the wave
            const T a = pick((ok2 >> q) & 1u, BWD ? opc(a2[q]) : a2[q], zero<T>());
            mac(acc, a, k4 + fk, Ys);
        }
    }
    if (half == 1) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q) Red[blk][a][lane][q] = acc[a][q];
    }
    __syncthreads();
    if (half == 1) return;
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[a][q] += Red[blk][a][lane][q];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = r0 + 16 * blk + rin(q);
        if (row >= d.b1 || c0 + fr >= d.k) continue;
        gstore(d.Xin + row + (int64_t)(c0 + fr) * d.ldx, xo[q] - value(acc, q));
    }
}

template <class T>
void launch_panel_step(const PanelStepDesc<T>* d, const int* task_start, int nd, int ntasks,
                       bool backward, bool conj, hipStream_t s) {
    if (nd <= 0 || ntasks <= 0) return;
    if (!backward)
        hipLaunchKernelGGL((k_panel_step<T, false, false>), dim3(ntasks), dim3(512), 0, s, d,
                           task_start, nd);
    else if (conj)
        hipLaunchKernelGGL((k_panel_step<T, true, true>), dim3(ntasks), dim3(512), 0, s, d,
                           task_start, nd);
    else
        hipLaunchKernelGGL((k_panel_step<T, true, false>), dim3(ntasks), dim3(512), 0, s, d,
                           task_start, nd);
}

// ---------------------------------------------------------------------------
// Solve helpers. Column j of an N x k block is blockIdx.y (k <= 65535 is
// checked by the host), rows are strided over blockIdx.x: no 64-bit index
// division per element.
// ---------------------------------------------------------------------------
static inline unsigned grid_for(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    if (b < 1) b = 1;
    return (unsigned)b;
}
static inline dim3 grid_cols(int N, int k) {
    unsigned gx = grid_for(N);
    if (gx > 512) gx = 512;
    return dim3(gx, (unsigned)k);
}

// xn(map[i], j) = x(i, j): reads of x (the wide type) coalesced, map[i] the
// nodal index of original row i
template <class T, class V>
__global__ void k_pull(const V* __restrict__ x, int64_t ldx, const int* __restrict__ map,
                       T* __restrict__ xn, int N) {
    const int j = blockIdx.y;
    const V* xc = x + (int64_t)j * ldx;
    T* yc = xn + (int64_t)j * N;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        yc[map[i]] = cvt<T>(xc[i]);
}
// x(i, j) = xn(map[i], j): writes of x coalesced
template <class T, class V>
__global__ void k_push(const T* __restrict__ xn, const int* __restrict__ map, V* __restrict__ x,
                       int64_t ldx, int N) {
    const int j = blockIdx.y;
    const T* xc = xn + (int64_t)j * N;
    V* yc = x + (int64_t)j * ldx;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        yc[i] = cvt<V>(xc[map[i]]);
}

template <class T, class V>
void launch_pull(const V* x, int64_t ldx, const int* map, T* xn, int N, int k, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL((k_pull<T, V>), grid_cols(N, k), dim3(256), 0, s, x, ldx, map, xn, N);
}
template <class T, class V>
void launch_push(const T* xn, const int* map, V* x, int64_t ldx, int N, int k, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL((k_push<T, V>), grid_cols(N, k), dim3(256), 0, s, xn, map, x, ldx, N);
}

// Right-hand-side columns a gather / solve extend-add thread handles: all of
// a thread's loads are issued before its stores (the destination may alias
// the source pool, so the compiler could not reorder them itself).
constexpr int RHS_CHUNK = 8;

template <class T>
__global__ void k_gather(const SolveSeg* __restrict__ segs, const int* __restrict__ row_start,
                         int nseg, int nrows, T* __restrict__ wpool, const T* __restrict__ xn,
                         int N, int k, const int* __restrict__ lowpool) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nrows) return;
    const int j0 = blockIdx.y * RHS_CHUNK;
    const int si = find_segment(row_start, nseg, g);
    const SolveSeg sg = segs[si];
    const int i = g - row_start[si];
    T* w = wpool + sg.w * k + i + (int64_t)j0 * sg.u;
    const T* src = xn + lowpool[sg.low + i] + (int64_t)j0 * N;
    T v[RHS_CHUNK];
#pragma unroll
    for (int q = 0; q < RHS_CHUNK; ++q)
        if (j0 + q < k) v[q] = src[(int64_t)q * N];
#pragma unroll
    for (int q = 0; q < RHS_CHUNK; ++q)
        if (j0 + q < k) w[(int64_t)q * sg.u] = v[q];
}
template <class T>
void launch_gather(const SolveSeg* segs, const int* row_start, int nseg, int nrows, T* wpool,
                   const T* xn, int N, int k, const int* lowpool, hipStream_t s) {
    if (nrows <= 0 || k <= 0) return;
    hipLaunchKernelGGL(k_gather<T>, dim3((nrows + 255) / 256, (k + RHS_CHUNK - 1) / RHS_CHUNK),
                       dim3(256), 0, s, segs, row_start, nseg, nrows, wpool, xn, N, k, lowpool);
}

// One thread per parent row and RHS_CHUNK columns, both children's rows added
// in one pass (see k_extend_add). Bound by launch and load latency: 15 launches
// of 3.4 us for a solve of a 30^3 problem instead of 30 of 3.3.
template <class T>
__global__ void k_solve_extend(const SolveExtend* __restrict__ ds, const int* __restrict__ row_start,
                               int nd, int nrows, T* __restrict__ wpool, T* __restrict__ xn, int N,
                               const int2* __restrict__ invpool, int k) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nrows) return;
    const int j0 = blockIdx.y * RHS_CHUNK;
    const int c = find_segment(row_start, nd, g);
    const SolveExtend d = ds[c];
    const int I = g - row_start[c] + d.i0;
    const int2 r = invpool[d.inv + I];
    if (r.x < 0 && r.y < 0) return;
    const T* w0 = wpool + d.wc[0] * k + max(r.x, 0) + (int64_t)j0 * d.uc[0];
    const T* w1 = wpool + d.wc[1] * k + max(r.y, 0) + (int64_t)j0 * d.uc[1];
    T* dst;
    int64_t ld;
    if (I < d.np) {
        dst = xn + d.offp + I;
        ld = N;
    } else {
        dst = wpool + d.wp * k + (I - d.np);
        ld = d.up;
    }
    dst += (int64_t)j0 * ld;
    T a0[RHS_CHUNK], a1[RHS_CHUNK], b[RHS_CHUNK];
#pragma unroll
    for (int q = 0; q < RHS_CHUNK; ++q)
        if (j0 + q < k) {
            if (r.x >= 0) a0[q] = w0[(int64_t)q * d.uc[0]];
            if (r.y >= 0) a1[q] = w1[(int64_t)q * d.uc[1]];
            b[q] = dst[(int64_t)q * ld];
        }
#pragma unroll
    for (int q = 0; q < RHS_CHUNK; ++q)
        if (j0 + q < k) {
            if (r.x >= 0) b[q] += a0[q];
            if (r.y >= 0) b[q] += a1[q];
            dst[(int64_t)q * ld] = b[q];
        }
}
template <class T>
void launch_solve_extend(const SolveExtend* d, const int* row_start, int nd, int nrows,
                         T* wpool, T* xn, int N, const int2* invpool, int k, hipStream_t s) {
    if (nrows <= 0 || k <= 0) return;
    hipLaunchKernelGGL(k_solve_extend<T>,
                       dim3((nrows + 255) / 256, (k + RHS_CHUNK - 1) / RHS_CHUNK), dim3(256), 0, s,
                       d, row_start, nd, nrows, wpool, xn, N, invpool, k);
}

// One thread per row: the pivot's reciprocal once, then its k columns
template <class T, class V>
__global__ void k_diag_solve(T* __restrict__ xn, const V* __restrict__ D, int N, int k,
                             int* status) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < N; p += gridDim.x * blockDim.x) {
        const V dv = D[p];
        if (is_zero_or_nonfinite(dv)) record_status(status, 2, -1, p);
        const V r = one<V>() / dv;
        T* xc = xn + p;
        for (int j = 0; j < k; ++j) xc[(int64_t)j * N] = cvt<T>(cvt<V>(xc[(int64_t)j * N]) * r);
    }
}
template <class T, class V>
void launch_diag_solve(T* xn, const V* D, int N, int k, int* d_status, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL((k_diag_solve<T, V>), dim3(grid_for(N)), dim3(256), 0, s, xn, D, N, k,
                       d_status);
}

// ---------------------------------------------------------------------------
// FP64 sparse kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ void atomic_max_nonneg(unsigned long long* p, double v) {
    atomicMax(p, (unsigned long long)__double_as_longlong(v));
}

// y := alpha A x + beta b over CSR rows (b = y when null); with colmax,
// colmax[j] = max(colmax[j], max_i |y(i, j)|). One thread per (row, 8
// right-hand sides). Bound by memory: what matters is the loads in flight, so
// for rows of at most 8 entries no load sits behind a branch of a lane (an
// entry past the row's end loads one that exists and its product is dropped;
// a divergent load would be waited for inside its branch) and the next two
// columns' loads are issued before a pair's products (16 complex right-hand
// sides of an 81 x 80 x 77 stencil, 325 MB: 138 -> 97 us; one column ahead
// 101, chunks of 4 columns 105, of 16 columns 163).
constexpr int SPMV_COLS = 8, SPMV_ROWNZ = 8;
// Row blocks whose column chunks run one after the other: their part of A is
// then read from L2 for every chunk but the first.
constexpr int SPMV_GROUP = 32;
// With xn, y is not written: row i of the result goes to xn(map[i], j) in the
// working type (the nodal right-hand side of a refinement solve), ld N.
template <class V, class T>
__global__ __launch_bounds__(256) void k_spmv(int N, const int64_t* __restrict__ rowoff,
                                              const int* __restrict__ cols,
                                              const V* __restrict__ vals, double alpha,
                                              const V* __restrict__ x, int64_t ldx, double beta,
                                              const V* __restrict__ b, int64_t ldb,
                                              V* __restrict__ y, int64_t ldy, int k,
                                              unsigned long long* colmax, T* __restrict__ xn,
                                              const int* __restrict__ map) {
    constexpr int SPMV_BATCH = 2;
    __shared__ double red[SPMV_COLS][4];
    // one-dimensional grid of (row block, column chunk) pairs, remapped so
    // each XCD runs a contiguous range of row blocks: the stencil's
    // neighbours in x then come from that XCD's L2
    const int rb = (N + 255) / 256, nch = (k + SPMV_COLS - 1) / SPMV_COLS;
    const int t = xcd_remap(blockIdx.x, gridDim.x);
    const int grp = t / (SPMV_GROUP * nch), in = t - grp * (SPMV_GROUP * nch);
    const int gw = min(SPMV_GROUP, rb - grp * SPMV_GROUP);
    const int i = (grp * SPMV_GROUP + in % gw) * 256 + threadIdx.x;
    const int j0 = (in / gw) * SPMV_COLS;
    const int nj = min(SPMV_COLS, k - j0);
    double m[SPMV_COLS];
#pragma unroll
    for (int q = 0; q < SPMV_COLS; ++q) m[q] = 0.0;
    if (i < N) {
        V acc[SPMV_COLS];
#pragma unroll
        for (int q = 0; q < SPMV_COLS; ++q) acc[q] = V{};
        const int64_t e0 = rowoff[i], e1 = rowoff[i + 1];
        const int ne = (int)(e1 - e0);
        const unsigned long long some = __ballot(ne > 0);
        if (some == 0) {
            // nothing stored in these rows
        } else if (!__any(ne > SPMV_ROWNZ)) {
            const int64_t safe = __shfl(e0, __ffsll(some) - 1);   // an entry that exists
            int c[SPMV_ROWNZ];
            V a[SPMV_ROWNZ];
#pragma unroll
            for (int u = 0; u < SPMV_ROWNZ; ++u) {
                const int64_t e = u < ne ? e0 + u : safe;
                c[u] = cols[e];
                a[u] = gload(vals + e);
            }
            const bool last = __any(ne == SPMV_ROWNZ);   // a stencil's rows have seven
            V xv[2][SPMV_BATCH][SPMV_ROWNZ];
            // columns past the last one load it again
            auto fetch = [&](int buf, int q0) {
#pragma unroll
                for (int q = 0; q < SPMV_BATCH; ++q) {
                    const V* xc = x + (int64_t)(j0 + min(q0 + q, nj - 1)) * ldx;
#pragma unroll
                    for (int u = 0; u < SPMV_ROWNZ - 1; ++u) xv[buf][q][u] = gload(xc + c[u]);
                    if (last) xv[buf][q][SPMV_ROWNZ - 1] = gload(xc + c[SPMV_ROWNZ - 1]);
                }
            };
            fetch(0, 0);
#pragma unroll
            for (int q0 = 0; q0 < SPMV_COLS; q0 += SPMV_BATCH) {
                const int buf = (q0 / SPMV_BATCH) & 1;
                if (q0 + SPMV_BATCH < nj) fetch(buf ^ 1, q0 + SPMV_BATCH);
#pragma unroll
                for (int q = 0; q < SPMV_BATCH; ++q) {
                    V sum = V{};
#pragma unroll
                    for (int u = 0; u < SPMV_ROWNZ - 1; ++u)
                        sum = pick(u < ne, sum + a[u] * xv[buf][q][u], sum);
                    if (last)
                        sum = pick(SPMV_ROWNZ - 1 < ne,
                                   sum + a[SPMV_ROWNZ - 1] * xv[buf][q][SPMV_ROWNZ - 1], sum);
                    acc[q0 + q] = sum;
                }
            }
        } else {
            for (int64_t e = e0; e < e1; ++e) {
                const V a = vals[e];
                const V* xc = x + cols[e] + (int64_t)j0 * ldx;
#pragma unroll
                for (int q = 0; q < SPMV_COLS; ++q)
                    if (q < nj) acc[q] = acc[q] + a * xc[q * ldx];
            }
        }
#pragma unroll
        for (int q = 0; q < SPMV_COLS; ++q) {
            if (q >= nj) break;
            V* py = y + i + (int64_t)(j0 + q) * ldy;
            V out = scale(acc[q], alpha);
            if (beta != 0.0) out = out + scale(b ? b[i + (int64_t)(j0 + q) * ldb] : *py, beta);
            if (xn) xn[map[i] + (int64_t)(j0 + q) * N] = cvt<T>(out);
            else *py = out;
            m[q] = abs1(out);
        }
    }
    if (colmax) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (int q = 0; q < SPMV_COLS; ++q) {
            double v = m[q];
            for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
            if (lane == 0) red[q][wave] = v;
        }
        __syncthreads();
        if (threadIdx.x < nj) {
            const int q = threadIdx.x;
            const double v = fmax(fmax(red[q][0], red[q][1]), fmax(red[q][2], red[q][3]));
            atomic_max_nonneg(colmax + j0 + q, v);
        }
    }
}
template <class V, class T>
static void launch_spmv_any(int N, const int64_t* rowoff, const int* cols, const V* vals,
                            double alpha, const V* x, int64_t ldx, double beta, const V* b,
                            int64_t ldb, V* y, int64_t ldy, int k, unsigned long long* colmax,
                            T* xn, const int* map, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    const int64_t blocks = (int64_t)((N + 255) / 256) * ((k + SPMV_COLS - 1) / SPMV_COLS);
    if (blocks > 0x7fffffff) throw Error(1, "SpMV grid too large");
    hipLaunchKernelGGL((k_spmv<V, T>), dim3((unsigned)blocks), dim3(256), 0, s, N, rowoff, cols,
                       vals, alpha, x, ldx, beta, b, ldb, y, ldy, k, colmax, xn, map);
}
template <class V>
void launch_spmv_ex(int N, const int64_t* rowoff, const int* cols, const V* vals, double alpha,
                    const V* x, int64_t ldx, double beta, const V* b, int64_t ldb, V* y,
                    int64_t ldy, int k, unsigned long long* colmax, hipStream_t s) {
    launch_spmv_any<V, V>(N, rowoff, cols, vals, alpha, x, ldx, beta, b, ldb, y, ldy, k, colmax,
                          nullptr, nullptr, s);
}
template <class T, class V>
void launch_residual_nodal(int N, const int64_t* rowoff, const int* cols, const V* vals,
                           const V* x, int64_t ldx, const V* b, int64_t ldb, int k,
                           unsigned long long* colmax, T* xn, const int* map, hipStream_t s) {
    launch_spmv_any<V, T>(N, rowoff, cols, vals, -1.0, x, ldx, 1.0, b, ldb, nullptr, 0, k, colmax,
                          xn, map, s);
}

// x(i, j) += xn(map[i], j) with colmax[j] = max(colmax[j], max_i |x(i, j)|)
template <class T, class V>
__global__ __launch_bounds__(256) void k_push_add_abs(const T* __restrict__ xn,
                                                      const int* __restrict__ map,
                                                      V* __restrict__ x, int64_t ldx, int N,
                                                      unsigned long long* colmax) {
    __shared__ double red[4];
    const T* xc = xn + (int64_t)blockIdx.y * N;
    V* yc = x + (int64_t)blockIdx.y * ldx;
    double m = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const V v = yc[i] + cvt<V>(xc[map[i]]);
        yc[i] = v;
        m = fmax(m, abs1(v));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        atomic_max_nonneg(colmax + blockIdx.y, fmax(fmax(red[0], red[1]), fmax(red[2], red[3])));
}
template <class T, class V>
void launch_push_add_abs(const T* xn, const int* map, V* x, int64_t ldx, int N, int k,
                         unsigned long long* colmax, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL((k_push_add_abs<T, V>), grid_cols(N, k), dim3(256), 0, s, xn, map, x, ldx,
                       N, colmax);
}
template <class V>
void launch_spmv(int N, const int64_t* rowoff, const int* cols, const V* vals, double alpha,
                 const V* x, int64_t ldx, double beta, V* y, int64_t ldy, int k, hipStream_t s) {
    launch_spmv_ex<V>(N, rowoff, cols, vals, alpha, x, ldx, beta, nullptr, 0, y, ldy, k, nullptr,
                      s);
}

template <class V>
__global__ void k_row_abs_sum_max(int N, const int64_t* __restrict__ rowoff,
                                  const V* __restrict__ vals, unsigned long long* out) {
    __shared__ double red[256];
    double m = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int64_t e = rowoff[i]; e < rowoff[i + 1]; ++e) s += abs1(vals[e]);
        m = fmax(m, s);
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) atomic_max_nonneg(out, red[0]);
}
template <class V>
void launch_row_abs_sum_max(int N, const int64_t* rowoff, const V* vals, unsigned long long* out,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_row_abs_sum_max<V>, dim3(grid_for(N) > 1024 ? 1024 : grid_for(N)),
                       dim3(256), 0, s, N, rowoff, vals, out);
}

template <class V>
__global__ void k_col_abs_max(const V* __restrict__ x, int64_t ldx, int N,
                              unsigned long long* out) {
    __shared__ double red[256];
    const int j = blockIdx.y;
    double m = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        m = fmax(m, abs1(x[i + j * ldx]));
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) atomic_max_nonneg(out + j, red[0]);
}
template <class V>
void launch_col_abs_max(const V* x, int64_t ldx, int N, int k, unsigned long long* out,
                        hipStream_t s) {
    unsigned gx = grid_for(N);
    if (gx > 256) gx = 256;
    hipLaunchKernelGGL(k_col_abs_max<V>, dim3(gx, k), dim3(256), 0, s, x, ldx, N, out);
}

template <class V>
__global__ void k_copy_cols(V* __restrict__ y, int64_t ldy, const V* __restrict__ x, int64_t ldx,
                            int N) {
    V* yc = y + (int64_t)blockIdx.y * ldy;
    const V* xc = x + (int64_t)blockIdx.y * ldx;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        yc[i] = xc[i];
}
template <class V>
void launch_copy_cols(V* y, int64_t ldy, const V* x, int64_t ldx, int N, int k, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL(k_copy_cols<V>, grid_cols(N, k), dim3(256), 0, s, y, ldy, x, ldx, N);
}

template <class V>
__global__ void k_adjoint_dA(int N, const int64_t* __restrict__ rowoff, const int* __restrict__ cols,
                             const V* __restrict__ lam, int64_t ldl, const V* __restrict__ x,
                             int64_t ldx, int k, bool conj, V* __restrict__ dA) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        for (int64_t e = rowoff[i]; e < rowoff[i + 1]; ++e) {
            const int c = cols[e];
            V acc = V{};
            for (int r = 0; r < k; ++r) acc = acc + lam[i + r * ldl] * cj(x[c + r * ldx], conj);
            dA[e] = -acc;
        }
    }
}
template <class V>
void launch_adjoint_dA(int N, const int64_t* rowoff, const int* cols, const V* lambda,
                       int64_t ldl, const V* x, int64_t ldx, int k, bool conj, V* dA,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_adjoint_dA<V>, dim3(grid_for(N)), dim3(256), 0, s, N, rowoff, cols, lambda,
                       ldl, x, ldx, k, conj, dA);
}

template <class T, class V>
__global__ void k_widen(const T* __restrict__ src, V* __restrict__ dst, int64_t n) {
    for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n;
         g += (int64_t)gridDim.x * blockDim.x)
        dst[g] = cvt<V>(src[g]);
}
template <class T, class V>
void launch_widen(const T* src, V* dst, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_widen<T, V>), dim3(grid_for(n)), dim3(256), 0, s, src, dst, n);
}

template <class V>
__global__ void k_permute_rows(const V* __restrict__ src, int64_t lds, V* __restrict__ dst,
                               int64_t ldd, const int* __restrict__ perm, int N, bool scatter) {
    const V* sc = src + (int64_t)blockIdx.y * lds;
    V* dc = dst + (int64_t)blockIdx.y * ldd;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < N; p += gridDim.x * blockDim.x) {
        if (scatter) dc[perm[p]] = sc[p];
        else dc[p] = sc[perm[p]];
    }
}
template <class V>
void launch_permute_rows(const V* src, int64_t lds, V* dst, int64_t ldd, const int* perm, int N,
                         int k, bool scatter, hipStream_t s) {
    if (N <= 0 || k <= 0) return;
    hipLaunchKernelGGL(k_permute_rows<V>, grid_cols(N, k), dim3(256), 0, s, src, lds, dst, ldd,
                       perm, N, scatter);
}

template <class V>
__global__ __launch_bounds__(256) void k_col_sumsq(const V* __restrict__ x, int64_t ldx, int N,
                                                   double* out) {
    __shared__ double red[256];
    const V* xc = x + (int64_t)blockIdx.x * ldx;
    double acc = 0.0;
    for (int i = threadIdx.x; i < N; i += 256) acc += sq_mod(xc[i]);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}
template <class V>
void launch_col_sumsq(const V* x, int64_t ldx, int N, int k, double* out, hipStream_t s) {
    if (k <= 0) return;
    hipLaunchKernelGGL(k_col_sumsq<V>, dim3(k), dim3(256), 0, s, x, ldx, N, out);
}

__global__ void k_fill_int(int* __restrict__ p, int n, int value) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        p[i] = value;
}
void launch_fill_int(int* p, int n, int value, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_int, dim3(grid_for(n)), dim3(256), 0, s, p, n, value);
}

// ---------------------------------------------------------------------------
// explicit instantiations
// ---------------------------------------------------------------------------
#define CQ_INST_T(T)                                                                           \
    template void launch_zero_segments<T>(const ZeroSeg<T>*, const int*, int, int, hipStream_t); \
    template void launch_copy2d<T>(const CopyDesc<T>*, const int*, int, int, hipStream_t);       \
    template void launch_reduce_slices<T>(const ReduceDesc<T>*, const int*, int, int, hipStream_t); \
    template void launch_zero_lower<T>(const ZeroLowerDesc<T>*, const int*, int, int, hipStream_t); \
    template void launch_gemm<T>(const GemmDesc<T>*, const int*, int, int, int, int, int, hipStream_t);   \
    template void launch_extend_add<T>(const ExtendDesc<T>*, const int*, int, int, hipStream_t); \
    template void launch_wide_inverse<T>(const WideInvDesc<T>*, int, hipStream_t);        \
    template void launch_gather<T>(const SolveSeg*, const int*, int, int, T*, const T*, int,    \
                                   int, const int*, hipStream_t);                               \
    template void launch_solve_extend<T>(const SolveExtend*, const int*, int, int, T*, T*, int, \
                                         const int2*, int, hipStream_t);                        \
    template void launch_panel_step<T>(const PanelStepDesc<T>*, const int*, int, int, bool, bool, \
                                       hipStream_t);

CQ_INST_T(float)
CQ_INST_T(double)
CQ_INST_T(cfloat)
CQ_INST_T(cdouble)

#define CQ_INST_TV(T, V)                                                                        \
    template void launch_assemble<T, V>(const V*, const int64_t*, int64_t, T*, bool, hipStream_t); \
    template void launch_pull<T, V>(const V*, int64_t, const int*, T*, int, int, hipStream_t);   \
    template void launch_push<T, V>(const T*, const int*, V*, int64_t, int, int, hipStream_t);   \
    template void launch_diag_solve<T, V>(T*, const V*, int, int, int*, hipStream_t);           \
    template void launch_widen<T, V>(const T*, V*, int64_t, hipStream_t);                        \
    template void launch_residual_nodal<T, V>(int, const int64_t*, const int*, const V*,         \
                                              const V*, int64_t, const V*, int64_t, int,         \
                                              unsigned long long*, T*, const int*, hipStream_t); \
    template void launch_push_add_abs<T, V>(const T*, const int*, V*, int64_t, int, int,         \
                                            unsigned long long*, hipStream_t);

CQ_INST_TV(float, double)
CQ_INST_TV(double, double)
CQ_INST_TV(cfloat, cdouble)
CQ_INST_TV(cdouble, cdouble)

#define CQ_INST_V(V)                                                                            \
    template void launch_spmv<V>(int, const int64_t*, const int*, const V*, double, const V*,   \
                                 int64_t, double, V*, int64_t, int, hipStream_t);              \
    template void launch_spmv_ex<V>(int, const int64_t*, const int*, const V*, double,          \
                                    const V*, int64_t, double, const V*, int64_t, V*, int64_t,  \
                                    int, unsigned long long*, hipStream_t);                    \
    template void launch_row_abs_sum_max<V>(int, const int64_t*, const V*, unsigned long long*, \
                                            hipStream_t);                                      \
    template void launch_col_abs_max<V>(const V*, int64_t, int, int, unsigned long long*,       \
                                        hipStream_t);                                          \
    template void launch_copy_cols<V>(V*, int64_t, const V*, int64_t, int, int, hipStream_t);   \
    template void launch_permute_rows<V>(const V*, int64_t, V*, int64_t, const int*, int, int,  \
                                         bool, hipStream_t);                                    \
    template void launch_col_sumsq<V>(const V*, int64_t, int, int, double*, hipStream_t);      \
    template void launch_adjoint_dA<V>(int, const int64_t*, const int*, const V*, int64_t,      \
                                       const V*, int64_t, int, bool, V*, hipStream_t);

CQ_INST_V(double)
CQ_INST_V(cdouble)

}  // namespace cliqg
