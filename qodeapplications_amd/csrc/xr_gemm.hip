// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4f64).
//
// C_b = alpha * op(A_b) op(B_b) + beta * C_b.  Split-K goes through a
// workspace and a fixed-order reduction; an unsplit product applies alpha and
// beta where it stores C.  256 threads = 4 waves per workgroup, whose 16-row
// (or 32-row) fragments of the output tile are dealt out to the waves in
// turn.  K advances 16 at a time through two LDS stages, one barrier per step.
// Workgroups are remapped so each XCD (own L2) receives a contiguous run of
// output tiles.
#include "xr_common.h"
#include "xr_gemm.h"
#include <vector>
#include <algorithm>
#include <type_traits>

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef double d2_t __attribute__((ext_vector_type(2)));

#define GEMM_BK 16
#define GEMM_THREADS 256
// s_waitcnt operand: vmcnt 0, the other counters unlimited
#define GEMM_WAIT_VMCNT0 0x0F70
// output row of accumulator element r for lane group fk (lane / 16) of
// v_mfma_f32_16x16x4f32 (checked on gfx950; the f64 variant differs)
#define XR_F32_ROW(fk, r) (4 * (fk) + (r))

// blockIdx.x -> logical tile id, so that the ids one XCD executes (hardware
// hands out workgroups round-robin over the 8 XCDs) are contiguous.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t total) {
    const int64_t nx = 8;
    int64_t q = total / nx, r = total % nx;
    int64_t x = b % nx, j = b / nx;
    int64_t base = (x < r) ? x * (q + 1) : r * (q + 1) + (x - r) * q;
    return base + j;
}

// 16 bytes of zeros: where a load of a tile's padding (k past K) points.
static __device__ __align__(16) double xr_zero_page[2] = {0.0, 0.0};

// One operand of a tile: BX rows of op(A) (columns of op(B)) by 16 of k.
// KC: K is contiguous in memory (A as stored, B transposed); otherwise the
// BX index is.  LDS layout, in 16-byte chunks of two doubles:
//   KC   row x holds its 8 chunks of k, chunk c at slot c ^ (x & 7);
//   !KC  row k holds BX doubles.
// Fragment reads are 16 bytes: with KC a lane takes two k of one row, else
// two neighbouring rows x of one k.  A product over k may take its k in any
// order that both operands share, so lane group fk supplies k = 8 s + 2 fk + h
// to MFMA (s, h).  The slot XOR puts the 64 lanes of a KC read on distinct
// banks (rows are 128 bytes apart, so without it 8 rows share one).
//
// DIRECT: the chunks go from memory straight into LDS
// (global_load_lds_dwordx4: no staging registers, no LDS stores), which needs
// 16-byte aligned rows: base, leading dimension and the extent along the
// contiguous index even.  Otherwise 8-byte loads pass through registers.
// Rows past the edge read the last row again (their results are not
// stored); k past K reads the zero page.
template <int BX, bool KC, bool DIRECT>
struct TileOperand {
    static constexpr int NI = BX / 32;                    // DIRECT: load instructions per wave and stage
    static constexpr int NE = BX * GEMM_BK / GEMM_THREADS;   // registers: elements per thread and stage
    const double* p[DIRECT ? NI : 1];
    const double* base;
    double r[DIRECT ? 1 : NE];
    int64_t ld, x0, X;
    int kofs[DIRECT ? NI : 1];

    __device__ __forceinline__ void init(const double* src, int64_t ld_, int64_t x0_, int64_t X_, int lane, int wave) {
        base = src;
        ld = ld_;
        x0 = x0_;
        X = X_;
        if constexpr (DIRECT) {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                if (KC) {
                    int64_t x = x0 + wave * (BX / 4) + i * 8 + (lane >> 3);
                    if (x > X - 1) x = X - 1;
                    kofs[i] = 2 * ((lane & 7) ^ (lane >> 3));
                    p[i] = src + x * ld + kofs[i];
                } else {
                    int64_t x = x0 + 2 * (lane % (BX / 2));
                    if (x > X - 2) x = X - 2;
                    kofs[i] = (wave * NI + i) * (128 / BX) + lane / (BX / 2);
                    p[i] = src + kofs[i] * ld + x;
                }
            }
        }
    }
    // DIRECT: queues the loads of the next 16 k into `dst`; tail: only the
    // first `krest` of them exist.  (The empty asm keeps the two branches
    // apart: merged, every load of every stage pays the tail's selects.)
    __device__ __forceinline__ void stage(double* dst, bool tail, int krest, int wave) {
        auto go = [&](int i, const double* q) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)q,
                                             (__attribute__((address_space(3))) void*)(dst + (wave * NI + i) * 128),
                                             16, 0, 0);
        };
        if (tail) {
            asm volatile("");
#pragma unroll
            for (int i = 0; i < NI; i++) go(i, kofs[i] < krest ? p[i] : xr_zero_page);
            asm volatile("");
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                go(i, p[i]);
                p[i] += KC ? GEMM_BK : GEMM_BK * ld;
            }
        }
    }
    // registers: loads of k in [k0, k0 + 16), then their LDS stores.  The
    // first krest of them exist.
    __device__ __forceinline__ void load(int64_t k0, int krest, int tid) {
        if (KC) {
            const int k = tid & 15, xlast = (int)(X - x0 < BX ? X - x0 : BX) - 1;
            int x = tid >> 4;
            int64_t off = (x0 + (x < xlast ? x : xlast)) * ld + k0 + k;
#pragma unroll
            for (int i = 0; i < NE; i++) {
                const double* q = base + off;
                if (k >= krest) q = xr_zero_page;
                r[i] = *q;
                const int up = xlast - x < 16 ? xlast - x : 16;   // rows left below the clamp
                off += (up > 0 ? up : 0) * ld;
                x += 16;
                asm("" : "+v"(off));
            }
        } else {
            int64_t x = x0 + tid % BX;
            if (x > X - 1) x = X - 1;
            int k = tid / BX;
            int64_t off = (k0 + k) * ld + x;
#pragma unroll
            for (int i = 0; i < NE; i++) {
                const double* q = base + off;
                if (k >= krest) q = xr_zero_page;
                r[i] = *q;
                off += (GEMM_THREADS / BX) * ld;
                k += GEMM_THREADS / BX;
                asm("" : "+v"(off));           // one running offset, not one kept register pair per row
            }
        }
    }
    __device__ __forceinline__ void store(double* dst, int tid) {
#pragma unroll
        for (int i = 0; i < NE; i++) {
            if (KC) {
                const int k = tid & 15, x = (tid >> 4) + 16 * i;
                dst[x * GEMM_BK + 2 * ((k >> 1) ^ (x & 7)) + (k & 1)] = r[i];
            } else {
                dst[(tid / BX + i * (GEMM_THREADS / BX)) * BX + tid % BX] = r[i];
            }
        }
    }
};

// Fragments of one operand for a wave: F MFMA fragments of 16 rows.  KC:
// fragment f covers rows (2 f + w) 16 + [0, 16).  !KC: fragments 2 g and
// 2 g + 1 cover the even and odd rows of (2 g + w) 32 + [0, 32).
template <int F, int BX, bool KC>
struct TileFrags {
    d2_t v[GEMM_BK / 8][F];       // KC: [s][f] = k pair;  !KC: [s][2 g + h] = row pair at k parity h
    __device__ __forceinline__ void read(const double* src, int w, int fr, int fk, int s) {
#pragma unroll
        for (int f = 0; f < F; f++) {
            if (KC) {
                const int x = (2 * f + w) * 16 + fr;
                v[s][f] = *(const d2_t*)(src + x * GEMM_BK + 2 * ((4 * s + fk) ^ (fr & 7)));
            } else {
                const int k = 8 * s + 2 * fk + (f & 1);
                v[s][f] = *(const d2_t*)(src + k * BX + (f - (f & 1) + w) * 32 + 2 * fr);
            }
        }
    }
    __device__ __forceinline__ double get(int s, int h, int f) const {
        return KC ? v[s][f][h] : v[s][f - (f & 1) + h][f & 1];
    }
    // fragments that touch rows below `rem`
    static __device__ __forceinline__ int valid(int64_t rem, int w) {
        int n = 0;
#pragma unroll
        for (int f = 0; f < F; f++) n += (KC ? (2 * f + w) * 16 : (f - (f & 1) + w) * 32) < rem ? 1 : 0;
        return n;
    }
    // row of element i (0..15) of fragment f
    static __device__ __forceinline__ int row(int f, int w, int i) {
        return KC ? (2 * f + w) * 16 + i : (f - (f & 1) + w) * 32 + 2 * i + (f & 1);
    }
};

// One BM x BN output tile at (m0, n0): C = alpha op(A) op(B) + beta C over [0, K).
//
// Bound by the matrix cores: a 16-deep step of a 128 x 128 tile is 64 MFMAs
// of 64 cycles per wave against 8 load instructions and 16 LDS reads.  The
// order inside a step keeps everything else off that path: the barrier
// that ends the previous step, all fragment reads of this stage, then the
// loads of the next stage (after the reads: the compiler makes a read wait
// for every load into LDS queued before it), then the MFMAs.  The accumulators live
// in ordinary registers (220 to 244 of 256 at two waves per SIMD), so alpha and beta
// cost nothing at the store.  Measured on 8192^3: 71.5 to 72.7 TFLOP/s by
// transposes (0.91 to 0.925 of the FP64 matrix peak), against 59.7 with guarded
// 8-byte loads through registers and two barriers per step.
// Fragments wholly past M or N are skipped, and neighbouring fragments
// belong to different waves, so an edge tile costs about its valid 16 or 32 row
// groups on every SIMD rather than the whole tile.
template <int BM, int BN, bool TA, bool TB, bool DIRECT>
__device__ __forceinline__ void dgemm_tile(int64_t M, int64_t N, int64_t K, double alpha,
                                           const double* __restrict__ A, int64_t lda,
                                           const double* __restrict__ B, int64_t ldb,
                                           double* __restrict__ C, int64_t ldc, int64_t m0, int64_t n0,
                                           double beta = 0.0) {
    constexpr int FM = BM / 32, FN = BN / 32;  // MFMA fragments per wave and side
    __shared__ __align__(1024) double As[2][BM * GEMM_BK];
    __shared__ __align__(1024) double Bs[2][BN * GEMM_BK];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int fr = lane & 15;   // row / column inside a fragment
    const int fk = lane >> 4;   // k group of a fragment
    typedef TileFrags<FM, BM, !TA> FragA;
    typedef TileFrags<FN, BN, TB> FragB;
    TileOperand<BM, !TA, DIRECT> oa;
    TileOperand<BN, TB, DIRECT> ob;
    oa.init(A, lda, m0, M, lane, wave);
    ob.init(B, ldb, n0, N, lane, wave);
    const int fmv = FragA::valid(M - m0, wm), fnv = FragB::valid(N - n0, wn);

    d4_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};

    FragA fa;
    FragB fb;
    // FULL: every fragment of the wave is inside; k outermost, so the first
    // MFMAs wait for the first fragments only.  Else skip the outside ones.
    auto mults = [&](auto FULL, int s0, int s1) {
        if constexpr (FULL.value) {
#pragma unroll
            for (int s = s0; s < s1; s++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int i = 0; i < FM; i++)
#pragma unroll
                        for (int j = 0; j < FN; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa.get(s, h, i), fb.get(s, h, j),
                                                                             acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j += 2)
                    if (i < fmv && j < fnv) {
#pragma unroll
                        for (int s = s0; s < s1; s++)
#pragma unroll
                            for (int h = 0; h < 2; h++)
#pragma unroll
                                for (int e = 0; e < 2; e++)
                                    acc[i][j + e] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                        fa.get(s, h, i), fb.get(s, h, j + e), acc[i][j + e], 0, 0, 0);
                    }
        }
    };
    const int steps = (int)((K + GEMM_BK - 1) / GEMM_BK);
    const int klast = (int)(K - (int64_t)(steps - 1) * GEMM_BK);      // k of the last step, 1..16
    auto queue = [&](int buf, int t) {         // the loads of step t into stage buf
        const bool tail = t == steps - 1 && klast < GEMM_BK;
        if constexpr (DIRECT) {
            oa.stage(As[buf], tail, klast, wave);
            ob.stage(Bs[buf], tail, klast, wave);
        } else {
            oa.load((int64_t)t * GEMM_BK, tail ? klast : GEMM_BK, tid);
            ob.load((int64_t)t * GEMM_BK, tail ? klast : GEMM_BK, tid);
        }
    };
    auto land = [&](int buf) {                 // registers only: the queued values into LDS
        if constexpr (!DIRECT) {
            oa.store(As[buf], tid);
            ob.store(Bs[buf], tid);
        }
    };
    auto step = [&](auto FULL, int cur, int tnext) {
        // this wave's loads into LDS have landed (vmcnt 0: a barrier waits for
        // its waves, not for their loads); after the barrier every wave's have, and the
        // other stage is free
        if constexpr (DIRECT) __builtin_amdgcn_s_waitcnt(GEMM_WAIT_VMCNT0);
        __syncthreads();
        if constexpr (DIRECT) {
#pragma unroll
            for (int s = 0; s < GEMM_BK / 8; s++) {
                fa.read(As[cur], wm, fr, fk, s);
                fb.read(Bs[cur], wn, fr, fk, s);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (tnext < steps) queue(cur ^ 1, tnext);
            __builtin_amdgcn_sched_barrier(0);
            mults(FULL, 0, GEMM_BK / 8);
        } else {
            // the staging registers leave room for the fragments of 8 k only
            if (tnext < steps) queue(cur ^ 1, tnext);
#pragma unroll
            for (int s = 0; s < GEMM_BK / 8; s++) {
                __builtin_amdgcn_sched_barrier(0);
                fa.read(As[cur], wm, fr, fk, s);
                fb.read(Bs[cur], wn, fr, fk, s);
                mults(FULL, s, s + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (tnext < steps) land(cur ^ 1);
        }
    };
    if (steps > 0) {
        queue(0, 0);
        land(0);
    }
    // the same barriers in both loops: waves of one workgroup may take either
    auto loop = [&](auto FULL) {
        for (int t = 0; t < steps; t += 2) {
            step(FULL, 0, t + 1);
            if (t + 1 < steps) step(FULL, 1, t + 2);
        }
    };
    if (fmv == FM && fnv == FN) loop(std::integral_constant<bool, true>());
    else loop(std::integral_constant<bool, false>());

    // D[row][col] of a 16x16 fragment (v_mfma_f64_16x16x4f64, checked on
    // gfx950): col = lane % 16, row = lane / 16 + 4 * r for element r.
    // All C values of a fragment row are loaded before any is stored: loads
    // and stores through the one C pointer would otherwise stay in program order.
    const bool pair = !TB && (ldc & 1) == 0 && ((uintptr_t)C & 15) == 0;   // fragments j, j + 1 adjacent in C
#pragma unroll
    for (int i = 0; i < FM; i++) {
        if (i >= fmv) continue;
        d2_t cv[FN / 2][4];
        if (beta != 0.0) {
#pragma unroll
            for (int j = 0; j < FN; j += 2)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t gm = m0 + FragA::row(i, wm, fk + 4 * r);
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int64_t gn = n0 + FragB::row(j + e, wn, fr);
                        cv[j / 2][r][e] = (gm < M && gn < N) ? C[gm * ldc + gn] : 0.0;
                    }
                }
        }
#pragma unroll
        for (int j = 0; j < FN; j += 2)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t gm = m0 + FragA::row(i, wm, fk + 4 * r);
                const int64_t gn = n0 + FragB::row(j, wn, fr), gn1 = n0 + FragB::row(j + 1, wn, fr);
                d2_t v = {alpha * acc[i][j][r], alpha * acc[i][j + 1][r]};
                if (beta != 0.0) v += beta * cv[j / 2][r];
                if (gm < M) {
                    if (pair && gn1 < N) {
                        *(d2_t*)(C + gm * ldc + gn) = v;
                    } else {
                        if (gn < N) C[gm * ldc + gn] = v[0];
                        if (gn1 < N) C[gm * ldc + gn1] = v[1];
                    }
                }
            }
    }
}

// Whether both operands' tiles can be loaded in 16-byte chunks (DIRECT):
// base, leading dimension, batch stride and the extent along the contiguous
// index even.
static inline bool gemm_direct(int ta, int tb, int64_t M, int64_t N, int64_t K, const double* A, int64_t lda,
                               int64_t sA, const double* B, int64_t ldb, int64_t sB) {
    const int64_t ea = ta ? M : K, eb = tb ? K : N;
    return ((((uintptr_t)A | (uintptr_t)B) & 15) | ((lda | ldb | sA | sB | ea | eb) & 1)) == 0;
}

// Waves per SIMD the register budget of a tile allows (LDS allows as many).
#define GEMM_WAVES(BM, BN) ((BM) * (BN) >= 128 * 128 ? 2 : ((BM) * (BN) >= 128 * 64 ? 3 : 4))

template <int BM, int BN, bool TA, bool TB, bool DIRECT>
__global__ __launch_bounds__(GEMM_THREADS, GEMM_WAVES(BM, BN)) void k_dgemm(
    int64_t M, int64_t N, int64_t K, double alpha, const double* __restrict__ A, int64_t lda,
    int64_t sA, const double* __restrict__ B, int64_t ldb, int64_t sB, double beta,
    double* __restrict__ C, int64_t ldc, int64_t sC, int64_t tiles_m, int64_t tiles_n,
    int64_t kchunk, int64_t sSplit, int upper) {
    const int64_t batch = blockIdx.z;
    A += batch * sA;
    B += batch * sB;
    C += batch * sC + (int64_t)blockIdx.y * sSplit;
    // split K: this workgroup covers [kbeg, kbeg + K) of the full K range
    const int64_t kbeg = (int64_t)blockIdx.y * kchunk;
    K = (K - kbeg < kchunk) ? (K - kbeg) : kchunk;
    if (TA) A += kbeg * lda; else A += kbeg;
    if (TB) B += kbeg; else B += kbeg * ldb;
    const int64_t tile = xcd_remap(blockIdx.x, (int64_t)gridDim.x);
    // groups of 8 tile rows walk the tile columns together (L2 reuse of B)
    const int64_t GROUP = 8;
    const int64_t per_group = GROUP * tiles_n;
    const int64_t g = tile / per_group;
    const int64_t first_m = g * GROUP;
    const int64_t gsize = (tiles_m - first_m < GROUP) ? (tiles_m - first_m) : GROUP;
    const int64_t tm = first_m + (tile % per_group) % gsize;
    const int64_t tn = (tile % per_group) / gsize;
    if (upper && tm > tn) return;              // symmetric product: the upper tiles only
    const int64_t m0 = tm * BM, n0 = tn * BN;

    dgemm_tile<BM, BN, TA, TB, DIRECT>(M, N, K, alpha, A, lda, B, ldb, C, ldc, m0, n0, beta);
}

// Small products: 32 x 32 output tiles, the four waves of a workgroup taking
// every fourth 8-deep chunk of K and adding their tiles through LDS in wave order.
// What bounds these is latency, not rate: a 64 x 64 tile that stages each
// 16 of K behind a barrier takes 0.7 us a step with one workgroup per CU
// whatever the tile holds.  Here a wave loads its fragments straight from
// memory (L2) into registers, four chunks ahead of their use, waits for
// nobody until the end, and does a quarter of K.
template <bool TA, bool TB>
__global__ __launch_bounds__(GEMM_THREADS) void k_dgemm_small(
    int64_t M, int64_t N, int64_t K, double alpha, const double* __restrict__ A, int64_t lda, int64_t sA,
    const double* __restrict__ B, int64_t ldb, int64_t sB, double beta, double* __restrict__ C, int64_t ldc,
    int64_t sC, int tiles_n, int64_t kchunk, int64_t sSplit, int upper) {
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - tm * tiles_n;
    if (upper && tm > tn) return;
    const int64_t batch = blockIdx.z;
    A += batch * sA;
    B += batch * sB;
    C += batch * sC + (int64_t)blockIdx.y * sSplit;
    const int64_t kbeg = (int64_t)blockIdx.y * kchunk;
    K = (K - kbeg < kchunk) ? (K - kbeg) : kchunk;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fk = lane >> 4;
    const int64_t m0 = (int64_t)tm * 32, n0 = (int64_t)tn * 32;
    // element (row, k) of op(A) at pa[f] + k * ka; rows past the edge repeat the last one
    const int64_t ka = TA ? lda : 1, kb = TB ? 1 : ldb;
    const double* pa[2];
    const double* pb[2];
#pragma unroll
    for (int f = 0; f < 2; f++) {
        int64_t m = m0 + 16 * f + fr, n = n0 + 16 * f + fr;
        if (m > M - 1) m = M - 1;
        if (n > N - 1) n = N - 1;
        pa[f] = A + (TA ? m : m * lda) + (kbeg + 8 * wave + 2 * fk) * ka;
        pb[f] = B + (TB ? n * ldb : n) + (kbeg + 8 * wave + 2 * fk) * kb;
    }
    d4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
    constexpr int U = 4;                       // chunks in flight
    double a[U][2][2], b[U][2][2];
    auto load = [&](int u) {
#pragma unroll
        for (int f = 0; f < 2; f++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                a[u][f][h] = pa[f][h * ka];
                b[u][f][h] = pb[f][h * kb];
            }
            pa[f] += 32 * ka;
            pb[f] += 32 * kb;
        }
    };
    auto mult = [&](int u) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][i][h], b[u][j][h], acc[i][j], 0, 0, 0);
    };
    const int64_t whole = K / 8;               // whole chunks: this wave's are wave, wave + 4, ...
    int64_t left = whole > wave ? (whole - wave + 3) / 4 : 0;
    if (left >= U) {
#pragma unroll
        for (int u = 0; u < U; u++) load(u);
        left -= U;
        for (; left >= U; left -= U) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                mult(u);
                load(u);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) mult(u);
    }
#pragma unroll
    for (int u = 0; u < U - 1; u++)
        if (u < left) load(u);
#pragma unroll
    for (int u = 0; u < U - 1; u++)
        if (u < left) mult(u);
    if ((K & 7) && (whole & 3) == wave) {      // the last chunk's K % 8
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const bool in = 8 * whole + 2 * fk + h < K;
                const double* qa = in ? pa[f] + h * ka : xr_zero_page;
                const double* qb = in ? pb[f] + h * kb : xr_zero_page;
                a[0][f][h] = *qa;
                b[0][f][h] = *qb;
            }
        mult(0);
    }
    __shared__ double red[4][16][64];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave][(i * 2 + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();
    // wave w finishes fragment (i, j) = (w >> 1, w & 1)
    const int64_t gn = n0 + (wave & 1) * 16 + fr;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int64_t gm = m0 + (wave >> 1) * 16 + fk + 4 * r;
        const int e = wave * 4 + r;
        double v = alpha * ((red[0][e][lane] + red[1][e][lane]) + (red[2][e][lane] + red[3][e][lane]));
        if (gm < M && gn < N) {
            if (beta != 0.0) v += beta * C[gm * ldc + gn];
            C[gm * ldc + gn] = v;
        }
    }
}

// Grouped GEMM: up to XR_GROUP_PROBS independent products C_q = alpha
// op(A_q) op(B_q) of uneven shapes in one launch, so the launch fills the
// chip evenly where the problems alone would leave a partly empty last
// round of workgroups.  Workgroups are handed to the 8 XCDs round-robin
// (blockIdx % 8); every problem's tiles are split evenly over the XCDs, each
// XCD taking a contiguous run of them (L2 reuse inside the run), and each
// XCD works through the problems in order: per-tile work differs between
// problems (K), and this keeps the XCDs' loads equal.  The host orders the
// problems by decreasing K, so the longest tiles start first.
#define XR_GROUP_PROBS 32
struct GemmProb {
    const double* A;
    const double* B;
    double* C;
    int64_t M, N, K, lda, ldb, ldc, tiles_m, tiles_n;
    const int* off;      // null, or: *off == 0 restricts k to [k0, k1) (even; A and B not transposed)
    int64_t k0, k1;
};
struct GemmGroup {
    int n;
    int lower;           // square products whose strictly upper tiles are skipped
    double alpha, beta;
    GemmProb p[XR_GROUP_PROBS];
};

template <int BM, int BN, bool TA, bool TB, bool DIRECT>
__global__ __launch_bounds__(GEMM_THREADS, GEMM_WAVES(BM, BN)) void k_dgemm_grouped(GemmGroup g) {
    const int x = (int)(blockIdx.x & 7);
    int64_t j = blockIdx.x >> 3, local = -1;
    int q = 0;
    for (; q < g.n; q++) {                       // this XCD's share of each problem, in order
        const int64_t T = g.lower ? g.p[q].tiles_m * (g.p[q].tiles_m + 1) / 2 : g.p[q].tiles_m * g.p[q].tiles_n;
        const int64_t base = T >> 3, r = T & 7;
        const int64_t share = base + (x < r ? 1 : 0);
        if (j < share) {
            local = x * base + (x < r ? x : r) + j;
            break;
        }
        j -= share;
    }
    if (local < 0) return;                       // padding workgroup (uneven XCD shares)
    const GemmProb& P = g.p[q];
    int64_t tm, tn;
    if (g.lower) {                               // the lower-triangle tiles (tm >= tn) row by row
        tm = (int64_t)((sqrt(8.0 * (double)local + 1.0) - 1.0) * 0.5);
        while ((tm + 1) * (tm + 2) / 2 <= local) tm++;
        while (tm * (tm + 1) / 2 > local) tm--;
        tn = local - tm * (tm + 1) / 2;
    } else {
        const int64_t GROUP = 8;
        const int64_t per_group = GROUP * P.tiles_n;
        const int64_t gi = local / per_group;
        const int64_t first_m = gi * GROUP;
        const int64_t gsize = (P.tiles_m - first_m < GROUP) ? (P.tiles_m - first_m) : GROUP;
        tm = first_m + (local % per_group) % gsize;
        tn = (local % per_group) / gsize;
    }
    const double *A = P.A, *B = P.B;
    int64_t K = P.K;
    if (!TA && !TB && P.off && *P.off == 0) {
        A += P.k0;
        B += P.k0 * P.ldb;
        K = P.k1 - P.k0;
    }
    dgemm_tile<BM, BN, TA, TB, DIRECT>(P.M, P.N, K, g.alpha, A, P.lda, B, P.ldb, P.C, P.ldc, tm * BM, tn * BN,
                                       g.beta);
}

// C = alpha * sum_s P[s * step] + beta * C, summed in split order.
__global__ void k_splitk_reduce(const double* __restrict__ P, int64_t splits, int64_t batch,
                                int64_t M, int64_t N, double alpha, double beta,
                                double* __restrict__ C, int64_t ldc, int64_t sC, int64_t step = 1) {
    const int64_t n = batch * M * N;
    XR_GRID_STRIDE(i, n) {
        int64_t b = i / (M * N), r = i - b * M * N;
        int64_t m = r / N, col = r - m * N;
        double acc = 0.0;
        for (int64_t s = 0; s < splits; s += step) acc += P[s * n + i];
        double* cp = C + b * sC + m * ldc + col;
        double v = alpha * acc;
        if (beta != 0.0) v += beta * (*cp);
        *cp = v;
    }
}

// First stage of a reduction over many splits on a small output: each
// group of SPLIT_FOLD consecutive partials is summed (in order) into its
// first one, so the final pass reads every SPLIT_FOLD-th partial.
#define SPLIT_FOLD 32
__global__ void k_splitk_fold(double* __restrict__ P, int64_t splits, int64_t n) {
    const int64_t groups = (splits + SPLIT_FOLD - 1) / SPLIT_FOLD;
    XR_GRID_STRIDE(i, groups * n) {
        const int64_t g = i / n, e = i - g * n;
        const int64_t s0 = g * SPLIT_FOLD, s1 = s0 + SPLIT_FOLD < splits ? s0 + SPLIT_FOLD : splits;
        double acc = 0.0;
        for (int64_t s = s0; s < s1; s++) acc += P[s * n + e];
        P[s0 * n + e] = acc;
    }
}

// C = alpha * (sum of the split partials in Cw) + beta * C: outputs that
// leave most of the chip idle fold groups of partials first.
static int splitk_reduce(xr_ctx* c, double* Cw, int64_t splits, int64_t batch, int64_t M, int64_t N,
                         double alpha, double beta, double* C, int64_t ldc, int64_t sC) {
    const int64_t n = batch * M * N;
    int64_t step = 1;
    if (splits > 2 * SPLIT_FOLD && n < (1 << 18)) {
        k_splitk_fold<<<xr_grid(ceil_div(splits, SPLIT_FOLD) * n), 256, 0, c->stream>>>(Cw, splits, n);
        XR_LAUNCH_CHECK(c);
        step = SPLIT_FOLD;
    }
    k_splitk_reduce<<<xr_grid(n), 256, 0, c->stream>>>(Cw, splits, batch, M, N, alpha, beta, C, ldc, sC, step);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// Tall-skinny product for N <= 8 with A row-major (M x K, the Davidson
// H X): memory bound on A, so each wave streams 4 rows of A once, reusing
// every loaded row of B for all 4, and reduces across lanes at the end.
template <int NB, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_skinny(int64_t M, int64_t N, int64_t K, double alpha,
                                                      const double* __restrict__ A, int64_t lda,
                                                      const double* __restrict__ B, int64_t ldb,
                                                      double beta, double* __restrict__ C,
                                                      int64_t ldc) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t r0 = wave * 4; r0 < M; r0 += nwaves * 4) {
        double acc[4][NB];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[r][j] = 0.0;
        const int nr = (M - r0 < 4) ? (int)(M - r0) : 4;
        for (int64_t k = lane; k < K; k += 64) {
            double b[NB];
#pragma unroll
            for (int j = 0; j < NB; j++) b[j] = (j < N) ? (TB ? B[j * ldb + k] : B[k * ldb + j]) : 0.0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                double a = (r < nr) ? A[(r0 + r) * lda + k] : 0.0;
#pragma unroll
                for (int j = 0; j < NB; j++) acc[r][j] = fma(a, b[j], acc[r][j]);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < NB; j++) {
                double v = acc[r][j];
                for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
                acc[r][j] = v;
            }
        if (lane == 0) {
            for (int r = 0; r < nr; r++)
                for (int j = 0; j < N; j++) {
                    double* cp = C + (r0 + r) * ldc + j;
                    double v = alpha * acc[r][j];
                    if (beta != 0.0) v += beta * (*cp);
                    *cp = v;
                }
        }
    }
}

// C = alpha A^T B + beta C for A (K x M) and B (K x N) row-major with K
// large and M <= 64, N <= 8 (Gram products of a tall block of vectors).
// Each block sums a contiguous run of rows (lane = column of A, the 4 waves
// take every 4th row) into a partial (64 x NB) tile; a second kernel adds
// the partials in block order (deterministic).
template <int NB>
__global__ __launch_bounds__(256) void k_dgemm_tn_skinny(int64_t M, int64_t N, int64_t K,
                                                         const double* __restrict__ A, int64_t lda,
                                                         const double* __restrict__ B, int64_t ldb,
                                                         int64_t rows, double* __restrict__ part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t k0 = (int64_t)blockIdx.x * rows;
    const int64_t k1 = (K - k0 < rows) ? K : k0 + rows;
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = 0.0;
#pragma unroll 4
    for (int64_t k = k0 + wave; k < k1; k += 4) {
        const double a = (lane < M) ? A[k * lda + lane] : 0.0;
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = fma(a, (j < N) ? B[k * ldb + j] : 0.0, acc[j]);
    }
    __shared__ double red[4][64][NB];
#pragma unroll
    for (int j = 0; j < NB; j++) red[wave][lane][j] = acc[j];
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            part[((int64_t)blockIdx.x * 64 + lane) * NB + j] =
                red[0][lane][j] + red[1][lane][j] + red[2][lane][j] + red[3][lane][j];
    }
}

// C[i, j] = alpha * sum_b part[b][i][j] + beta C: one workgroup per output
// entry, the threads stride over the partial tiles and a fixed butterfly
// adds their sums (same order on every run).
__global__ __launch_bounds__(256) void k_tn_reduce(const double* __restrict__ part, int64_t nblk, int64_t M,
                                                   int64_t N, int nb, double alpha, double beta,
                                                   double* __restrict__ C, int64_t ldc) {
    const int64_t t = blockIdx.x;
    const int64_t i = t / N, j = t - (t / N) * N;
    double s = 0.0;
    for (int64_t b = threadIdx.x; b < nblk; b += 256) s += part[(b * 64 + i) * nb + j];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = alpha * ((red[0] + red[1]) + (red[2] + red[3]));
        if (beta != 0.0) v += beta * C[i * ldc + j];
        C[i * ldc + j] = v;
    }
}

// Gram products with M <= 8 columns: the rows are spread over all 256
// threads (coalesced reads of A and B), each thread keeps the M x NB sums,
// and the block adds them through LDS into the same partial layout as above.
template <int MB, int NB>
__global__ __launch_bounds__(256) void k_dgemm_tn_small(int64_t M, int64_t N, int64_t K,
                                                        const double* __restrict__ A, int64_t lda,
                                                        const double* __restrict__ B, int64_t ldb,
                                                        int64_t rows, double* __restrict__ part) {
    const int64_t k0 = (int64_t)blockIdx.x * rows;
    const int64_t k1 = (K - k0 < rows) ? K : k0 + rows;
    double acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = 0.0;
#pragma unroll 4
    for (int64_t k = k0 + threadIdx.x; k < k1; k += 256) {
        double a[MB], b[NB];
#pragma unroll
        for (int i = 0; i < MB; i++) a[i] = (i < M) ? A[k * lda + i] : 0.0;
#pragma unroll
        for (int j = 0; j < NB; j++) b[j] = (j < N) ? B[k * ldb + j] : 0.0;
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[i][j] = fma(a[i], b[j], acc[i][j]);
    }
    __shared__ double red[256];
    for (int i = 0; i < MB; i++)
        for (int j = 0; j < NB; j++) {
            double v = acc[i][j];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
            __syncthreads();
            if (threadIdx.x == 0)
                part[((int64_t)blockIdx.x * 64 + i) * NB + j] = red[0] + red[1] + red[2] + red[3];
            __syncthreads();
        }
}

// C = alpha A op(B) + beta C for tall A (M x K row-major, row stride lda)
// with K <= 64 and N <= 8.  A block stages 64 rows of A through LDS with
// coalesced loads (the rows' K values are contiguous), then 4 threads per
// row sum interleaved k and combine with two shuffles.
template <int NB, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_rows_lds(int64_t M, int64_t N, int64_t K, double alpha,
                                                        const double* __restrict__ A, int64_t lda,
                                                        const double* __restrict__ B, int64_t ldb,
                                                        double beta, double* __restrict__ C, int64_t ldc) {
    __shared__ double tile[64 * 64];
    __shared__ double bs[64 * NB];
    const int tid = threadIdx.x;
    const int Ki = (int)K;
    for (int e = tid; e < Ki * NB; e += 256) {
        const int k = e / NB, j = e - (e / NB) * NB;
        bs[e] = (j < N) ? (TB ? B[(int64_t)j * ldb + k] : B[(int64_t)k * ldb + j]) : 0.0;
    }
    const int row = tid >> 2, part = tid & 3;
    for (int64_t r0 = (int64_t)blockIdx.x * 64; r0 < M; r0 += (int64_t)gridDim.x * 64) {
        const int nrows = (M - r0 < 64) ? (int)(M - r0) : 64;
        __syncthreads();
        for (int e = tid; e < nrows * Ki; e += 256) {
            const int r = e / Ki, k = e - (e / Ki) * Ki;
            tile[e] = A[(r0 + r) * lda + k];
        }
        __syncthreads();
        double acc[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = 0.0;
        if (row < nrows) {
            for (int k = part; k < Ki; k += 4) {
                const double a = tile[row * Ki + k];
#pragma unroll
                for (int j = 0; j < NB; j++) acc[j] = fma(a, bs[k * NB + j], acc[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            acc[j] += __shfl_xor(acc[j], 1, 64);
            acc[j] += __shfl_xor(acc[j], 2, 64);
        }
        if (part == 0 && row < nrows) {
#pragma unroll
            for (int j = 0; j < NB; j++) {
                if (j < N) {
                    double v = alpha * acc[j];
                    if (beta != 0.0) v += beta * C[(r0 + row) * ldc + j];
                    C[(r0 + row) * ldc + j] = v;
                }
            }
        }
    }
}

// C = alpha A op(B) + beta C for tall A (M x K row-major) with K <= 4 and
// N <= 8: one thread per output row (the K values of consecutive rows are
// adjacent, so a wave reads one contiguous run).
template <int NB, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_rows_small(int64_t M, int64_t N, int64_t K, double alpha,
                                                          const double* __restrict__ A, int64_t lda,
                                                          const double* __restrict__ B, int64_t ldb,
                                                          double beta, double* __restrict__ C, int64_t ldc) {
    double bs[4][NB];
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            bs[k][j] = (k < K && j < N) ? (TB ? B[(int64_t)j * ldb + k] : B[(int64_t)k * ldb + j]) : 0.0;
    XR_GRID_STRIDE(r, M) {
        double acc[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = 0.0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k < K) {
                const double a = A[r * lda + k];
#pragma unroll
                for (int j = 0; j < NB; j++) acc[j] = fma(a, bs[k][j], acc[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (j < N) {
                double v = alpha * acc[j];
                if (beta != 0.0) v += beta * C[r * ldc + j];
                C[r * ldc + j] = v;
            }
        }
    }
}

// C = alpha A^T op(B) + beta C for A stored K x M (row-major, lda) with
// K <= 64 and M large, N <= 8: the product of a block of vectors stored one
// per row with a small coefficient matrix.  One thread per output row reads
// column r of A, so consecutive threads read consecutive addresses.
template <int NB, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_tn_tall(int64_t M, int64_t N, int64_t K, double alpha,
                                                       const double* __restrict__ A, int64_t lda,
                                                       const double* __restrict__ B, int64_t ldb,
                                                       double beta, double* __restrict__ C, int64_t ldc) {
    __shared__ double bs[64 * NB];
    for (int e = threadIdx.x; e < (int)K * NB; e += 256) {
        const int k = e / NB, j = e - (e / NB) * NB;
        bs[e] = (j < N) ? (TB ? B[(int64_t)j * ldb + k] : B[(int64_t)k * ldb + j]) : 0.0;
    }
    __syncthreads();
    XR_GRID_STRIDE(r, M) {
        double acc[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) acc[j] = 0.0;
        for (int k = 0; k < (int)K; k++) {
            const double a = A[(int64_t)k * lda + r];
#pragma unroll
            for (int j = 0; j < NB; j++) acc[j] = fma(a, bs[k * NB + j], acc[j]);
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (j < N) {
                double v = alpha * acc[j];
                if (beta != 0.0) v += beta * C[r * ldc + j];
                C[r * ldc + j] = v;
            }
        }
    }
}

// C = alpha A B + beta C for A (M x K row-major) with M <= 64 / NB, N <= NB
// and K large (Gram products of vectors stored one per row).  Each block
// sums a contiguous run of k; wave w owns rows [w RB, w RB + RB) and its
// lanes read consecutive k of those rows (few accumulators per thread, so
// many waves stay resident to keep loads in flight).  The per-block sums go
// to a partial tile; k_tn_reduce adds the partials in block order.
template <int RB, int NB>
__global__ __launch_bounds__(256) void k_dgemm_nn_gram(int64_t M, int64_t N, int64_t K,
                                                       const double* __restrict__ A, int64_t lda,
                                                       const double* __restrict__ B, int64_t ldb,
                                                       int64_t rows, double* __restrict__ part) {
    const int lane = threadIdx.x & 63;
    const int i0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * RB;
    const int64_t k0 = (int64_t)blockIdx.x * rows;
    const int64_t k1 = (K - k0 < rows) ? K : k0 + rows;
    double acc[RB][NB];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[r][j] = 0.0;
#pragma unroll 2
    for (int64_t k = k0 + lane; k < k1; k += 64) {
        double b[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) b[j] = (j < N) ? B[k * ldb + j] : 0.0;
#pragma unroll
        for (int r = 0; r < RB; r++) {
            if (i0 + r < M) {
                const double a = A[(int64_t)(i0 + r) * lda + k];
#pragma unroll
                for (int j = 0; j < NB; j++) acc[r][j] = fma(a, b[j], acc[r][j]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            double v = acc[r][j];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            if (lane == 0 && i0 + r < M) part[((int64_t)blockIdx.x * 64 + i0 + r) * NB + j] = v;
        }
}

static int launch_tn_skinny(xr_ctx* c, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
                            int64_t lda, const double* B, int64_t ldb, double beta, double* C,
                            int64_t ldc) {
    const int nb = N <= 1 ? 1 : (N <= 2 ? 2 : (N <= 4 ? 4 : 8));
    int64_t nblk = ceil_div(K, 2048);
    if (nblk > 1024) nblk = 1024;
    const int64_t rows = ceil_div(K, nblk);
    nblk = ceil_div(K, rows);
    double* part = (double*)xr_workspace(c, 52, nblk * 64 * nb * sizeof(double));
    if (!part) return xr_fail(c, XR_ENOMEM, "workspace (Gram)");
    ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
    prof.shape(M, N, K, 1, 1, 0);
#define XR_TN_SMALL(MB_)                                                                                  \
    if (nb == 1) k_dgemm_tn_small<MB_, 1><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part); \
    else if (nb == 2) k_dgemm_tn_small<MB_, 2><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part); \
    else if (nb == 4) k_dgemm_tn_small<MB_, 4><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part); \
    else k_dgemm_tn_small<MB_, 8><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part)
    if (M <= 1) { XR_TN_SMALL(1); }
    else if (M <= 2) { XR_TN_SMALL(2); }
    else if (M <= 4) { XR_TN_SMALL(4); }
    else if (M <= 8) { XR_TN_SMALL(8); }
    else if (nb == 1) k_dgemm_tn_skinny<1><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part);
    else if (nb == 2) k_dgemm_tn_skinny<2><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part);
    else if (nb == 4) k_dgemm_tn_skinny<4><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part);
    else k_dgemm_tn_skinny<8><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part);
#undef XR_TN_SMALL
    XR_LAUNCH_CHECK(c);
    k_tn_reduce<<<(unsigned)(M * N), 256, 0, c->stream>>>(part, nblk, M, N, nb, alpha, beta, C, ldc);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// Workgroups of 256 threads of `kernel` resident on the device at once (CUs
// x occupancy): a grid of that size runs in one round.
static int64_t resident_blocks(const void* kernel) {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 256, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 1024;
    }
    return (int64_t)(cus > 0 ? cus : 256) * (per > 0 ? per : 1);
}

// Runs the Gram kernel with RB x NB accumulators per thread: one contiguous
// run of k per workgroup, as many workgroups as are resident at once (no
// partly filled second round); the partial tiles go to the workspace.
template <int RB, int NB>
static int nn_gram_go(xr_ctx* c, int64_t M, int64_t N, int64_t K, const double* A, int64_t lda,
                      const double* B, int64_t ldb, int64_t* nblk_out, double** part_out) {
    static const int64_t res = resident_blocks(reinterpret_cast<const void*>(&k_dgemm_nn_gram<RB, NB>));
    int64_t nblk = ceil_div(K, 2048);
    if (nblk > res) nblk = res;
    const int64_t rows = ceil_div(K, nblk);
    nblk = ceil_div(K, rows);
    double* part = (double*)xr_workspace(c, 52, nblk * 64 * NB * sizeof(double));
    if (!part) return xr_fail(c, XR_ENOMEM, "workspace (Gram)");
    k_dgemm_nn_gram<RB, NB><<<(unsigned)nblk, 256, 0, c->stream>>>(M, N, K, A, lda, B, ldb, rows, part);
    *nblk_out = nblk;
    *part_out = part;
    return XR_OK;
}

static int launch_nn_gram(xr_ctx* c, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
                          int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc) {
    const int nb = N <= 1 ? 1 : (N <= 2 ? 2 : (N <= 4 ? 4 : 8));
    const int64_t q = ceil_div(M, 4);             // rows per wave
    const int rb = q <= 1 ? 1 : (q <= 2 ? 2 : (q <= 4 ? 4 : (q <= 8 ? 8 : 16)));
    ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
    prof.shape(M, N, K, 1, 0, 0);
    int64_t nblk = 0;
    double* part = nullptr;
    int rc;
#define XR_GRAM_GO(RB_, NB_) rc = nn_gram_go<RB_, NB_>(c, M, N, K, A, lda, B, ldb, &nblk, &part)
    if (nb == 1) {
        if (rb == 1) XR_GRAM_GO(1, 1);
        else if (rb == 2) XR_GRAM_GO(2, 1);
        else if (rb == 4) XR_GRAM_GO(4, 1);
        else if (rb == 8) XR_GRAM_GO(8, 1);
        else XR_GRAM_GO(16, 1);
    } else if (nb == 2) {
        if (rb == 1) XR_GRAM_GO(1, 2);
        else if (rb == 2) XR_GRAM_GO(2, 2);
        else if (rb == 4) XR_GRAM_GO(4, 2);
        else XR_GRAM_GO(8, 2);
    } else if (nb == 4) {
        if (rb == 1) XR_GRAM_GO(1, 4);
        else if (rb == 2) XR_GRAM_GO(2, 4);
        else XR_GRAM_GO(4, 4);
    } else {
        if (rb == 1) XR_GRAM_GO(1, 8);
        else XR_GRAM_GO(2, 8);
    }
#undef XR_GRAM_GO
    if (rc) return rc;
    XR_LAUNCH_CHECK(c);
    k_tn_reduce<<<(unsigned)(M * N), 256, 0, c->stream>>>(part, nblk, M, N, nb, alpha, beta, C, ldc);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// ---------------------------------------------------------------------------
// Choice of tile shape and K split
// ---------------------------------------------------------------------------
// Tile 0: 128 x 128, 1: 128 x 64, 2: 64 x 128, 3: 64 x 64, 4: 32 x 32 (k_dgemm_small).
struct GemmTile { int bm, bn, resident; double eff, alone; };
// resident: workgroups the model takes a CU to hold; eff: share of the FP64
// matrix peak with the CU full; alone: us one 16-deep step takes over its
// MFMAs when a workgroup has the CU to itself (load latency and the barrier).  Set from
// products of 64 x 324 x 64 to 8192^3; measured at rest on 8192 x 8192 x 4096: 72.2, 71.5, 71.7 and 71.3
// TFLOP/s for tiles 0 to 3 (0.91 to 0.92 of the peak, so eff is a little low for all alike), and
// 137, 75, 76 and 45 us for 64, 128, 128 and 256 workgroups of 1024^3.  By their registers the 64 x 64
// kernels of unaligned rows with B transposed hold four workgroups, and the 32 x 32
// one two, unless B alone is transposed: past that many the wait is modelled too short.
static const GemmTile GEMM_TILES[5] = {
    {128, 128, 2, 0.90, 0.50}, {128, 64, 3, 0.89, 0.40}, {64, 128, 3, 0.89, 0.40}, {64, 64, 5, 0.87, 0.26}, {32, 32, 4, 0.60, 0.10}};
#define GEMM_STAGING_MAX ((int64_t)64 << 20)   // bytes of split-K partial tiles

static int device_cus() {
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();
            return 256;
        }
        return cus > 0 ? cus : 256;
    }();
    return n;
}

// Modelled time (us) of a product with the given tile and K split.  The
// busiest CU takes n = ceil(workgroups / CUs) of them: either its matrix
// cores are busy throughout (padding past the 16-row and 32-column fragments is
// skipped), or it waits out the steps of one workgroup after another.  A
// split adds the reduction's launch and its traffic.
static double gemm_cost(const GemmTile& t, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t s, bool upper,
                        int cus) {
    const int64_t tm = ceil_div(M, t.bm), tn = ceil_div(N, t.bn);
    const int64_t tiles = upper ? tm * (tm + 1) / 2 : tm * tn;
    const int64_t units = tiles * batch * s;
    const double n = std::ceil((double)units / cus);
    const double fill = (double)(ceil_div(M, 16) * 16) * (double)(ceil_div(N, 32) * 32) /
                        ((double)(tm * t.bm) * (double)(tn * t.bn));
    const double steps = std::ceil((double)K / (double)s / GEMM_BK);
    const double step = t.bm * t.bn * (2.0 * GEMM_BK) / 128.0 / 2400.0;    // us of MFMA per step at full rate
    const double busy = n * steps * step * std::min(1.0, fill) / t.eff;
    const double wait = std::ceil(n / t.resident) * steps * (step + t.alone);
    double us = 3.0 + std::max(busy, wait);
    if (s > 1) us += 4.0 + (double)(s + 1) * 8.0 * M * N * batch / 4.0e6;
    return us;
}

// The tile and K split of least modelled time.  Each split keeps at least 64
// of K, and the partial tiles stay within `room` and the staging array of the
// no-allocation entry point, so both entry points choose alike.
static void gemm_choose(int64_t M, int64_t N, int64_t K, int64_t batch, bool direct, bool upper, size_t room,
                        int* tile, int64_t* splits) {
    static const int S[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512};
    const int cus = device_cus();
    const int64_t most = (int64_t)std::min<size_t>(room, GEMM_STAGING_MAX);
    double best = 1e300;
    *tile = 3;
    *splits = 1;
    for (int t = 0; t < 5; t++) {
        if (!direct && t < 3) continue;                 // unaligned rows: 64 x 64 and 32 x 32 only
        if (upper && GEMM_TILES[t].bm != GEMM_TILES[t].bn) continue;
        for (const int s : S) {
            if (s > 1 && (K / s < 64 || 8 * s * M * N * batch > most)) break;
            const double c = gemm_cost(GEMM_TILES[t], M, N, K, batch, s, upper, cus);
            if (c < best) { best = c; *tile = t; *splits = s; }
        }
    }
}

// Bytes of staging a product counts as needing when memory is capped: the
// rule by which xr_gemm_f64_noalloc, a pinned context and one with a memory
// limit refuse a call.  It is stated in the sizes (K splits toward full rounds of
// workgroups, and a staged beta over a large output) and not in how the product
// runs, so a faster split or an epilogue that needs no staging does not
// change what a caller can rely on.
static int64_t gemm_refusal_bytes(int64_t M, int64_t N, int64_t K, bool beta, int64_t batch, bool upper) {
    const int64_t cus = device_cus();
    auto choice = [&](int64_t units, int64_t slots, int64_t* splits, int64_t kmin) {
        auto score = [&](int64_t s) {
            const double rounds = std::ceil((double)(units * s) / (double)slots);
            const double ideal = (double)units * (double)K / (double)slots;
            const double t = rounds * ((double)K / (double)s + 32.0);
            return ideal / t / (1.0 + (s > 1 ? (double)(s + 1) * 46.0 / (double)K : 0.0));
        };
        double best = score(1);
        *splits = 1;
        if (K < 512 || units >= 4 * slots) return best;
        const int64_t smax = std::min<int64_t>(std::min<int64_t>(512, std::max<int64_t>(64, 2 * slots / units)), K / kmin);
        for (int64_t s = 2; s <= smax; s++) {
            const double e = score(s);
            if (e > best) { best = e; *splits = s; }
        }
        return best;
    };
    int64_t bm = 64, bn = 64, per = 4, s = 1;
    const int64_t big = ceil_div(M, 128) * ceil_div(N, 128) * batch;
    if (upper) { bm = bn = 128; per = 2; }
    else if (beta && K <= 64) { bm = bn = 64; }
    else if (big >= 512 || (M > 64 && N > 64 && choice(big, 2 * cus, &s, 256) >= 0.8)) { bm = bn = 128; per = 2; }
    else if (big >= 64 && N <= 64 && M > 64) { bm = 128; per = 3; }
    else if (big >= 64 && M <= 64 && N > 64) { bn = 128; per = 3; }
    const int64_t tm = ceil_div(M, bm), tn = ceil_div(N, bn), units = tm * tn * batch;
    choice(units, per * cus, &s, (tm == 1 || tn == 1) ? 64 : 256);
    if (s > 1) s = ceil_div(K, ceil_div(ceil_div(K, s), GEMM_BK) * GEMM_BK);
    const bool staged = s > 1 || (beta && !(2 * units <= per * cus || K <= 256));
    return staged ? 8 * s * batch * M * N : 0;
}

// One product with an explicit tile and K split (0: unsplit).
static int launch_cfg(xr_ctx* c, int tile, int64_t splits, int ta, int tb, int64_t M, int64_t N, int64_t K,
                      double alpha, const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb,
                      int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int64_t batch,
                      bool upper = false) {
    const bool direct = gemm_direct(ta, tb, M, N, K, A, lda, sA, B, ldb, sB);
    if (!direct && tile < 3) tile = 3;
    int64_t kchunk = K;
    double* Cw = C;
    if (splits > 1) {
        const int64_t unit = tile == 4 ? 32 : GEMM_BK;
        kchunk = ceil_div(ceil_div(K, splits), unit) * unit;
        splits = ceil_div(K, kchunk);
    }
    if (splits < 1) splits = 1;
    if (splits > 1) {
        const int64_t need = splits * batch * M * N * (int64_t)sizeof(double);
        Cw = (double*)xr_workspace(c, 50, need);
        if (!Cw) return xr_fail(c, XR_ENOMEM, "workspace (split-K)");
    }
    const GemmTile& T = GEMM_TILES[tile];
    const int64_t tm = ceil_div(M, T.bm), tn = ceil_div(N, T.bn), tiles = tm * tn;
    if (tiles > 0x7fffffff || batch > 65535) return xr_fail(c, XR_EUNSUPPORTED, "GEMM grid too large");
    const bool staged = splits > 1;
    const int64_t ldw = staged ? N : ldc, sCw = staged ? M * N : sC, sSplit = staged ? batch * M * N : 0;
    const double aw = staged ? 1.0 : alpha, bw = staged ? 0.0 : beta;
    dim3 grid((unsigned)tiles, (unsigned)splits, (unsigned)batch);
    {
        ProfScope prof(c, XR_K_GEMM_F64, 2.0 * M * N * K * batch, 8.0 * (M * K + K * N + M * N) * batch);
        prof.shape(M, N, K, batch, ta, tb);
#define XR_GEMM_ARGS M, N, K, aw, A, lda, sA, B, ldb, sB, bw, Cw, ldw, sCw
#define XR_GEMM_LAUNCH(BM_, BN_, TA_, TB_, D_)                                                             \
    k_dgemm<BM_, BN_, TA_, TB_, D_><<<grid, GEMM_THREADS, 0, c->stream>>>(XR_GEMM_ARGS, tm, tn, kchunk, sSplit, \
                                                                          upper ? 1 : 0)
#define XR_GEMM_TRANS(BM_, BN_, D_)                           \
    if (ta && tb) XR_GEMM_LAUNCH(BM_, BN_, true, true, D_);   \
    else if (ta) XR_GEMM_LAUNCH(BM_, BN_, true, false, D_);   \
    else if (tb) XR_GEMM_LAUNCH(BM_, BN_, false, true, D_);   \
    else XR_GEMM_LAUNCH(BM_, BN_, false, false, D_)
#define XR_GEMM_SMALL(TA_, TB_)                                                                            \
    k_dgemm_small<TA_, TB_><<<grid, GEMM_THREADS, 0, c->stream>>>(XR_GEMM_ARGS, (int)tn, kchunk, sSplit, upper ? 1 : 0)
        if (tile == 4) {
            if (ta && tb) XR_GEMM_SMALL(true, true);
            else if (ta) XR_GEMM_SMALL(true, false);
            else if (tb) XR_GEMM_SMALL(false, true);
            else XR_GEMM_SMALL(false, false);
        } else if (!direct) { XR_GEMM_TRANS(64, 64, false); }
        else if (tile == 0) { XR_GEMM_TRANS(128, 128, true); }
        else if (tile == 1) { XR_GEMM_TRANS(128, 64, true); }
        else if (tile == 2) { XR_GEMM_TRANS(64, 128, true); }
        else { XR_GEMM_TRANS(64, 64, true); }
#undef XR_GEMM_SMALL
#undef XR_GEMM_TRANS
#undef XR_GEMM_LAUNCH
#undef XR_GEMM_ARGS
        XR_LAUNCH_CHECK(c);
    }
    if (staged) {
        ProfScope prof(c, XR_K_OTHER, 0.0, 8.0 * (splits + 2) * batch * M * N);
        return splitk_reduce(c, Cw, splits, batch, M, N, alpha, beta, C, ldc, sC);
    }
    return XR_OK;
}

// Refuses a product whose staging (gemm_refusal_bytes, or a tuned split's) is
// more than the context may hold.  An admitted one leaves that much behind in the
// workspace slot, up to the most any split needs: a later product admitted because a larger
// one ran before the pin then finds room for its own partial tiles.
static int gemm_admit(xr_ctx* c, int64_t bytes) {
    if (bytes == 0 || (!c->noalloc && bytes <= c->gemm_staging)) return XR_OK;
    if ((size_t)bytes > xr_workspace_room(c, 50)) {
        c->noalloc_blocked = c->noalloc;
        c->pin_blocked = !c->noalloc && c->pins > 0;
        return xr_fail(c, XR_ENOMEM, "workspace (split-K)");
    }
    if (!c->noalloc && xr_workspace(c, 50, std::min(bytes, GEMM_STAGING_MAX))) c->gemm_staging = bytes;
    return XR_OK;
}

// One product with the configuration chosen for its sizes, kept in a small
// direct-mapped table of the context (a pure function of the sizes: an entry
// never goes stale; at most 1024 of them).  Where a cap leaves less room than its
// partial tiles take, the best of the splits that fit runs instead.
static int launch_chosen(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
                         int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB, double beta, double* C,
                         int64_t ldc, int64_t sC, int64_t batch, bool upper = false) {
    const bool direct = gemm_direct(ta, tb, M, N, K, A, lda, sA, B, ldb, sB);
    const std::array<int64_t, 5> key{M, N, K, batch, (direct ? 1 : 0) | (upper ? 2 : 0) | (beta != 0.0 ? 4 : 0)};
    uint64_t h = 0;
    for (int64_t v : key) h = (h ^ (uint64_t)v) * 0x9E3779B97F4A7C15ull;
    if (c->gemm_choice.empty()) c->gemm_choice.resize(1024);
    auto& e = c->gemm_choice[h >> 54];
    if (e.key != key) {
        gemm_choose(M, N, K, batch, direct, upper, SIZE_MAX, &e.tile, &e.splits);
        e.staging = gemm_refusal_bytes(M, N, K, beta != 0.0, batch, upper);
        e.key = key;
    }
    const int rc = gemm_admit(c, e.staging);
    if (rc) return rc;
    int tile = e.tile;
    int64_t splits = e.splits;
    const size_t room = splits > 1 ? xr_workspace_room(c, 50) : SIZE_MAX;
    if ((size_t)(8 * splits * M * N * batch) > room)
        gemm_choose(M, N, K, batch, direct, upper, room, &tile, &splits);
    return launch_cfg(c, tile, splits, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch,
                      upper);
}

// C[i][j] = C[j][i] for i > j: the lower triangle from the upper one (32 x 32
// tiles through LDS; a workgroup writes one lower tile and reads its mirror,
// which no workgroup writes).
__global__ __launch_bounds__(256) void k_mirror_upper(double* __restrict__ C, int64_t n, int64_t ldc) {
    const int64_t a = blockIdx.y, b = blockIdx.x;     // target tile rows a, columns b
    if (a < b) return;
    __shared__ double T[32][33];
    const int tx = threadIdx.x, ty = threadIdx.y;
    for (int j = ty; j < 32; j += 8) {                // T[j][tx] = C[b*32 + j][a*32 + tx]
        const int64_t r = b * 32 + j, col = a * 32 + tx;
        if (r < n && col < n) T[j][tx] = C[r * ldc + col];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {                // C[a*32 + j][b*32 + tx] = C[b*32 + tx][a*32 + j]
        const int64_t r = a * 32 + j, col = b * 32 + tx;
        if (r < n && col < n && r > col) C[r * ldc + col] = T[tx][j];
    }
}

// C = alpha A^T A for A (K x n, leading dimension lda): the tile GEMM on the
// upper tiles only, then the lower triangle mirrored.
int xr_dgemm_syrk_tn(xr_ctx* c, int64_t n, int64_t K, double alpha, const double* A, int64_t lda, double* C,
                     int64_t ldc) {
    if (n <= 0) return XR_OK;
    int rc = launch_chosen(c, 1, 0, n, n, K, alpha, A, lda, 0, A, lda, 0, 0.0, C, ldc, 0, 1, true);
    if (rc) return rc;
    const int64_t t = ceil_div(n, 32);
    if (t > 65535) return xr_fail(c, XR_EUNSUPPORTED, "matrix too large for the mirror grid");
    ProfScope prof(c, XR_K_OTHER, 0.0, 8.0 * n * n);
    k_mirror_upper<<<dim3((unsigned)t, (unsigned)t), dim3(32, 8), 0, c->stream>>>(C, n, ldc);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// C = alpha A A^T for A (n x K, leading dimension lda): the same upper-tile
// product and mirror.
int xr_dgemm_syrk_nt(xr_ctx* c, int64_t n, int64_t K, double alpha, const double* A, int64_t lda, double* C,
                     int64_t ldc) {
    if (n <= 0) return XR_OK;
    int rc = launch_chosen(c, 0, 1, n, n, K, alpha, A, lda, 0, A, lda, 0, 0.0, C, ldc, 0, 1, true);
    if (rc) return rc;
    const int64_t t = ceil_div(n, 32);
    if (t > 65535) return xr_fail(c, XR_EUNSUPPORTED, "matrix too large for the mirror grid");
    ProfScope prof(c, XR_K_OTHER, 0.0, 8.0 * n * n);
    k_mirror_upper<<<dim3((unsigned)t, (unsigned)t), dim3(32, 8), 0, c->stream>>>(C, n, ldc);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

extern "C" int xr_gemm_syrk(xr_ctx* c, int trans, int64_t n, int64_t K, double alpha, const double* A, int64_t lda,
                            double* C, int64_t ldc) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (n < 0 || K < 0) return xr_fail(c, XR_EINVAL, "negative size");
    if (ldc < n) return xr_fail(c, XR_ESHAPE, "ldc < n");
    if ((trans ? lda < n : lda < K) && n > 0 && K > 0) return xr_fail(c, XR_ESHAPE, "lda too small");
    if (n == 0) return XR_OK;
    return trans ? xr_dgemm_syrk_tn(c, n, K, alpha, A, lda, C, ldc) : xr_dgemm_syrk_nt(c, n, K, alpha, A, lda, C, ldc);
}

// Shapes xr_dgemm_launch gives to the bandwidth kernels.
static bool gemm_skinny(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t batch) {
    if (batch != 1 || N > 8) return false;
    return (!ta && M >= 1024) || (ta && !tb && M <= 64 && K >= 4096) || (ta && M >= 1024 && K <= 64) ||
           (!ta && !tb && K >= 4096 && M * (N <= 1 ? 1 : (N <= 2 ? 2 : (N <= 4 ? 4 : 8))) <= 64);
}

// The bandwidth kernels for tall-skinny shapes, else the autotuned
// configuration when the shape has one, else the modelled choice.
int xr_dgemm_launch(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                    const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb,
                    int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int64_t batch) {
    if (M <= 0 || N <= 0 || batch <= 0) return XR_OK;
    if (ta && !tb && batch == 1 && M <= 64 && N <= 8 && K >= 4096)
        return launch_tn_skinny(c, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    if (ta && batch == 1 && M >= 1024 && K <= 64 && N <= 8) {
        ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
        prof.shape(M, N, K, batch, ta, tb);
#define XR_TN_TALL(NB_)                                                                                 \
        if (tb) k_dgemm_tn_tall<NB_, true><<<xr_grid(M), 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc); \
        else k_dgemm_tn_tall<NB_, false><<<xr_grid(M), 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc)
        if (N <= 1) { XR_TN_TALL(1); }
        else if (N <= 2) { XR_TN_TALL(2); }
        else if (N <= 4) { XR_TN_TALL(4); }
        else { XR_TN_TALL(8); }
#undef XR_TN_TALL
        XR_LAUNCH_CHECK(c);
        return XR_OK;
    }
    if (!ta && !tb && batch == 1 && N <= 8 && K >= 4096 && M * (N <= 1 ? 1 : (N <= 2 ? 2 : (N <= 4 ? 4 : 8))) <= 64)
        return launch_nn_gram(c, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    if (N <= 8 && !ta && batch == 1 && M >= 1024 && K <= 4) {
        ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
        prof.shape(M, N, K, batch, ta, tb);
#define XR_ROWS_SMALL(NB_)                                                                              \
        if (tb) k_dgemm_rows_small<NB_, true><<<xr_grid(M), 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc); \
        else k_dgemm_rows_small<NB_, false><<<xr_grid(M), 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc)
        if (N <= 1) { XR_ROWS_SMALL(1); }
        else if (N <= 2) { XR_ROWS_SMALL(2); }
        else if (N <= 4) { XR_ROWS_SMALL(4); }
        else { XR_ROWS_SMALL(8); }
#undef XR_ROWS_SMALL
        XR_LAUNCH_CHECK(c);
        return XR_OK;
    }
    if (N <= 8 && !ta && batch == 1 && M >= 1024 && K <= 64) {
        ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
        prof.shape(M, N, K, batch, ta, tb);
        const unsigned rgrid = (unsigned)(ceil_div(M, 64) < (1 << 20) ? ceil_div(M, 64) : (1 << 20));
#define XR_ROWWISE(NB_)                                                                                 \
        if (tb) k_dgemm_rows_lds<NB_, true><<<rgrid, 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc); \
        else k_dgemm_rows_lds<NB_, false><<<rgrid, 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc)
        if (N <= 1) { XR_ROWWISE(1); }
        else if (N <= 2) { XR_ROWWISE(2); }
        else if (N <= 4) { XR_ROWWISE(4); }
        else { XR_ROWWISE(8); }
#undef XR_ROWWISE
        XR_LAUNCH_CHECK(c);
        return XR_OK;
    }
    if (N <= 8 && !ta && batch == 1 && M >= 1024 && K > 64) {
        ProfScope prof(c, XR_K_GEMM_BW, 2.0 * M * N * K, 8.0 * (M * K + K * N + M * N));
        prof.shape(M, N, K, batch, ta, tb);
        unsigned grid = xr_grid(ceil_div(M, 4) * 64);
#define XR_SKINNY(NB_)                                                                                  \
        if (tb) k_dgemm_skinny<NB_, true><<<grid, 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc); \
        else k_dgemm_skinny<NB_, false><<<grid, 256, 0, c->stream>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc)
        if (N <= 1) { XR_SKINNY(1); }
        else if (N <= 2) { XR_SKINNY(2); }
        else if (N <= 4) { XR_SKINNY(4); }
        else { XR_SKINNY(8); }
#undef XR_SKINNY
        XR_LAUNCH_CHECK(c);
        return XR_OK;
    }
    auto it = c->tune.find(std::array<int64_t, 6>{ta, tb, M, N, K, batch});
    if (it != c->tune.end()) {
        const int64_t sp = it->second.second;
        const int rc = gemm_admit(c, sp > 1 ? 8 * sp * M * N * batch : 0);
        if (rc) return rc;
        return launch_cfg(c, it->second.first, sp, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC,
                          batch);
    }
    return launch_chosen(c, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch);
}

extern "C" int xr_gemm_f64(xr_ctx* c, int transA, int transB, int64_t M, int64_t N, int64_t K,
                           double alpha, const double* A, int64_t lda, int64_t sA,
                           const double* B, int64_t ldb, int64_t sB, double beta, double* C,
                           int64_t ldc, int64_t sC, int64_t batch) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (M < 0 || N < 0 || K < 0 || batch < 0) return xr_fail(c, XR_EINVAL, "negative GEMM size");
    if (ldc < N) return xr_fail(c, XR_ESHAPE, "ldc < N");
    if ((transA ? lda < M : lda < K) && M > 0 && K > 0) return xr_fail(c, XR_ESHAPE, "lda too small");
    if ((transB ? ldb < K : ldb < N) && N > 0 && K > 0) return xr_fail(c, XR_ESHAPE, "ldb too small");
    return xr_dgemm_launch(c, transA, transB, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                           sC, batch);
}

// Launches the problems of one tile shape, XR_GROUP_PROBS per grid
// (C_q = alpha op(A_q) op(B_q) + beta C_q; DIRECT: every problem passes gemm_direct;
// lower: square products with BM == BN whose grids hold only the tiles on
// and below the diagonal; kind: the profiler class of the launches).
template <int BM, int BN, bool DIRECT = true>
static int launch_grouped(xr_ctx* c, const std::vector<int>& ids, int ta, int tb, const int64_t* M,
                          const int64_t* N, const int64_t* K, double alpha, const double* const* A,
                          const int64_t* lda, const double* const* B, const int64_t* ldb, double* const* C,
                          const int64_t* ldc, double beta = 0.0, int lower = 0, int kind = XR_K_GEMM_GROUPED,
                          const int* off = nullptr, const int64_t* k0 = nullptr, const int64_t* k1 = nullptr) {
    if (lower && BM != BN) return xr_fail(c, XR_EUNSUPPORTED, "lower-triangle grids need square tiles");
    // launches of equal problem counts, problems by decreasing K
    std::vector<int> order(ids);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return K[a] > K[b]; });
    const size_t nl = (order.size() + XR_GROUP_PROBS - 1) / XR_GROUP_PROBS;
    for (size_t l = 0; l < nl; l++) {
        GemmGroup g;
        g.n = 0;
        g.lower = lower;
        g.alpha = alpha;
        g.beta = beta;
        int64_t slots = 0;                         // workgroups per XCD
        double flops = 0.0, bytes = 0.0;
        for (size_t t = l; t < order.size(); t += nl) {
            const int q = order[t];
            if (DIRECT && !gemm_direct(ta, tb, M[q], N[q], K[q], A[q], lda[q], 0, B[q], ldb[q], 0))
                return xr_fail(c, XR_EINVAL, "grouped GEMM: rows not 16-byte aligned");
            GemmProb& P = g.p[g.n++];
            P = GemmProb{A[q], B[q], C[q], M[q], N[q], K[q], lda[q], ldb[q], ldc[q],
                         ceil_div(M[q], BM), ceil_div(N[q], BN), off, off ? k0[q] : 0, off ? k1[q] : 0};
            if (lower && M[q] != N[q]) return xr_fail(c, XR_EUNSUPPORTED, "lower-triangle grid of a non-square C");
            slots += ceil_div(lower ? P.tiles_m * (P.tiles_m + 1) / 2 : P.tiles_m * P.tiles_n, 8);
            flops += (lower ? 1.0 : 2.0) * M[q] * N[q] * K[q];
            bytes += 8.0 * (M[q] * K[q] + K[q] * N[q] + M[q] * N[q]);
        }
        if (8 * slots > 0x7fffffff) return xr_fail(c, XR_EUNSUPPORTED, "GEMM grid too large");
        ProfScope prof(c, kind, flops, bytes);
        // no shape in the class of the single products: the tuner would time it as one
        if (kind != XR_K_GEMM_F64) prof.shape(g.p[0].M, g.p[0].N, g.p[0].K, g.n, ta, tb);
        const dim3 grid((unsigned)(8 * slots));
#define XR_GROUPED(TA_, TB_) \
    k_dgemm_grouped<BM, BN, TA_, TB_, DIRECT><<<grid, GEMM_THREADS, 0, c->stream>>>(g)
        if (ta && tb) XR_GROUPED(true, true);
        else if (ta) XR_GROUPED(true, false);
        else if (tb) XR_GROUPED(false, true);
        else XR_GROUPED(false, false);
#undef XR_GROUPED
        XR_LAUNCH_CHECK(c);
    }
    return XR_OK;
}

// launch_grouped for problems of any alignment: those that cannot be loaded
// in 16-byte chunks run on 64 x 64 tiles.
template <int BM, int BN>
static int launch_grouped_any(xr_ctx* c, const std::vector<int>& ids, int ta, int tb, const int64_t* M,
                              const int64_t* N, const int64_t* K, double alpha, const double* const* A,
                              const int64_t* lda, const double* const* B, const int64_t* ldb, double* const* C,
                              const int64_t* ldc, double beta = 0.0, int lower = 0, int kind = XR_K_GEMM_GROUPED) {
    std::vector<int> even, odd;
    for (int q : ids)
        (gemm_direct(ta, tb, M[q], N[q], K[q], A[q], lda[q], 0, B[q], ldb[q], 0) ? even : odd).push_back(q);
    const int rc = launch_grouped<BM, BN>(c, even, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc, beta, lower, kind);
    if (rc) return rc;
    return launch_grouped<64, 64, false>(c, odd, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc, beta, lower, kind);
}

// C_q = alpha op(A_q) op(B_q) for n independent problems (row-major, the
// same transposes).  Problems with N > 64 share 128 x 128 tile grids, those
// with 8 < N <= 64 share 128 x 64 grids (both with M > 64; 64 x 64 ones when
// their rows are not 16-byte aligned); the rest (the
// tall-skinny and small shapes) go to the single-product dispatch, whose
// bandwidth kernels suit them.  No K split and no beta: every C_q is
// overwritten.
extern "C" int xr_gemm_grouped(xr_ctx* c, int n, int ta, int tb, const int64_t* M, const int64_t* N,
                               const int64_t* K, double alpha, const double* const* A, const int64_t* lda,
                               const double* const* B, const int64_t* ldb, double* const* C,
                               const int64_t* ldc) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> lock(c->mu);
    if (n < 0) return xr_fail(c, XR_EINVAL, "negative problem count");
    std::vector<int> wide, narrow;
    for (int q = 0; q < n; q++) {
        if (M[q] < 0 || N[q] < 0 || K[q] < 0) return xr_fail(c, XR_EINVAL, "negative GEMM size");
        if (ldc[q] < N[q]) return xr_fail(c, XR_ESHAPE, "ldc < N");
        if ((ta ? lda[q] < M[q] : lda[q] < K[q]) && M[q] > 0 && K[q] > 0)
            return xr_fail(c, XR_ESHAPE, "lda too small");
        if ((tb ? ldb[q] < K[q] : ldb[q] < N[q]) && N[q] > 0 && K[q] > 0)
            return xr_fail(c, XR_ESHAPE, "ldb too small");
    }
    for (int q = 0; q < n; q++) {
        if (M[q] == 0 || N[q] == 0) continue;
        if (M[q] > 64 && N[q] > 64) wide.push_back(q);
        else if (M[q] > 64 && N[q] > 8) narrow.push_back(q);
        else {
            const int rc = xr_dgemm_launch(c, ta, tb, M[q], N[q], K[q], alpha, A[q], lda[q], 0, B[q], ldb[q], 0,
                                           0.0, C[q], ldc[q], 0, 1);
            if (rc) return rc;
        }
    }
    // At most two 64 x 64 tiles a compute unit in all: one launch of that tile for
    // every width and alignment.  One workgroup then walks each K alone, so the
    // small tile's shorter step counts and a second launch costs a whole walk more.
    // Operator on one vector, 21 x 16 x 30 states: 219 -> 146 us, on eight, 23 x 15 x 8:
    // 265 -> 131; two fragments (60 us) unchanged.
    std::vector<int> all(wide);
    all.insert(all.end(), narrow.begin(), narrow.end());
    int64_t tiles = 0;
    bool direct = true;
    for (int q : all) {
        tiles += ceil_div(M[q], 64) * ceil_div(N[q], 64);
        direct = direct && gemm_direct(ta, tb, M[q], N[q], K[q], A[q], lda[q], 0, B[q], ldb[q], 0);
    }
    if (!all.empty() && tiles <= 2 * device_cus())
        return direct ? launch_grouped<64, 64>(c, all, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc)
                      : launch_grouped<64, 64, false>(c, all, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc);
    int rc = launch_grouped_any<128, 128>(c, wide, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc);
    if (rc) return rc;
    return launch_grouped_any<128, 64>(c, narrow, ta, tb, M, N, K, alpha, A, lda, B, ldb, C, ldc);
}

int xr_dgemm_blocks(xr_ctx* c, int n, const int64_t* row, int64_t K, int64_t N, const double* A, int64_t lda,
                    const double* B, int64_t ldb, double* C, int64_t ldc, const int* off) {
    std::vector<int> ids;
    std::vector<int64_t> M(n), Ns(n, N), Ks(n, K), la(n, lda), lb(n, ldb), lc(n, ldc), k0(n), k1(n);
    std::vector<const double*> As(n), Bs(n, B);
    std::vector<double*> Cs(n);
    bool direct = true;
    for (int q = 0; q < n; q++) {
        M[q] = row[q + 1] - row[q];
        As[q] = A + row[q] * lda;
        Cs[q] = C + row[q] * ldc;
        k0[q] = row[q] & ~(int64_t)1;                         // whole 16-byte chunks of A's rows
        k1[q] = std::min<int64_t>(K, (row[q + 1] + 1) & ~(int64_t)1);
        if (M[q] > 0) ids.push_back(q);
        direct = direct && gemm_direct(0, 0, M[q], N, K, As[q], lda, 0, B, ldb, 0);
    }
    // 64 x 64 tiles: a block's k range is short (154 or 324 of 630), so a
    // tile's first loads and its stores are a large part of it, and five tiles a CU
    // hide them better than two (18 orbitals, 64 states: 3.35 ms with 128 x 128, 3.2 with 128 x 64, 3.0)
    if (direct)
        return launch_grouped<64, 64>(c, ids, 0, 0, M.data(), Ns.data(), Ks.data(), 1.0, As.data(), la.data(),
                                      Bs.data(), lb.data(), Cs.data(), lc.data(), 0.0, 0, XR_K_GEMM_F64, off,
                                      k0.data(), k1.data());
    return launch_grouped<64, 64, false>(c, ids, 0, 0, M.data(), Ns.data(), Ks.data(), 1.0, As.data(), la.data(),
                                         Bs.data(), lb.data(), Cs.data(), lc.data(), 0.0, 0, XR_K_GEMM_F64, off,
                                         k0.data(), k1.data());
}

// ---------------------------------------------------------------------------
// Autotuner: times every tile shape with a ladder of K splits on scratch
// operands of the given shape (HIP events on the context stream) and keeps
// the fastest in the context's table, which xr_dgemm_launch consults.
// ---------------------------------------------------------------------------
extern "C" int xr_gemm_tune(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t batch,
                            int reps, int* tile_out, int* splits_out, double* ms_out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0 || reps <= 0) return xr_fail(c, XR_EINVAL, "bad tune shape");
    if (gemm_skinny(ta, tb, M, N, K, batch)) {           // bandwidth kernels, not tiled
        if (tile_out) *tile_out = -1;
        if (splits_out) *splits_out = 0;
        if (ms_out) *ms_out = 0.0;
        return XR_OK;
    }
    const int64_t na = M * K * batch, nb = K * N * batch, nc = M * N * batch;
    if ((na + nb + nc) * 8 > (int64_t)16 << 30) return xr_fail(c, XR_EUNSUPPORTED, "shape too large to tune");
    double* A = (double*)xr_workspace(c, 60, na * sizeof(double));
    double* B = (double*)xr_workspace(c, 61, nb * sizeof(double));
    double* C = (double*)xr_workspace(c, 62, nc * sizeof(double));
    if (!A || !B || !C) return xr_fail(c, XR_ENOMEM, "workspace (tune)");
    int rc;
    if ((rc = xr_fill(c, A, na, 1e-3)) || (rc = xr_fill(c, B, nb, 1e-3))) return rc;
    const int64_t lda = ta ? M : K, ldb = tb ? K : N;
    const int64_t sA = batch > 1 ? M * K : 0, sB = batch > 1 ? K * N : 0, sC = batch > 1 ? M * N : 0;
    hipEvent_t e0, e1;
    XR_HIP(c, hipEventCreate(&e0));
    XR_HIP(c, hipEventCreate(&e1));
    const bool prof = c->prof;
    c->prof = false;
    const std::array<int64_t, 6> key{ta, tb, M, N, K, batch};
    c->tune.erase(key);
    // the untuned dispatch is the first candidate: a table entry is kept
    // only for a configuration that beats it
    double best = 1e300;
    int best_tile = -1, best_split = 0;
    rc = xr_dgemm_launch(c, ta, tb, M, N, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, C, N, sC, batch);
    if (!rc) {
        XR_HIP(c, hipEventRecord(e0, c->stream));
        for (int r = 0; r < reps; r++)
            rc |= xr_dgemm_launch(c, ta, tb, M, N, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, C, N, sC, batch);
        XR_HIP(c, hipEventRecord(e1, c->stream));
        XR_HIP(c, hipEventSynchronize(e1));
        float ms = 0.f;
        XR_HIP(c, hipEventElapsedTime(&ms, e0, e1));
        best = ms / reps;
    }
    for (int tile = 0; tile < 4 && !rc; tile++) {   // the untuned choice covers the 32 x 32 kernel
        for (int sp = 1; sp <= 64; sp *= 2) {
            if (sp > 1 && (K / sp < 64 || 8 * sp * M * N * batch > GEMM_STAGING_MAX)) break;
            rc = launch_cfg(c, tile, sp, ta, tb, M, N, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, C, N, sC, batch);
            if (rc) break;
            XR_HIP(c, hipEventRecord(e0, c->stream));
            for (int r = 0; r < reps; r++)
                rc |= launch_cfg(c, tile, sp, ta, tb, M, N, K, 1.0, A, lda, sA, B, ldb, sB, 0.0, C, N, sC, batch);
            XR_HIP(c, hipEventRecord(e1, c->stream));
            XR_HIP(c, hipEventSynchronize(e1));
            float ms = 0.f;
            XR_HIP(c, hipEventElapsedTime(&ms, e0, e1));
            if (rc) break;
            if (ms / reps < best) { best = ms / reps; best_tile = tile; best_split = sp; }
        }
        if (rc) break;
    }
    c->prof = prof;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (best_tile >= 0) c->tune[key] = std::make_pair(best_tile, best_split);
    if (tile_out) *tile_out = best_tile;
    if (splits_out) *splits_out = best_split;
    if (ms_out) *ms_out = best;
    return XR_OK;
}

extern "C" int xr_gemm_tune_reset(xr_ctx* c) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    c->tune.clear();
    return XR_OK;
}

// ---------------------------------------------------------------------------
// Split-FP32 GEMM on v_mfma_f32_16x16x4f32 with FP64 accumulation.
//
// While an operand tile is staged in LDS, every group of 8 consecutive k
// values of one row of A (one column of B) is put on a common power-of-two
// grid g = 2^(e-10), e = exponent of the group's largest |x|:
//   hi = rint(x / g) * g      (|hi / g| <= 2^10: 11 significant bits)
//   lo = fp32(x - hi)         (|lo| <= g/2, 24 significant bits)
// A hi*hi product is an integer multiple of ga*gb below 2^20 of it, so the
// 8 products of one group (two chained MFMAs) sum to < 2^23 grid units and
// the FP32 matrix core forms them EXACTLY; that sum is then added into the
// FP64 accumulator.  The remaining terms hi_a*lo_b + lo_a*(hi_b + lo_b) are
// ~2^-11 of the group's scale and go through FP32 accumulation over one
// 16-deep LDS tile; their rounding, and the 24-bit lo, leave a relative
// error of a few 2^-35 of max|a|*max|b| per group.
// ---------------------------------------------------------------------------
typedef float f4_t __attribute__((ext_vector_type(4)));

// Biased exponent field of |x|.
__device__ __forceinline__ int xr_expo(double x) {
    return (int)((__double_as_longlong(x) >> 52) & 0x7ff);
}

// Split x on the grid of a group whose largest biased exponent is eb.  A
// group whose largest value is below 2^-1012 (or zero) is flushed to zero.
__device__ __forceinline__ void xr_split(double x, int eb, float& hi, float& lo) {
    if (eb < 12) { hi = 0.f; lo = 0.f; return; }
    const double s = __longlong_as_double((long long)(2055 - eb) << 52);   // 2^(1032-eb) = 1/g
    const double gi = __longlong_as_double((long long)(eb - 9) << 52);     // 2^(eb-1032) = g
    const double h = rint(x * s) * gi;
    hi = (float)h;
    lo = (float)(x - h);
}

// Max over the 8 lanes (aligned) that hold one group.
__device__ __forceinline__ int xr_group8_max(int e) {
    e = max(e, __shfl_xor(e, 1));
    e = max(e, __shfl_xor(e, 2));
    e = max(e, __shfl_xor(e, 4));
    return e;
}

// BM x BM tiles on 4 * BM threads (4 elements of each operand per thread
// and 16-deep k step): 128 x 128 as 8 waves of 64 x 32, 64 x 64 as 4 waves
// of 32 x 32.
template <bool TA, bool TB, int BM>
__global__ __launch_bounds__(4 * BM) void k_dgemm_split(
    int64_t M, int64_t N, int64_t K, const double* __restrict__ A, int64_t lda, int64_t sA,
    const double* __restrict__ B, int64_t ldb, int64_t sB, double* __restrict__ C, int64_t ldc,
    int64_t sC, int64_t tiles_m, int64_t tiles_n, int64_t kchunk, int64_t sSplit) {
    constexpr int THREADS = 4 * BM, BN = BM, PAD = 4;
    constexpr int WGN = (BM == 128) ? 4 : 2, WGM = THREADS / 64 / WGN;
    constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
    constexpr int PER = BM * GEMM_BK / THREADS;
    static_assert(PER == 4 && (BM == 128 || BM == 64), "4 elements per thread and operand");
    __shared__ float Ah[GEMM_BK][BM + PAD], Al[GEMM_BK][BM + PAD];
    __shared__ float Bh[GEMM_BK][BN + PAD], Bl[GEMM_BK][BN + PAD];
    const int64_t batch = blockIdx.z;
    A += batch * sA;
    B += batch * sB;
    C += batch * sC + (int64_t)blockIdx.y * sSplit;
    const int64_t kbeg = (int64_t)blockIdx.y * kchunk;
    K = (K - kbeg < kchunk) ? (K - kbeg) : kchunk;
    if (TA) A += kbeg * lda; else A += kbeg;
    if (TB) B += kbeg; else B += kbeg * ldb;
    const int64_t tile = xcd_remap(blockIdx.x, (int64_t)gridDim.x);
    const int64_t GROUP = 8, per_group = GROUP * tiles_n, g = tile / per_group, first_m = g * GROUP;
    const int64_t gsize = (tiles_m - first_m < GROUP) ? (tiles_m - first_m) : GROUP;
    const int64_t tm = first_m + (tile % per_group) % gsize, tn = (tile % per_group) / gsize;
    const int64_t m0 = tm * BM, n0 = tn * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WGN, wn = wave % WGN;
    // Element i of a thread as (row, k) inside a BM x 16 tile.  Operands
    // stored k-major (A transposed, B plain) give lanes t and t^1 the two
    // halves of one row's 8-deep group; row-major ones give 8 aligned lanes
    // one k each of a row's group.
    auto pos = [&](bool kmajor, int i, int& row, int& kk) {
        if (kmajor) { row = (tid >> 1) & (BM - 1); kk = (tid / (2 * BM)) * 8 + (tid & 1) * 4 + i; }
        else { kk = tid % GEMM_BK; row = tid / GEMM_BK + i * (THREADS / GEMM_BK); }
    };
    auto group_max = [&](bool kmajor, int* e) {
        if (kmajor) {
            int m = max(max(e[0], e[1]), max(e[2], e[3]));
            m = max(m, __shfl_xor(m, 1));
#pragma unroll
            for (int i = 0; i < PER; i++) e[i] = m;
        } else {
#pragma unroll
            for (int i = 0; i < PER; i++) e[i] = xr_group8_max(e[i]);
        }
    };
    double ra[PER], rb[PER];
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int mm, kk;
            pos(TA, i, mm, kk);
            int64_t gm = m0 + mm, gk = k0 + kk;
            ra[i] = (gm < M && gk < K) ? (TA ? A[gk * lda + gm] : A[gm * lda + gk]) : 0.0;
        }
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int nn, kk;
            pos(!TB, i, nn, kk);
            int64_t gn = n0 + nn, gk = k0 + kk;
            rb[i] = (gn < N && gk < K) ? (TB ? B[gn * ldb + gk] : B[gk * ldb + gn]) : 0.0;
        }
    };
    auto store = [&]() {
        int ea[PER], eb[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) { ea[i] = xr_expo(ra[i]); eb[i] = xr_expo(rb[i]); }
        group_max(TA, ea);
        group_max(!TB, eb);
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int mm, kk;
            pos(TA, i, mm, kk);
            xr_split(ra[i], ea[i], Ah[kk][mm], Al[kk][mm]);
            pos(!TB, i, mm, kk);
            xr_split(rb[i], eb[i], Bh[kk][mm], Bl[kk][mm]);
        }
    };
    d4_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
    const int64_t nk = (K + GEMM_BK - 1) / GEMM_BK;
    const int fr = lane & 15, fk = lane >> 4;
    if (nk > 0) { load(0); store(); __syncthreads(); }
    const f4_t z4 = {0.f, 0.f, 0.f, 0.f};
    for (int64_t kt = 0; kt < nk; kt++) {
        if (kt + 1 < nk) load((kt + 1) * GEMM_BK);
#pragma unroll
        for (int grp = 0; grp < GEMM_BK / 8; grp++) {
            float ah[2][FM], al[2][FM], bh[2][FN], bl[2][FN], bs[2][FN];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int k = grp * 8 + s * 4 + fk;
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    ah[s][i] = Ah[k][wm * WM + i * 16 + fr];
                    al[s][i] = Al[k][wm * WM + i * 16 + fr];
                }
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    bh[s][j] = Bh[k][wn * WN + j * 16 + fr];
                    bl[s][j] = Bl[k][wn * WN + j * 16 + fr];
                    bs[s][j] = bh[s][j] + bl[s][j];
                }
            }
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    f4_t hh = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[0][i], bh[0][j], z4, 0, 0, 0);
                    hh = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[1][i], bh[1][j], hh, 0, 0, 0);
                    f4_t x = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[0][i], bl[0][j], z4, 0, 0, 0);
                    x = __builtin_amdgcn_mfma_f32_16x16x4f32(al[0][i], bs[0][j], x, 0, 0, 0);
                    x = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[1][i], bl[1][j], x, 0, 0, 0);
                    x = __builtin_amdgcn_mfma_f32_16x16x4f32(al[1][i], bs[1][j], x, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] += (double)hh[r] + (double)x[r];
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        if (kt + 1 < nk) { store(); __syncthreads(); }
    }
    // D[row][col] of v_mfma_f32_16x16x4f32: col = lane % 16, row = XR_F32_ROW(fk, r)
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                int64_t gm = m0 + wm * WM + i * 16 + XR_F32_ROW(fk, r);
                int64_t gn = n0 + wn * WN + j * 16 + fr;
                if (gm < M && gn < N) C[gm * ldc + gn] = acc[i][j][r];
            }
}

template <int BM>
static void split_go(xr_ctx* c, int ta, int tb, dim3 grid, int64_t M, int64_t N, int64_t K, const double* A,
                     int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB, double* Cw,
                     int64_t tm, int64_t tn, int64_t kchunk, int64_t batch) {
    const int nt = 4 * BM;
    if (ta && tb) k_dgemm_split<true, true, BM><<<grid, nt, 0, c->stream>>>(M, N, K, A, lda, sA, B, ldb, sB, Cw, N, M * N, tm, tn, kchunk, batch * M * N);
    else if (ta) k_dgemm_split<true, false, BM><<<grid, nt, 0, c->stream>>>(M, N, K, A, lda, sA, B, ldb, sB, Cw, N, M * N, tm, tn, kchunk, batch * M * N);
    else if (tb) k_dgemm_split<false, true, BM><<<grid, nt, 0, c->stream>>>(M, N, K, A, lda, sA, B, ldb, sB, Cw, N, M * N, tm, tn, kchunk, batch * M * N);
    else k_dgemm_split<false, false, BM><<<grid, nt, 0, c->stream>>>(M, N, K, A, lda, sA, B, ldb, sB, Cw, N, M * N, tm, tn, kchunk, batch * M * N);
}

// Split-FP32 product (always staged: partial tiles go to a workspace and the
// fixed-order reduction applies beta).
int xr_dgemm_split_launch(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                          const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb,
                          int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int64_t batch) {
    if (M <= 0 || N <= 0 || batch <= 0) return XR_OK;
    // 64 x 64 tiles, with a K split (chunks of at least 256) toward 1024
    // workgroups when the tiles are few.  The 128 x 128 variant needs more
    // than the 256 registers a lane has at two waves per SIMD (it spilled 27)
    // and ran the c3 split iteration 6% slower.
    const int bm = 64;
    int64_t tm = ceil_div(M, bm), tn = ceil_div(N, bm), tiles = tm * tn;
    if (tiles > 0x7fffffff || batch > 65535) return xr_fail(c, XR_EUNSUPPORTED, "GEMM grid too large");
    int64_t splits = 1, kchunk = K;
    if (tiles * batch < 512 && K >= 512) {
        splits = ceil_div(1024, tiles * batch);
        int64_t max_split = K / 256;
        if (splits > max_split) splits = max_split;
        if (splits > 512) splits = 512;
        if (splits < 1) splits = 1;
        kchunk = ceil_div(ceil_div(K, splits), GEMM_BK) * GEMM_BK;
        splits = ceil_div(K, kchunk);
    }
    double* Cw = (double*)xr_workspace(c, 51, splits * batch * M * N * sizeof(double));
    if (!Cw) return xr_fail(c, XR_ENOMEM, "workspace (split-FP32)");
    dim3 grid((unsigned)tiles, (unsigned)splits, (unsigned)batch);
    {
        ProfScope prof(c, XR_K_GEMM_SPLIT, 2.0 * M * N * K * batch, 8.0 * (M * K + K * N + M * N) * batch);
        prof.shape(M, N, K, batch, ta, tb);
        split_go<64>(c, ta, tb, grid, M, N, K, A, lda, sA, B, ldb, sB, Cw, tm, tn, kchunk, batch);
        XR_LAUNCH_CHECK(c);
    }
    return splitk_reduce(c, Cw, splits, batch, M, N, alpha, beta, C, ldc, sC);
}

// The contraction GEMMs of the two-electron terms go through here: FP64,
// split-FP32 or split-int8 depending on the context's precision setting
// (split-int8 for the products where it pays, xr_i8_pays; FP64 for the rest).
int xr_gemm_2e(xr_ctx* c, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
               const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB,
               double beta, double* C, int64_t ldc, int64_t sC, int64_t batch) {
    if (c->precision == XR_PREC_SPLIT_F32)
        return xr_dgemm_split_launch(c, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                                     sC, batch);
    if (c->precision == XR_PREC_SPLIT_I8 && xr_i8_pays(M, N, K, batch))
        return xr_dgemm_i8_launch(c, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch);
    return xr_dgemm_launch(c, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch);
}

extern "C" int xr_set_precision(xr_ctx* c, int mode) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (mode != XR_PREC_F64 && mode != XR_PREC_SPLIT_F32 && mode != XR_PREC_SPLIT_I8)
        return xr_fail(c, XR_EINVAL, "unknown precision mode");
    c->precision = mode;
    return XR_OK;
}

extern "C" int xr_gemm_split_f32(xr_ctx* c, int transA, int transB, int64_t M, int64_t N, int64_t K,
                                 double alpha, const double* A, int64_t lda, int64_t sA,
                                 const double* B, int64_t ldb, int64_t sB, double beta, double* C,
                                 int64_t ldc, int64_t sC, int64_t batch) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (M < 0 || N < 0 || K < 0 || batch < 0) return xr_fail(c, XR_EINVAL, "negative GEMM size");
    if (ldc < N) return xr_fail(c, XR_ESHAPE, "ldc < N");
    return xr_dgemm_split_launch(c, transA, transB, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                                 sC, batch);
}

// ---------------------------------------------------------------------------
// No-allocation FP64 GEMM
// ---------------------------------------------------------------------------
// Staging memory of xr_gemm_f64_noalloc (the split-K partial tiles and the
// partial sums of the tall-skinny kernels): one 64 MiB array per device,
// held until the process ends and shared by every such call on that device.
// Host code never passes the array's name to a kernel (in host code it is a
// host-side stand-in); it uses the device address xr_noalloc_init stores in
// the context.
#define XR_NOALLOC_SCRATCH_BYTES ((size_t)64 << 20)
static __device__ __align__(256) double scratch[XR_NOALLOC_SCRATCH_BYTES / sizeof(double)];

// Called by xr_create with the context's device current: the device address
// of this device's copy of `scratch`.
int xr_noalloc_init(xr_ctx* c) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        (void)hipGetLastError();
        return xr_fail(c, XR_EHIP, "hipGetSymbolAddress(scratch) failed");
    }
    c->scratch = p;
    c->scratch_bytes = XR_NOALLOC_SCRATCH_BYTES;
    return XR_OK;
}

extern "C" int xr_gemm_f64_noalloc(xr_ctx* c, int transA, int transB, int64_t M, int64_t N, int64_t K,
                                   double alpha, const double* A, int64_t lda, int64_t sA,
                                   const double* B, int64_t ldb, int64_t sB, double beta, double* C,
                                   int64_t ldc, int64_t sC, int64_t batch) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (M < 0 || N < 0 || K < 0 || batch < 0) return xr_fail(c, XR_EINVAL, "negative GEMM size");
    if (ldc < N) return xr_fail(c, XR_ESHAPE, "ldc < N");
    if ((transA ? lda < M : lda < K) && M > 0 && K > 0) return xr_fail(c, XR_ESHAPE, "lda too small");
    if ((transB ? ldb < K : ldb < N) && N > 0 && K > 0) return xr_fail(c, XR_ESHAPE, "ldb too small");
    if (!c->scratch) return xr_fail(c, XR_EHIP, "no scratch address for this device");
    // the same kernels and choices as xr_gemm_f64, with every staging buffer
    // taken from the scratch array; the launch timers are off for the call
    // (they would create events)
    const bool prof = c->prof;
    c->prof = false;
    c->noalloc = true;
    c->noalloc_blocked = false;
    int rc = xr_dgemm_launch(c, transA, transB, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC,
                             batch);
    c->noalloc = false;
    c->noalloc_blocked = false;
    c->prof = prof;
    return rc;
}
