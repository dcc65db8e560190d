// Transition densities as gather-GEMMs on the matrix cores.
//
// The reference walks every (ket determinant, operator-index tuple) and
// scatters a rank-1 update into all state pairs (general-XRCC/
// density_tensors.c:142-556).  Here an operator string is split as
// L * R with L pure creators (possibly empty) and R pure annihilators or
// pure creators, and a resolution of the identity over the complete
// determinant space K between them is inserted:
//
//   <I| L_l R_t |J> = sum_K <I|L_l|K> <K|R_t|J>
//                   = sum_K X[K, l, I] * Y[K, t, J]
//
//   X[K, l, I] = sum_P <K| L_l^+ |P> zbra[I, P]   (one P per (K, l))
//   Y[K, t, J] = sum_Q <K| R_t |Q> zket[J, Q]     (one Q per (K, t))
//
// l and t run over sorted index tuples only (operators of one kind
// anticommute), so X and Y are signed gathers of coefficient rows driven by
// integer excitation tables, and the contraction over K is one dense FP64
// GEMM.  An expand pass writes the full antisymmetric dim^k layout.  When L
// is empty, K is the bra space itself and X = zbra^T.
#include "xr_common.h"
#include "xr_gemm.h"
#include "xr_density.h"
#include <algorithm>

// ---------------------------------------------------------------------------
// operator plans
// ---------------------------------------------------------------------------
int xr_plan_op(const char* ops, OpPlan* p) {
    struct Row { const char* s; OpPlan p; };
    // side: {k, is_c, slots}; slots name the tuple entry each operator of
    // the side string uses, leftmost operator first.
    static const Row rows[] = {
        {"a",    {1, 0, {0, 0, {0}}, {1, 0, {0}}}},
        {"c",    {1, 1, {1, 0, {0}}, {0, 0, {0}}}},
        {"aa",   {2, 0, {0, 0, {0}}, {2, 0, {0, 1}}}},
        {"cc",   {2, 1, {2, 0, {1, 0}}, {0, 0, {0}}}},
        {"ca",   {2, 1, {1, 0, {0}}, {1, 0, {0}}}},
        {"caa",  {3, 1, {1, 0, {0}}, {2, 0, {0, 1}}}},
        {"cca",  {3, 1, {2, 0, {1, 0}}, {1, 0, {0}}}},
        {"ccaa", {4, 1, {2, 0, {1, 0}}, {2, 0, {0, 1}}}},
        {"caaa", {4, 1, {1, 0, {0}}, {3, 0, {0, 1, 2}}}},
        {"ccca", {4, 1, {3, 0, {2, 1, 0}}, {1, 0, {0}}}},
        // the 5-operator strings of XR order 1 (Be-states/densities.py:83-88;
        // Be-states/_attic_/deprecated/density_tensors.c:690-836)
        {"ccaaa", {5, 1, {2, 0, {1, 0}}, {3, 0, {0, 1, 2}}}},
        {"cccaa", {5, 1, {3, 0, {2, 1, 0}}, {2, 0, {0, 1}}}},
    };
    if (!ops) return 0;
    for (const Row& r : rows) {
        if (strcmp(ops, r.s) == 0) {
            *p = r.p;
            int d = 0;
            for (const char* q = ops; *q; q++) d += (*q == 'c') ? 1 : -1;
            p->delta = d;
            return 1;
        }
    }
    return 0;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t d_from_valence(uint64_t v, int n_orbs, int n_core) {
    if (n_core == 0) return v;
    int nv = n_orbs - n_core;
    uint64_t m = (nv >= 64) ? ~0ull : ((1ull << nv) - 1);
    uint64_t a = (v & m) << n_core;
    uint64_t b = ((v >> nv) & m) << (n_orbs + n_core);
    return a | b | d_core_mask(n_orbs, n_core);
}

__device__ __forceinline__ void k_unrank_space_elem(int64_t i, uint64_t* masks, int64_t n, int n_orbs, int n_core, int n_elec) {
    int nval = 2 * (n_orbs - n_core);
    masks[i] = d_from_valence(d_lex_unrank(i, nval, n_elec - 2 * n_core), n_orbs, n_core);
}

__global__ void k_unrank_space(uint64_t* masks, int64_t n, int n_orbs, int n_core, int n_elec) {
    XR_GRID_STRIDE(i, n) k_unrank_space_elem(i, masks, n, n_orbs, n_core, n_elec);
}

// One entry per (K, t): the source determinant the side string maps onto K,
// as sign * (valence rank + 1), or 0 when the string annihilates it.
__device__ __forceinline__ void k_side_table_elem(int64_t i, SidePlan sd, const uint64_t* __restrict__ Km, int64_t nK, int dim,
                             int n_orbs, int n_core, int64_t nT, int32_t* __restrict__ tab) {
    int64_t K = i / nT, t = i - K * nT;
    uint64_t km = Km[K];
    uint64_t tm = d_lex_unrank(t, dim, sd.k);
    int orb[3] = {0, 0, 0};
    {
        uint64_t x = tm;
        for (int j = 0; j < sd.k; j++) {
            orb[j] = __ffsll((unsigned long long)x) - 1;
            x &= x - 1;
        }
    }
    uint64_t src;
    if (!sd.is_c) {
        if (km & tm) { tab[i] = 0; return; }
        src = km | tm;
    } else {
        if ((km & tm) != tm) { tab[i] = 0; return; }
        src = km & ~tm;
    }
    uint64_t core = d_core_mask(n_orbs, n_core);
    if ((src & core) != core) { tab[i] = 0; return; }
    uint64_t cur = src;
    int sg = 1;
    for (int j = sd.k - 1; j >= 0; j--) {
        int o = orb[sd.slot[j]];
        sg *= d_sign_above(cur, o);
        cur ^= 1ull << o;
    }
    int64_t r = d_lex_rank(d_to_valence(src, n_orbs, n_core), dim - 2 * n_core);
    tab[i] = sg * (int32_t)(r + 1);
}

// Spin-class order of the pairs p < q of dim = 2 n spin orbitals (alpha
// first): the alpha-alpha pairs, the alpha-beta ones, the beta-beta ones, each
// lexical.  A two-body part that conserves the spin projection couples no two
// classes, so in this order its antisymmetrised pair matrix is block diagonal.
__host__ __device__ __forceinline__ int pair_pos(int p, int q, int n) {
    const int aa = n * (n - 1) / 2;
    if (q < n) return p * n - p * (p + 1) / 2 + (q - p - 1);
    if (p < n) return aa + p * n + (q - n);
    p -= n;
    q -= n;
    return aa + n * n + p * n - p * (p + 1) / 2 + (q - p - 1);
}
__device__ __forceinline__ void pair_at(int pos, int n, int* p, int* q) {
    const int aa = n * (n - 1) / 2;
    int base = 0;
    if (pos >= aa && pos < aa + n * n) {
        pos -= aa;
        *p = pos / n;
        *q = n + (pos - *p * n);
        return;
    }
    if (pos >= aa) { pos -= aa + n * n; base = n; }
    int a = 0;
    while (pos >= n - 1 - a) { pos -= n - 1 - a; a++; }
    *p = base + a;
    *q = base + a + 1 + pos;
}
__device__ __forceinline__ int pair_class(int pos, int n) {
    const int aa = n * (n - 1) / 2;
    return pos < aa ? 0 : (pos < aa + n * n ? 1 : 2);
}

// The entries of k_side_table for a pair string, pair-major: tab[u * nK + K]
// with u in spin-class order (and a row of zeros where the number of pairs is odd).
__global__ void k_pair_table(SidePlan sd, const uint64_t* __restrict__ Km, int64_t nK, int dim, int n_orbs,
                             int n_core, int64_t nU, int32_t* __restrict__ tab) {
    const uint64_t core = d_core_mask(n_orbs, n_core);
    XR_GRID_STRIDE(i, nU * nK) {
        const int64_t u = i / nK, K = i - u * nK;
        int orb[2];
        if (u >= n_orbs * (2 * n_orbs - 1)) { tab[i] = 0; continue; }      // padding row
        pair_at((int)u, n_orbs, &orb[0], &orb[1]);
        const uint64_t km = Km[K], tm = (1ull << orb[0]) | (1ull << orb[1]);
        const uint64_t src = sd.is_c ? (km & ~tm) : (km | tm);
        if ((sd.is_c ? (km & tm) != tm : (km & tm) != 0) || (src & core) != core) {
            tab[i] = 0;
            continue;
        }
        uint64_t cur = src;
        int sg = 1;
        for (int j = 1; j >= 0; j--) {
            const int o = orb[sd.slot[j]];
            sg *= d_sign_above(cur, o);
            cur ^= 1ull << o;
        }
        tab[i] = sg * (int32_t)(d_lex_rank(d_to_valence(src, n_orbs, n_core), dim - 2 * n_core) + 1);
    }
}

__global__ void k_side_table(SidePlan sd, const uint64_t* __restrict__ Km, int64_t nK, int dim,
                             int n_orbs, int n_core, int64_t nT, int32_t* __restrict__ tab) {
    XR_GRID_STRIDE(i, nK * nT) k_side_table_elem(i, sd, Km, nK, dim, n_orbs, n_core, nT, tab);
}

// zT[c * nS + s] = z[s * nC + c] for the side blockIdx.z picks
struct TransposeSide { const double* z; double* zT; int64_t nS, nC; };
__global__ void k_transpose(TransposeSide t0, TransposeSide t1) {
    const TransposeSide t = blockIdx.z ? t1 : t0;
    __shared__ double tile[32][33];
    const int64_t c0 = (int64_t)blockIdx.x * 32, s0 = (int64_t)blockIdx.y * 32;
    if (c0 >= t.nC || s0 >= t.nS) return;
    const int tx = threadIdx.x, ty = threadIdx.y;  // 32 x 8
    for (int j = ty; j < 32; j += 8) {
        const int64_t s = s0 + j, c = c0 + tx;
        if (s < t.nS && c < t.nC) tile[j][tx] = t.z[s * t.nC + c];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {
        const int64_t c = c0 + j, s = s0 + tx;
        if (s < t.nS && c < t.nC) t.zT[c * t.nS + s] = tile[tx][j];
    }
}

// Signed row gather: row r of the output (nS states) is sign * row |e| - 1
// of zT for e = tab[r], zero for e = 0.  A wave copies 64 / SP rows at a time
// (SP = nS rounded up to a power of two, at most 64; lanes (row, s)), so
// every row is one contiguous read and one contiguous write, and
// GATHER_ROWS such sets are in flight: all table entries are loaded, then all
// source rows, then all are stored.  Bound by HBM writes: with one set in
// flight (one dependent table and row load per store) it wrote 2.0 TB/s on
// 630 x 7140 rows of 64 states.
// blockIdx.y picks the side: both factors of a density in one launch.  Element
// (configuration c, state s) of the coefficients is z[c * sC + s * sS].
#define GATHER_ROWS 4
struct GatherSide {
    const int32_t* tab;
    const double* z;
    double* out;
    int64_t rows, nS, sC, sS;
};
template <int SP>
__global__ __launch_bounds__(256) void k_gather_rows(GatherSide g0, GatherSide g1) {
    constexpr int RPW = 64 / SP;                 // rows per wave and set
    const GatherSide S = blockIdx.y ? g1 : g0;
    const int lane = threadIdx.x & 63;
    const int sub = lane / SP, s0 = lane % SP;
    const int64_t wave = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (RPW * GATHER_ROWS);
    const int64_t step = (int64_t)gridDim.x * 4 * (RPW * GATHER_ROWS);
    for (int64_t r0 = wave; r0 < S.rows; r0 += step) {
        int32_t e[GATHER_ROWS];
#pragma unroll
        for (int g = 0; g < GATHER_ROWS; g++) {
            const int64_t r = r0 + g * RPW + sub;
            e[g] = r < S.rows ? S.tab[r] : 0;
        }
        for (int64_t s = s0; s < S.nS; s += SP) {
            double v[GATHER_ROWS];
#pragma unroll
            for (int g = 0; g < GATHER_ROWS; g++) {
                const int32_t a = e[g] > 0 ? e[g] : -e[g];
                v[g] = a ? S.z[(int64_t)(a - 1) * S.sC + s * S.sS] : 0.0;
            }
#pragma unroll
            for (int g = 0; g < GATHER_ROWS; g++) {
                const int64_t r = r0 + g * RPW + sub;
                if (r < S.rows) S.out[r * S.nS + s] = e[g] < 0 ? -v[g] : v[g];
            }
        }
    }
}


// For each flat index (d_0 ... d_{k-1}) in [0, dim^k): the lexical rank of
// the sorted tuple and the parity of the sort, as sign * (rank + 1); 0 if an
// index repeats.
__device__ __forceinline__ void k_index_table_elem(int64_t i, int k, int dim, int64_t n, int32_t* tab) {
    int d[3];
    int64_t x = i;
    for (int j = k - 1; j >= 0; j--) {
        d[j] = (int)(x % dim);
        x /= dim;
    }
    int inv = 0;
    uint64_t m = 0;
    for (int a = 0; a < k; a++) {
        for (int b = a + 1; b < k; b++) {
            if (d[a] == d[b]) { tab[i] = 0; return; }
            if (d[a] > d[b]) inv++;
        }
        m |= 1ull << d[a];
    }
    int32_t r = (int32_t)d_lex_rank(m, dim);
    tab[i] = ((inv & 1) ? -1 : 1) * (r + 1);
}

__global__ void k_index_table(int k, int dim, int64_t n, int32_t* tab) {
    XR_GRID_STRIDE(i, n) k_index_table_elem(i, k, dim, n, tab);
}

// out[((I*nJ + J)*nL + iL)*nR + iR] from the compressed GEMM result
// Cc[(l*nI + I) * ldc + t*nJ + J], through the signed index tables
// tab[i] = sign * (sorted-tuple rank + 1), 0 for a repeated index.
// blockIdx.x walks the (I, J) planes (J fastest, remapped so that each XCD
// takes a contiguous run of planes) and blockIdx.y 1024-element chunks of a
// plane: the blocks in flight on one XCD write contiguous chunks of
// neighbouring planes and read the same Cc rows for consecutive J, so one
// cache line of Cc serves 8 planes in that XCD's L2.  Plane offsets are 32-bit.
__global__ __launch_bounds__(256) void k_expand_planes(
    const double* __restrict__ Cc, int64_t ldc, int64_t nI, int64_t nJ,
    const int32_t* __restrict__ tabL, uint32_t nL, const int32_t* __restrict__ tabR, uint32_t nR,
    double* __restrict__ out) {
    const uint32_t plane = nL * nR;
    const int64_t n_planes = nI * nJ;
    const int64_t lstride = nI * ldc;
    for (int64_t b = blockIdx.x; b < n_planes; b += gridDim.x) {
        const int64_t pl = (b - blockIdx.x) + xcd_remap(blockIdx.x, gridDim.x);
        if (pl >= n_planes) continue;
        const int64_t I = pl / nJ, J = pl - I * nJ;
        const double* src = Cc + I * ldc + J;
        double* dst = out + pl * (int64_t)plane;
        for (uint32_t base = blockIdx.y * 1024u; base < plane; base += gridDim.y * 1024u) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t e = base + k * 256u + threadIdx.x;
                if (e >= plane) break;
                const uint32_t iL = e / nR, iR = e - iL * nR;
                const int32_t eL = tabL ? tabL[iL] : 1;
                const int32_t eR = tabR ? tabR[iR] : 1;
                double v = 0.0;
                if (eL != 0 && eR != 0) {
                    const int64_t l = (eL > 0 ? eL : -eL) - 1, t = (eR > 0 ? eR : -eR) - 1;
                    v = src[l * lstride + t * nJ];
                    if ((eL < 0) != (eR < 0)) v = -v;
                }
                dst[e] = v;
            }
        }
    }
}

// The same expansion turned through LDS: a workgroup takes JB consecutive J
// of one I and LC consecutive left indices iL, reads the Cc rows of those along J
// (JB doubles at a time), and writes LC * nR contiguous doubles of each of
// its planes.  Bound by HBM (8 B written and about 4 read per element); the walk
// plane by plane above reads Cc one 8-byte element per cache line and counts
// on L2 for the other planes' share.  caa, 13 orbitals, 32 x 32 states (17576
// per plane): 100 -> 45 us; 18 orbitals, 64 states: 1.10 -> 0.50 ms.
// nT sorted right tuples; LDS rows of ntp (odd) doubles.
template <int JB>
__global__ __launch_bounds__(256) void k_expand_tile(
    const double* __restrict__ Cc, int64_t ldc, int64_t nI, int64_t nJ, const int32_t* __restrict__ tabL, int nL,
    const int32_t* __restrict__ tabR, int nR, int nT, int ntp, int LC, double* __restrict__ out) {
    extern __shared__ double T[];              // [c][j][t]
    const int jb = (int)((nJ + JB - 1) / JB);
    const int64_t I = blockIdx.x / jb, J0 = (int64_t)(blockIdx.x - I * jb) * JB;
    const int iL0 = blockIdx.y * LC, lc = nL - iL0 < LC ? nL - iL0 : LC;
    const int tid = threadIdx.x;
    {
        const int j = tid % JB, t0 = tid / JB;
        const int64_t J = J0 + j < nJ ? J0 + j : nJ - 1;
        for (int c = 0; c < lc; c++) {
            const int eL = tabL ? tabL[iL0 + c] : 1;
            if (eL == 0) continue;
            const double* src = Cc + (int64_t)((eL > 0 ? eL : -eL) - 1) * nI * ldc + I * ldc + J;
            double* dst = T + (c * JB + j) * ntp;
#pragma unroll 4
            for (int t = t0; t < nT; t += 256 / JB) {
                const double v = src[(int64_t)t * nJ];
                dst[t] = eL < 0 ? -v : v;
            }
        }
    }
    __syncthreads();
    const int len = lc * nR;
    for (int x = tid; x < len; x += 256) {
        const int c = x / nR, iR = x - c * nR;
        const int eL = tabL ? tabL[iL0 + c] : 1, eR = tabR ? tabR[iR] : 1;
        const int t = (eR > 0 ? eR : -eR) - 1;
        const double* src = T + c * JB * ntp + (t < 0 ? 0 : t);
        double* dst = out + (I * nJ + J0) * (int64_t)nL * nR + (int64_t)iL0 * nR + x;
#pragma unroll
        for (int j = 0; j < JB; j++) {
            if (J0 + j >= nJ) break;
            double v = 0.0;
            if (eL != 0 && eR != 0) v = eR < 0 ? -src[j * ntp] : src[j * ntp];
            dst[(int64_t)j * nL * nR] = v;
        }
    }
}

// Veff[u, w] for pairs u = (p<q), w = (a<b) in spin-class order:
//   V[p,q,b,a] - V[q,p,b,a] - V[p,q,a,b] + V[q,p,a,b]
// (rows of ld >= nU doubles, the padding zero).  h (or null): adds the
// one-body part as a two-body one on states of N electrons, hs = 1 / (N - 1):
//   hs (h[p,b] d(q,a) - h[p,a] d(q,b) - h[q,b] d(p,a) + h[q,a] d(p,b)),
// from h_xy c_x a_y = hs sum_z h_xy c_x c_z a_z a_y there.
// transposed: Ve holds Veff[w, u] instead.
// off (or null): set to 1 when an element between two spin classes is not zero.
__global__ void k_veff(const double* __restrict__ V, const double* __restrict__ h, double hs, int dim, int64_t nU,
                       int64_t ld, int transposed, double* __restrict__ Ve, int* __restrict__ off) {
    const int64_t D = dim;
    const int n = dim / 2;
    XR_GRID_STRIDE(i, nU * ld) {
        const int64_t u = i / ld, w = i - u * ld;
        if (w >= nU) { Ve[i] = 0.0; continue; }
        int p, q, a, b;
        pair_at((int)(transposed ? w : u), n, &p, &q);
        pair_at((int)(transposed ? u : w), n, &a, &b);
        auto at = [&](int64_t x0, int64_t x1, int64_t x2, int64_t x3) {
            return V[((x0 * D + x1) * D + x2) * D + x3];
        };
        double v = at(p, q, b, a) - at(q, p, b, a) - at(p, q, a, b) + at(q, p, a, b);
        if (h) {
            double o = 0.0;
            if (q == a) o += h[p * D + b];
            if (q == b) o -= h[p * D + a];
            if (p == a) o -= h[q * D + b];
            if (p == b) o += h[q * D + a];
            v += hs * o;
        }
        Ve[i] = v;
        if (off && v != 0.0 && pair_class((int)u, n) != pair_class((int)w, n)) *off = 1;
    }
}

__global__ void k_set_int(int* p, int v) { *p = v; }

static inline int64_t even_up(int64_t n) { return n + (n & 1); }

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
int xr_space_masks(xr_ctx* c, int n_orbs, int n_core, int n_elec, const uint64_t** masks,
                   int64_t* n) {
    auto key = std::make_pair(n_orbs * 1024 + n_core, n_elec);
    auto it = c->kspace.find(key);
    if (it != c->kspace.end()) {
        *masks = it->second.first;
        *n = it->second.second;
        return XR_OK;
    }
    int64_t cnt = h_binom(2 * (n_orbs - n_core), n_elec - 2 * n_core);
    if (cnt <= 0) return xr_fail(c, XR_EINVAL, "empty determinant space");
    uint64_t* p = nullptr;
    XR_HIP(c, hipMalloc(&p, cnt * sizeof(uint64_t)));
    k_unrank_space<<<xr_grid(cnt), 256, 0, c->stream>>>(p, cnt, n_orbs, n_core, n_elec);
    XR_LAUNCH_CHECK(c);
    c->kspace[key] = std::make_pair(p, cnt);
    *masks = p;
    *n = cnt;
    return XR_OK;
}

// Coefficients as a gather reads them: the stored (n_states x n_configs)
// array, or a copy with the state index fastest.
struct Coeffs { const double* z; int64_t sC, sS; };

// Up to this many bytes of coefficients are gathered as they are stored, which
// saves the transposing launch: ca of 9 orbitals, 3 electrons, 8 x 8 states, 18.9 us
// with it, 15.8 without (both gathers in one launch save 0.4 us of that, within the spread).
#define GATHER_DIRECT_BYTES (1 << 20)

// The two blocks' coefficients for a gather, those of size > GATHER_DIRECT_BYTES
// transposed (one launch; one copy for a block with itself).  A null z is not wanted.
static int coeffs_for_gather(xr_ctx* c, int slot0, int slot1, int64_t nI, int64_t nP, const double* zbra, int64_t nJ,
                             int64_t nQ, const double* zket, Coeffs* b, Coeffs* k) {
    const bool same = zbra && zbra == zket && nI == nJ && nP == nQ;
    *b = Coeffs{zbra, 1, nP};
    *k = Coeffs{zket, 1, nQ};
    TransposeSide t[2];
    int n = 0;
    if (zbra && nI * nP * (int64_t)sizeof(double) > GATHER_DIRECT_BYTES) {
        double* zT = (double*)xr_workspace(c, slot0, nP * nI * sizeof(double));
        if (!zT) return xr_fail(c, XR_ENOMEM, "workspace (coefficients)");
        t[n++] = TransposeSide{zbra, zT, nI, nP};
        *b = Coeffs{zT, nI, 1};
    }
    if (same) *k = *b;
    else if (zket && nJ * nQ * (int64_t)sizeof(double) > GATHER_DIRECT_BYTES) {
        double* zT = (double*)xr_workspace(c, slot1, nQ * nJ * sizeof(double));
        if (!zT) return xr_fail(c, XR_ENOMEM, "workspace (coefficients)");
        t[n++] = TransposeSide{zket, zT, nJ, nQ};
        *k = Coeffs{zT, nJ, 1};
    }
    if (n == 0) return XR_OK;
    if (n == 1) t[1] = t[0];
    const dim3 grid((unsigned)ceil_div(std::max(t[0].nC, t[1].nC), 32), (unsigned)ceil_div(std::max(t[0].nS, t[1].nS), 32),
                    (unsigned)n);
    k_transpose<<<grid, dim3(32, 8), 0, c->stream>>>(t[0], t[1]);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// The side table of (sd, K space) depends on the determinant spaces only:
// built on first use and kept for the context's lifetime (*tab; nullptr
// for an empty table).
int xr_side_table(xr_ctx* c, const SidePlan& sd, const uint64_t* Km, int64_t nK, int n_orbs,
                  int n_core, int32_t** tab) {
    int64_t nT = h_binom(2 * n_orbs, sd.k);
    int64_t n = nK * nT;
    *tab = nullptr;
    if (n <= 0) return XR_OK;
    const std::array<int64_t, 12> key{sd.k, sd.is_c, sd.slot[0], sd.slot[1], sd.slot[2],
                                      (int64_t)(uintptr_t)Km, nK, n_orbs, n_core, -1, 0, 0};
    auto it = c->sidetab.find(key);
    if (it != c->sidetab.end()) {
        *tab = it->second.first;
        return XR_OK;
    }
    int32_t* p = nullptr;
    XR_HIP(c, hipMalloc(&p, n * sizeof(int32_t)));
    c->sidetab[key] = std::make_pair(p, n);
    ProfScope prof(c, XR_K_TABLE, 0.0, 4.0 * n);
    k_side_table<<<xr_grid(n), 256, 0, c->stream>>>(sd, Km, nK, 2 * n_orbs, n_orbs, n_core, nT, p);
    XR_LAUNCH_CHECK(c);
    *tab = p;
    return XR_OK;
}

// The pair-major table of a pair string (k_pair_table), kept like the above.
static int pair_table(xr_ctx* c, const SidePlan& sd, const uint64_t* Km, int64_t nK, int n_orbs, int n_core,
                      int32_t** tab) {
    const int64_t nU = even_up(h_binom(2 * n_orbs, 2)), n = nK * nU;
    *tab = nullptr;
    if (n <= 0) return XR_OK;
    const std::array<int64_t, 12> key{sd.k, sd.is_c, sd.slot[0], sd.slot[1], sd.slot[2],
                                      (int64_t)(uintptr_t)Km, nK, n_orbs, n_core, -2, 0, 0};
    auto it = c->sidetab.find(key);
    if (it != c->sidetab.end()) {
        *tab = it->second.first;
        return XR_OK;
    }
    int32_t* p = nullptr;
    XR_HIP(c, hipMalloc(&p, n * sizeof(int32_t)));
    c->sidetab[key] = std::make_pair(p, n);
    ProfScope prof(c, XR_K_TABLE, 0.0, 4.0 * n);
    k_pair_table<<<xr_grid(n), 256, 0, c->stream>>>(sd, Km, nK, 2 * n_orbs, n_orbs, n_core, nU, p);
    XR_LAUNCH_CHECK(c);
    *tab = p;
    return XR_OK;
}

// One or two sides gathered (k_gather_rows): in one launch up to
// GATHER_DIRECT_BYTES of output, where the launch is most of it.  Larger ones go one
// after the other, since two at once share L2: 67 us apart against 72 together (13
// orbitals, 32 states), 692 against 745 (18 orbitals, 64 states).
static int gather(xr_ctx* c, const GatherSide* g, int n) {
    if (n == 2 && (g[0].rows * g[0].nS + g[1].rows * g[1].nS) * (int64_t)sizeof(double) > GATHER_DIRECT_BYTES) {
        const int rc = gather(c, g, 1);
        return rc ? rc : gather(c, g + 1, 1);
    }
    int64_t elems = 0, rows = 0, nS = 1;
    for (int q = 0; q < n; q++) {
        elems += g[q].rows * g[q].nS;
        rows = std::max(rows, g[q].rows);
        nS = std::max(nS, g[q].nS);
    }
    if (elems <= 0) return XR_OK;
    ProfScope prof(c, XR_K_GATHER, 0.0, 8.0 * elems);
    const int sp = nS <= 1 ? 1 : nS <= 2 ? 2 : nS <= 4 ? 4 : nS <= 8 ? 8 : nS <= 16 ? 16 : nS <= 32 ? 32 : 64;
    const dim3 grid(xr_grid(ceil_div(rows, (64 / sp) * GATHER_ROWS) * 64), (unsigned)n);
    const GatherSide &a = g[0], &b = g[n - 1];
    switch (sp) {
    case 1: k_gather_rows<1><<<grid, 256, 0, c->stream>>>(a, b); break;
    case 2: k_gather_rows<2><<<grid, 256, 0, c->stream>>>(a, b); break;
    case 4: k_gather_rows<4><<<grid, 256, 0, c->stream>>>(a, b); break;
    case 8: k_gather_rows<8><<<grid, 256, 0, c->stream>>>(a, b); break;
    case 16: k_gather_rows<16><<<grid, 256, 0, c->stream>>>(a, b); break;
    case 32: k_gather_rows<32><<<grid, 256, 0, c->stream>>>(a, b); break;
    default: k_gather_rows<64><<<grid, 256, 0, c->stream>>>(a, b); break;
    }
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}
static GatherSide gather_side(const int32_t* tab, int64_t rows, const Coeffs& z, int64_t nS, double* out) {
    return GatherSide{tab, z.z, out, rows, nS, z.sC, z.sS};
}

// The signed index table of k indices (k_index_table) depends on (k, dim)
// only: built on first use and kept (nullptr for k = 0).
static int index_table(xr_ctx* c, int k, int dim, const int32_t** tab) {
    *tab = nullptr;
    if (!k) return XR_OK;
    int64_t n = 1;
    for (int j = 0; j < k; j++) n *= dim;
    const std::array<int64_t, 12> key{k, dim, 0, 0, 0, 0, 0, 0, 0, -3, 0, 0};
    auto it = c->sidetab.find(key);
    if (it != c->sidetab.end()) {
        *tab = it->second.first;
        return XR_OK;
    }
    int32_t* p = nullptr;
    XR_HIP(c, hipMalloc(&p, n * sizeof(int32_t)));
    c->sidetab[key] = std::make_pair(p, n);
    k_index_table<<<xr_grid(n), 256, 0, c->stream>>>(k, dim, n, p);
    XR_LAUNCH_CHECK(c);
    *tab = p;
    return XR_OK;
}

static int check_spaces(xr_ctx* c, const OpPlan& pl, int n_orbs, int n_core, int n_elec_ket,
                        int64_t nP, int64_t nQ, int* n_elec_bra) {
    if (n_orbs <= 0 || 2 * n_orbs > XR_MAX_SO) return xr_fail(c, XR_EUNSUPPORTED, "need 0 < 2*n_orbs <= 64");
    if (n_core < 0 || n_core > n_orbs) return xr_fail(c, XR_EINVAL, "bad n_core");
    int nb = n_elec_ket + pl.delta;
    if (n_elec_ket < 2 * n_core || n_elec_ket > 2 * n_orbs || nb < 2 * n_core || nb > 2 * n_orbs)
        return xr_fail(c, XR_EINVAL, "electron counts incompatible with orbitals / core");
    int nval = 2 * (n_orbs - n_core);
    if (nQ != h_binom(nval, n_elec_ket - 2 * n_core))
        return xr_fail(c, XR_ESHAPE, "ket coefficient columns != size of the ket determinant space");
    if (nP != h_binom(nval, nb - 2 * n_core))
        return xr_fail(c, XR_ESHAPE, "bra coefficient columns != size of the bra determinant space");
    if (nP >= 0x7fffffff || nQ >= 0x7fffffff) return xr_fail(c, XR_EUNSUPPORTED, "determinant space >= 2^31");
    *n_elec_bra = nb;
    return XR_OK;
}

// ---------------------------------------------------------------------------
// entry points
// ---------------------------------------------------------------------------
enum { WS_ZTB = 0, WS_ZTK, WS_OFF, WS_X = 4, WS_Y, WS_C, WS_VE = 9, WS_W };
enum { WS_GC = 40, WS_XB, WS_YB, WS_ZBT, WS_WB, WS_VEB, WS_GS };

// The two factors of a density: X (nK x nLt*nI) from the bra coefficients
// and Y (nK x nT*nJ) from the ket coefficients, over the K space that sits
// between L and R: the bra space when there is no L, the ket space when there
// is no R, else every determinant with n_ket - |R| electrons.  Without L
// (R) the factor is the transpose of the coefficients as they are stored: xT
// (yT) says that X (Y) points at those, nI x nK (nJ x nK) with rows of ldx (ldy).
struct Factors {
    const uint64_t* Km = nullptr;
    int64_t nK = 0, nLt = 1, nT = 1;
    int kspace_core = 0;
    const double* X = nullptr;
    const double* Y = nullptr;
    int xT = 0, yT = 0;
    int64_t ldx = 0, ldy = 0;
};

static int prepare_factors(xr_ctx* c, const OpPlan& pl, int n_orbs, int n_core, int n_elec_ket,
                           int nb, int64_t nI, int64_t nP, const double* zbra, int64_t nJ,
                           int64_t nQ, const double* zket, Factors* f) {
    const int dim = 2 * n_orbs;
    int rc;
    f->nT = pl.R.k ? h_binom(dim, pl.R.k) : 1;
    f->nLt = pl.L.k ? h_binom(dim, pl.L.k) : 1;
    f->ldx = f->nLt * nI;
    f->ldy = f->nT * nJ;
    if (!pl.L.k) {
        if ((rc = xr_space_masks(c, n_orbs, n_core, nb, &f->Km, &f->nK))) return rc;
        f->X = zbra;
        f->xT = 1;
        f->ldx = nP;
        f->kspace_core = n_core;
    } else if (!pl.R.k) {
        if ((rc = xr_space_masks(c, n_orbs, n_core, n_elec_ket, &f->Km, &f->nK))) return rc;
        f->Y = zket;
        f->yT = 1;
        f->ldy = nQ;
        f->kspace_core = n_core;
    } else {
        if ((rc = xr_space_masks(c, n_orbs, 0, n_elec_ket - pl.R.k, &f->Km, &f->nK))) return rc;
        f->kspace_core = 0;
    }
    Coeffs cb, ck;
    if ((rc = coeffs_for_gather(c, WS_ZTB, WS_ZTK, nI, nP, pl.L.k ? zbra : nullptr, nJ, nQ,
                                pl.R.k ? zket : nullptr, &cb, &ck)))
        return rc;
    GatherSide g[2];
    int n = 0;
    int32_t *tabL = nullptr, *tabR = nullptr;
    if (pl.L.k) {
        double* Xb = (double*)xr_workspace(c, WS_X, f->nK * f->nLt * nI * sizeof(double));
        if (!Xb) return xr_fail(c, XR_ENOMEM, "workspace (bra gather)");
        if ((rc = xr_side_table(c, pl.L, f->Km, f->nK, n_orbs, n_core, &tabL))) return rc;
        g[n++] = gather_side(tabL, f->nK * f->nLt, cb, nI, Xb);
        f->X = Xb;
    }
    if (pl.R.k) {
        if ((rc = xr_side_table(c, pl.R, f->Km, f->nK, n_orbs, n_core, &tabR))) return rc;
        if (pl.L.k && tabR == tabL && zbra == zket && nI == nJ && nP == nQ) {
            f->Y = f->X;                    // a block with itself through one table: the same factor
        } else {
            double* Yb = (double*)xr_workspace(c, WS_Y, f->nK * f->nT * nJ * sizeof(double));
            if (!Yb) return xr_fail(c, XR_ENOMEM, "workspace (ket gather)");
            g[n++] = gather_side(tabR, f->nK * f->nT, ck, nJ, Yb);
            f->Y = Yb;
        }
    }
    return n ? gather(c, g, n) : XR_OK;
}

int xr_density_impl(xr_ctx* c, const char* ops, int n_orbs, int n_core, int n_elec_ket,
                    int64_t nI, int64_t nP, const double* zbra, int64_t nJ, int64_t nQ,
                    const double* zket, double* out) {
    OpPlan pl;
    if (!xr_plan_op(ops, &pl)) return xr_fail(c, XR_EUNSUPPORTED, std::string("operator string not supported: ") + (ops ? ops : "(null)"));
    int nb = 0;
    int rc = check_spaces(c, pl, n_orbs, n_core, n_elec_ket, nP, nQ, &nb);
    if (rc) return rc;
    const int dim = 2 * n_orbs;
    if (nI <= 0 || nJ <= 0) return XR_OK;
    int64_t out_size = nI * nJ;
    for (int j = 0; j < pl.k; j++) out_size *= dim;
    if (pl.L.k && pl.R.k && (n_elec_ket - pl.R.k < 0))  // R annihilates more electrons than the ket has
        return xr_fill(c, out, out_size, 0.0);
    Factors f;
    if ((rc = prepare_factors(c, pl, n_orbs, n_core, n_elec_ket, nb, nI, nP, zbra, nJ, nQ, zket, &f)))
        return rc;
    const int64_t Mg = f.nLt * nI, Ng = f.nT * nJ;
    double* Cc = (double*)xr_workspace(c, WS_C, Mg * Ng * sizeof(double));
    if (!Cc) return xr_fail(c, XR_ENOMEM, "workspace (compressed density)");
    if (f.X == f.Y && Mg == Ng && Mg > 512) {
        // a block with itself through one factor: Cc = X^T X is symmetric (a
        // small one is bound by launches, and the mirror is one more)
        if ((rc = xr_dgemm_syrk_tn(c, Mg, f.nK, 1.0, f.X, Mg, Cc, Ng))) return rc;
    } else if ((rc = xr_dgemm_launch(c, f.xT ? 0 : 1, f.yT, Mg, Ng, f.nK, 1.0, f.X, f.ldx, 0, f.Y, f.ldy, 0, 0.0, Cc,
                                     Ng, 0, 1))) {
        return rc;
    }
    int64_t nIL = 1, nIR = 1;
    for (int j = 0; j < pl.L.k; j++) nIL *= dim;
    for (int j = 0; j < pl.R.k; j++) nIR *= dim;
    const int32_t *idxL = nullptr, *idxR = nullptr;
    if ((rc = index_table(c, pl.L.k, dim, &idxL)) || (rc = index_table(c, pl.R.k, dim, &idxR))) return rc;
    int64_t total = nI * nJ * nIL * nIR;
    ProfScope prof(c, XR_K_EXPAND, 0.0, 8.0 * total);
    if (nIL * nIR > 0xffffffffLL - 65536LL * 1024) return xr_fail(c, XR_EUNSUPPORTED, "density plane too large");
    // through LDS where a tile of JB planes and at least one left index fits
    // in 48 KB (64 KB for JB = 8); triples on the right (nT > 1000) go plane by plane
    const int ntp = (int)(f.nT | 1);
    const int JB = nJ > 8 && 16 * ntp * 8 <= (48 << 10) ? 16 : 8;
    if ((int64_t)JB * ntp * 8 <= (64 << 10) && nIL * nIR < (1LL << 30)) {
        const int64_t gx = nI * ceil_div(nJ, JB);
        int64_t lc = std::max<int64_t>(1, (48 << 10) / ((int64_t)JB * ntp * 8));
        lc = std::min(lc, std::max<int64_t>(1, nIL * gx / 512));     // enough workgroups first
        lc = std::min(lc, nIL);
        const int64_t gy = ceil_div(nIL, lc);
        if (gx <= 0x7fffffffLL && gy <= 65535) {
            const dim3 grid((unsigned)gx, (unsigned)gy);
            const size_t lds = (size_t)lc * JB * ntp * 8;
            if (JB == 16)
                k_expand_tile<16><<<grid, 256, lds, c->stream>>>(Cc, Ng, nI, nJ, idxL, (int)nIL, idxR, (int)nIR,
                                                                 (int)f.nT, ntp, (int)lc, out);
            else
                k_expand_tile<8><<<grid, 256, lds, c->stream>>>(Cc, Ng, nI, nJ, idxL, (int)nIL, idxR, (int)nIR,
                                                                (int)f.nT, ntp, (int)lc, out);
            XR_LAUNCH_CHECK(c);
            return XR_OK;
        }
    }
    const int64_t planes = nI * nJ;
    const int64_t chunks = ceil_div(nIL * nIR, 1024);
    dim3 grid((unsigned)(planes < (1LL << 30) ? planes : (1LL << 30)),
              (unsigned)(chunks < 65535 ? chunks : 65535));
    k_expand_planes<<<grid, 256, 0, c->stream>>>(Cc, Ng, nI, nJ, idxL, (uint32_t)nIL, idxR,
                                                 (uint32_t)nIR, out);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

extern "C" int xr_density(xr_ctx* c, const char* ops, int n_orbs, int n_core, int n_elec_ket,
                          int64_t nI, int64_t nP, const double* zbra, int64_t nJ, int64_t nQ,
                          const double* zket, double* out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    return xr_density_impl(c, ops, n_orbs, n_core, n_elec_ket, nI, nP, zbra, nJ, nQ, zket, out);
}

// The pair matrix Ve (rows padded to an even length Kp; transposed: Veff^T)
// and the product W = Ve Y of the two-electron terms, Y (Kp x N, the pairs
// in spin-class order, its padding row zero).
//
// With h (the FCI sigma) the product is FP64 in every precision mode: the
// matrix then carries the one-electron term, which the split modes leave
// in FP64, and which being the larger part would also set the split's grids.
//
// In FP64 a product of at least VEFF_CLASS_FLOPS runs one problem per spin
// class, each over its own class's rows of Y when k_veff found no element
// between classes (on the device: the host does not wait): integrals that
// conserve the spin projection then cost (2 aa^2 + ab^2) / nU^2 = 0.385 of the dense
// product (aa, ab pairs of a class).  18 orbitals, 64 states, 5 electrons (630 x 457k x 630): 5.5 -> 3.0 ms.
// Smaller products are bound by launches and run dense in one.
#define VEFF_CLASS_FLOPS 5e8
static int veff_product(xr_ctx* c, const double* V, const double* h, double hs, int dim, bool transposed,
                        const double* Y, int64_t N, double* W) {
    const int64_t nU = h_binom(dim, 2), Kp = even_up(nU);
    const int64_t n = dim / 2, aa = n * (n - 1) / 2;
    double* Ve = (double*)xr_workspace(c, WS_VE, nU * Kp * sizeof(double));
    int* off = (int*)xr_workspace(c, WS_OFF, 256);
    if (!Ve || !off) return xr_fail(c, XR_ENOMEM, "workspace (pair matrix)");
    const bool f64 = h || c->precision == XR_PREC_F64;
    const bool classes = f64 && 2.0 * nU * nU * N >= VEFF_CLASS_FLOPS;
    if (classes) {
        k_set_int<<<1, 1, 0, c->stream>>>(off, 0);
        XR_LAUNCH_CHECK(c);
    }
    k_veff<<<xr_grid(nU * Kp), 256, 0, c->stream>>>(V, h, hs, dim, nU, Kp, transposed ? 1 : 0, Ve,
                                                   classes ? off : nullptr);
    XR_LAUNCH_CHECK(c);
    if (!classes)
        return (f64 ? xr_dgemm_launch : xr_gemm_2e)(c, 0, 0, nU, N, Kp, 1.0, Ve, Kp, 0, Y, N, 0, 0.0, W, N, 0, 1);
    const int64_t row[4] = {0, aa, aa + n * n, nU};
    return xr_dgemm_blocks(c, 3, row, Kp, N, Ve, Kp, Y, N, W, N, off);
}

// Wkeep: caller's buffer for W = Veff Y (nU * nK * nJ doubles, w_len), which
// the adjoint can take instead of recomputing it; nullptr: a workspace.
static int monomer_2e_impl(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI, int64_t nP,
                           const double* zbra, int64_t nJ, int64_t nQ, const double* zket,
                           const double* V, double* out, double* Wkeep, int64_t w_len) {
    OpPlan pl;
    xr_plan_op("ccaa", &pl);
    int nb = 0;
    int rc = check_spaces(c, pl, n_orbs, n_core, n_elec, nP, nQ, &nb);
    if (rc) return rc;
    if (nI <= 0 || nJ <= 0) return XR_OK;
    const int dim = 2 * n_orbs;
    if (n_elec < 2) return xr_fill(c, out, nI * nJ, 0.0);
    Coeffs cb, ck;
    if ((rc = coeffs_for_gather(c, WS_ZTB, WS_ZTK, nI, nP, zbra, nJ, nQ, zket, &cb, &ck))) return rc;
    const uint64_t* Km = nullptr;
    int64_t nK = 0;
    if ((rc = xr_space_masks(c, n_orbs, 0, n_elec - 2, &Km, &nK))) return rc;
    const int64_t nU = h_binom(dim, 2), Kp = even_up(nU);
    int32_t *tabL = nullptr, *tabR = nullptr;
    // a block with itself: the two sides' tables differ only by the order of
    // the two annihilators, so X = sg Y and one gather serves both
    const double sg = (pl.L.slot[0] == pl.R.slot[0]) ? 1.0 : -1.0;
    const bool same = zbra == zket && nI == nJ && nP == nQ;
    if (Wkeep && w_len != nU * nK * nJ) return xr_fail(c, XR_ESHAPE, "sigma factor buffer size");
    double* X = same ? nullptr : (double*)xr_workspace(c, WS_X, nU * nK * nI * sizeof(double));
    double* Y = (double*)xr_workspace(c, WS_Y, Kp * nK * nJ * sizeof(double));
    double* W = Wkeep ? Wkeep : (double*)xr_workspace(c, WS_W, nU * nK * nJ * sizeof(double));
    if ((!same && !X) || !Y || !W) return xr_fail(c, XR_ENOMEM, "workspace (sigma)");
    if ((rc = pair_table(c, pl.R, Km, nK, n_orbs, n_core, &tabR))) return rc;
    if (!same && (rc = pair_table(c, pl.L, Km, nK, n_orbs, n_core, &tabL))) return rc;
    GatherSide g[2] = {gather_side(tabR, Kp * nK, ck, nJ, Y), GatherSide()};     // Y[w][K][J]
    if (!same) g[1] = gather_side(tabL, nU * nK, cb, nI, X);                     // X[u][K][I]
    if ((rc = gather(c, g, same ? 1 : 2))) return rc;
    // W[u][K*nJ + J] = sum_w Ve[u,w] Y[w][K*nJ + J]
    if ((rc = veff_product(c, V, nullptr, 0.0, dim, false, Y, nK * nJ, W))) return rc;
    // E[I,J] = sum_{(u,K)} X[(u,K), I] W[(u,K), J]
    return xr_gemm_2e(c, 1, 0, nI, nJ, nU * nK, same ? sg : 1.0, same ? Y : X, nI, 0, W, nJ, 0, 0.0, out, nJ, 0, 1);
}

extern "C" int xr_monomer_2e(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI, int64_t nP,
                             const double* zbra, int64_t nJ, int64_t nQ, const double* zket,
                             const double* V, double* out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    return monomer_2e_impl(c, n_orbs, n_core, n_elec, nI, nP, zbra, nJ, nQ, zket, V, out, nullptr, 0);
}

extern "C" int xr_monomer_2e_keep(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI, int64_t nP,
                                  const double* zbra, int64_t nJ, int64_t nQ, const double* zket,
                                  const double* V, double* out, double* W, int64_t w_len) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (!W) return xr_fail(c, XR_EINVAL, "null sigma factor buffer");
    return monomer_2e_impl(c, n_orbs, n_core, n_elec, nI, nP, zbra, nJ, nQ, zket, V, out, W, w_len);
}

// ---------------------------------------------------------------------------
// adjoints
// ---------------------------------------------------------------------------
// Orbitals of the lexicographic k-tuple of rank r (ascending).
__device__ __forceinline__ void tuple_orbs(int64_t r, int dim, int k, int* o) {
    if (!k) return;
    uint64_t m = d_lex_unrank(r, dim, k);
    for (int j = 0; j < k; j++) { o[j] = __ffsll((unsigned long long)m) - 1; m &= m - 1; }
}

// Sum over the index orderings of the sorted tuples lo (kL) and ro (kR) of
// sign * plane[iL * nIR + iR].
__device__ __forceinline__ double compress_sum(const double* __restrict__ plane, const int* lo, const int* ro,
                                               int kL, int kR, int dim, int64_t nIR) {
    const int P3[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
    const int S3[6] = {1, -1, -1, 1, 1, -1};
    const int P2[2][3] = {{0, 1, 0}, {1, 0, 0}};
    const int S2[2] = {1, -1};
    const int nPL = kL == 3 ? 6 : (kL == 2 ? 2 : 1);
    const int nPR = kR == 3 ? 6 : (kR == 2 ? 2 : 1);
    double acc = 0.0;
    for (int a = 0; a < nPL; a++) {
        int64_t iL = 0;
        for (int j = 0; j < kL; j++) iL = iL * dim + lo[kL == 3 ? P3[a][j] : (kL == 2 ? P2[a][j] : 0)];
        const int sL = kL == 3 ? S3[a] : (kL == 2 ? S2[a] : 1);
        for (int b = 0; b < nPR; b++) {
            int64_t iR = 0;
            for (int j = 0; j < kR; j++) iR = iR * dim + ro[kR == 3 ? P3[b][j] : (kR == 2 ? P2[b][j] : 0)];
            const int sR = kR == 3 ? S3[b] : (kR == 2 ? S2[b] : 1);
            acc += (double)(sL * sR) * plane[iL * nIR + iR];
        }
    }
    return acc;
}

// Transpose of k_expand: Gc[(l*nI + I) * ldc + t*nJ + J] = sum over the index
// orderings of l and t of sign * Rbar[I, J, iL, iR].  Rbar is read along t
// inside one (I, J) plane and Gc written along J: a workgroup takes 32
// consecutive J by 32 consecutive t for one (l, I) and turns the tile
// through LDS.  blockIdx.x = (I, J tile), blockIdx.y = l, blockIdx.z = t tile.
__global__ __launch_bounds__(256) void k_compress(
    const double* __restrict__ Rbar, int64_t nI, int64_t nJ, int kL, int kR, int dim, int64_t nT,
    double* __restrict__ Gc, int64_t ldc) {
    __shared__ double tile[32][33];
    const int64_t jt = (nJ + 31) / 32;
    const int64_t I = blockIdx.x / jt, J0 = (blockIdx.x - I * jt) * 32;
    const int64_t l = blockIdx.y, t0 = (int64_t)blockIdx.z * 32;
    int64_t nIL = 1, nIR = 1;
    for (int j = 0; j < kL; j++) nIL *= dim;
    for (int j = 0; j < kR; j++) nIR *= dim;
    int lo[3] = {0, 0, 0}, ro[3] = {0, 0, 0};
    tuple_orbs(l, dim, kL, lo);
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int64_t t = t0 + tx;
    if (t < nT) tuple_orbs(t, dim, kR, ro);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int jj = ty + 8 * q;
        const int64_t J = J0 + jj;
        if (t < nT && J < nJ)
            tile[jj][tx] = compress_sum(Rbar + (I * nJ + J) * nIL * nIR, lo, ro, kL, kR, dim, nIR);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int tt = ty + 8 * q;
        const int64_t J = J0 + tx;
        if (t0 + tt < nT && J < nJ) Gc[(l * nI + I) * ldc + (t0 + tt) * nJ + J] = tile[tx][tt];
    }
}

// Transpose of k_gather through the side table: for each source determinant
// S (state space, mask Sm[S]) and state s,
//   zbar[S, s] = sum_t sign(K, t) * Ybar[K(S,t), t, s]
// where t runs over the tuples the side string removes from S (annihilators)
// or adds to it (creators), and K is their image in the K space.  Each
// output is owned by one thread: deterministic, no atomics.
// One (tuple of K ascending orbitals o[0] < o[1] < o[2]) term of the side
// adjoint: sign of applying the string (slot order) to src, K's rank, t's rank.
// Encoded as sign * (row + 1) with row the Ybar row (K, t) in the given
// layout (0: [K][t], 2: [t][K] for pairs t in spin-class order), 0 where K
// falls outside the K space.
template <int K>
__device__ __forceinline__ int64_t side_code(const SidePlan& sd, uint64_t src, const int* o, int n_orbs,
                                            uint64_t kcore, int kspace_core, int nK_val, int dim,
                                            int64_t nK, int64_t nT, int layout) {
    uint64_t tm = 0;
#pragma unroll
    for (int j = 0; j < K; j++) tm |= 1ull << o[j];
    const uint64_t km = sd.is_c ? (src | tm) : (src & ~tm);
    if ((km & kcore) != kcore) return 0;
    uint64_t cur = src;
    int sg = 1;
#pragma unroll
    for (int j = K - 1; j >= 0; j--) {
        const int sl = sd.slot[j];
        const int oo = (sl == 0) ? o[0] : ((sl == 1) ? o[1 < K ? 1 : 0] : o[2 < K ? 2 : 0]);
        sg *= d_sign_above(cur, oo);
        cur ^= 1ull << oo;
    }
    const int64_t Kr = d_lex_rank(d_to_valence(km, n_orbs, kspace_core), nK_val);
    const int64_t t = layout == 2 ? pair_pos(o[0], o[1], n_orbs) : d_lex_rank(tm, dim);
    const int64_t row = layout == 0 ? Kr * nT + t : t * nK + Kr;
    return sg * (row + 1);
}

template <int K>
__device__ __forceinline__ double side_term(const SidePlan& sd, uint64_t src, const int* o, int n_orbs,
                                            uint64_t kcore, int kspace_core, int nK_val, int dim,
                                            int64_t nK, int64_t nT, const double* __restrict__ Ybar,
                                            int64_t nS, int64_t s, int layout) {
    const int64_t e = side_code<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, layout);
    if (!e) return 0.0;
    const double y = Ybar[((e > 0 ? e : -e) - 1) * nS + s];
    return e > 0 ? y : -y;
}

// The codes of side_code for every source determinant S and tuple j (in the
// enumeration order of k_side_adjoint): tab[S * nTup + j].  One thread per S.
template <int K>
__global__ void k_side_index(SidePlan sd, const uint64_t* __restrict__ Sm, int64_t nS_cfg, int n_orbs,
                             int kspace_core, int64_t nK, int64_t nT, int layout, int64_t nTup,
                             int32_t* __restrict__ tab) {
    XR_GRID_STRIDE(S, nS_cfg) {
        const int dim = 2 * n_orbs;
        const uint64_t src = Sm[S];
        const uint64_t full = (dim >= 64) ? ~0ull : ((1ull << dim) - 1);
        const uint64_t pool = sd.is_c ? (~src & full) : src;
        const uint64_t kcore = d_core_mask(n_orbs, kspace_core);
        const int nK_val = dim - 2 * kspace_core;
        int32_t* out = tab + S * nTup;
        int64_t j = 0;
        int o[3] = {0, 0, 0};
        for (uint64_t p1 = pool; p1; p1 &= p1 - 1) {
            o[0] = __ffsll((unsigned long long)p1) - 1;
            if (K == 1) {
                if (j < nTup) out[j++] = (int32_t)side_code<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, layout);
                continue;
            }
            for (uint64_t p2 = p1 & (p1 - 1); p2; p2 &= p2 - 1) {
                o[1] = __ffsll((unsigned long long)p2) - 1;
                if (K == 2) {
                    if (j < nTup) out[j++] = (int32_t)side_code<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, layout);
                    continue;
                }
                for (uint64_t p3 = p2 & (p2 - 1); p3; p3 &= p3 - 1) {
                    o[2] = __ffsll((unsigned long long)p3) - 1;
                    if (j < nTup) out[j++] = (int32_t)side_code<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, layout);
                }
            }
        }
        for (; j < nTup; j++) out[j] = 0;
    }
}

// zbarT[S, s] = sum_j sign_j Ybar[row_j, s] over the tuples of S, in the
// tuple order of k_side_adjoint (same sums, same order); the codes of one S
// are shared by the lanes of its states.
__global__ __launch_bounds__(256) void k_side_adjoint_tab(const int32_t* __restrict__ tab, int64_t nS_cfg,
                                                          int64_t nTup, const double* __restrict__ Ybar,
                                                          int64_t nS, double* __restrict__ zbarT) {
    XR_GRID_STRIDE(i, nS_cfg * nS) {
        const int64_t S = i / nS, s = i - S * nS;
        const int32_t* e = tab + S * nTup;
        double acc = 0.0;
#pragma unroll 8
        for (int64_t j = 0; j < nTup; j++) {
            const int32_t v = e[j];
            if (v) {
                const double y = Ybar[(int64_t)((v > 0 ? v : -v) - 1) * nS + s];
                acc += v > 0 ? y : -y;
            }
        }
        zbarT[i] = acc;
    }
}

// Each output (S, s) is owned by one thread (deterministic, no atomics); the
// state index s is fastest, so the threads of a wave share S and walk the
// same tuples in lockstep while reading consecutive s.  Tuples are
// enumerated as nested ascending bit loops over the orbitals the string may
// touch, in the lexicographic order of (o[0], o[1], o[2]).
template <int K>
__global__ void k_side_adjoint(SidePlan sd, const uint64_t* __restrict__ Sm, int64_t nS_cfg,
                               int n_orbs, int n_core, int kspace_core, int64_t nK, int64_t nT,
                               const double* __restrict__ Ybar, int64_t nS, int layout,
                               double* __restrict__ zbarT) {
    XR_GRID_STRIDE(i, nS_cfg * nS) {
        const int dim = 2 * n_orbs;
        const int64_t S = i / nS, s = i - (i / nS) * nS;
        const uint64_t src = Sm[S];
        const uint64_t full = (dim >= 64) ? ~0ull : ((1ull << dim) - 1);
        const uint64_t pool = sd.is_c ? (~src & full) : src;
        const uint64_t kcore = d_core_mask(n_orbs, kspace_core);
        const int nK_val = dim - 2 * kspace_core;
        double acc = 0.0;
        int o[3] = {0, 0, 0};
        for (uint64_t p1 = pool; p1; p1 &= p1 - 1) {
            o[0] = __ffsll((unsigned long long)p1) - 1;
            if (K == 1) {
                acc += side_term<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, Ybar, nS, s, layout);
                continue;
            }
            for (uint64_t p2 = p1 & (p1 - 1); p2; p2 &= p2 - 1) {
                o[1] = __ffsll((unsigned long long)p2) - 1;
                if (K == 2) {
                    acc += side_term<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, Ybar, nS, s, layout);
                    continue;
                }
                for (uint64_t p3 = p2 & (p2 - 1); p3; p3 &= p3 - 1) {
                    o[2] = __ffsll((unsigned long long)p3) - 1;
                    acc += side_term<K>(sd, src, o, n_orbs, kcore, kspace_core, nK_val, dim, nK, nT, Ybar, nS, s, layout);
                }
            }
        }
        zbarT[S * nS + s] = acc;
    }
}

// zbar[s * nC + c] += zbarT[c * nS + s] (= without add)
__global__ void k_add_transpose(const double* __restrict__ zT, int64_t nS, int64_t nC,
                                double* __restrict__ z, int add) {
    __shared__ double tile[32][33];
    int64_t c0 = (int64_t)blockIdx.x * 32, s0 = (int64_t)blockIdx.y * 32;
    int tx = threadIdx.x, ty = threadIdx.y;
    for (int j = ty; j < 32; j += 8) {
        int64_t c = c0 + j, s = s0 + tx;
        if (s < nS && c < nC) tile[j][tx] = zT[c * nS + s];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {
        int64_t s = s0 + j, c = c0 + tx;
        if (s < nS && c < nC) z[s * nC + c] = add ? z[s * nC + c] + tile[tx][j] : tile[tx][j];
    }
}

// S = G + G^T for a square n x n matrix (32 x 32 tiles, the transposed tile
// through LDS).
__global__ void k_sym_sum(const double* __restrict__ G, int64_t n, double* __restrict__ S) {
    __shared__ double tile[32][33];
    const int64_t c0 = (int64_t)blockIdx.x * 32, r0 = (int64_t)blockIdx.y * 32;
    const int tx = threadIdx.x, ty = threadIdx.y;
    for (int j = ty; j < 32; j += 8) {            // tile[j][tx] = G[c0 + j][r0 + tx]
        const int64_t r = c0 + j, col = r0 + tx;
        if (r < n && col < n) tile[j][tx] = G[r * n + col];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {            // S[r0 + j][c0 + tx] = G[r0 + j][c0 + tx] + G[c0 + tx][r0 + j]
        const int64_t r = r0 + j, col = c0 + tx;
        if (r < n && col < n) S[r * n + col] = G[r * n + col] + tile[tx][j];
    }
}

// Whether the scratch of a call's side adjoints, na and nb elements, is there
// (the larger serves both).
static bool side_scratch(xr_ctx* c, int64_t na, int64_t nb) {
    const int64_t n = std::max(na, nb);
    return n == 0 || xr_workspace(c, WS_ZBT, n * sizeof(double));
}

static int side_adjoint(xr_ctx* c, const SidePlan& sd, int n_orbs, int n_core, int kspace_core,
                        int n_elec_src, int64_t nK, int64_t nT, const double* Ybar, int64_t nS,
                        int layout, double* zbar, bool add = true) {
    const uint64_t* Sm = nullptr;
    int64_t nS_cfg = 0;
    int rc;
    if (sd.k < 1 || sd.k > 3) return xr_fail(c, XR_EINVAL, "side string of 1 to 3 operators expected");
    if ((rc = xr_space_masks(c, n_orbs, n_core, n_elec_src, &Sm, &nS_cfg))) return rc;
    int64_t n = nS_cfg * nS;
    // index table of the (S, tuple) terms: built once per side string and
    // spaces, then every call is a signed gather-sum
    const int dim = 2 * n_orbs;
    const int64_t pool = sd.is_c ? dim - n_elec_src : n_elec_src;
    const int64_t nTup = h_binom((int)pool, sd.k);
    const std::array<int64_t, 12> key{sd.k, sd.is_c, sd.slot[0], sd.slot[1], sd.slot[2], n_orbs, n_core,
                                      kspace_core, n_elec_src, layout, nK, nT};
    int32_t* tab = nullptr;
    auto it = c->sidetab.find(key);
    if (it != c->sidetab.end()) {
        tab = it->second.first;
    } else if (nK * nT < 0x7fffffffLL && nS_cfg * nTup > 0 && nS_cfg * nTup <= (1LL << 28)) {
        XR_HIP(c, hipMalloc(&tab, nS_cfg * nTup * sizeof(int32_t)));
        c->sidetab[key] = std::make_pair(tab, nS_cfg * nTup);
        ProfScope prof(c, XR_K_TABLE, 0.0, 4.0 * nS_cfg * nTup);
        if (sd.k == 1)
            k_side_index<1><<<xr_grid(nS_cfg), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, kspace_core, nK, nT, layout, nTup, tab);
        else if (sd.k == 2)
            k_side_index<2><<<xr_grid(nS_cfg), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, kspace_core, nK, nT, layout, nTup, tab);
        else
            k_side_index<3><<<xr_grid(nS_cfg), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, kspace_core, nK, nT, layout, nTup, tab);
        XR_LAUNCH_CHECK(c);
    }
    double* tmpT = (double*)xr_workspace(c, WS_ZBT, n * sizeof(double));
    if (!tmpT) return xr_fail(c, XR_ENOMEM, "workspace (side adjoint)");
    if (tab) {
        ProfScope prof(c, XR_K_GATHER, 0.0, 8.0 * n + 4.0 * nS_cfg * nTup);
        k_side_adjoint_tab<<<xr_grid(n), 256, 0, c->stream>>>(tab, nS_cfg, nTup, Ybar, nS, tmpT);
        XR_LAUNCH_CHECK(c);
    } else {
        ProfScope prof(c, XR_K_GATHER, 0.0, 8.0 * n);
        if (sd.k == 1)
            k_side_adjoint<1><<<xr_grid(n), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, n_core, kspace_core,
                                                                 nK, nT, Ybar, nS, layout, tmpT);
        else if (sd.k == 2)
            k_side_adjoint<2><<<xr_grid(n), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, n_core, kspace_core,
                                                                 nK, nT, Ybar, nS, layout, tmpT);
        else
            k_side_adjoint<3><<<xr_grid(n), 256, 0, c->stream>>>(sd, Sm, nS_cfg, n_orbs, n_core, kspace_core,
                                                                 nK, nT, Ybar, nS, layout, tmpT);
        XR_LAUNCH_CHECK(c);
    }
    dim3 grid((unsigned)ceil_div(nS_cfg, 32), (unsigned)ceil_div(nS, 32));
    k_add_transpose<<<grid, dim3(32, 8), 0, c->stream>>>(tmpT, nS, nS_cfg, zbar, add ? 1 : 0);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// Vbar[p,q,b,a] += Veb[u,w], Vbar[q,p,b,a] -= .., Vbar[p,q,a,b] -= .., Vbar[q,p,a,b] += ..
// (transpose of k_veff); one thread per (u, w), distinct targets.
__global__ void k_veff_adjoint(const double* __restrict__ Veb, int dim, int64_t nU,
                               double* __restrict__ Vbar) {
    const int64_t D = dim;
    XR_GRID_STRIDE(i, nU * nU) {
        const int64_t u = i / nU, w = i - u * nU;
        int p, q, a, b;
        pair_at((int)u, dim / 2, &p, &q);
        pair_at((int)w, dim / 2, &a, &b);
        const double g = Veb[i];
        auto at = [&](int64_t x0, int64_t x1, int64_t x2, int64_t x3) -> double& {
            return Vbar[((x0 * D + x1) * D + x2) * D + x3];
        };
        at(p, q, b, a) += g;
        at(q, p, b, a) -= g;
        at(p, q, a, b) -= g;
        at(q, p, a, b) += g;
    }
}

// Wgiven: W = Veff Y as xr_monomer_2e_keep left it (same V and ket), used
// instead of recomputing the product; nullptr: recomputed.
static int monomer_2e_adjoint_impl(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI,
                                   int64_t nP, const double* zbra, int64_t nJ, int64_t nQ,
                                   const double* zket, const double* V, const double* Ebar,
                                   double* zbar_bra, double* zbar_ket, double* Vbar,
                                   const double* Wgiven, int64_t w_len) {
    OpPlan pl;
    xr_plan_op("ccaa", &pl);
    int nb = 0;
    int rc = check_spaces(c, pl, n_orbs, n_core, n_elec, nP, nQ, &nb);
    if (rc) return rc;
    if (nI <= 0 || nJ <= 0 || n_elec < 2) return XR_OK;
    if (!zbar_bra && !zbar_ket && !Vbar) return XR_OK;
    const int dim = 2 * n_orbs;
    const uint64_t* Km = nullptr;
    int64_t nK = 0;
    if ((rc = xr_space_masks(c, n_orbs, 0, n_elec - 2, &Km, &nK))) return rc;
    const int64_t nU = h_binom(dim, 2), Kp = even_up(nU);
    int32_t *tabL = nullptr, *tabR = nullptr;
    // A block with itself into one adjoint buffer: both sides remove two
    // electrons from the same states, and their tables differ only by the
    // order of the two annihilators (sg = -1 when the slots are swapped), so
    // X = sg Y.  When the caller guarantees a Hermitian two-body part
    // (V[pqrs] = V[rspq], xr_assume_hermitian_v), Ve is symmetric, hence
    // Ybar = Ve^T Wbar = sg W Ebar with W = Ve Y, side_R = sg side_L, and the
    // two side adjoints add up to side_L(W (Ebar + Ebar^T)): one gather, no
    // Ve^T Wbar product, one side adjoint.
    const double sg = (pl.L.slot[0] == pl.R.slot[0]) ? 1.0 : -1.0;
    const bool mirror = c->hermitian_v && zbra == zket && nI == nJ && nP == nQ && zbar_bra == zbar_ket && zbar_ket;
    // what the wanted outputs need: W and Xbar for the bra's adjoint, X and
    // Wbar for the ket's and V's, Y for W and for V's
    const bool need_w = mirror || zbar_bra, need_wbar = (zbar_ket && !mirror) || Vbar;
    const bool need_y = (need_w && !Wgiven) || Vbar || (mirror && need_wbar);
    if (Wgiven && w_len != nU * nK * nJ) return xr_fail(c, XR_ESHAPE, "sigma factor buffer size");
    const size_t szI = Kp * nK * nI * sizeof(double), szJ = Kp * nK * nJ * sizeof(double);
    double* X = need_wbar && !mirror ? (double*)xr_workspace(c, WS_X, szI) : nullptr;
    double* Y = need_y ? (double*)xr_workspace(c, WS_Y, szJ) : nullptr;
    double* W = !need_w ? nullptr : Wgiven ? const_cast<double*>(Wgiven) : (double*)xr_workspace(c, WS_W, szJ);
    double* Xbar = need_w ? (double*)xr_workspace(c, WS_XB, szI) : nullptr;
    double* Ybar = zbar_ket && !mirror ? (double*)xr_workspace(c, WS_YB, szJ) : nullptr;
    double* Wbar = need_wbar ? (double*)xr_workspace(c, WS_WB, szJ) : nullptr;
    double* Veb = Vbar ? (double*)xr_workspace(c, WS_VEB, nU * nU * sizeof(double)) : nullptr;
    if ((need_wbar && !mirror && !X) || (need_y && !Y) || (need_w && (!W || !Xbar)) ||
        (zbar_ket && !mirror && !Ybar) || (need_wbar && !Wbar) || (Vbar && !Veb) ||
        !side_scratch(c, zbar_bra ? nP * nI : 0, zbar_ket && !mirror ? nQ * nJ : 0))
        return xr_fail(c, XR_ENOMEM, "workspace (sigma adjoint)");
    Coeffs cb, ck;
    if ((rc = coeffs_for_gather(c, WS_ZTB, WS_ZTK, nI, nP, X ? zbra : nullptr, nJ, nQ, Y ? zket : nullptr, &cb, &ck)))
        return rc;
    GatherSide g[2];
    int ng = 0;
    if (X) {                                                                   // X[u][K][I]
        if ((rc = pair_table(c, pl.L, Km, nK, n_orbs, n_core, &tabL))) return rc;
        g[ng++] = gather_side(tabL, Kp * nK, cb, nI, X);
    }
    if (Y) {                                                                   // Y[w][K][J]
        if ((rc = pair_table(c, pl.R, Km, nK, n_orbs, n_core, &tabR))) return rc;
        g[ng++] = gather_side(tabR, Kp * nK, ck, nJ, Y);
    }
    if (ng && (rc = gather(c, g, ng))) return rc;
    const int64_t KJ = nK * nJ;
    // W = Ve Y (nU x KJ)
    if (need_w && !Wgiven && (rc = veff_product(c, V, nullptr, 0.0, dim, false, Y, KJ, W))) return rc;
    if (mirror) {
        double* Es = (double*)xr_workspace(c, WS_GS, nI * nI * sizeof(double));
        if (!Es) return xr_fail(c, XR_ENOMEM, "workspace (sigma adjoint)");
        dim3 grid((unsigned)ceil_div(nI, 32), (unsigned)ceil_div(nI, 32));
        k_sym_sum<<<grid, dim3(32, 8), 0, c->stream>>>(Ebar, nI, Es);   // Es = Ebar + Ebar^T
        XR_LAUNCH_CHECK(c);
        // Xbar[(u,K), I] = sum_J W[(u,K), J] Es[I, J]
        if ((rc = xr_gemm_2e(c, 0, 1, nU * nK, nI, nJ, 1.0, W, nJ, 0, Es, nJ, 0, 0.0, Xbar, nI, 0, 1)))
            return rc;
    } else if (need_w) {
        // Xbar[(u,K), I] = sum_J W[(u,K), J] Ebar[I, J]    ((nU nK) x nI)
        if ((rc = xr_gemm_2e(c, 0, 1, nU * nK, nI, nJ, 1.0, W, nJ, 0, Ebar, nJ, 0, 0.0, Xbar, nI, 0, 1)))
            return rc;
    }
    // Wbar[(u,K), J] = sum_I X[(u,K), I] Ebar[I, J], X = sg Y for a block with itself (zero in the padding row)
    if (need_wbar && (rc = xr_gemm_2e(c, 0, 0, Kp * nK, nJ, nI, mirror ? sg : 1.0, mirror ? Y : X, nI, 0, Ebar, nJ, 0,
                                      0.0, Wbar, nJ, 0, 1)))
        return rc;
    // every product before the first output is added to: a call that is refused
    // memory (a limit, a pin) leaves all outputs as they were
    // Veb = Wbar Y^T (nU x nU), Ybar = Ve^T Wbar (nU x KJ)
    if (Vbar && (rc = xr_gemm_2e(c, 0, 1, nU, nU, KJ, 1.0, Wbar, KJ, 0, Y, KJ, 0, 0.0, Veb, nU, 0, 1))) return rc;
    if (Ybar && (rc = veff_product(c, V, nullptr, 0.0, dim, true, Wbar, KJ, Ybar))) return rc;
    if (Vbar) {
        k_veff_adjoint<<<xr_grid(nU * nU), 256, 0, c->stream>>>(Veb, dim, nU, Vbar);
        XR_LAUNCH_CHECK(c);
    }
    if (Ybar && (rc = side_adjoint(c, pl.R, n_orbs, n_core, 0, n_elec, nK, nU, Ybar, nJ, 2, zbar_ket))) return rc;
    if (zbar_bra && (rc = side_adjoint(c, pl.L, n_orbs, n_core, 0, n_elec, nK, nU, Xbar, nI, 2, zbar_bra)))
        return rc;
    return XR_OK;
}

// out[v, P] = <P| H |Z_v> (overwritten) for H = sum h_pq p+ q + sum V_pqrs p+ q+ s r.
// With n_elec >= 2 the one-body part is carried by the two-body one
// (k_veff), so a pass is one gather of Z over the pairs it loses, one pair-matrix product and one side
// adjoint.  13 orbitals, 5 electrons, 21 vectors: 1.86 -> 0.22 ms against the two adjoints it replaces, whose
// one-body weight was a dense delta_IJ h over all vector pairs and whose
// ket-side products were computed and dropped.
extern "C" int xr_fci_sigma(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nv, int64_t nC, const double* Z,
                            const double* h, const double* V, double* out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    OpPlan pl;
    xr_plan_op("ccaa", &pl);
    int nb = 0;
    int rc = check_spaces(c, pl, n_orbs, n_core, n_elec, nC, nC, &nb);
    if (rc) return rc;
    if (nv <= 0) return XR_OK;
    const int dim = 2 * n_orbs;
    if (n_elec == 0) return xr_fill(c, out, nv * nC, 0.0);
    // one electron (no core): the determinants are the spin orbitals in order
    if (n_elec == 1) return xr_dgemm_launch(c, 0, 1, nv, dim, dim, 1.0, Z, dim, 0, h, dim, 0, 0.0, out, dim, 0, 1);
    const uint64_t* Km = nullptr;
    int64_t nK = 0;
    if ((rc = xr_space_masks(c, n_orbs, 0, n_elec - 2, &Km, &nK))) return rc;
    const int64_t nU = h_binom(dim, 2), Kp = even_up(nU), N = nK * nv;
    double* Y = (double*)xr_workspace(c, WS_Y, Kp * N * sizeof(double));
    double* W = (double*)xr_workspace(c, WS_W, nU * N * sizeof(double));
    if (!Y || !W) return xr_fail(c, XR_ENOMEM, "workspace (FCI sigma)");
    int32_t* tab = nullptr;
    Coeffs cz, none;
    if ((rc = coeffs_for_gather(c, WS_ZTB, WS_ZTK, nv, nC, Z, 0, 0, nullptr, &cz, &none)) ||
        (rc = pair_table(c, pl.R, Km, nK, n_orbs, n_core, &tab)))
        return rc;
    const GatherSide gs = gather_side(tab, Kp * nK, cz, nv, Y);
    if ((rc = gather(c, &gs, 1)) || (rc = veff_product(c, V, h, 1.0 / (n_elec - 1), dim, false, Y, N, W))) return rc;
    return side_adjoint(c, pl.L, n_orbs, n_core, 0, n_elec, nK, nU, W, nv, 2, out, false);
}

extern "C" int xr_monomer_2e_adjoint(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI,
                                     int64_t nP, const double* zbra, int64_t nJ, int64_t nQ,
                                     const double* zket, const double* V, const double* Ebar,
                                     double* zbar_bra, double* zbar_ket, double* Vbar) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    return monomer_2e_adjoint_impl(c, n_orbs, n_core, n_elec, nI, nP, zbra, nJ, nQ, zket, V, Ebar, zbar_bra,
                                   zbar_ket, Vbar, nullptr, 0);
}

extern "C" int xr_monomer_2e_adjoint_keep(xr_ctx* c, int n_orbs, int n_core, int n_elec, int64_t nI,
                                          int64_t nP, const double* zbra, int64_t nJ, int64_t nQ,
                                          const double* zket, const double* V, const double* Ebar,
                                          double* zbar_bra, double* zbar_ket, double* Vbar,
                                          const double* W, int64_t w_len) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (!W) return xr_fail(c, XR_EINVAL, "null sigma factor buffer");
    return monomer_2e_adjoint_impl(c, n_orbs, n_core, n_elec, nI, nP, zbra, nJ, nQ, zket, V, Ebar, zbar_bra,
                                   zbar_ket, Vbar, W, w_len);
}

extern "C" int xr_density_adjoint(xr_ctx* c, const char* ops, int n_orbs, int n_core,
                                  int n_elec_ket, int64_t nI, int64_t nP, const double* zbra,
                                  int64_t nJ, int64_t nQ, const double* zket, const double* Rbar,
                                  double* zbar_bra, double* zbar_ket) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    OpPlan pl;
    if (!xr_plan_op(ops, &pl)) return xr_fail(c, XR_EUNSUPPORTED, "operator string not supported");
    int nb = 0;
    int rc = check_spaces(c, pl, n_orbs, n_core, n_elec_ket, nP, nQ, &nb);
    if (rc) return rc;
    if (nI <= 0 || nJ <= 0) return XR_OK;
    if (pl.L.k && pl.R.k && n_elec_ket - pl.R.k < 0) return XR_OK;  // density identically zero
    if (!zbar_bra && !zbar_ket) return XR_OK;
    const int dim = 2 * n_orbs;
    Factors f;
    if ((rc = prepare_factors(c, pl, n_orbs, n_core, n_elec_ket, nb, nI, nP, zbra, nJ, nQ, zket, &f)))
        return rc;
    const int64_t Mg = f.nLt * nI, Ng = f.nT * nJ;
    double* Gc = (double*)xr_workspace(c, WS_GC, Mg * Ng * sizeof(double));
    const bool mirror = ops[0] == 'c' && ops[1] == 'a' && ops[2] == 0 && zbra == zket && nI == nJ &&
                        nP == nQ && Mg == Ng && zbar_bra == zbar_ket && zbar_ket && pl.R.k;
    double* Xbar = zbar_bra && !mirror && pl.L.k ? (double*)xr_workspace(c, WS_XB, f.nK * Mg * sizeof(double)) : nullptr;
    double* Ybar = zbar_ket && pl.R.k ? (double*)xr_workspace(c, WS_YB, f.nK * Ng * sizeof(double)) : nullptr;
    if (!Gc || (zbar_bra && !mirror && pl.L.k && !Xbar) || (zbar_ket && pl.R.k && !Ybar) ||
        !side_scratch(c, Xbar ? nP * nI : 0, Ybar ? nQ * nJ : 0))
        return xr_fail(c, XR_ENOMEM, "workspace (adjoint)");
    {
        int64_t n = Mg * Ng;
        ProfScope prof(c, XR_K_EXPAND, 0.0, 8.0 * n * (pl.k > 2 ? 4 : 2));
        if (nI * ceil_div(nJ, 32) > 0x7fffffffLL || f.nLt > 65535 || ceil_div(f.nT, 32) > 65535)
            return xr_fail(c, XR_EUNSUPPORTED, "density adjoint grid too large");
        dim3 grid((unsigned)(nI * ceil_div(nJ, 32)), (unsigned)f.nLt, (unsigned)ceil_div(f.nT, 32));
        k_compress<<<grid, 256, 0, c->stream>>>(Rbar, nI, nJ, pl.L.k, pl.R.k, dim, f.nT, Gc, Ng);
        XR_LAUNCH_CHECK(c);
    }
    // One-body string 'ca' between a block and itself, adjoints into one
    // buffer: X = Y (both sides remove one electron from the same states,
    // through the same table) and the two side adjoints are the same map, so
    // side(Y Gc^T) + side(X Gc) = side(X (Gc + Gc^T)): one GEMM, one side
    // adjoint.
    if (mirror) {
        double* Gs = (double*)xr_workspace(c, WS_GS, Mg * Ng * sizeof(double));
        if (!Gs) return xr_fail(c, XR_ENOMEM, "workspace (adjoint)");
        dim3 grid((unsigned)ceil_div(Mg, 32), (unsigned)ceil_div(Mg, 32));
        k_sym_sum<<<grid, dim3(32, 8), 0, c->stream>>>(Gc, Mg, Gs);   // Gs = Gc + Gc^T
        XR_LAUNCH_CHECK(c);
        if ((rc = xr_dgemm_launch(c, 0, 0, f.nK, Ng, Mg, 1.0, f.X, Mg, 0, Gs, Ng, 0, 0.0, Ybar, Ng, 0, 1)))
            return rc;
        return side_adjoint(c, pl.R, n_orbs, n_core, f.kspace_core, n_elec_ket, f.nK, f.nT, Ybar, nJ, 0,
                            zbar_ket);
    }
    // Every product that can be refused memory (a limit, a pin) and every read of
    // the coefficients comes before the first output is added to.
    // Ybar = X Gc (nK x Ng), Xbar = Y Gc^T (nK x Mg)
    if (Ybar && (rc = xr_dgemm_launch(c, f.xT, 0, f.nK, Ng, Mg, 1.0, f.X, f.ldx, 0, Gc, Ng, 0, 0.0, Ybar, Ng, 0, 1)))
        return rc;
    if (Xbar && (rc = xr_dgemm_launch(c, f.yT, 1, f.nK, Mg, Ng, 1.0, f.Y, f.ldy, 0, Gc, Ng, 0, 0.0, Xbar, Mg, 0, 1)))
        return rc;
    // without R, Y = zket^T: zbar_ket (nJ x nQ) += Gc^T X^T; without L, X = zbra^T:
    // zbar_bra (nI x nP) += Gc Y^T
    if (zbar_ket && !pl.R.k &&
        (rc = xr_dgemm_launch(c, 1, 1, nJ, nQ, Mg, 1.0, Gc, Ng, 0, f.X, f.ldx, 0, 1.0, zbar_ket, nQ, 0, 1)))
        return rc;
    if (zbar_bra && !pl.L.k &&
        (rc = xr_dgemm_launch(c, 0, 1, nI, nP, Ng, 1.0, Gc, Ng, 0, f.Y, f.ldy, 0, 1.0, zbar_bra, nP, 0, 1)))
        return rc;
    // then the transposes of the gathers
    if (Ybar && (rc = side_adjoint(c, pl.R, n_orbs, n_core, f.kspace_core, n_elec_ket, f.nK, f.nT, Ybar, nJ, 0,
                                   zbar_ket)))
        return rc;
    if (Xbar && (rc = side_adjoint(c, pl.L, n_orbs, n_core, f.kspace_core, nb, f.nK, f.nLt, Xbar, nI, 0, zbar_bra)))
        return rc;
    return XR_OK;
}
