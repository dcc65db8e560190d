// Vector kernels of the block-Davidson eigensolver (the matrix-free XR
// solve and the dense fallback): the diagonal preconditioner's divide, the
// residual block with its column norms, column sums of squares, and the
// transposed store of a block of vectors into the basis kept one vector per
// row.  Each is one pass over the n x b block; the column reductions go
// through fixed-order partial sums (the same result on every run).
// ---------------------------------------------------------------------------
#define XR_SOLVER_MAXB 32
enum { WS_SOLVER_PART = 90 };

// Y[i, j] = X[i, j] / d with d = s (lam[i] - theta[j]), replaced by +floor
// where |d| < floor.  X and Y may be the same array.
__global__ void k_precond_divide(int64_t n, int64_t b, const double* X, int64_t ldx, double* Y, int64_t ldy,
                                 const double* __restrict__ lam, const double* __restrict__ theta, double s,
                                 double floor_) {
    XR_GRID_STRIDE(e, n * b) {
        const int64_t i = e / b, j = e - i * b;
        double d = s * (lam[i] - theta[j]);
        if (fabs(d) < floor_) d = floor_;
        Y[i * ldy + j] = X[i * ldx + j] / d;
    }
}

// Fixed-order sum of one value per thread over the block (256 threads).
__device__ __forceinline__ double block_sum256(double v, double* red) {
    const int tid = threadIdx.x;
    red[tid] = v;
    __syncthreads();
#pragma unroll
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

// R = AX - X diag(theta) (row-major n x NB blocks, row strides ldx / ldax /
// ldr; R may be null), and part[block][j] = the block's sum of R[i][j]^2 for
// j < k (R[i][j] = A[i][j] when X is null: plain column sums of squares).
template <int NB>
__global__ __launch_bounds__(256) void k_residual_part(int64_t n, int b, int k, const double* X, int64_t ldx,
                                                       const double* A, int64_t lda,
                                                       const double* __restrict__ theta, double* R, int64_t ldr,
                                                       double* __restrict__ part) {
    __shared__ double red[256];
    double acc[NB];
    double th[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        acc[j] = 0.0;
        th[j] = (X && j < b) ? theta[j] : 0.0;
    }
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (j < b) {
                double r = A[i * lda + j];
                if (X) r -= X[i * ldx + j] * th[j];
                if (R) R[i * ldr + j] = r;
                if (j < k) acc[j] += r * r;
            }
        }
    }
    for (int j = 0; j < k; j++) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < NB; q++)
            if (q == j) v = acc[q];
        const double s = block_sum256(v, red);
        if (threadIdx.x == 0) part[(int64_t)blockIdx.x * k + j] = s;
    }
}

// out[j] = sum over blocks of part[block][j], or its root: one workgroup per
// column, each thread summing every 256th partial in order, then the fixed
// block tree.
__global__ __launch_bounds__(256) void k_residual_final(const double* __restrict__ part, int64_t nblk, int k,
                                                        double* out, int root) {
    __shared__ double red[256];
    const int j = blockIdx.x;
    double s = 0.0;
    for (int64_t q = threadIdx.x; q < nblk; q += 256) s += part[q * k + j];
    s = block_sum256(s, red);
    if (threadIdx.x == 0) out[j] = root ? sqrt(s) : s;
}

// B[j][i] = A[i][j] for an rows x cols block (32 x 32 tiles through LDS;
// grid x over the rows, which may be many, y over the columns).
__global__ __launch_bounds__(256) void k_transpose(int64_t rows, int64_t cols, const double* __restrict__ A,
                                                   int64_t lda, double* __restrict__ B, int64_t ldb) {
    __shared__ double t[32][33];
    const int64_t tr = (int64_t)blockIdx.x * 32, tc = (int64_t)blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int64_t i = tr + r, j = tc + tx;
        if (i < rows && j < cols) t[r][tx] = A[i * lda + j];
    }
    __syncthreads();
    for (int c = ty; c < 32; c += 8) {
        const int64_t j = tc + c, i = tr + tx;
        if (i < rows && j < cols) B[j * ldb + i] = t[tx][c];
    }
}

// The same for cols <= NB (a block of a few vectors): one thread per row
// reads its NB values and writes them to NB rows of B (coalesced over i).
template <int NB>
__global__ __launch_bounds__(256) void k_transpose_narrow(int64_t rows, int cols, const double* __restrict__ A,
                                                          int64_t lda, double* __restrict__ B, int64_t ldb) {
    XR_GRID_STRIDE(i, rows) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (j < cols) B[j * ldb + i] = A[i * lda + j];
    }
}

static int residual_go(xr_ctx* c, int64_t n, int b, int k, const double* X, int64_t ldx, const double* A,
                       int64_t lda, const double* theta, double* R, int64_t ldr, double* out, int root) {
    const int64_t nblk = std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256 * 4), 1024));
    double* part = nullptr;
    if (k > 0) {
        part = (double*)xr_workspace(c, WS_SOLVER_PART, (size_t)(nblk * k * sizeof(double)));
        if (!part) return xr_fail(c, XR_ENOMEM, "workspace (column norms)");
    }
    ProfScope prof(c, XR_K_OTHER, 0.0, 8.0 * n * b * (X ? 3 : 1));
#define XR_RES(NB_) k_residual_part<NB_><<<(unsigned)nblk, 256, 0, c->stream>>>(n, b, k, X, ldx, A, lda, theta, R, ldr, part)
    if (b <= 1) { XR_RES(1); }
    else if (b <= 2) { XR_RES(2); }
    else if (b <= 4) { XR_RES(4); }
    else if (b <= 8) { XR_RES(8); }
    else if (b <= 16) { XR_RES(16); }
    else { XR_RES(32); }
#undef XR_RES
    XR_LAUNCH_CHECK(c);
    if (k > 0) {
        k_residual_final<<<(unsigned)k, 256, 0, c->stream>>>(part, nblk, k, out, root);
        XR_LAUNCH_CHECK(c);
    }
    return XR_OK;
}

extern "C" int xr_precond_divide(xr_ctx* c, int64_t n, int64_t b, const double* X, int64_t ldx, double* Y,
                                 int64_t ldy, const double* lam, const double* theta, double sign, double floor_) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (n < 0 || b < 0) return xr_fail(c, XR_EINVAL, "negative size");
    if (n == 0 || b == 0) return XR_OK;
    if (ldx < b || ldy < b) return xr_fail(c, XR_ESHAPE, "row stride below the block width");
    if (!(floor_ > 0.0)) return xr_fail(c, XR_EINVAL, "floor must be positive");
    ProfScope prof(c, XR_K_OTHER, 0.0, 16.0 * n * b);
    k_precond_divide<<<xr_grid(n * b), 256, 0, c->stream>>>(n, b, X, ldx, Y, ldy, lam, theta, sign, floor_);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

extern "C" int xr_residual(xr_ctx* c, int64_t n, int b, int k, const double* X, int64_t ldx, const double* AX,
                           int64_t ldax, const double* theta, double* R, int64_t ldr, double* norms) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (n < 0 || b < 0 || k < 0 || k > b) return xr_fail(c, XR_EINVAL, "bad residual sizes (0 <= k <= b)");
    if (b > XR_SOLVER_MAXB) return xr_fail(c, XR_EUNSUPPORTED, "residual block wider than 32 columns");
    if (ldx < b || ldax < b || ldr < b) return xr_fail(c, XR_ESHAPE, "row stride below the block width");
    if (n == 0 || b == 0) return XR_OK;
    if (!X || !AX || !theta || !R || (k > 0 && !norms)) return xr_fail(c, XR_EINVAL, "null residual operand");
    return residual_go(c, n, b, k, X, ldx, AX, ldax, theta, R, ldr, norms, 1);
}

extern "C" int xr_column_norms(xr_ctx* c, int64_t n, int b, const double* A, int64_t lda, double* out,
                               int squared) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (n < 0 || b < 0) return xr_fail(c, XR_EINVAL, "negative size");
    if (b > XR_SOLVER_MAXB) return xr_fail(c, XR_EUNSUPPORTED, "more than 32 columns");
    if (lda < b) return xr_fail(c, XR_ESHAPE, "row stride below the block width");
    if (b == 0) return XR_OK;
    if (!A || !out) return xr_fail(c, XR_EINVAL, "null operand");
    return residual_go(c, n, b, b, nullptr, 0, A, lda, nullptr, nullptr, 0, out, squared ? 0 : 1);
}

extern "C" int xr_transpose(xr_ctx* c, int64_t rows, int64_t cols, const double* A, int64_t lda, double* B,
                            int64_t ldb) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (rows < 0 || cols < 0) return xr_fail(c, XR_EINVAL, "negative size");
    if (rows == 0 || cols == 0) return XR_OK;
    if (lda < cols || ldb < rows) return xr_fail(c, XR_ESHAPE, "leading dimension too small");
    ProfScope prof(c, XR_K_OTHER, 0.0, 16.0 * rows * cols);
    if (cols <= 8) {
#define XR_TN(NB_) k_transpose_narrow<NB_><<<xr_grid(rows), 256, 0, c->stream>>>(rows, (int)cols, A, lda, B, ldb)
        if (cols <= 1) { XR_TN(1); }
        else if (cols <= 2) { XR_TN(2); }
        else if (cols <= 4) { XR_TN(4); }
        else { XR_TN(8); }
#undef XR_TN
        XR_LAUNCH_CHECK(c);
        return XR_OK;
    }
    if (ceil_div(rows, 32) > 0x7fffffff || ceil_div(cols, 32) > 65535)
        return xr_fail(c, XR_EUNSUPPORTED, "transpose grid too large");
    k_transpose<<<dim3((unsigned)ceil_div(rows, 32), (unsigned)ceil_div(cols, 32)), 256, 0, c->stream>>>(
        rows, cols, A, lda, B, ldb);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// ---------------------------------------------------------------------------
// Diagonal of the XR operator in the product eigenbasis, one sector tuple at
// a time: out[i] = sum_m e_m[j_m] + sum_(m<n) pd_mn[j_m, j_n] for the
// row-major digits (j_0, ..., j_{nf-1}) of i, the terms summed in that order.
// ---------------------------------------------------------------------------
#define XR_DIAG_MAXF 8
enum { WS_COLDOT = 93 };

struct DiagTuple {
    int nf;
    int64_t size;
    int64_t dims[XR_DIAG_MAXF];
    const double* e[XR_DIAG_MAXF];
    const double* pd[XR_DIAG_MAXF * (XR_DIAG_MAXF - 1) / 2];
};

__global__ __launch_bounds__(256) void k_sector_diag(DiagTuple t, double* __restrict__ out) {
    XR_GRID_STRIDE(i, t.size) {
        int64_t j[XR_DIAG_MAXF];
        int64_t r = i;
        for (int m = t.nf - 1; m >= 0; m--) {
            const int64_t q = r / t.dims[m];
            j[m] = r - q * t.dims[m];
            r = q;
        }
        double v = 0.0;
        for (int m = 0; m < t.nf; m++) v += t.e[m][j[m]];
        int p = 0;
        for (int m = 0; m < t.nf; m++)
            for (int n = m + 1; n < t.nf; n++, p++) v += t.pd[p][j[m] * t.dims[n] + j[n]];
        out[i] = v;
    }
}

extern "C" int xr_sector_diag(xr_ctx* c, int nf, int ntup, const int64_t* dims, const int64_t* off,
                              const double* const* e, const double* const* pd, double* out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (nf < 1 || nf > XR_DIAG_MAXF) return xr_fail(c, XR_EUNSUPPORTED, "1 to 8 fragments");
    if (ntup < 0) return xr_fail(c, XR_EINVAL, "negative tuple count");
    if (ntup == 0) return XR_OK;
    if (!dims || !off || !e || (nf > 1 && !pd) || !out) return xr_fail(c, XR_EINVAL, "null argument");
    const int np = nf * (nf - 1) / 2;
    for (int q = 0; q < ntup; q++) {
        DiagTuple t{};
        t.nf = nf;
        t.size = 1;
        for (int m = 0; m < nf; m++) {
            const int64_t d = dims[(int64_t)q * nf + m];
            if (d < 1) return xr_fail(c, XR_EINVAL, "empty tuple axis");
            t.dims[m] = d;
            t.size *= d;
            t.e[m] = e[(int64_t)q * nf + m];
            if (!t.e[m]) return xr_fail(c, XR_EINVAL, "null monomer diagonal");
        }
        for (int p = 0; p < np; p++) {
            t.pd[p] = pd[(int64_t)q * np + p];
            if (!t.pd[p]) return xr_fail(c, XR_EINVAL, "null pair diagonal");
        }
        ProfScope prof(c, XR_K_OTHER, 0.0, 8.0 * t.size);
        k_sector_diag<<<xr_grid(t.size), 256, 0, c->stream>>>(t, out + off[q]);
        XR_LAUNCH_CHECK(c);
    }
    return XR_OK;
}

// out[j] = sum_i A[i, j] B[i, j] for rows x cols blocks: partial sums over
// chunks of 64 rows (one thread per column, in row order), then the chunks
// in order (deterministic).
__global__ __launch_bounds__(256) void k_coldot_part(int64_t rows, int64_t cols, const double* __restrict__ A,
                                                     int64_t lda, const double* __restrict__ B, int64_t ldb,
                                                     double* __restrict__ part) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.y * 64;
    if (j >= cols) return;
    const int64_t r1 = r0 + 64 < rows ? r0 + 64 : rows;
    double s = 0.0;
    for (int64_t i = r0; i < r1; i++) s += A[i * lda + j] * B[i * ldb + j];
    part[(int64_t)blockIdx.y * cols + j] = s;
}

__global__ __launch_bounds__(256) void k_coldot_final(const double* __restrict__ part, int64_t nchunk, int64_t cols,
                                                      double* __restrict__ out) {
    XR_GRID_STRIDE(j, cols) {
        double s = 0.0;
        for (int64_t q = 0; q < nchunk; q++) s += part[q * cols + j];
        out[j] = s;
    }
}

extern "C" int xr_column_dots(xr_ctx* c, int64_t rows, int64_t cols, const double* A, int64_t lda, const double* B,
                              int64_t ldb, double* out) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    if (rows < 0 || cols < 0) return xr_fail(c, XR_EINVAL, "negative size");
    if (cols == 0) return XR_OK;
    if (lda < cols || ldb < cols) return xr_fail(c, XR_ESHAPE, "leading dimension below the column count");
    if (!A || !B || !out) return xr_fail(c, XR_EINVAL, "null operand");
    const int64_t nchunk = std::max<int64_t>(1, ceil_div(rows, 64));
    if (nchunk > 65535 || ceil_div(cols, 256) > 0x7fffffff) return xr_fail(c, XR_EUNSUPPORTED, "block too large");
    double* part = (double*)xr_workspace(c, WS_COLDOT, sizeof(double) * (size_t)(nchunk * cols));
    if (!part) return xr_fail(c, XR_ENOMEM, "workspace (column dots)");
    ProfScope prof(c, XR_K_OTHER, 2.0 * rows * cols, 16.0 * rows * cols);
    if (rows == 0) {
        k_coldot_final<<<xr_grid(cols), 256, 0, c->stream>>>(part, 0, cols, out);
    } else {
        k_coldot_part<<<dim3((unsigned)ceil_div(cols, 256), (unsigned)nchunk), 256, 0, c->stream>>>(rows, cols, A, lda,
                                                                                                   B, ldb, part);
        XR_LAUNCH_CHECK(c);
        k_coldot_final<<<xr_grid(cols), 256, 0, c->stream>>>(part, nchunk, cols, out);
    }
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// ---------------------------------------------------------------------------
// Lanczos with full reorthogonalisation for the lowest root of a dense
// symmetric A (n x n).  One step is one pass over A and two classical
// Gram-Schmidt passes over the basis V (one vector per row):
//   k_root_matvec   V_j = r / |r|, w = A V_j - |r| V_(j-1)
//   k_root_dots     c = V w,  k_root_update  w -= V^T c        (twice; |w|^2 in parts)
// Every sum has a fixed order, so a root is the same bits on every run.  Bound by
// launches for n of some hundreds (A sits in L2) and by A's bytes above; the
// second pass keeps V orthogonal to rounding, without which the alpha / beta
// factors of a step would amplify the loss.
// ---------------------------------------------------------------------------
#define LZ_COLS 64                     // columns of an update block (and of a norm part)
#define LZ_MAXPART 128                 // n <= LZ_COLS * LZ_MAXPART

__device__ __forceinline__ double wave_sum64(double v) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
    return v;
}

// start vector in (-1, 1) from the index (splitmix64's mix), with its norm parts
__global__ __launch_bounds__(LZ_COLS) void k_root_start(int64_t n, double* __restrict__ r, double* __restrict__ part) {
    const int64_t i = (int64_t)blockIdx.x * LZ_COLS + threadIdx.x;
    uint64_t z = (uint64_t)(i + 1) * 0x9e3779b97f4a7c15ULL;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    z ^= z >> 31;
    const double v = i < n ? (double)(int64_t)z * 0x1p-63 : 0.0;
    if (i < n) r[i] = v;
    const double t = wave_sum64(v * v);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// one wave a row; every wave adds up the nb norm parts of r by itself
__global__ __launch_bounds__(256) void k_root_matvec(int64_t n, const double* __restrict__ A, int64_t lda,
                                                   const double* __restrict__ r, const double* __restrict__ part,
                                                   int nb, double* __restrict__ Vj, const double* __restrict__ Vp,
                                                   double* __restrict__ beta, double* __restrict__ w) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    double sq = 0.0;
    for (int p = lane; p < nb; p += 64) sq += part[p];
    const double b = sqrt(wave_sum64(sq)), inv = b > 0.0 ? 1.0 / b : 0.0;
    const double* a = A + row * lda;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int64_t i = lane;
    for (; i + 192 < n; i += 256) {
        s0 += a[i] * r[i];
        s1 += a[i + 64] * r[i + 64];
        s2 += a[i + 128] * r[i + 128];
        s3 += a[i + 192] * r[i + 192];
    }
    for (; i < n; i += 64) s0 += a[i] * r[i];
    const double s = wave_sum64((s0 + s1) + (s2 + s3));
    if (lane == 0) {
        Vj[row] = r[row] * inv;
        w[row] = s * inv - (Vp ? b * Vp[row] : 0.0);
        if (row == 0 && beta) *beta = b;
    }
}

// c[q] = <V_q, w>, one workgroup a basis vector
__global__ __launch_bounds__(256) void k_root_dots(int64_t n, const double* __restrict__ V, int64_t ldv,
                                                 const double* __restrict__ w, double* __restrict__ out) {
    __shared__ double red[4];
    const double* v = V + (int64_t)blockIdx.x * ldv;
    double s0 = 0.0, s1 = 0.0;
    int64_t i = threadIdx.x;
    for (; i + 256 < n; i += 512) {
        s0 += v[i] * w[i];
        s1 += v[i + 256] * w[i + 256];
    }
    if (i < n) s0 += v[i] * w[i];
    const double s = wave_sum64(s0 + s1);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// w = base - sum_q c_q V_q (base null: + sum) over 64 columns a workgroup, the
// vectors dealt to 16 waves.  part: |w|^2 of these columns.  alpha = c[m-1] (+ prev[m-1]).
__global__ __launch_bounds__(1024) void k_root_update(int64_t n, const double* __restrict__ V, int64_t ldv, int m,
                                                    const double* __restrict__ c, const double* base,
                                                    double* w, double* __restrict__ part,
                                                    const double* __restrict__ prev, double* __restrict__ alpha) {
    __shared__ double red[16][LZ_COLS];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * LZ_COLS + lane;
    double s = 0.0;
    if (i < n) {
#pragma unroll 4
        for (int q = wv; q < m; q += 16) s += c[q] * V[(int64_t)q * ldv + i];
    }
    red[wv][lane] = s;
    __syncthreads();
    if (wv == 0) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 16; q++) t += red[q][lane];
        double v = 0.0;
        if (i < n) {
            v = base ? base[i] - t : t;
            w[i] = v;
        }
        if (part) {
            const double sq = wave_sum64(v * v);
            if (lane == 0) part[blockIdx.x] = sq;
        }
        if (alpha && blockIdx.x == 0 && lane == 0) *alpha = c[m - 1] + prev[m - 1];
    }
}

// out = {y.w, |w - (y.w) y|} for |y| = 1; one workgroup
__global__ __launch_bounds__(256) void k_root_check(int64_t n, const double* __restrict__ y,
                                                  const double* __restrict__ w, double* __restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 256) s += y[i] * w[i];
    const double th = block_sum256(s, red);
    s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const double d = w[i] - th * y[i];
        s += d * d;
    }
    const double rr = block_sum256(s, red);
    if (threadIdx.x == 0) {
        out[0] = th;
        out[1] = sqrt(rr);
    }
}

// work: alpha[cap], beta[cap] (beta[j] couples j - 1 and j, beta[0] the start's
// norm), the norm parts of the next vector [LZ_MAXPART], c, c' [cap each], two vectors [n each]
struct LzWork { double *alpha, *beta, *part, *c0, *c1, *w[2]; };
static LzWork lz_work(double* p, int64_t cap, int64_t n) {
    LzWork k;
    k.alpha = p;
    k.beta = p + cap;
    k.part = p + 2 * cap;
    k.c0 = k.part + LZ_MAXPART;
    k.c1 = k.c0 + cap;
    k.w[0] = k.c1 + cap;
    k.w[1] = k.w[0] + n;
    return k;
}
static int lz_args(xr_ctx* c, int64_t n, const double* A, int64_t lda, int64_t cap, const double* V, int64_t ldv,
                   const double* work) {
    if (n < 1 || n > (int64_t)LZ_COLS * LZ_MAXPART || cap < 1 || cap > n)
        return xr_fail(c, XR_EUNSUPPORTED, "Lanczos: 1 <= steps <= n <= 8192 expected");
    if (lda < n || ldv < n) return xr_fail(c, XR_ESHAPE, "row stride below n");
    if (!A || !V || !work) return xr_fail(c, XR_EINVAL, "null operand");
    return XR_OK;
}

extern "C" int xr_lanczos_steps(xr_ctx* c, int64_t n, const double* A, int64_t lda, int64_t j0, int64_t j1,
                                int64_t cap, double* V, int64_t ldv, double* work) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    const int rc = lz_args(c, n, A, lda, cap, V, ldv, work);
    if (rc) return rc;
    if (j0 < 0 || j1 < j0 || j1 > cap) return xr_fail(c, XR_EINVAL, "Lanczos: step range");
    const LzWork k = lz_work(work, cap, n);
    const int nb = (int)ceil_div(n, LZ_COLS);
    ProfScope prof(c, XR_K_OTHER, 2.0 * n * n * (j1 - j0), 8.0 * n * n * (j1 - j0));
    if (j0 == 0) k_root_start<<<nb, LZ_COLS, 0, c->stream>>>(n, k.w[0], k.part);
    for (int64_t j = j0; j < j1; j++) {
        double *r = k.w[j & 1], *w = k.w[(j + 1) & 1];
        k_root_matvec<<<(unsigned)ceil_div(n, 4), 256, 0, c->stream>>>(n, A, lda, r, k.part, nb, V + j * ldv,
                                                                     j ? V + (j - 1) * ldv : nullptr, k.beta + j, w);
        const unsigned m = (unsigned)(j + 1);
        k_root_dots<<<m, 256, 0, c->stream>>>(n, V, ldv, w, k.c0);
        k_root_update<<<nb, 1024, 0, c->stream>>>(n, V, ldv, (int)m, k.c0, w, w, nullptr, nullptr, nullptr);
        k_root_dots<<<m, 256, 0, c->stream>>>(n, V, ldv, w, k.c1);
        k_root_update<<<nb, 1024, 0, c->stream>>>(n, V, ldv, (int)m, k.c1, w, w, k.part, k.c0, k.alpha + j);
    }
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// s (device, m): y = V^T s normalised -> v; {Rayleigh quotient, residual norm} -> work's first two doubles
extern "C" int xr_lanczos_root(xr_ctx* c, int64_t n, const double* A, int64_t lda, int64_t m, int64_t cap,
                               const double* V, int64_t ldv, const double* s, double* work, double* v) {
    if (!c) return XR_EINVAL;
    std::lock_guard<std::mutex> g(c->mu);
    const int rc = lz_args(c, n, A, lda, cap, V, ldv, work);
    if (rc) return rc;
    if (m < 1 || m > cap) return xr_fail(c, XR_EINVAL, "Lanczos: basis size");
    if (!s || !v) return xr_fail(c, XR_EINVAL, "null operand");
    const LzWork k = lz_work(work, cap, n);
    const int nb = (int)ceil_div(n, LZ_COLS);
    ProfScope prof(c, XR_K_OTHER, 2.0 * n * n, 8.0 * n * n);
    k_root_update<<<nb, 1024, 0, c->stream>>>(n, V, ldv, (int)m, s, nullptr, k.w[0], k.part, nullptr, nullptr);
    k_root_matvec<<<(unsigned)ceil_div(n, 4), 256, 0, c->stream>>>(n, A, lda, k.w[0], k.part, nb, v, nullptr, nullptr,
                                                                 k.w[1]);
    k_root_check<<<1, 256, 0, c->stream>>>(n, v, k.w[1], k.alpha);
    XR_LAUNCH_CHECK(c);
    return XR_OK;
}

// Lowest eigenpair of the m x m symmetric tridiagonal (d, e), on the host:
// Sturm bisection, then the vector from a twisted factorisation (top-down
// and bottom-up LDL^T of T - theta joined where the pivot is least), which keeps small
// components accurate; the last one decides convergence.  out: theta, the
// largest |eigenvalue| bound (Gershgorin), |last component|; s[m] normalised.
extern "C" int xr_tridiag_lowest(int64_t m, const double* d, const double* e, double* out, double* s, double* scratch) {
    if (m < 1 || !d || (m > 1 && !e) || !out || !s || !scratch) return XR_EINVAL;
    double lo = 0.0, hi = 0.0;
    for (int64_t i = 0; i < m; i++) {
        const double rad = (i ? fabs(e[i - 1]) : 0.0) + (i + 1 < m ? fabs(e[i]) : 0.0);
        if (!(fabs(d[i]) + rad <= 1e300)) return XR_EINVAL;           // NaN or infinite
        lo = i ? fmin(lo, d[i] - rad) : d[i] - rad;
        hi = i ? fmax(hi, d[i] + rad) : d[i] + rad;
    }
    const double nrm = fmax(fabs(lo), fabs(hi)), tiny = fmax(nrm, 1e-280) * 0x1p-106;
    double a = lo, b = hi;                       // lowest eigenvalue in [a, b]
    for (int it = 0; it < 128; it++) {
        const double x = 0.5 * (a + b);
        if (x <= a || x >= b) break;
        bool below = false;                      // an eigenvalue under x
        double q = 1.0;
        for (int64_t i = 0; i < m && !below; i++) {
            q = d[i] - x - (i ? e[i - 1] * e[i - 1] / q : 0.0);
            if (fabs(q) < tiny) q = -tiny;
            below = q < 0.0;
        }
        if (below) b = x; else a = x;
    }
    const double th = a;
    double *p = scratch, *q = scratch + m;       // pivots from the top and from the bottom
    for (int64_t i = 0; i < m; i++) {
        p[i] = d[i] - th - (i ? e[i - 1] * e[i - 1] / p[i - 1] : 0.0);
        if (fabs(p[i]) < tiny) p[i] = tiny;
    }
    for (int64_t i = m - 1; i >= 0; i--) {
        q[i] = d[i] - th - (i + 1 < m ? e[i] * e[i] / q[i + 1] : 0.0);
        if (fabs(q[i]) < tiny) q[i] = tiny;
    }
    int64_t r = 0;
    double best = 0.0;
    for (int64_t i = 0; i < m; i++) {
        const double gam = fabs(p[i] + q[i] - (d[i] - th));
        if (i == 0 || gam < best) {
            best = gam;
            r = i;
        }
    }
    s[r] = 1.0;
    for (int64_t i = r - 1; i >= 0; i--) s[i] = -e[i] * s[i + 1] / p[i];
    for (int64_t i = r + 1; i < m; i++) s[i] = -e[i - 1] * s[i - 1] / q[i];
    double nn = 0.0;
    for (int64_t i = 0; i < m; i++) nn += s[i] * s[i];
    nn = 1.0 / sqrt(nn);
    for (int64_t i = 0; i < m; i++) s[i] *= nn;
    out[0] = th;
    out[1] = nrm;
    out[2] = fabs(s[m - 1]);
    return XR_OK;
}
