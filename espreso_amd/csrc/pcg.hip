// Kernels of the projected PCG on K interleaved dual vectors (x[l K + v], v < K
// load cases; K = 1 is the single solve): gathers between lambda space and the
// boundary DOFs, the projector P = I - G^T (G G^T)^-1 G (itersolver.cpp:
// 5541-5623), the sparse preconditioners (itersolvercpu.cpp:520-602) and the
// vector updates with their dot products (itersolver.cpp:1537-1684).
//
// These passes move a few MB: what bounds them is the number of launches and
// the chains of dependent loads, not bytes.  So the K cases share one launch
// (a gather by lambda reads the K values of a line together), a dot product is
// summed by the kernel that produces its operand (one partial per workgroup
// and case) and finished by the kernel that needs the scalar, and the rows of
// the coarse basis are stored row-major beside per-entry offsets (one indexed
// load instead of a chain of subdomain tables).
#include <hip/hip_runtime.h>

#include "dual.h"

namespace esp {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

static inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// threads of a workgroup as lines of K values: thread (li, v), li < per
struct Lines {
    int per, li, v;
    bool on;
};
__device__ __forceinline__ Lines lines_of(int K) {
    Lines L;
    if (K == 1) {
        L.per = blockDim.x;
        L.li = threadIdx.x;
        L.v = 0;
        L.on = true;
    } else {
        L.per = blockDim.x / K;
        L.li = threadIdx.x / K;
        L.v = threadIdx.x - L.li * K;
        L.on = L.li < L.per;
    }
    return L;
}

// sum of `val` over the lines of the workgroup, per case: sh[v] (blockDim
// doubles of LDS), in a fixed order; every thread may read sh[v] afterwards
__device__ __forceinline__ void lines_sum(double val, const Lines &L, int K, double *sh) {
    __syncthreads();
    sh[threadIdx.x] = L.on ? val : 0.0;
    __syncthreads();
    int h = 1;
    while (2 * h < L.per) h *= 2;
    for (; h > 0; h >>= 1) {
        if (L.on && L.li < h && L.li + h < L.per) sh[threadIdx.x] += sh[threadIdx.x + h * K];
        __syncthreads();
    }
}

// sum of np partials per case, part[b K + v], into sh[v]
__device__ __forceinline__ void partials_sum(const double *__restrict__ part, int np, const Lines &L, int K,
                                             double *sh) {
    double a = 0.0;
    if (L.on)
        for (int b = L.li; b < np; b += L.per) a += part[(int64_t)b * K + L.v];
    lines_sum(a, L, K, sh);
}

constexpr int LINE_THREADS_1 = 256, LINE_THREADS_K = 512;
static inline int line_threads(int K) { return K == 1 ? LINE_THREADS_1 : LINE_THREADS_K; }
// workgroups of a pass over n lines that sums a dot product: one partial each.
// At most 4 (K = 1) or 2 workgroups per CU: the consumer of the partials reads
// them all in every workgroup
int dot_blocks(int64_t n, int K) {
    const int64_t per = line_threads(K) / K;
    return (int)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, K == 1 ? 1024 : 512));
}
static inline unsigned line_grid(int64_t n, int K) {
    const int64_t per = line_threads(K) / K;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, 4096));
}

// ---- set-up of the derived maps ----
// bl_row[q]: boundary DOF of entry q of the boundary -> lambda CSR
__global__ void k_entry_rows(int64_t nb, const int64_t *bl_ptr, int *bl_row) {
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < nb; j += (int64_t)gridDim.x * blockDim.x)
        for (int64_t q = bl_ptr[j]; q < bl_ptr[j + 1]; q++) bl_row[q] = (int)j;
}

// row-major copy of the per-subdomain bases (m_s x k_s column-major at roff[s])
__global__ void __launch_bounds__(256) k_basis_rows(const int *M, const int *kcols, const int64_t *roff,
                                                    const double *R, double *RT) {
    const int s = blockIdx.y, m = M[s], k = kcols[s];
    const double *src = R + roff[s];
    double *dst = RT + roff[s];
    for (int j = blockIdx.x * 256 + threadIdx.x; j < m; j += gridDim.x * 256)
        for (int a = 0; a < k; a++) dst[(int64_t)j * k + a] = src[j + (int64_t)a * m];
}

// the coarse-basis row and coarse offset of every lambda entry
__global__ void k_lambda_coarse(int nlam, const int *cnt, const int64_t *lb, const int *lsub, const int64_t *boff,
                                const int64_t *rtoff, const int *ck, const int *cblk, const int *coff, LamCoarse *le) {
    for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < nlam; l += gridDim.x * blockDim.x)
        for (int q = 0; q < 2; q++) {
            LamCoarse c{0, 0, 0};
            if (q < cnt[l]) {
                const int s = lsub[2 * (int64_t)l + q];
                c.k = ck[s];
                c.row = rtoff[s] + (lb[2 * (int64_t)l + q] - boff[s]) * c.k;
                c.off = coff[cblk[s]];
            }
            le[2 * (int64_t)l + q] = c;
        }
}

void launch_entry_rows(int64_t nb, const int64_t *bl_ptr, int *bl_row, hipStream_t st) {
    hipLaunchKernelGGL(k_entry_rows, dim3(std::max(1u, std::min(cdiv(nb, 256), 4096u))), dim3(256), 0, st, nb, bl_ptr,
                       bl_row);
}
void launch_basis_rows(int nsub, int max_m, const int *M, const int *kcols, const int64_t *roff, const double *R,
                       double *RT, hipStream_t st) {
    hipLaunchKernelGGL(k_basis_rows, dim3(std::max(1u, cdiv(max_m, 256)), nsub), dim3(256), 0, st, M, kcols, roff, R,
                       RT);
}
void launch_lambda_coarse(const DualDev &D, LamCoarse *le, hipStream_t st) {
    hipLaunchKernelGGL(k_lambda_coarse, dim3(std::max(1u, std::min(cdiv(D.nlam, 256), 4096u))), dim3(256), 0, st,
                       D.nlam, D.le_cnt, D.le_b, D.le_sub, D.boff, D.rtoff, D.ck, D.cblk, D.coff, le);
}

// ---- gathers ----
// yb[(boff + j) K + v] = sum of the partials of the items of subdomain s that
// cover j.  A partial starts at its item's first row j0, so the interleaved
// index i = j K + v of the item's own values is i - j0 K: no division, and the
// item list is uniform over the workgroup (scalar loads).  grid (chunks, subdomains)
__global__ void __launch_bounds__(256) k_part_reduce(const SymvItem *__restrict__ items, const int *__restrict__ item0,
                                                     const int *__restrict__ nitems, const int *__restrict__ M,
                                                     const int64_t *__restrict__ boff, int R, int K,
                                                     const double *__restrict__ ypart, double *__restrict__ yb) {
    const int s = blockIdx.y;
    const int64_t n = (int64_t)M[s] * K;
    const int i0 = item0[s], ni = nitems[s];
    double *y = yb + boff[s] * K;
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        double v = 0.0;
        for (int q = 0; q < ni; q++) {
            const SymvItem it = items[i0 + q];
            const int64_t lo = (int64_t)it.t0 * R * K;
            if (i >= lo) v += ypart[it.part_off * K + i - lo];
        }
        y[i] = v;
    }
}

// y[l K + v] = sum_e coef_e yb[b_e K + v]; with `a`, part gets the partial dot
// products of y with a
__global__ void k_lambda_gather(int nlam, int K, const int *__restrict__ cnt, const int64_t *__restrict__ lb,
                                const double *__restrict__ coef, const double *__restrict__ yb, double *__restrict__ y,
                                const double *__restrict__ a, double *__restrict__ part) {
    extern __shared__ double sh[];
    const Lines L = lines_of(K);
    double dot = 0.0;
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < nlam; l += (int64_t)gridDim.x * L.per) {
            double v = 0.0;
            const int c = cnt[l];
            for (int e = 0; e < c; e++) v += coef[2 * l + e] * yb[lb[2 * l + e] * K + L.v];
            y[l * K + L.v] = v;
            if (a) dot += v * a[l * K + L.v];
        }
    if (!a) return;  // uniform
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// xb[j K + v] = sum coef x[lambda K + v]
__global__ void k_boundary_gather(int64_t nb, int K, const int64_t *__restrict__ bl_ptr,
                                  const int *__restrict__ bl_lam, const double *__restrict__ coef,
                                  const double *__restrict__ x, double *__restrict__ xb) {
    const Lines L = lines_of(K);
    if (!L.on) return;
    for (int64_t j = (int64_t)blockIdx.x * L.per + L.li; j < nb; j += (int64_t)gridDim.x * L.per) {
        double v = 0.0;
        const int64_t q1 = bl_ptr[j + 1];
        for (int64_t q = bl_ptr[j]; q < q1; q++) v += coef[q] * x[(int64_t)bl_lam[q] * K + L.v];
        xb[j * K + L.v] = v;
    }
}

// yb = K_bb xb (lumped preconditioner).  One case: 16 lanes read a CSR row
// together (a thread per row chains its 27 or 81 entries: 19 us at 64
// subdomains of 5^3 elasticity); several cases: a thread per row and case, the
// K values of a column read together.
__global__ void __launch_bounds__(256) k_kbb_rows(int64_t nb, const int64_t *__restrict__ ptr,
                                                  const int64_t *__restrict__ col, const double *__restrict__ val,
                                                  const double *__restrict__ xb, double *__restrict__ yb) {
    const int l = threadIdx.x & 15;
    for (int64_t j = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4); j < nb; j += (int64_t)gridDim.x * 16) {
        double v = 0.0;
        const int64_t q1 = ptr[j + 1];
        for (int64_t q = ptr[j] + l; q < q1; q += 16) v += val[q] * xb[col[q]];
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
        if (l == 0) yb[j] = v;
    }
}
__global__ void k_kbb_lines(int64_t nb, int K, const int64_t *__restrict__ ptr, const int64_t *__restrict__ col,
                            const double *__restrict__ val, const double *__restrict__ xb, double *__restrict__ yb) {
    const Lines L = lines_of(K);
    if (!L.on) return;
    for (int64_t j = (int64_t)blockIdx.x * L.per + L.li; j < nb; j += (int64_t)gridDim.x * L.per) {
        double v = 0.0;
        const int64_t q1 = ptr[j + 1];
        for (int64_t q = ptr[j]; q < q1; q++) v += val[q] * xb[col[q] * K + L.v];
        yb[j * K + L.v] = v;
    }
}

// SUPER_DIRICHLET (clustercpu.cpp:243-314): S = K_bb - K_bi diag(K_ii)^-1 K_ib
// applied from the sparse blocks: t = diag(K_nn)^-1 K_nb x_b for the interior
// DOFs next to the boundary, then y_b = K_bb x_b - K_bn t
__global__ void k_superdir_near(int64_t n_near, int K, const int64_t *ptr, const int64_t *col, const double *val,
                                const double *diag, const double *xb, double *t) {
    const Lines L = lines_of(K);
    if (!L.on) return;
    for (int64_t g = (int64_t)blockIdx.x * L.per + L.li; g < n_near; g += (int64_t)gridDim.x * L.per) {
        double v = 0.0;
        for (int64_t q = ptr[g]; q < ptr[g + 1]; q++) v += val[q] * xb[col[q] * K + L.v];
        t[g * K + L.v] = v / diag[g];
    }
}
__global__ void k_superdir_bnd(int64_t nb, int K, const int64_t *kptr, const int64_t *kcol, const double *kval,
                               const int64_t *ptr, const int64_t *col, const double *val, const double *xb,
                               const double *t, double *yb) {
    const Lines L = lines_of(K);
    if (!L.on) return;
    for (int64_t j = (int64_t)blockIdx.x * L.per + L.li; j < nb; j += (int64_t)gridDim.x * L.per) {
        double v = 0.0;
        for (int64_t q = kptr[j]; q < kptr[j + 1]; q++) v += kval[q] * xb[kcol[q] * K + L.v];
        double w = 0.0;
        for (int64_t q = ptr[j]; q < ptr[j + 1]; q++) w += val[q] * t[col[q] * K + L.v];
        yb[j * K + L.v] = v - w;
    }
}

// ---- projector ----
// per subdomain s: out[(outoff[s] + a) K + v] = -sum over its lambda entries of
// sign R_s(j, a) x_lambda,v for a < k[s] (R_s row-major at RT + roff[s]): with the
// coarse basis this is G x = -(B R)^T x per subdomain.  The entries of a
// subdomain are one run of the boundary -> lambda CSR, so index, sign and row
// come coalesced and only x and the row of R depend on them (a thread per
// boundary DOF would chain three loads: 24 us at 512 x 10^3 with 1024 threads,
// 40 us at 2000 heat subdomains of ~330 entries).  One workgroup per subdomain.
// stop != null (first pass of an iteration): workgroup 0 copies the stop flags
// that the previous iteration decided (slot PCG_NEXT) to the ones this one obeys.
template <bool ONE>
__global__ void k_apply_G(const int *__restrict__ M, const int64_t *__restrict__ boff, const int *__restrict__ kcols,
                          const int64_t *__restrict__ outoff, const int64_t *__restrict__ roff,
                          const double *__restrict__ RT, const int64_t *__restrict__ bl_ptr,
                          const int *__restrict__ bl_lam, const int *__restrict__ bl_row,
                          const double *__restrict__ sign, int K, const double *__restrict__ x,
                          double *__restrict__ out, double *stop) {
    constexpr int KB = 8;  // columns per pass
    extern __shared__ double sh[];
    const int s = blockIdx.x, k = kcols[s];
    if (stop && s == 0 && (int)threadIdx.x < K)
        stop[threadIdx.x * PCG_SLOTS + PCG_STOP] = stop[threadIdx.x * PCG_SLOTS + PCG_NEXT];
    const int64_t b0 = boff[s], q0 = bl_ptr[b0], q1 = bl_ptr[b0 + M[s]];
    const double *Rs = RT + roff[s];
    const Lines L = lines_of(ONE ? 1 : K);
    for (int a0 = 0; a0 < k; a0 += KB) {
        const int kb = min(KB, k - a0);
        double acc[KB];
#pragma unroll
        for (int a = 0; a < KB; a++) acc[a] = 0.0;
        if (L.on) {
#pragma unroll 4
            for (int64_t q = q0 + L.li; q < q1; q += L.per) {
                const double xv = sign[q] * x[(int64_t)bl_lam[q] * (ONE ? 1 : K) + L.v];
                const double *r = Rs + (bl_row[q] - b0) * k + a0;
#pragma unroll
                for (int a = 0; a < KB; a++)
                    if (a < kb) acc[a] += r[a] * xv;
            }
        }
        if constexpr (ONE) {
            const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
            for (int a = 0; a < KB; a++) {
                if (a >= kb) break;
                double v = acc[a];
                for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
                if (lane == 0) sh[a * 16 + w] = v;
            }
            __syncthreads();
            if ((int)threadIdx.x < kb) {
                double v = 0.0;
                for (int q = 0; q < nw; q++) v += sh[threadIdx.x * 16 + q];
                out[outoff[s] + a0 + threadIdx.x] = -v;
            }
            __syncthreads();
        } else {
            for (int a = 0; a < kb; a++) {
                double v = 0.0;
#pragma unroll
                for (int b = 0; b < KB; b++)
                    if (b == a) v = acc[b];
                lines_sum(v, L, K, sh);
                if ((int)threadIdx.x < K) out[(outoff[s] + a0 + a) * K + threadIdx.x] = -sh[threadIdx.x];
            }
        }
    }
}

// d[(coff[b] + a) K + v] = sum over the subdomains of coarse block b of their
// partials (hybrid: several subdomains per block); a thread per (block, column, case)
__global__ void k_block_sum(int nblk, int K, const int *blk_ptr, const int *blk_sub, const int64_t *subpart_off,
                            const int *ck, const int *coff, const double *part, double *d) {
    // blocks hold at most 64 columns
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nblk * 64 * K; e += gridDim.x * blockDim.x) {
        const int b = e / (64 * K), a = e / K & 63, c = e % K;
        const int q0 = blk_ptr[b], q1 = blk_ptr[b + 1];
        if (a >= ck[blk_sub[q0]]) continue;
        double v = 0.0;
        for (int q = q0; q < q1; q++) v += part[(subpart_off[blk_sub[q]] + a) * K + c];
        d[(int64_t)(coff[b] + a) * K + c] = v;
    }
}

// e = GGinv d (symmetric, column access), one case
__global__ void __launch_bounds__(256) k_coarse_gemv(int nc, const double *__restrict__ Ginv,
                                                     const double *__restrict__ d, double *__restrict__ e) {
    __shared__ double red[4];
    const int i = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double *col = Ginv + (int64_t)i * nc;
    double v = 0.0;
#pragma unroll 4
    for (int j = threadIdx.x; j < nc; j += 256) v += col[j] * d[j];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) red[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) e[i] = (red[0] + red[1]) + (red[2] + red[3]);
}

// e = GGinv d for K <= 16 cases on MFMA (the N dimension of v_mfma_f64_16x16x4f64):
// GGinv is read once for all cases.  One workgroup per 16 rows, its four waves
// take every fourth chunk of 16 columns and meet in LDS in a fixed order.  A lane
// loads four consecutive columns of its row (32 B of the 128 B line that four
// lanes share) and the matching rows of d; products of columns past nc are zero.
__global__ void __launch_bounds__(256) k_coarse_block(int nc, int K, const double *__restrict__ Ginv,
                                                      const double *__restrict__ d, double *__restrict__ e) {
    __shared__ double sum[4][256];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, kq = lane >> 4;
    const int i0 = blockIdx.x * 16;
    const double *row = Ginv + (int64_t)min(i0 + l16, nc - 1) * nc;
    const int v = min(l16, K - 1);
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 16 * w; k0 < nc; k0 += 64) {
        double a[4], b[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int k = k0 + 4 * kq + s;
            const bool ok = k < nc;
            const double av = row[ok ? k : 0], bv = d[(int64_t)(ok ? k : 0) * K + v];
            a[s] = ok ? av : 0.0;
            b[s] = ok ? bv : 0.0;
        }
#pragma unroll
        for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) sum[w][(kq + 4 * q) * 16 + l16] = acc[q];
    __syncthreads();
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    if (i0 + r < nc && c < K)
        e[(int64_t)(i0 + r) * K + c] =
            (sum[0][threadIdx.x] + sum[1][threadIdx.x]) + (sum[2][threadIdx.x] + sum[3][threadIdx.x]);
}

// mode 0: y = x - G^T e ; mode 1: y = G^T e, (G^T e)_l = -sum_entries sign Rt(row) e_blk.
// with `part`: partial dot products of y with a (a == null: with y itself)
__global__ void k_project_finish(int nlam, int K, const int *__restrict__ cnt, const LamCoarse *__restrict__ lc,
                                 const double *__restrict__ sign, const double *__restrict__ RT,
                                 const double *__restrict__ e, const double *x, double *y, int mode,
                                 const double *__restrict__ a, double *__restrict__ part) {
    extern __shared__ double sh[];
    const Lines L = lines_of(K);
    double dot = 0.0;
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < nlam; l += (int64_t)gridDim.x * L.per) {
            double g = 0.0;
            const int c = cnt[l];
            for (int q = 0; q < c; q++) {
                const LamCoarse t = lc[2 * l + q];
                const double *r = RT + t.row, *es = e + (int64_t)t.off * K + L.v;
                double acc = 0.0;
                if (t.k == 6) {  // rigid motions in space: the row as three 16-byte loads
                    const d2u r0 = *(const d2u *)r, r1 = *(const d2u *)(r + 2), r2 = *(const d2u *)(r + 4);
                    acc = r0[0] * es[0] + r0[1] * es[K] + r1[0] * es[2 * K] + r1[1] * es[3 * K] + r2[0] * es[4 * K] +
                          r2[1] * es[5 * K];
                } else {
                    for (int b = 0; b < t.k; b++) acc += r[b] * es[(int64_t)b * K];
                }
                g -= sign[2 * l + q] * acc;
            }
            const double v = mode == 0 ? x[l * K + L.v] - g : g;
            y[l * K + L.v] = v;
            if (part) dot += v * (a ? a[l * K + L.v] : v);
        }
    if (!part) return;  // uniform
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// ---- dots and updates ----
__global__ void k_dot_lines(int64_t n, int K, const double *__restrict__ a, const double *__restrict__ b,
                            double *__restrict__ part) {
    extern __shared__ double sh[];
    const Lines L = lines_of(K);
    double dot = 0.0;
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per)
            dot += a[l * K + L.v] * b[l * K + L.v];
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// tolerance and flags of a PCG from the partials of ||P r0||^2 and ||b||^2:
// tol = precision min(||P r0||, ||b||), or tol_abs when that is positive
__global__ void __launch_bounds__(256) k_pcg_init(int K, const double *part_r, const double *part_b, int np,
                                                  double precision, double tol_abs, double *scal, PcgRecord *rec) {
    __shared__ double sh[256], rr[16];
    const Lines L = lines_of(K);
    partials_sum(part_r, np, L, K, sh);
    const int v = threadIdx.x;
    if (v < K) rr[v] = sh[v];
    partials_sum(part_b, np, L, K, sh);
    if (v >= K) return;
    double *s = scal + v * PCG_SLOTS;
    s[PCG_YW] = s[PCG_YW_PREV] = s[PCG_PAP] = s[PCG_WW] = 0.0;
    s[PCG_STOP] = s[PCG_NEXT] = s[PCG_ITERS] = s[PCG_COUNT] = 0.0;
    const double tol = tol_abs > 0.0 ? tol_abs : precision * fmin(sqrt(rr[v]), sqrt(sh[v]));
    s[PCG_TOL] = tol;
    rec->tol[v] = tol;
    rec->bb[v] = sh[v];
}

// beta = yw / yw_prev (first: 0), p = y + beta p of the cases that still run,
// from the partials of y.w; workgroup 0 finishes ||w||^2, decides the stop flags
// of the next iteration (||w|| < tol, or not finite) and reports to the host
// record (pinned memory): the host queues the next iteration, or not, while the
// dual operator of this one runs, so the stop test costs no wait on either side.
__global__ void k_p_update(int64_t n, int K, double *__restrict__ p, const double *__restrict__ y,
                           const double *__restrict__ part_yw, const double *__restrict__ part_ww, int np, int first,
                           double *scal, PcgRecord *rec) {
    extern __shared__ double sh[];
    const Lines L = lines_of(K);
    partials_sum(part_yw, np, L, K, sh);
    const double yw = sh[L.v], prev = scal[L.v * PCG_SLOTS + PCG_YW_PREV];
    const bool run = L.on && scal[L.v * PCG_SLOTS + PCG_STOP] == 0.0;
    const double beta = first ? 0.0 : yw / prev;
    if (run)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per)
            p[l * K + L.v] = first ? y[l * K + L.v] : y[l * K + L.v] + beta * p[l * K + L.v];
    if (blockIdx.x) return;
    partials_sum(part_ww, np, L, K, sh);
    if (threadIdx.x >= 64) return;
    const int v = threadIdx.x;
    int active = 0;
    if (v < K) {
        double *s = scal + v * PCG_SLOTS;
        if (run) {
            const double ww = sh[v];
            const bool stop = sqrt(ww) < s[PCG_TOL] || !isfinite(ww);
            s[PCG_YW] = yw;
            s[PCG_WW] = ww;
            s[PCG_ITERS] += 1.0;
            s[PCG_NEXT] = stop ? 1.0 : 0.0;
            rec->ww[v] = ww;
            rec->iters[v] = (int)s[PCG_ITERS];
            active = !stop;
        }
    }
    const unsigned long long any = __ballot(active);
    if (v == 0) {
        scal[PCG_COUNT] += 1.0;
        rec->active = any != 0;
    }
    __threadfence_system();
    if (v == 0) __hip_atomic_store(&rec->count, (int)scal[PCG_COUNT], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// alpha = yw / pAp; x += alpha p; r -= alpha Ap of the cases that still run
__global__ void k_xr_update(int64_t n, int K, double *__restrict__ x, double *__restrict__ r,
                            const double *__restrict__ p, const double *__restrict__ Ap,
                            const double *__restrict__ part_pAp, int np, double *scal) {
    extern __shared__ double sh[];
    const Lines L = lines_of(K);
    partials_sum(part_pAp, np, L, K, sh);
    const double yw = scal[L.v * PCG_SLOTS + PCG_YW], alpha = yw / sh[L.v];
    const bool run = L.on && scal[L.v * PCG_SLOTS + PCG_STOP] == 0.0;
    if (!run) return;
    for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) {
        x[l * K + L.v] += alpha * p[l * K + L.v];
        r[l * K + L.v] -= alpha * Ap[l * K + L.v];
    }
    if (blockIdx.x == 0 && (int)threadIdx.x < K) {
        scal[threadIdx.x * PCG_SLOTS + PCG_PAP] = sh[threadIdx.x];
        scal[threadIdx.x * PCG_SLOTS + PCG_YW_PREV] = yw;  // read by the next iteration only
    }
}

// y_v -= c for every case
__global__ void k_sub_lines(int64_t n, int K, double *__restrict__ y, const double *__restrict__ c) {
    const Lines L = lines_of(K);
    if (!L.on) return;
    for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) y[l * K + L.v] -= c[l];
}

// ------------------------------------------------------------ launchers ----
void launch_sub_lines(int64_t n, int K, double *y, const double *c, hipStream_t st) {
    hipLaunchKernelGGL(k_sub_lines, dim3(line_grid(n, K)), dim3(line_threads(K)), 0, st, n, K, y, c);
}

void launch_part_reduce(const DualDev &D, const SymvItem *items, const int *item0, const int *nitems, int R, int K,
                        const double *ypart, double *yb, hipStream_t st) {
    const unsigned g = std::max(1u, std::min(cdiv((int64_t)D.max_m * K, 256), 64u));
    hipLaunchKernelGGL(k_part_reduce, dim3(g, D.nsub), dim3(256), 0, st, items, item0, nitems, D.m, D.boff, R, K, ypart,
                       yb);
}

void launch_lambda_gather(const DualDev &D, int K, const double *yb, bool scaled, double *y, hipStream_t st,
                          const double *a, double *part) {
    const int T = line_threads(K);
    hipLaunchKernelGGL(k_lambda_gather, dim3(part ? (unsigned)dot_blocks(D.nlam, K) : line_grid(D.nlam, K)), dim3(T),
                       part ? T * sizeof(double) : 0, st, D.nlam, K, D.le_cnt, D.le_b,
                       scaled ? D.le_sscale : D.le_sign, yb, y, a, part);
}

void launch_boundary_gather(const DualDev &D, int K, const double *x, bool scaled, double *xb, hipStream_t st) {
    hipLaunchKernelGGL(k_boundary_gather, dim3(line_grid(D.nbnd, K)), dim3(line_threads(K)), 0, st, D.nbnd, K, D.bl_ptr,
                       D.bl_lam, scaled ? D.bl_sscale : D.bl_sign, x, xb);
}

void launch_kbb(const DualDev &D, int K, const double *xb, double *yb, hipStream_t st) {
    if (K == 1)
        hipLaunchKernelGGL(k_kbb_rows, dim3(std::max(1u, std::min(cdiv(D.nbnd, 16), 8192u))), dim3(256), 0, st, D.nbnd,
                           D.kbb_ptr, D.kbb_col, D.kbb_val, xb, yb);
    else
        hipLaunchKernelGGL(k_kbb_lines, dim3(line_grid(D.nbnd, K)), dim3(line_threads(K)), 0, st, D.nbnd, K, D.kbb_ptr,
                           D.kbb_col, D.kbb_val, xb, yb);
}

void launch_superdir(const DualDev &D, int K, int64_t n_near, const int64_t *sib_ptr, const int64_t *sib_col,
                     const double *sib_val, const double *sdiag, const int64_t *sbi_ptr, const int64_t *sbi_col,
                     const double *sbi_val, double *t, const double *xb, double *yb, hipStream_t st) {
    if (n_near > 0)
        hipLaunchKernelGGL(k_superdir_near, dim3(line_grid(n_near, K)), dim3(line_threads(K)), 0, st, n_near, K, sib_ptr,
                           sib_col, sib_val, sdiag, xb, t);
    hipLaunchKernelGGL(k_superdir_bnd, dim3(line_grid(D.nbnd, K)), dim3(line_threads(K)), 0, st, D.nbnd, K, D.kbb_ptr,
                       D.kbb_col, D.kbb_val, sbi_ptr, sbi_col, sbi_val, xb, t, yb);
}

// out[(outoff[s] + a) K + v] = -R_s^T (B_s^T x_v).  Threads per subdomain: about
// two entries each, 256 to 1024 (2000 heat subdomains of 330 lambda entries fill
// the GPU in one round with 256; 64 to 512 subdomains of 2000 and more need the
// loads in flight)
static void apply_G(const DualDev &D, int K, const int *kcols, const int64_t *outoff, const int64_t *roff,
                    const double *RT, const double *x, double *out, double *stop, hipStream_t st) {
    const int64_t e = D.nle * K / std::max(D.nsub, 1) / 2;
    const int T = e <= 256 ? 256 : e <= 512 ? 512 : 1024;
    if (K == 1)
        hipLaunchKernelGGL(k_apply_G<true>, dim3(D.nsub), dim3(T), 8 * 16 * sizeof(double), st, D.m, D.boff, kcols,
                           outoff, roff, RT, D.bl_ptr, D.bl_lam, D.bl_row, D.bl_sign, 1, x, out, stop);
    else
        hipLaunchKernelGGL(k_apply_G<false>, dim3(D.nsub), dim3(T), T * sizeof(double), st, D.m, D.boff, kcols, outoff,
                           roff, RT, D.bl_ptr, D.bl_lam, D.bl_row, D.bl_sign, K, x, out, stop);
}

void launch_project(const DualDev &D, int K, const double *x, double *y, int mode, hipStream_t st, const double *a,
                    double *part, double *stop) {
    // mode 0: y = P x;  mode 1: y = G^T GGinv x (x coarse);  mode 2: y = GGinv G x (coarse out)
    const double *din = x;
    if (mode != 1) {
        apply_G(D, K, D.ck, D.dsub_off, D.rtoff, D.RtT, x, D.dsub, stop, st);
        // one subdomain per coarse block in coarse order (TOTAL_FETI): the
        // subdomain results are the coarse vector
        din = D.coarse_direct ? D.dsub : D.cd;
        if (!D.coarse_direct)
            hipLaunchKernelGGL(k_block_sum, dim3(std::max(1u, std::min(cdiv((int64_t)D.nblk * 64 * K, 256), 4096u))),
                               dim3(256), 0, st, D.nblk, K, D.blk_ptr, D.blk_sub, D.dsub_off, D.ck, D.coff, D.dsub,
                               D.cd);
    }
    double *eout = mode == 2 ? y : D.ce;
    if (K == 1)
        hipLaunchKernelGGL(k_coarse_gemv, dim3(D.ncoarse), dim3(256), 0, st, D.ncoarse, D.GGinv, din, eout);
    else
        hipLaunchKernelGGL(k_coarse_block, dim3(cdiv(D.ncoarse, 16)), dim3(256), 0, st, D.ncoarse, K, D.GGinv, din,
                           eout);
    if (mode == 2) return;
    const int T = line_threads(K);
    hipLaunchKernelGGL(k_project_finish, dim3(part ? (unsigned)dot_blocks(D.nlam, K) : line_grid(D.nlam, K)), dim3(T),
                       part ? T * sizeof(double) : 0, st, D.nlam, K, D.le_cnt, D.le_coarse, D.le_sign, D.RtT, D.ce, x,
                       y, mode, a, part);
}

void launch_subdomain_kernel_dots(const DualDev &D, int K, const double *x, double *out, hipStream_t st) {
    apply_G(D, K, D.kdim, D.asub, D.rboff, D.RbT, x, out, nullptr, st);
}

void launch_dot_lines(int64_t n, int K, const double *a, const double *b, double *part, hipStream_t st) {
    const int T = line_threads(K);
    hipLaunchKernelGGL(k_dot_lines, dim3(dot_blocks(n, K)), dim3(T), T * sizeof(double), st, n, K, a, b, part);
}

void launch_pcg_init(int K, const double *part_r, const double *part_b, int np, double precision, double tol_abs,
                     double *scal, PcgRecord *rec, hipStream_t st) {
    hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(256), 0, st, K, part_r, part_b, np, precision, tol_abs, scal, rec);
}

// the update passes read every partial in each workgroup: two workgroups per CU
static unsigned update_grid(int64_t n, int K) { return std::min(line_grid(n, K), 512u); }

void launch_p_update(int64_t n, int K, double *p, const double *y, const double *part_yw, const double *part_ww,
                     int np, bool first, double *scal, PcgRecord *rec, hipStream_t st) {
    const int T = line_threads(K);
    hipLaunchKernelGGL(k_p_update, dim3(update_grid(n, K)), dim3(T), T * sizeof(double), st, n, K, p, y, part_yw,
                       part_ww, np, first ? 1 : 0, scal, rec);
}

void launch_xr_update(int64_t n, int K, double *x, double *r, const double *p, const double *Ap,
                      const double *part_pAp, int np, double *scal, hipStream_t st) {
    const int T = line_threads(K);
    hipLaunchKernelGGL(k_xr_update, dim3(update_grid(n, K)), dim3(T), T * sizeof(double), st, n, K, x, r, p, Ap,
                       part_pAp, np, scal);
}

}  // namespace esp
