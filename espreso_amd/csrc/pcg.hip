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

// Threads of a workgroup as lines of K values, W consecutive cases a thread (W = 2:
// 16-byte accesses, K even): thread (li, v), li < per, v the first case of the thread,
// `width` threads a line, K / W or (pad) the next power of two, so that no line straddles
// a wave.  Pairs of cases halve the instructions and requests of a pass, which is what
// bounds it once thousands of workgroups are in flight: at 669000 lines of 16 cases (86
// MB a vector) lambda gather 100 -> 48 us, boundary gather 99 -> 79, projector finish
// 152 -> 47, partial sums 128 -> 76 (5 TB/s); several lines a thread gain nothing more.
constexpr int LINE_CASES = 16;  // largest K
template <int W>
struct Lines {
    int per, li, v, width;
    bool on;
    __device__ __forceinline__ explicit Lines(int K, bool pad = false) {
        width = K / W;
        if (pad) width = width > 8 ? 16 : width > 4 ? 8 : width > 2 ? 4 : width;
        per = blockDim.x;
        li = threadIdx.x;
        v = 0;
        if (width > 1) {
            per = blockDim.x / width;
            li = threadIdx.x / width;
            v = (threadIdx.x - li * width) * W;
        }
        on = li < per && v < K;
        if (!on) v = 0;
    }
};
template <int W>
struct Vals {
    double d[W];
};
template <int W>
__device__ __forceinline__ Vals<W> line_load(const double *p) {
    Vals<W> r;
    if constexpr (W == 2) {
        const double2 x = *(const double2 *)p;
        r.d[0] = x.x;
        r.d[1] = x.y;
    } else {
        r.d[0] = *p;
    }
    return r;
}
template <int W>
__device__ __forceinline__ void line_store(double *p, const Vals<W> &x) {
    if constexpr (W == 2) *(double2 *)p = make_double2(x.d[0], x.d[1]);
    else *p = x.d[0];
}

// sum of `val` over the lines of the workgroup, per case, into sh[v], in a fixed
// order (lines that divide a wave: a butterfly, then the waves; else a tree in LDS);
// every thread may read sh[v] afterwards.  sh: LINE_SUM doubles of LDS
constexpr int LINE_SUM = 512 + LINE_CASES;
template <int W>
__device__ __forceinline__ void lines_sum(Vals<W> val, const Lines<W> &L, int K, double *sh) {
    if ((L.width & (L.width - 1)) == 0) {
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
        for (int i = 0; i < W; i++)
            for (int o = 32; o >= L.width; o >>= 1) val.d[i] += __shfl_xor(val.d[i], o, 64);
        __syncthreads();
        if (lane < L.width)
#pragma unroll
            for (int i = 0; i < W; i++) sh[(w + 1) * K + L.v + i] = val.d[i];
        __syncthreads();
        if ((int)threadIdx.x < K) {
            double s = 0.0;
            for (int i = 1; i <= nw; i++) s += sh[i * K + threadIdx.x];
            sh[threadIdx.x] = s;
        }
        __syncthreads();
        return;
    }
    // at most 512 threads: the second value of a thread in a second turn
    double *t = sh + LINE_CASES;
    double sum[W];
#pragma unroll
    for (int i = 0; i < W; i++) {
        __syncthreads();
        t[threadIdx.x] = L.on ? val.d[i] : 0.0;
        __syncthreads();
        int h = 1;
        while (2 * h < L.per) h *= 2;
        for (; h > 0; h >>= 1) {
            if (L.on && L.li < h && L.li + h < L.per) t[threadIdx.x] += t[threadIdx.x + h * L.width];
            __syncthreads();
        }
        sum[i] = t[threadIdx.x];
    }
    if (L.li == 0)
#pragma unroll
        for (int i = 0; i < W; i++) sh[L.v + i] = sum[i];
    __syncthreads();
}

// sum of np partials per case, part[b K + v], into sh[v]
template <int W>
__device__ __forceinline__ void partials_sum(const double *__restrict__ part, int np, const Lines<W> &L, int K,
                                             double *sh) {
    Vals<W> a = {};
    if (L.on)
#pragma unroll 4
        for (int b = L.li; b < np; b += L.per) {
            const Vals<W> x = line_load<W>(part + (int64_t)b * K + L.v);
#pragma unroll
            for (int i = 0; i < W; i++) a.d[i] += x.d[i];
        }
    lines_sum(a, L, K, sh);
}

constexpr int LINE_THREADS_1 = 256, LINE_THREADS_K = 512;
static inline int line_threads(int K) { return K == 1 ? LINE_THREADS_1 : LINE_THREADS_K; }
// lines per workgroup
static inline int64_t line_per(int K) { return line_threads(K) / (K % 2 ? K : K / 2); }
// workgroups of a pass over n lines that sums a dot product: one partial each.
// At most 4 (K = 1) or 2 workgroups per CU: the consumer of the partials reads
// them all in every workgroup
int dot_blocks(int64_t n, int K) {
    const int64_t per = line_per(K);
    return (int)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, K == 1 ? 1024 : 512));
}
static inline unsigned line_grid(int64_t n, int K) {
    const int64_t per = line_per(K);
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, 4096));
}
// kernel<W> for K cases
#define ESP_LINES(KERNEL, K, grid, ...)                                                                            \
    do {                                                                                                           \
        if ((K) % 2)                                                                                               \
            hipLaunchKernelGGL(KERNEL<1>, dim3(grid), dim3(line_threads(K)), 0, st, __VA_ARGS__);                  \
        else                                                                                                       \
            hipLaunchKernelGGL(KERNEL<2>, dim3(grid), dim3(line_threads(K)), 0, st, __VA_ARGS__);                  \
    } while (0)

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
// item list is uniform over the workgroup (scalar loads).  An item that starts
// below i is read at its start and left out (no branch between the loads).  grid
// (chunks, subdomains); bound by the partials (16 cases: 2.4 times the result)
template <int W>
__global__ void __launch_bounds__(256) k_part_reduce(const SymvItem *__restrict__ items, const int *__restrict__ item0,
                                                     const int *__restrict__ nitems, const int *__restrict__ M,
                                                     const int64_t *__restrict__ boff, int R, int K,
                                                     const double *__restrict__ ypart, double *__restrict__ yb) {
    const int s = blockIdx.y;
    const int64_t n = (int64_t)M[s] * K;
    const int i0 = item0[s], ni = nitems[s];
    double *y = yb + boff[s] * K;
    for (int64_t i = (blockIdx.x * 256 + threadIdx.x) * W; i < n; i += (int64_t)gridDim.x * 256 * W) {
        Vals<W> v = {};
#pragma unroll 4
        for (int q = 0; q < ni; q++) {
            const SymvItem it = items[i0 + q];
            const int64_t lo = (int64_t)it.t0 * R * K;
            const Vals<W> x = line_load<W>(ypart + it.part_off * K + (i >= lo ? i - lo : 0));
#pragma unroll
            for (int k = 0; k < W; k++) v.d[k] += i >= lo ? x.d[k] : 0.0;
        }
        line_store<W>(y + i, v);
    }
}

// y[l K + v] = sum_e coef_e yb[b_e K + v] (one or two entries); with `a`, part gets
// the partial dot products of y with a
template <int W>
__global__ void k_lambda_gather(int nlam, int K, const int *__restrict__ cnt, const int64_t *__restrict__ lb,
                                const double *__restrict__ coef, const double *__restrict__ yb, double *__restrict__ y,
                                const double *__restrict__ a, double *__restrict__ part) {
    __shared__ double sh[LINE_SUM];
    const Lines<W> L(K);
    Vals<W> dot = {};
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < nlam; l += (int64_t)gridDim.x * L.per) {
            const bool two = cnt[l] > 1;
            const int64_t b0 = lb[2 * l], b1 = lb[2 * l + 1];
            const double c0 = coef[2 * l], c1 = coef[2 * l + 1];
            const Vals<W> x0 = line_load<W>(yb + b0 * K + L.v), x1 = line_load<W>(yb + (two ? b1 : b0) * K + L.v);
            Vals<W> v, av = {};
            if (a) av = line_load<W>(a + l * K + L.v);
#pragma unroll
            for (int i = 0; i < W; i++) {
                v.d[i] = c0 * x0.d[i];
                if (two) v.d[i] += c1 * x1.d[i];
                dot.d[i] += v.d[i] * av.d[i];
            }
            line_store<W>(y + l * K + L.v, v);
        }
    if (!a) return;  // uniform
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// xb[j K + v] = sum coef x[lambda K + v]
template <int W>
__global__ void k_boundary_gather(int64_t nb, int K, const int64_t *__restrict__ bl_ptr,
                                  const int *__restrict__ bl_lam, const double *__restrict__ coef,
                                  const double *__restrict__ x, double *__restrict__ xb) {
    const Lines<W> L(K);
    if (!L.on) return;
    for (int64_t j = (int64_t)blockIdx.x * L.per + L.li; j < nb; j += (int64_t)gridDim.x * L.per) {
        Vals<W> v = {};
        const int64_t q1 = bl_ptr[j + 1];
        for (int64_t q = bl_ptr[j]; q < q1; q++) {
            const double c = coef[q];
            const Vals<W> xl = line_load<W>(x + (int64_t)bl_lam[q] * K + L.v);
#pragma unroll
            for (int i = 0; i < W; i++) v.d[i] += c * xl.d[i];
        }
        line_store<W>(xb + j * K + L.v, v);
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
    const Lines<1> L(K);
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
    const Lines<1> L(K);
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
    const Lines<1> L(K);
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
// KB columns of the basis per pass (heat has one, elasticity six); one case reduces
// them together (a butterfly per column is 6 shuffles each).  Bound by the gather of x
// and the rows: 16 cases at 2000 heat subdomains 140 -> 47 us, 5 cases at 512 elasticity
// subdomains 56 -> 28 us (rows as 16-byte loads without a branch, cases in pairs, one LDS
// exchange for all columns), one case at 512 of 1806 boundary DOFs 25.6 -> 18.3 us.
template <int W, int KB>
__global__ void k_apply_G(const int *__restrict__ M, const int64_t *__restrict__ boff, const int *__restrict__ kcols,
                          const int64_t *__restrict__ outoff, const int64_t *__restrict__ roff,
                          const double *__restrict__ RT, const int64_t *__restrict__ bl_ptr,
                          const int *__restrict__ bl_lam, const int *__restrict__ bl_row,
                          const double *__restrict__ sign, int K, const double *__restrict__ x,
                          double *__restrict__ out, double *stop) {
    __shared__ double sh[KB * 16 * LINE_CASES];  // [column][wave][case]
    const int s = blockIdx.x, k = kcols[s];
    if (stop && s == 0 && (int)threadIdx.x < K)
        stop[threadIdx.x * PCG_SLOTS + PCG_STOP] = stop[threadIdx.x * PCG_SLOTS + PCG_NEXT];
    const int64_t b0 = boff[s], q0 = bl_ptr[b0];
    const int n = (int)(bl_ptr[b0 + M[s]] - q0);
    const double *Rs = RT + roff[s];
    const Lines<W> L(K, true);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    constexpr int UNR = W == 2 ? 2 : 4;  // four pairs take so many registers that one workgroup fits a CU (62 us, not 47)
    for (int a0 = 0; a0 < k; a0 += KB) {
        const int kb = min(KB, k - a0);
        Vals<W> acc[KB] = {};
        if (L.on) {
            auto entry = [&](int q, bool full) {
                const double sg = sign[q0 + q];
                const Vals<W> xv = line_load<W>(x + (int64_t)bl_lam[q0 + q] * K + L.v);
                const double *r = Rs + (bl_row[q0 + q] - b0) * k + a0;
                double ra[KB];
                if (full) {
                    if constexpr (KB % 2 == 0) {
#pragma unroll
                        for (int a = 0; a < KB; a += 2) {
                            const d2u rr = *(const d2u *)(r + a);
                            ra[a] = rr[0];
                            ra[a + 1] = rr[1];
                        }
                    } else {
                        ra[0] = r[0];
                    }
                } else {
#pragma unroll
                    for (int a = 0; a < KB; a++) ra[a] = a < kb ? r[a] : 0.0;
                }
#pragma unroll
                for (int a = 0; a < KB; a++)
#pragma unroll
                    for (int i = 0; i < W; i++) acc[a].d[i] += ra[a] * (sg * xv.d[i]);
            };
            // no branch between the loads of the usual case
            if (kb == KB) {
#pragma unroll UNR
                for (int q = L.li; q < n; q += L.per) entry(q, true);
            } else {
                for (int q = L.li; q < n; q += L.per) entry(q, false);
            }
        }
        __syncthreads();
        if (KB == 6 && W == 1 && L.width == 1) {
            double v[8];
#pragma unroll
            for (int a = 0; a < 8; a++) v[a] = a < KB ? acc[a % KB].d[0] : 0.0;
            const double t = wave_rows_reduce<8, double>(v, lane);
            if ((lane & 7) == 0 && lane < 8 * KB) sh[(lane >> 3) * 16 + w] = t;
        } else {
#pragma unroll
            for (int a = 0; a < KB; a++)
                if (a < kb)
#pragma unroll
                    for (int i = 0; i < W; i++) {
                        double v = acc[a].d[i];
                        for (int o = 32; o >= L.width; o >>= 1) v += __shfl_xor(v, o, 64);
                        if (lane < L.width && L.on) sh[(a * 16 + w) * K + L.v + i] = v;
                    }
        }
        __syncthreads();
        for (int c = threadIdx.x; c < kb * K; c += blockDim.x) {
            const int a = c / K, v = c - a * K;
            double t = 0.0;
            for (int q = 0; q < nw; q++) t += sh[(a * 16 + q) * K + v];
            out[(outoff[s] + a0 + a) * K + v] = -t;
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
// GGinv is read once for all cases.  One workgroup per 16 rows, its 16 waves take every
// 16th chunk of 16 columns, four chunks' loads at a time, and meet in LDS in a fixed
// order; products of columns past nc are zero.  GGinv is symmetric, so 16 lanes read 128
// consecutive bytes of a column; lanes along a row touch 16 lines a load, and one workgroup
// a CU then gets 12 GB/s: 47 us with four waves and 32 with 16 at 3072 columns (75 MB) and 5
// cases, now 20; 33, 23 and 15 at 2000 and 16.
__global__ void __launch_bounds__(1024) k_coarse_block(int nc, int K, const double *__restrict__ Ginv,
                                                      const double *__restrict__ d, double *__restrict__ e) {
    __shared__ double sum[16][256];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, kq = lane >> 4;
    const int i0 = blockIdx.x * 16;
    const double *col = Ginv + min(i0 + l16, nc - 1);
    const int v = min(l16, K - 1);
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    constexpr int U = 4;  // chunks loaded before the first is used
    for (int k0 = 16 * w; k0 < nc; k0 += 256 * U) {
        double a[U][4], b[U][4];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int k = k0 + 256 * u + 4 * s + kq;
                const bool ok = k < nc;
                const double av = col[(int64_t)(ok ? k : 0) * nc], bv = d[(int64_t)(ok ? k : 0) * K + v];
                a[u][s] = ok ? av : 0.0;
                b[u][s] = ok ? bv : 0.0;
            }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][s], b[u][s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) sum[w][(kq + 4 * q) * 16 + l16] = acc[q];
    __syncthreads();
    if (threadIdx.x >= 256) return;
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    double v2 = 0.0;
#pragma unroll
    for (int q = 0; q < 16; q++) v2 += sum[q][threadIdx.x];
    if (i0 + r < nc && c < K) e[(int64_t)(i0 + r) * K + c] = v2;
}

// mode 0: y = x - G^T e ; mode 1: y = G^T e, (G^T e)_l = -sum_entries sign Rt(row) e_blk.
// with `part`: partial dot products of y with a (a == null: with y itself)
template <int W>
__global__ void k_project_finish(int nlam, int K, const int *__restrict__ cnt, const LamCoarse *__restrict__ lc,
                                 const double *__restrict__ sign, const double *__restrict__ RT,
                                 const double *__restrict__ e, const double *x, double *y, int mode,
                                 const double *__restrict__ a, double *__restrict__ part) {
    __shared__ double sh[LINE_SUM];
    const Lines<W> L(K);
    Vals<W> dot = {};
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < nlam; l += (int64_t)gridDim.x * L.per) {
            // both entries, x and a are loaded before the first is used
            LamCoarse t[2] = {lc[2 * l], lc[2 * l + 1]};
            if (cnt[l] < 2) t[1].k = 0;
            const double sg[2] = {sign[2 * l], sign[2 * l + 1]};
            Vals<W> g = {}, v = {}, av = {};
            if (mode == 0) v = line_load<W>(x + l * K + L.v);
            if (a) av = line_load<W>(a + l * K + L.v);
            if (t[0].k <= 1 && t[1].k <= 1) {  // one column (heat) or none (any value is read, and not used)
                double r[2];
                Vals<W> ev[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const bool on = t[q].k > 0;
                    r[q] = *(on ? RT + t[q].row : sign);
                    ev[q] = line_load<W>(on ? e + (int64_t)t[q].off * K + L.v : y + l * K + L.v);
                }
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if (t[q].k > 0)
#pragma unroll
                        for (int i = 0; i < W; i++) g.d[i] -= sg[q] * (r[q] * ev[q].d[i]);
            } else {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const double *r = RT + t[q].row, *es = e + (int64_t)t[q].off * K + L.v;
                    Vals<W> acc = {};
                    if (t[q].k == 6) {  // rigid motions in space: the row as three 16-byte loads
                        const d2u rr[3] = {*(const d2u *)r, *(const d2u *)(r + 2), *(const d2u *)(r + 4)};
                        Vals<W> ev[6];
#pragma unroll
                        for (int b = 0; b < 6; b++) ev[b] = line_load<W>(es + b * K);
#pragma unroll
                        for (int b = 0; b < 6; b++)
#pragma unroll
                            for (int i = 0; i < W; i++) acc.d[i] += rr[b >> 1][b & 1] * ev[b].d[i];
                    } else {
                        for (int b = 0; b < t[q].k; b++) {
                            const Vals<W> ev = line_load<W>(es + b * K);
#pragma unroll
                            for (int i = 0; i < W; i++) acc.d[i] += r[b] * ev.d[i];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < W; i++) g.d[i] -= sg[q] * acc.d[i];
                }
            }
#pragma unroll
            for (int i = 0; i < W; i++) {
                v.d[i] = mode == 0 ? v.d[i] - g.d[i] : g.d[i];
                if (part) dot.d[i] += v.d[i] * (a ? av.d[i] : v.d[i]);
            }
            line_store<W>(y + l * K + L.v, v);
        }
    if (!part) return;  // uniform
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// ---- dots and updates ----
template <int W>
__global__ void k_dot_lines(int64_t n, int K, const double *__restrict__ a, const double *__restrict__ b,
                            double *__restrict__ part) {
    __shared__ double sh[LINE_SUM];
    const Lines<W> L(K);
    Vals<W> dot = {};
    if (L.on)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) {
            const Vals<W> x = line_load<W>(a + l * K + L.v), z = line_load<W>(b + l * K + L.v);
#pragma unroll
            for (int i = 0; i < W; i++) dot.d[i] += x.d[i] * z.d[i];
        }
    lines_sum(dot, L, K, sh);
    if ((int)threadIdx.x < K) part[(int64_t)blockIdx.x * K + threadIdx.x] = sh[threadIdx.x];
}

// tolerance and flags of a PCG from the partials of ||P r0||^2 and ||b||^2:
// tol = precision min(||P r0||, ||b||), or tol_abs when that is positive
__global__ void __launch_bounds__(256) k_pcg_init(int K, const double *part_r, const double *part_b, int np,
                                                  double precision, double tol_abs, double *scal, PcgRecord *rec) {
    __shared__ double sh[LINE_SUM], rr[LINE_CASES];
    const Lines<1> L(K);
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
template <int W>
__global__ void k_p_update(int64_t n, int K, double *__restrict__ p, const double *__restrict__ y,
                           const double *__restrict__ part_yw, const double *__restrict__ part_ww, int np, int first,
                           double *scal, PcgRecord *rec) {
    __shared__ double sh[LINE_SUM], yws[LINE_CASES];
    const Lines<W> L(K);
    partials_sum(part_yw, np, L, K, sh);
    if ((int)threadIdx.x < K) yws[threadIdx.x] = sh[threadIdx.x];
    double beta[W];
    bool run[W], any_run = false;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const double *s = scal + (L.v + i) * PCG_SLOTS;
        run[i] = L.on && s[PCG_STOP] == 0.0;
        beta[i] = first ? 0.0 : sh[L.v + i] / s[PCG_YW_PREV];
        any_run |= run[i];
    }
    if (any_run)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) {
            const Vals<W> yv = line_load<W>(y + l * K + L.v);
            Vals<W> pv = line_load<W>(p + l * K + L.v);
#pragma unroll
            for (int i = 0; i < W; i++)
                if (run[i]) pv.d[i] = first ? yv.d[i] : yv.d[i] + beta[i] * pv.d[i];
            line_store<W>(p + l * K + L.v, pv);
        }
    if (blockIdx.x) return;
    partials_sum(part_ww, np, L, K, sh);
    if (threadIdx.x >= 64) return;
    const int v = threadIdx.x;
    int active = 0;
    if (v < K) {
        double *s = scal + v * PCG_SLOTS;
        if (s[PCG_STOP] == 0.0) {
            const double ww = sh[v];
            const bool stop = sqrt(ww) < s[PCG_TOL] || !isfinite(ww);
            s[PCG_YW] = yws[v];
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
template <int W>
__global__ void k_xr_update(int64_t n, int K, double *__restrict__ x, double *__restrict__ r,
                            const double *__restrict__ p, const double *__restrict__ Ap,
                            const double *__restrict__ part_pAp, int np, double *scal) {
    __shared__ double sh[LINE_SUM];
    const Lines<W> L(K);
    partials_sum(part_pAp, np, L, K, sh);
    double alpha[W];
    bool run[W], any = false;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const double *s = scal + (L.v + i) * PCG_SLOTS;
        run[i] = L.on && s[PCG_STOP] == 0.0;
        alpha[i] = s[PCG_YW] / sh[L.v + i];
        any |= run[i];
    }
    if (any)
        for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) {
            const int64_t o = l * K + L.v;
            const Vals<W> pv = line_load<W>(p + o), Av = line_load<W>(Ap + o);
            Vals<W> xv = line_load<W>(x + o), rv = line_load<W>(r + o);
#pragma unroll
            for (int i = 0; i < W; i++)
                if (run[i]) {
                    xv.d[i] += alpha[i] * pv.d[i];
                    rv.d[i] -= alpha[i] * Av.d[i];
                }
            line_store<W>(x + o, xv);
            line_store<W>(r + o, rv);
        }
    if (blockIdx.x == 0 && (int)threadIdx.x < K) {
        double *s = scal + threadIdx.x * PCG_SLOTS;
        if (s[PCG_STOP] == 0.0) {
            s[PCG_PAP] = sh[threadIdx.x];
            s[PCG_YW_PREV] = s[PCG_YW];  // read by the next iteration only
        }
    }
}

// y_v -= c for every case
__global__ void k_sub_lines(int64_t n, int K, double *__restrict__ y, const double *__restrict__ c) {
    const Lines<1> L(K);
    if (!L.on) return;
    for (int64_t l = (int64_t)blockIdx.x * L.per + L.li; l < n; l += (int64_t)gridDim.x * L.per) y[l * K + L.v] -= c[l];
}

// ------------------------------------------------------------ launchers ----
void launch_sub_lines(int64_t n, int K, double *y, const double *c, hipStream_t st) {
    hipLaunchKernelGGL(k_sub_lines, dim3(line_grid(n, K)), dim3(line_threads(K)), 0, st, n, K, y, c);
}

void launch_part_reduce(const DualDev &D, const SymvItem *items, const int *item0, const int *nitems, int R, int K,
                        const double *ypart, double *yb, hipStream_t st) {
    const int W = K % 2 ? 1 : 2;
    const unsigned g = std::max(1u, std::min(cdiv((int64_t)D.max_m * K, 256 * W), 64u));
    if (W == 1)
        hipLaunchKernelGGL(k_part_reduce<1>, dim3(g, D.nsub), dim3(256), 0, st, items, item0, nitems, D.m, D.boff, R, K,
                           ypart, yb);
    else
        hipLaunchKernelGGL(k_part_reduce<2>, dim3(g, D.nsub), dim3(256), 0, st, items, item0, nitems, D.m, D.boff, R, K,
                           ypart, yb);
}

void launch_lambda_gather(const DualDev &D, int K, const double *yb, bool scaled, double *y, hipStream_t st,
                          const double *a, double *part) {
    ESP_LINES(k_lambda_gather, K, part ? (unsigned)dot_blocks(D.nlam, K) : line_grid(D.nlam, K), D.nlam, K, D.le_cnt,
              D.le_b, scaled ? D.le_sscale : D.le_sign, yb, y, a, part);
}

void launch_boundary_gather(const DualDev &D, int K, const double *x, bool scaled, double *xb, hipStream_t st) {
    ESP_LINES(k_boundary_gather, K, line_grid(D.nbnd, K), D.nbnd, K, D.bl_ptr, D.bl_lam,
              scaled ? D.bl_sscale : D.bl_sign, x, xb);
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
#define ESP_APPLY_G(W, KB)                                                                                          \
    hipLaunchKernelGGL((k_apply_G<W, KB>), dim3(D.nsub), dim3(T), 0, st, D.m, D.boff, kcols, outoff, roff, RT, D.bl_ptr, \
                       D.bl_lam, D.bl_row, D.bl_sign, K, x, out, stop)
    if (D.max_k == 1) {
        if (K % 2) ESP_APPLY_G(1, 1);
        else ESP_APPLY_G(2, 1);
    } else {
        if (K % 2) ESP_APPLY_G(1, 6);
        else ESP_APPLY_G(2, 6);
    }
#undef ESP_APPLY_G
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
        hipLaunchKernelGGL(k_coarse_block, dim3(cdiv(D.ncoarse, 16)), dim3(1024), 0, st, D.ncoarse, K, D.GGinv, din,
                           eout);
    if (mode == 2) return;
    ESP_LINES(k_project_finish, K, part ? (unsigned)dot_blocks(D.nlam, K) : line_grid(D.nlam, K), D.nlam, K, D.le_cnt,
              D.le_coarse, D.le_sign, D.RtT, D.ce, x, y, mode, a, part);
}

void launch_subdomain_kernel_dots(const DualDev &D, int K, const double *x, double *out, hipStream_t st) {
    apply_G(D, K, D.kdim, D.asub, D.rboff, D.RbT, x, out, nullptr, st);
}

void launch_dot_lines(int64_t n, int K, const double *a, const double *b, double *part, hipStream_t st) {
    ESP_LINES(k_dot_lines, K, dot_blocks(n, K), n, K, a, b, part);
}

void launch_pcg_init(int K, const double *part_r, const double *part_b, int np, double precision, double tol_abs,
                     double *scal, PcgRecord *rec, hipStream_t st) {
    hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(256), 0, st, K, part_r, part_b, np, precision, tol_abs, scal, rec);
}

// the update passes read every partial in each workgroup: two workgroups per CU
static unsigned update_grid(int64_t n, int K) { return std::min(line_grid(n, K), 512u); }

void launch_p_update(int64_t n, int K, double *p, const double *y, const double *part_yw, const double *part_ww,
                     int np, bool first, double *scal, PcgRecord *rec, hipStream_t st) {
    ESP_LINES(k_p_update, K, update_grid(n, K), n, K, p, y, part_yw, part_ww, np, first ? 1 : 0, scal, rec);
}

void launch_xr_update(int64_t n, int K, double *x, double *r, const double *p, const double *Ap,
                      const double *part_pAp, int np, double *scal, hipStream_t st) {
    ESP_LINES(k_xr_update, K, update_grid(n, K), n, K, x, r, p, Ap, part_pAp, np, scal);
}

}  // namespace esp
