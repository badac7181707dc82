// Dual-space kernels of the FETI iteration: the dual operator
// F x = sum_i B_i F_i B_i^T x (itersolvercpu.cpp:9-114) for one and for several
// cases, the cluster correction of hybrid FETI, new loads and the primal recovery
// (itersolver.cpp:372-431) with their interior band solves, and the KKT report.
// The passes of the PCG between two operator applies are in pcg.hip.
//
// F_i and S_D live in HBM in the packed-strip layout (see internal.h): one
// pass over the upper triangle applies both triangles.  A workgroup owns a
// contiguous range of strips of one subdomain; B_i^T x is gathered straight
// from lambda space into LDS, row and column contributions accumulate in LDS,
// and each workgroup writes one partial vector that a second pass sums and
// scatters back to lambda space in a fixed order (no global atomics).  The
// waves of a workgroup meet in 64-bit fixed-point accumulators (integer adds,
// so the order in which the waves arrive does not change a bit of the result:
// repeated applies are bitwise equal).
#include <hip/hip_runtime.h>

#include "dual.h"

namespace esp {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Acc { typedef float type; };
template <>
struct Acc<double> { typedef double type; };

template <typename T, typename A>
__device__ __forceinline__ A load_cvt(T v) { return (A)v; }
template <>
__device__ __forceinline__ float load_cvt<uint16_t, float>(uint16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// Fixed-point accumulation of the SYMV: value v enters the accumulators as
// rint(v 2^k).  With 2^e <= 2 ||F_s||_inf max|x| (the bound of every partial
// sum, doubled against the rounding of the stored values) and k = 60 - e,
// every accumulator stays below 2^60 in magnitude; one unit is 2^-59 of
// ||F_s||_inf max|x| or less, below the rounding of an FP64 sum of the same
// terms.
__device__ __forceinline__ unsigned long long to_fixed(double v, int k) {
    return (unsigned long long)(long long)__builtin_rint(ldexp(v, k));
}

template <typename T, int R>
__global__ void __launch_bounds__(256) k_symv(const SymvItem *__restrict__ items, const int *__restrict__ M,
                                              const int64_t *__restrict__ boff, const T *__restrict__ pool,
                                              const int64_t *__restrict__ poff, const float *__restrict__ fscale,
                                              const double *__restrict__ nrm, const int64_t *__restrict__ bl_ptr,
                                              const int *__restrict__ bl_lam, const double *__restrict__ coef,
                                              const double *__restrict__ x, int gather, double *__restrict__ ypart) {
    typedef typename Acc<T>::type A;
    extern __shared__ unsigned char smem[];
    __shared__ double wmax[4];
    const SymvItem it = items[blockIdx.x];
    const int s = it.sub, m = M[s];
    const int j0 = it.t0 * R, len = m - j0;
    unsigned long long *ys = (unsigned long long *)smem;  // len fixed-point sums
    A *xs = (A *)(ys + len);  // len + R entries: x of the columns, zero padding past m
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t b0 = boff[s] + j0;
    double xm = 0.0;
    for (int j = tid; j < len; j += 256) {
        double v;
        if (gather) {
            v = 0.0;
            for (int64_t q = bl_ptr[b0 + j]; q < bl_ptr[b0 + j + 1]; q++) v += coef[q] * x[bl_lam[q]];
        } else {
            v = x[b0 + j];
        }
        xs[j] = (A)v;
        ys[j] = 0ull;
        xm = fmax(xm, fabs(v));
    }
    if (tid < R) xs[len + tid] = (A)0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) xm = fmax(xm, __shfl_xor(xm, o, 64));
    if (lane == 0) wmax[wave] = xm;
    __syncthreads();
    xm = fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3]));
    const double sc = fscale ? (double)fscale[s] : 1.0;
    const double bound = 2.0 * nrm[s] / sc * xm;
    // a non-finite x or operator gives NaN outputs (the fixed point would hide it)
    const bool finite = bound <= 1.7976931348623157e308;
    const int k = (finite && bound > 0.0) ? 60 - ilogb(bound) : 0;
    const T *base = pool + poff[s];
    for (int t = it.t0 + wave; t < it.t1; t += 4) {
        const int r0 = t * R;
        const int ncol = m - r0;
        const T *S = base + strip_offset(m, R, t);
        // the strip-row x: FP64 keeps it in registers (R = 16 values per lane);
        // BF16 (64 rows) keeps it in one register, row r in lane r, broadcast
        // with readlane (no LDS reads and waits in the chunk loop); FP32
        // (32 rows) reads it from LDS, which measured faster there
        constexpr bool XREG = sizeof(T) == 8, XLANE = sizeof(T) == 2;
        A racc[R], xr[XREG ? R : 1];
#pragma unroll
        for (int r = 0; r < R; r++) {
            racc[r] = (A)0;
            if constexpr (XREG) xr[r] = xs[r0 + r - j0];
        }
        const float xlane = XLANE ? (lane < R ? (float)xs[r0 + lane - j0] : 0.0f) : 0.0f;
        const A *xrow = xs + (r0 - j0);  // x of the strip rows (FP32: LDS broadcast reads)
        constexpr int VEC = 16 / (int)sizeof(T);
        constexpr int NV = R / VEC;
        for (int c0 = 0; c0 < ncol; c0 += 64) {
            const int w = min(64, ncol - c0);
            if (lane < w) {
                // chunk [R/VEC][w][VEC]: the q-th 16-byte load of lane l sits at (q*w + l)*VEC
                const u32x4 *src = (const u32x4 *)(S + (int64_t)c0 * R) + lane;
                u32x4 raw[NV];
#pragma unroll
                for (int q = 0; q < NV; q++) raw[q] = __builtin_nontemporal_load(src + (int64_t)q * w);
                const T *a = (const T *)raw;
                const int c = c0 + lane;
                const A xc = xs[r0 + c - j0];
                // four independent chains for the column sum (latency of the FMA chain)
                A col[4] = {(A)0, (A)0, (A)0, (A)0};
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const A av = load_cvt<T, A>(a[r]);
                    if constexpr (XREG) {
                        col[r & 3] = fma(av, xr[r], col[r & 3]);
                    } else if constexpr (XLANE) {
                        const A xrr = __builtin_bit_cast(
                            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, xlane), r));
                        col[r & 3] = fma(av, xrr, col[r & 3]);
                    } else {
                        col[r & 3] = fma(av, xrow[r], col[r & 3]);
                    }
                    racc[r] = fma(av, xc, racc[r]);
                }
                atomicAdd(&ys[r0 + c - j0], to_fixed((double)((col[0] + col[1]) + (col[2] + col[3])), k));
            }
        }
        const A rs = wave_rows_reduce<R, A>(racc, lane);
        const int row = lane / (64 / R);
        if ((lane & (64 / R - 1)) == 0 && r0 + row < m) atomicAdd(&ys[r0 + row - j0], to_fixed((double)rs, k));
    }
    __syncthreads();
    for (int j = tid; j < len; j += 256)
        ypart[it.part_off + j] = finite ? ldexp((double)(long long)ys[j], -k) * sc : __builtin_nan("");
}

// Block SYMV on MFMA (v_mfma_f64_16x16x4f64): up to 16 right-hand sides, the
// MFMA's N dimension (lanes of right-hand sides past nr carry zeros).  An
// item is at most BLOCK_STRIPS strips of one subdomain; wave w owns strips 2w
// and 2w + 1 and walks the 16-column blocks of the item (a grid common to all
// strips, which start at multiples of 16), the four waves in step:
//   column product  Dc[c][v] += sum_r A[r][c] x[r][v]   (A op: lane (c, row slot))
//   row product     Dr[r][v] += sum_c A[r][c] x[c][v]   (A op: lane (r, column slot))
// The 16-byte loads give the first operand layout; per-wave LDS tiles
// transpose the blocks for the second.  Row sums and the x of a wave's rows stay
// in registers; the column sums of a step meet in LDS, where thread (column, case)
// adds the four waves' in order and writes the item's partial (fixed order, so
// repeated applies are bitwise equal).  x and the partials are interleaved by
// right-hand side with stride nr.
// What bounds it: a step of 16 columns moves 16 KB of F_i, 2 KB of x and, at 16 cases,
// 2 KB of partials, and takes 0.93 us a CU, 5 TB/s like a copy; 71 of the 596 us below
// are the starts and ends of items.  (F_i of 2000 uneven heat subdomains is 2.0 GB: 303 us
// read alone; the MFMAs take 216.)  So the next step's blocks are loaded before the
// current ones are used, by loads without a branch (blocks left of a strip's diagonal,
// past the item's strips or past the last column repeat stored values and are zeroed
// when used: at a branch the compiler waits for every load in flight) and without
// 64-bit address arithmetic per lane, four workgroups share a CU, waves whose strips
// start right of a block only keep step, and items are launched longest first.  x is
// read up to 15 lines past the last column: its buffers are that much longer.
// Waves owning columns instead of strips, one block's loads in flight, took 745 us at
// those subdomains and 16 cases (now 596), 421 at 512 uneven elasticity subdomains and 5
// cases (now 290).  Two steps ahead, 64 columns a load, 16 strips an item, two waves with four
// strips or eight with one and x in LDS all take 594 to 659 and 290 to 327 us.
typedef double v4d __attribute__((ext_vector_type(4)));

// loads with a scalar base and one 32-bit lane offset (no 64-bit address arithmetic per lane)
__device__ __forceinline__ u32x4 stream_load(const u32x4 *p, unsigned at) {
    asm volatile("" : "+s"(p));
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4 *)p + at);
}
__device__ __forceinline__ double line_value(const double *p, unsigned at) {
    asm volatile("" : "+s"(p));
    return ((const __attribute__((address_space(1))) double *)p)[at];
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// workgroup barrier that orders LDS accesses only: the full barrier also waits for
// every global load in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__global__ void __launch_bounds__(256, 4) k_symv_mfma(const SymvItem *__restrict__ items, const int *__restrict__ M,
                                                      const int64_t *__restrict__ boff,
                                                      const double *__restrict__ pool,
                                                      const int64_t *__restrict__ poff, const double *__restrict__ xb,
                                                      int nr, double *ypart) {
    constexpr int R = STRIP_F64, W = BLOCK_STRIPS / 4, TL = 18;  // W strips per wave; TL: leading dimension of T
    __shared__ double T[4][W][16 * TL], slot[2][4][256];
    const SymvItem it = items[blockIdx.x];
    const int s = it.sub, m = M[s];
    const int ns = it.t1 - it.t0, r0i = it.t0 * R;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, l16 = lane & 15, lv = min(l16, nr - 1);
    const double *xs = xb + boff[s] * nr;
    const int nblk = (m - r0i + 15) / 16;
    // the wave's strips (clamped to the item's), where they start and their columns
    const u32x4 *strip[W];
    int r0[W];
    double xr[W][4];  // x of the strip rows: row slot q of call (j, e) is row 2q + 8j + e
    v4d dr[W];
#pragma unroll
    for (int k = 0; k < W; k++) {
        const int t = it.t0 + min(W * wave + k, ns - 1);
        strip[k] = (const u32x4 *)(pool + poff[s] + strip_offset(m, R, t));
        r0[k] = t * R;
        dr[k] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int row = r0[k] + 2 * q + 8 * (j >> 1) + (j & 1);
            const double v = xs[(int64_t)min(row, m - 1) * nr + lv];
            xr[k][j] = (row < m && l16 < nr) ? v : 0.0;
        }
    }
    // column block cb of the wave's strips: rows 2q, 2q+1 and 2q+8, 2q+9 of column
    // c0 + l16; and the row product's B operand x[c0 + q + 4j][l16]
    struct Step {
        u32x4 p[W][2];
        double x[4];
    } st[2];
    int qw[W];  // q times the width of the last chunk of columns
    unsigned xo[4];
#pragma unroll
    for (int k = 0; k < W; k++) qw[k] = q * (((m - r0[k] - 1) & 63) + 1);
#pragma unroll
    for (int j = 0; j < 4; j++) xo[j] = (q + 4 * j) * nr + lv;
    auto load = [&](Step &n, int cb) {
        const int c0 = r0i + 16 * min(cb, nblk - 1);
#pragma unroll
        for (int k = 0; k < W; k++) {
            const int cl = max(0, c0 - r0[k]), ch = cl & ~63, w = min(64, m - r0[k] - ch);
            const unsigned at = (w == 64 ? 64 * q : qw[k]) + min(cl - ch + l16, w - 1);
            const u32x4 *chunk = strip[k] + (int64_t)ch * (R / 2);
            n.p[k][0] = stream_load(chunk, at);
            n.p[k][1] = stream_load(chunk + 4 * w, at);
        }
        const double *x = xs + (int64_t)c0 * nr;  // past the last column: not used
#pragma unroll
        for (int j = 0; j < 4; j++) n.x[j] = line_value(x, xo[j]);
    };
    auto step = [&](Step &c, int cb, int buf) {
        const int c0 = r0i + 16 * cb;
        if (cb < BLOCK_STRIPS || c0 + 16 > m || ns < BLOCK_STRIPS) {  // uniform: values to zero
            const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int k = 0; k < W; k++) {
                const bool in = W * wave + k <= min(cb, ns - 1) && c0 + l16 < m;
                c.p[k][0] = in ? c.p[k][0] : zero;
                c.p[k][1] = in ? c.p[k][1] : zero;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) c.x[j] = c0 + q + 4 * j < m ? c.x[j] : 0.0;
        }
        // waves whose strips start right of the block only keep step
        double dc[4] = {0.0, 0.0, 0.0, 0.0};
        if (W * wave <= min(cb, ns - 1)) {
            v4d d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < W; k++) {
                *(u32x4 *)(T[wave][k] + l16 * TL + 2 * q) = c.p[k][0];
                *(u32x4 *)(T[wave][k] + l16 * TL + 2 * q + 8) = c.p[k][1];
            }
            double a[W][4];
            __builtin_memcpy(a, c.p, sizeof(a));
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int k = 0; k < W; k++) d = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][j], xr[k][j], d, 0, 0, 0);
            wave_lds_sync();
            // row product: column slot q of call j is column q + 4j
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int k = 0; k < W; k++)
                    dr[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(T[wave][k][(q + 4 * j) * TL + l16], c.x[j], dr[k], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) dc[i] = d[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) slot[buf][wave][(q + 4 * i) * 16 + l16] = dc[i];
        lds_barrier();  // a slot is written again two steps on, behind the next barrier
        const int col = c0 + (tid >> 4), v = tid & 15;
        if (col < m && v < nr)
            ypart[(it.part_off + col - r0i) * nr + v] =
                (slot[buf][0][tid] + slot[buf][1][tid]) + (slot[buf][2][tid] + slot[buf][3][tid]);
    };
    load(st[0], 0);
    for (int cb = 0; cb < nblk; cb += 2) {
        load(st[1], cb + 1);
        step(st[0], cb, 0);
        if (cb + 1 >= nblk) break;
        load(st[0], cb + 2);
        step(st[1], cb + 1, 1);
    }
    // the row sums join the column sums of the item's own rows: lane holds D[strip row q + 4i][l16]
    __syncthreads();
    double own[W][4];
#pragma unroll
    for (int k = 0; k < W; k++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            own[k][i] = ypart[(it.part_off + min(r0[k] + q + 4 * i, m - 1) - r0i) * nr + lv];
#pragma unroll
    for (int k = 0; k < W; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = r0[k] + q + 4 * i;
            if (W * wave + k < ns && row < m && l16 < nr)
                ypart[(it.part_off + row - r0i) * nr + l16] = own[k][i] + dr[k][i];
        }
}

__device__ __forceinline__ double block_sum(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double r = 0.0;
    const int nw = blockDim.x >> 6;
    for (int w = 0; w < nw; w++) r += red[w];
    return r;
}

// ---- hybrid FETI: cluster correction of K^+ (cluster.cpp:796-916) ----
// g0 = B0 y_b, t = F0^-1 g0, alpha = Sa^-1 (G0 t - e0), lambda0 = F0^-1 (g0 - G0^T alpha) = t - H alpha
// with H = F0^-1 G0^T precomputed at setup.

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One case, first kernel: g0 gathered from the SYMV output and alpha = Sa^-1 (H^T g0 - e0)
// (H^T = G0 F0^-1), one workgroup per cluster, so that t is not needed before alpha
// and the kernel that computes t finishes lambda0.  Both are chains of latency beside
// the few MB of F0^-1: 38 us (t, each workgroup with the gather) + 28 us (alpha from t, one
// column a thread, then lambda0) at 64 clusters of 8 subdomains of 10^3 elasticity, now 18 + 21.
__global__ void __launch_bounds__(1024) k_cluster_alpha_one(const ClusterDev C, const double *yb, const double *e0s) {
    extern __shared__ double t2[];
    const int c = blockIdx.x;
    const int n0 = C.n0[c], kt = C.kt[c];
    const int64_t ro = C.rowoff[c];
    double *g0 = C.g0 + ro;
    for (int r = threadIdx.x; r < n0; r += 1024) {
        double v = 0.0;
        for (int64_t e = C.re_ptr[ro + r]; e < C.re_ptr[ro + r + 1]; e++) v += C.re_c[e] * yb[C.re_b[e]];
        g0[r] = v;
    }
    __syncthreads();
    const double *H = C.H + C.g0off[c];  // n0 x kt
    const double *e0 = e0s + C.eoff[c];  // cluster-contiguous subdomain partials
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int a = w; a < kt; a += 16) {
        double v = 0.0;
#pragma unroll 4
        for (int r = lane; r < n0; r += 64) v += H[r + (int64_t)a * n0] * g0[r];
        v = wave_sum(v);
        if (lane == 0) t2[a] = v - e0[a];
    }
    __syncthreads();
    const double *Sai = C.Sainv + C.saoff[c];  // symmetric: column a is row a
    for (int a = w; a < kt; a += 16) {
        double v = 0.0;
        for (int b = lane; b < kt; b += 64) v += Sai[b + (int64_t)a * kt] * t2[b];
        v = wave_sum(v);
        if (lane == 0) C.alphaK[C.eoff[c] + a] = v;
    }
}

// lambda0 = F0^-1 g0 - H alpha: 32 rows per workgroup (8 per wave, accumulated together
// for memory-level parallelism), each row a dot over a column of the symmetric F0^-1
__global__ void __launch_bounds__(256) k_cluster_lambda0(const ClusterDev C) {
    extern __shared__ double g0[];
    const int c = blockIdx.y;
    const int n0 = C.n0[c], kt = C.kt[c];
    const int rb = blockIdx.x * 32;
    if (rb >= n0) return;  // uniform over the workgroup
    const int64_t ro = C.rowoff[c];
    for (int r = threadIdx.x; r < n0; r += 256) g0[r] = C.g0[ro + r];
    __syncthreads();
    const double *F = C.F0inv + C.f0off[c], *H = C.H + C.g0off[c], *al = C.alphaK + C.eoff[c];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r0 = rb + w * 8;
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.0;
    for (int a = lane; a < kt; a += 64) {
        const double x = al[a];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] -= H[min(r0 + i, n0 - 1) + (int64_t)a * n0] * x;
    }
    for (int q = lane; q < n0; q += 64) {
        const double gq = g0[q];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] += F[q + (int64_t)min(r0 + i, n0 - 1) * n0] * gq;
    }
    const double s = wave_rows_reduce<8, double>(v, lane);
    if ((lane & 7) == 0 && r0 + (lane >> 3) < n0) C.lambda0[ro + r0 + (lane >> 3)] = s;
}

// Several cases: one workgroup per cluster and case: alpha = Sa^-1 (G0 t - e0), lambda0 = t - H alpha (in place over t);
// e0s interleaved by case, lam0 and alphaK at strides lstr and astr
__global__ void __launch_bounds__(1024) k_cluster_alpha(const ClusterDev C, const double *e0s, double *lam0,
                                                        int64_t lstr, double *alphaK, int64_t astr) {
    extern __shared__ double sh[];
    const int c = blockIdx.x, K = gridDim.y;
    lam0 += blockIdx.y * lstr;
    alphaK += blockIdx.y * astr;
    const int n0 = C.n0[c], kt = C.kt[c];
    double *t2 = sh, *al = sh + C.max_kt;
    const int64_t ro = C.rowoff[c];
    const double *t = lam0 + ro;
    const double *G0T = C.G0T + C.g0off[c];  // n0 x kt
    const double *e0 = e0s + C.eoff[c] * K + blockIdx.y;  // cluster-contiguous subdomain partials
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int a = w; a < kt; a += 16) {
        double v = 0.0;
        for (int r = lane; r < n0; r += 64) v += G0T[r + (int64_t)a * n0] * t[r];
        v = wave_sum(v);
        if (lane == 0) t2[a] = v - e0[(int64_t)a * K];
    }
    __syncthreads();
    const double *Sai = C.Sainv + C.saoff[c];
    for (int a = threadIdx.x; a < kt; a += 1024) {
        double v = 0.0;
        for (int b = 0; b < kt; b++) v += Sai[a + (int64_t)b * kt] * t2[b];
        al[a] = v;
        alphaK[C.eoff[c] + a] = v;
    }
    __syncthreads();
    const double *H = C.H + C.g0off[c];  // n0 x kt
    for (int r = threadIdx.x; r < n0; r += 1024) {
        double v = t[r];
        for (int a = 0; a < kt; a++) v -= H[r + (int64_t)a * n0] * al[a];
        lam0[ro + r] = v;
    }
}

// ---- hybrid FETI set-up on the device (cluster.cpp:1293-2016) ----
// F0 = sum over the cluster's subdomains of their corner blocks; one workgroup
// per cluster, subdomains in order (rows of one subdomain are distinct).
__global__ void __launch_bounds__(256) k_f0_assemble(const ClusterDev C, double *F0) {
    const int c = blockIdx.x;
    const int n0 = C.n0[c];
    double *F = F0 + C.f0off[c];
    const int64_t nn = (int64_t)n0 * n0;
    for (int64_t e = threadIdx.x; e < nn; e += 256) F[e] = 0.0;
    __syncthreads();
    const int64_t ro = C.rowoff[c];
    for (int s = C.sfirst[c]; s < C.sfirst[c] + C.scount[c]; s++) {
        const int nq = C.nq[s];
        const int *qr = C.qrow + C.qoff[s];
        const double *Fc = C.Fcc + C.fccoff[s];
        for (int e = threadIdx.x; e < nq * nq; e += 256) {
            const int q1 = e % nq, q2 = e / nq;
            F[(qr[q1] - ro) + (qr[q2] - ro) * (int64_t)n0] += Fc[e];
        }
        __syncthreads();
    }
}

// H(:, a) = F0^-1 G0^T(:, a): grid (kt, clusters), F0^-1 symmetric so rows are read along columns
__global__ void __launch_bounds__(256) k_cluster_h(const ClusterDev C) {
    extern __shared__ double g[];
    const int c = blockIdx.y, a = blockIdx.x;
    const int n0 = C.n0[c], kt = C.kt[c];
    if (a >= kt || n0 == 0) return;  // uniform
    const double *G0T = C.G0T + C.g0off[c] + (int64_t)a * n0;
    for (int r = threadIdx.x; r < n0; r += 256) g[r] = G0T[r];
    __syncthreads();
    const double *F = C.F0inv + C.f0off[c];
    double *H = C.H + C.g0off[c] + (int64_t)a * n0;
    for (int r = threadIdx.x; r < n0; r += 256) {
        double v = 0.0;
        for (int q = 0; q < n0; q++) v += F[r + (int64_t)q * n0] * g[q];
        H[r] = v;
    }
}

// Sa = G0 H + rho N N^T (rho = max diag of G0 H, 1 if that is not positive); one workgroup per cluster
__global__ void __launch_bounds__(256) k_cluster_sa(const ClusterDev C, double *Sa) {
    __shared__ double red[4];
    __shared__ double rho;
    const int c = blockIdx.x;
    const int n0 = C.n0[c], kt = C.kt[c], kn = C.kn[c];
    const double *G0T = C.G0T + C.g0off[c];
    const double *H = C.H + C.g0off[c];
    double *S = Sa + C.saoff[c];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int o = w; o < kt * kt; o += 4) {
        const int i = o % kt, j = o / kt;
        double v = 0.0;
        for (int r = lane; r < n0; r += 64) v += G0T[r + (int64_t)i * n0] * H[r + (int64_t)j * n0];
        v = wave_sum(v);
        if (lane == 0) S[o] = v;
    }
    __syncthreads();
    double m = 0.0;
    for (int i = threadIdx.x; i < kt; i += 256) m = fmax(m, S[i + (int64_t)i * kt]);
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if (lane == 0) red[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
        if (!(r > 0.0)) {
            // no corner rows (G0 empty): the scale of the cluster's own S_i, so
            // that the kernel term R Sa^-1 R^T stays within the size of K^+
            for (int q = 0; q < C.scount[c]; q++) r = fmax(r, C.rho_s[C.sfirst[c] + q]);
        }
        rho = r > 0.0 ? r : 1.0;
    }
    __syncthreads();
    const double *N = C.Nc + C.ncoff[c];  // kt x kn
    for (int o = threadIdx.x; o < kt * kt; o += 256) {
        const int i = o % kt, j = o / kt;
        double v = 0.0;
        for (int b = 0; b < kn; b++) v += N[i + (int64_t)b * kt] * N[j + (int64_t)b * kt];
        S[o] += rho * v;
    }
}

// y_b += -FB0_s lambda0 + addR * R_b alphaK; grid (row chunks of 256, subdomains);
// FB0 is C.FB0 (FP64) or C.FB0f (the low-precision F_i's columns)
template <typename T>
__global__ void __launch_bounds__(256) k_cluster_apply(const ClusterDev C, const T *FB0, const int *M,
                                                       const int64_t *boff, const int *kdim, const int64_t *rboff,
                                                       const double *Rb, const double *lambda0, const double *alphaK,
                                                       int addR, double *yb) {
    __shared__ double lam[256];
    const int s = blockIdx.y, m = M[s];
    if (blockIdx.x * 256 >= m) return;  // uniform
    const int nq = C.nq[s];
    const int64_t q0 = C.qoff[s];
    for (int q = threadIdx.x; q < nq; q += 256) lam[q] = lambda0[C.qrow[q0 + q]];
    __syncthreads();
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    const T *FB = FB0 + C.fb0off[s] + j;
    // eight independent chains: all loads of a group issue before their use
    double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int q = 0;
    for (; q + 8 <= nq; q += 8) {
        T f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = FB[(int64_t)(q + i) * m];
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] -= (double)f[i] * lam[q + i];
    }
    for (; q < nq; q++) acc[q & 7] -= (double)FB[(int64_t)q * m] * lam[q];
    double v = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    if (addR) {
        const double *R = Rb + rboff[s] + j;
        const double *al = alphaK + C.asub[s];
        for (int a = 0; a < kdim[s]; a++) v += R[(int64_t)a * m] * al[a];
    }
    yb[boff[s] + j] += v;
}

// FB0f = FB0 rounded to FP32.  With FP32 storage these are exactly the columns
// of the stored F_i, so the inner operator stays symmetric.  With BF16 storage
// they are not rounded to BF16: F0 = B0 F_i B0^T is built from the FP64 F_i,
// and the correction cancels the corner directions only when one of its two
// factors matches F0; a BF16-rounded pair leaves an indefinite error of the
// BF16 rounding on them (PCG then stalls).  grid (chunks, subdomains)
__global__ void __launch_bounds__(256) k_fb0_round(const ClusterDev C, const int *M) {
    const int s = blockIdx.y;
    const int64_t n = (int64_t)M[s] * C.nq[s];
    const double *src = C.FB0 + C.fb0off[s];
    float *dst = C.FB0f + C.fb0off[s];
    for (int64_t e = blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) dst[e] = (float)src[e];
}

void launch_fb0_round(const DualDev &D, const ClusterDev &C, hipStream_t st) {
    hipLaunchKernelGGL(k_fb0_round, dim3(64, D.nsub), dim3(256), 0, st, C, D.m);
}

// ---- the cluster correction for up to 8 cases per pass (block re-solve):
// F0^-1 and F_i B0^T are read once per pass instead of once per case.
// t_v = F0^-1 g0_v, g0_v gathered from the case's SYMV output; 4 rows per
// wave, kc <= 8 cases (g0 of the kc cases in LDS); grid (rows/16, clusters).
__global__ void __launch_bounds__(256) k_cluster_t_multi(const ClusterDev C, const double *yb, int64_t K,
                                                         int kc, double *t, int64_t tstr) {
    extern __shared__ double g0[];  // n0 x kc
    const int c = blockIdx.y;
    const int n0 = C.n0[c];
    const int rb = blockIdx.x * 16;
    if (rb >= n0) return;  // uniform over the workgroup
    const int64_t ro = C.rowoff[c];
    for (int e = threadIdx.x; e < n0 * kc; e += 256) {
        const int r = e / kc, v = e % kc;
        double g = 0.0;
        for (int64_t q = C.re_ptr[ro + r]; q < C.re_ptr[ro + r + 1]; q++) g += C.re_c[q] * yb[C.re_b[q] * K + v];
        g0[e] = g;
    }
    __syncthreads();
    const double *F = C.F0inv + C.f0off[c];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r0 = rb + w * 4;
    double acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int v = 0; v < 8; v++) acc[i][v] = 0.0;
    for (int q = lane; q < n0; q += 64) {
        double f[4];
#pragma unroll
        for (int i = 0; i < 4; i++) f[i] = r0 + i < n0 ? F[q + (int64_t)(r0 + i) * n0] : 0.0;
#pragma unroll
        for (int v = 0; v < 8; v++) {
            if (v < kc) {
                const double gq = g0[q * kc + v];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i][v] += f[i] * gq;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int v = 0; v < 8; v++) {
            if (v < kc) {
                const double sv = wave_sum(acc[i][v]);
                if (lane == 0 && r0 + i < n0) t[v * tstr + ro + r0 + i] = sv;
            }
        }
}

// y_b,v += -FB0_s lambda0_v + addR * R_b alphaK_v for kc <= 8 cases;
// grid (row chunks of 256, subdomains)
__global__ void __launch_bounds__(256) k_cluster_apply_multi(const ClusterDev C, const int *M, const int64_t *boff,
                                                             const int *kdim, const int64_t *rboff, const double *Rb,
                                                             const double *lambda0, int64_t lstr,
                                                             const double *alphaK, int64_t astr, int addR, int kc,
                                                             double *yb, int64_t K) {
    __shared__ double lam[256 * 8];
    const int s = blockIdx.y, m = M[s];
    if (blockIdx.x * 256 >= m) return;  // uniform
    const int nq = C.nq[s];
    const int64_t q0 = C.qoff[s];
    for (int e = threadIdx.x; e < nq * kc; e += 256) {
        const int q = e / kc, v = e % kc;
        lam[e] = lambda0[v * lstr + C.qrow[q0 + q]];
    }
    __syncthreads();
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    const double *FB = C.FB0 + C.fb0off[s] + j;
    double acc[8];
#pragma unroll
    for (int v = 0; v < 8; v++) acc[v] = 0.0;
    for (int q = 0; q < nq; q++) {
        const double f = FB[(int64_t)q * m];
#pragma unroll
        for (int v = 0; v < 8; v++)
            if (v < kc) acc[v] -= f * lam[q * kc + v];
    }
    const double *R = Rb + rboff[s] + j;
    for (int v = 0; v < kc; v++) {
        double val = acc[v];
        if (addR) {
            const double *al = alphaK + v * astr + C.asub[s];
            for (int a = 0; a < kdim[s]; a++) val += R[(int64_t)a * m] * al[a];
        }
        yb[(boff[s] + j) * K + v] += val;
    }
}

// alpha_tot_v(s) = addK * alphaK_v(s) + N_s alpha_coarse,v(block(s)), a thread per subdomain and case
// (alpha_coarse interleaved by case, alphaK and alpha_tot at stride astr)
__global__ void k_alpha_combine(int nsub, int K, const int *kdim, const int *ck, const int *cblk, const int *coff,
                                const int64_t *asub, const int64_t *noff, const double *N, const double *alphaK,
                                int addK, const double *alpha_coarse, double *alpha_tot, int64_t astr) {
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nsub * K; e += gridDim.x * blockDim.x) {
        const int s = e / K, v = e % K;
        const int k = kdim[s], kc = ck[s];
        const double *Ns = N + noff[s];  // k x kc column-major
        const double *ac = alpha_coarse + (int64_t)coff[cblk[s]] * K + v;
        for (int a = 0; a < k; a++) {
            double t = addK ? alphaK[v * astr + asub[s] + a] : 0.0;
            for (int b = 0; b < kc; b++) t += Ns[a + (int64_t)b * k] * ac[(int64_t)b * K];
            alpha_tot[v * astr + asub[s] + a] = t;
        }
    }
}

// ---- vector kernels ----
__global__ void __launch_bounds__(256) k_dot_partial(const double *a, const double *b, int64_t n, double *partial) {
    __shared__ double red[4];
    double v = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        v += a[i] * b[i];
    v = block_sum(v, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = v;
}
__global__ void __launch_bounds__(256) k_dot_final(const double *partial, int np, double *out) {
    __shared__ double red[4];
    double v = 0.0;
    for (int i = threadIdx.x; i < np; i += 256) v += partial[i];
    v = block_sum(v, red);
    if (threadIdx.x == 0) *out = v;
}

__global__ void k_axpby(double *y, const double *a, const double *b, int64_t n, double alpha, double beta) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = alpha * a[i] + beta * b[i];
}
__global__ void k_symmetrize(double *A, int n) {
    const int64_t nn = (int64_t)n * n;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nn; e += (int64_t)gridDim.x * blockDim.x) {
        int i = (int)(e % n), j = (int)(e / n);
        if (i < j) A[e] = A[j + (int64_t)i * n];
    }
}


// ------------------------------------------------------------ launchers ----
static inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }
static inline unsigned vgrid(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(n, 256), 4096)); }

void launch_symv(const DualDev &D, bool sd, int prec, const double *x, int gather, bool scaled, hipStream_t st,
                 hipEvent_t ev0, hipEvent_t ev1) {
    if (sd) prec = D.sd_prec;
    const SymvItem *items = D.launch_items[prec];
    const int n_items = D.n_items[prec];
    const double *coef = scaled ? D.bl_sscale : D.bl_sign;
    const double *nrm = sd ? D.sdnrm : D.fnrm;
    const size_t shm = symv_lds_bytes(D.max_m, prec);
    if (ev0) (void)hipEventRecord(ev0, st);
    if (prec == 0) {
        const double *pool = sd ? D.SD : D.Fd;
        const int64_t *off = sd ? D.sdoff : D.foff;
        hipLaunchKernelGGL((k_symv<double, STRIP_F64>), dim3(n_items), dim3(256), shm, st, items, D.m, D.boff, pool,
                           off, (const float *)nullptr, nrm, D.bl_ptr, D.bl_lam, coef, x, gather, D.ypart);
    } else if (prec == 1) {
        hipLaunchKernelGGL((k_symv<float, STRIP_F32>), dim3(n_items), dim3(256), shm, st, items, D.m, D.boff,
                           sd ? D.SDf : D.Ff, D.poff[1], (const float *)nullptr, nrm, D.bl_ptr, D.bl_lam, coef, x,
                           gather, D.ypart);
    } else {
        hipLaunchKernelGGL((k_symv<uint16_t, STRIP_B16>), dim3(n_items), dim3(256), shm, st, items, D.m, D.boff,
                           sd ? D.SDh : D.Fh, D.poff[2], (const float *)(sd ? D.sdscale : D.fscale), nrm, D.bl_ptr,
                           D.bl_lam, coef, x, gather, D.ypart);
    }
    if (ev1) (void)hipEventRecord(ev1, st);
    launch_part_reduce(D, D.items[prec], D.item0[prec], D.nitems[prec], strip_rows(prec), 1, D.ypart, D.yb, st);
}

void launch_symv_mfma(const DualDev &D, const SymvBlock &B, bool sd, int nr, const double *xb, double *yb,
                      hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    if (nr < 1 || nr > 16) throw Error(ESPRESO_ERR_ARG, "block SYMV: 1 to 16 right-hand sides");
    const double *pool = sd ? D.SD : D.Fd;
    const int64_t *off = sd ? D.sdoff : D.foff;
    if (ev0) (void)hipEventRecord(ev0, st);
    hipLaunchKernelGGL(k_symv_mfma, dim3(B.n_items), dim3(256), 0, st, B.launch_items, D.m, D.boff, pool, off, xb, nr,
                       B.ypart);
    if (ev1) (void)hipEventRecord(ev1, st);
    launch_part_reduce(D, B.items, B.item0, B.nitems, STRIP_F64, nr, B.ypart, yb, st);
}

void launch_cluster_correction(const DualDev &D, const ClusterDev &C, const double *e0s, double *yb, int addR,
                               hipStream_t st, bool lowp) {
    hipLaunchKernelGGL(k_cluster_alpha_one, dim3(C.ncl), dim3(1024), (size_t)std::max(C.max_kt, 1) * 8, st, C, yb, e0s);
    if (C.max_n0 > 0)
        hipLaunchKernelGGL(k_cluster_lambda0, dim3((C.max_n0 + 31) / 32, C.ncl), dim3(256), (size_t)C.max_n0 * 8, st, C);
    if (lowp && C.FB0f)
        hipLaunchKernelGGL(k_cluster_apply<float>, dim3((D.max_m + 255) / 256, D.nsub), dim3(256), 0, st, C,
                           (const float *)C.FB0f, D.m, D.boff, D.kdim, D.rboff, D.Rb, C.lambda0, C.alphaK, addR, yb);
    else
        hipLaunchKernelGGL(k_cluster_apply<double>, dim3((D.max_m + 255) / 256, D.nsub), dim3(256), 0, st, C,
                           (const double *)C.FB0, D.m, D.boff, D.kdim, D.rboff, D.Rb, C.lambda0, C.alphaK, addR, yb);
}

// the correction of nr interleaved cases: F0^-1 and F_i B0^T read once per 8 cases
void launch_cluster_correction_multi(const DualDev &D, const ClusterDev &C, int nr, const double *e0s, double *lam0,
                                     int64_t lstr, double *alphaK, int64_t astr, double *yb, int addR,
                                     hipStream_t st) {
    if (C.max_n0 > 0) {
        const int kc_max = (int)std::max<int64_t>(1, std::min<int64_t>(8, 6144 / C.max_n0));
        for (int v0 = 0; v0 < nr; v0 += kc_max) {
            const int kc = std::min(kc_max, nr - v0);
            hipLaunchKernelGGL(k_cluster_t_multi, dim3((C.max_n0 + 15) / 16, C.ncl), dim3(256),
                               (size_t)C.max_n0 * kc * 8, st, C, yb + v0, (int64_t)nr, kc, lam0 + v0 * lstr, lstr);
        }
    }
    hipLaunchKernelGGL(k_cluster_alpha, dim3(C.ncl, nr), dim3(1024), 2 * (size_t)std::max(C.max_kt, 1) * 8, st, C, e0s,
                       lam0, lstr, alphaK, astr);
    for (int v0 = 0; v0 < nr; v0 += 8) {
        const int kc = std::min(8, nr - v0);
        hipLaunchKernelGGL(k_cluster_apply_multi, dim3((D.max_m + 255) / 256, D.nsub), dim3(256), 0, st, C, D.m,
                           D.boff, D.kdim, D.rboff, D.Rb, lam0 + v0 * lstr, lstr, alphaK + v0 * astr, astr, addR, kc,
                           yb + v0, (int64_t)nr);
    }
}

void launch_cluster_setup_f0(const ClusterDev &C, hipStream_t st) {
    hipLaunchKernelGGL(k_f0_assemble, dim3(C.ncl), dim3(256), 0, st, C, C.F0inv);
}

void launch_cluster_setup_sa(const ClusterDev &C, double *Sa, hipStream_t st) {
    if (C.max_n0 > 0 && C.max_kt > 0)
        hipLaunchKernelGGL(k_cluster_h, dim3(C.max_kt, C.ncl), dim3(256), (size_t)C.max_n0 * 8, st, C);
    hipLaunchKernelGGL(k_cluster_sa, dim3(C.ncl), dim3(256), 0, st, C, Sa);
}

void launch_alpha_combine(const DualDev &D, int K, const double *alphaK, int64_t astr, bool hybrid,
                          const double *alpha_coarse, double *alpha_tot, hipStream_t st) {
    hipLaunchKernelGGL(k_alpha_combine, dim3(vgrid((int64_t)D.nsub * K)), dim3(256), 0, st, D.nsub, K, D.kdim, D.ck,
                       D.cblk, D.coff, D.asub, D.noff, D.N, alphaK, hybrid ? 1 : 0, alpha_coarse, alpha_tot, astr);
}

void launch_dot(const double *a, const double *b, int64_t n, double *partial, double *out, hipStream_t st) {
    const int np = 512;
    hipLaunchKernelGGL(k_dot_partial, dim3(np), dim3(256), 0, st, a, b, n, partial);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(256), 0, st, partial, np, out);
}

void launch_axpby(double *y, const double *a, const double *b, int64_t n, double alpha, double beta, hipStream_t st) {
    hipLaunchKernelGGL(k_axpby, dim3(vgrid(n)), dim3(256), 0, st, y, a, b, n, alpha, beta);
}

void launch_symmetrize(double *A, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_symmetrize, dim3(vgrid((int64_t)n * n)), dim3(256), 0, st, A, n);
}

__global__ void k_copy(const double4 *__restrict__ src, double4 *__restrict__ dst, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// read-only stream: each thread sums 4 independent 16-byte nontemporal loads
// per step; one double per workgroup keeps the loads alive
__global__ void __launch_bounds__(256) k_stream_read(const u32x4 *__restrict__ src, int64_t n, double *out) {
    __shared__ double red[4];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    unsigned acc = 0;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const u32x4 a = __builtin_nontemporal_load(src + i), b = __builtin_nontemporal_load(src + i + stride),
                    c = __builtin_nontemporal_load(src + i + 2 * stride),
                    d = __builtin_nontemporal_load(src + i + 3 * stride);
        acc ^= (a.x ^ b.y) ^ (c.z ^ d.w);
    }
    for (; i < n; i += stride) acc ^= __builtin_nontemporal_load(src + i).x;
    const double v = block_sum((double)acc, red);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

void launch_stream_read(const double *src, int64_t n, int wgs, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_stream_read, dim3(wgs), dim3(256), 0, st, (const u32x4 *)src, n / 2, out);
}

void launch_copy(const double *src, double *dst, int64_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, st, (const double4 *)src, (double4 *)dst, n / 4);
}

// ---- banded interior solves (K_ii = L L^T) for K <= 16 vectors at once,
// interleaved z[r K + v].  L is a lower band of width bw >= 63 stored by columns,
// L(c + d, c) at L[c w + d], w = bw + 1, except that the 64 x 64 diagonal blocks
// hold their inverses, so a block of the solution is a product and not a chain of 64
// divisions.  One workgroup per subdomain walks the blocks; all products are MFMA
// tiles whose N dimension is the case (lanes past K repeat case K - 1 and store
// nothing), read straight from the band:
//   lower: u = Dinv z_block (wave w: row tile w & 3, every second half of the columns),
//     then wave w takes the 16-row tiles w, w + 8, ... below: z -= L u
//   upper: wave w sums the columns of tile w & 3 over every second 16-row block below
//     the diagonal, then z_block = Dinv^T (z - sums)
// with the partial sums and u in LDS and the first tiles of a step loaded before the
// values they meet are known.  One kernel serves all K, so a band is read once for up
// to 16 cases: at K = 1 the idle MFMA lanes cost less than the memory takes.  What
// bounds it is a step's latency (load, two LDS exchanges, a barrier), 13 us a step and
// direction at bw = 270; 16 waves a workgroup gain nothing (943 against 890 us at 64
// subdomains, 2010 against 1780 at 512).  Chains of 64 divisions and one row a thread
// took, for the two directions: 3.7 ms at 512 subdomains of 2187 interior DOFs (now
// 1.78), 2.95 ms at 64 of them (now 0.89), 13.2 ms at 2000 uneven heat subdomains
// (4 to 14 elements an edge) and 16 cases (now 1.3 and, without the gather, 1.1).
// PRIMAL: z = K_ib u_b on entry; z <- L^-T (yf - L^-1 z).  Else z = f_int,
// yf = L^-1 z, z <- L^-T yf.
// p[off] with a scalar base: the offset of a lane is the same for every load of a step
__device__ __forceinline__ double band_load(const double *p, unsigned off) {
    asm volatile("" : "+s"(p));
    return ((const __attribute__((address_space(1))) double *)p)[off];
}
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void band_load4(double (&a)[4], const double *p, unsigned off) {
    asm volatile("" : "+s"(p));
    auto *s = (const __attribute__((address_space(1))) d2u *)((const __attribute__((address_space(1))) double *)p + off);
    const d2u lo = s[0], hi = s[1];
    a[0] = lo.x;
    a[1] = lo.y;
    a[2] = hi.x;
    a[3] = hi.y;
}

// Element (c, r) of the block at column c0 is Lc[c (w - 1) + r], r counted from c0.  Elements
// outside the band or the matrix are replaced when used: their loads stay inside the
// storage, which ends with BAND_PAD columns that belong to no subdomain.
struct BandTile {  // 16 rows x 64 columns of the band as A operands, and z of the rows
    double a[16], z[4];
};

__device__ __forceinline__ void band_tile_load(BandTile &b, const double *Lc, int w, int ni, int c0, int r, unsigned off,
                                               const double *z, int K, int lv, int q) {
#pragma unroll
    for (int j = 0; j < 16; j++) b.a[j] = band_load(Lc + r + 4 * j * (int64_t)(w - 1), off);
#pragma unroll
    for (int i = 0; i < 4; i++) b.z[i] = z[(unsigned)(min(c0 + r + q + 4 * i, ni - 1) * K + lv)];
}

constexpr int BAND_WAVES = 8;
template <bool PRIMAL>
__global__ void __launch_bounds__(64 * BAND_WAVES, 4)
    k_band_solves(const PrimalDev P, int K, const double *f, int64_t fstr, double *yf, int64_t ystr, double *work) {
    const int s = blockIdx.x;
    const int ni = P.ni[s], bw = P.bw[s];
    if (ni == 0) return;
    int w = bw + 1;
    const double *L = P.band + P.band_off[s];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int l16 = lane & 15, q = lane >> 4;
    const int lv = min(l16, K - 1);
    const int rt = wave & 3, h = wave >> 2;  // 16-row (16-column) tile of the block and part of the sum
    constexpr int NW = BAND_WAVES, H = NW / 4, E = 16 / NW;  // parts of a sum, values of a block per thread
    double *z = work + P.work_off[s] * K;
    yf += P.yf_off[s];
    __shared__ double u[64 * 16], part[H][64 * 16];
    if (!PRIMAL) {
        const int *perm = P.perm + P.perm_off[s];
        const double *fs = f + P.perm_off[s];
        for (int i = tid; i < ni * K; i += 64 * NW) z[i] = fs[(i % K) * fstr + perm[i / K]];
        __syncthreads();
    }
    for (int c0 = 0; c0 < ni; c0 += 64) {
        asm volatile("" : "+s"(w), "+v"(q), "+v"(l16));  // no offsets kept over the loop (they spill)
        const double *Lc = L + (int64_t)c0 * w;
        const int nb = min(64, ni - c0);
        const int below = nb == 64 ? min(bw, ni - c0 - 64) : 0;
        const int nt = (below + 15) >> 4;
        const unsigned off = q * (w - 1) + l16;
        double a[16 / H], x[16 / H], y[E];
#pragma unroll
        for (int j = 0; j < 16 / H; j++) {
            const int c = 64 / H * h + 4 * j;
            a[j] = band_load(Lc + 16 * rt + c * (int64_t)(w - 1), off);
            x[j] = z[(unsigned)((c0 + min(c + q, nb - 1)) * K + lv)];
        }
#pragma unroll
        for (int e = 0; e < E; e++)
            if (PRIMAL) y[e] = yf[lv * ystr + c0 + min((tid >> 4) + 4 * NW * e, nb - 1)];
        BandTile b;
        band_tile_load(b, Lc, w, ni, c0, 64 + 16 * wave, off, z, K, lv, q);
        v4d d0 = {0.0, 0.0, 0.0, 0.0}, d1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 16 / H; j++) {
            const int c = 64 / H * h + 4 * j + q;
            const double av = 16 * rt + l16 >= c && c < nb ? a[j] : 0.0;
            if (j & 1) d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, x[j], d1, 0, 0, 0);
            else d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av, x[j], d0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) part[h][(16 * rt + q + 4 * i) * 16 + l16] = d0[i] + d1[i];
        lds_barrier();
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int k = tid + 64 * NW * e, r = k >> 4;
            double v = part[0][k];
#pragma unroll
            for (int g = 1; g < H; g++) v += part[g][k];
            u[k] = v;
            if (r < nb && l16 < K) {
                z[(unsigned)((c0 + r) * K + l16)] = PRIMAL ? y[e] - v : v;
                if (!PRIMAL) yf[l16 * ystr + c0 + r] = v;
            }
        }
        lds_barrier();
        for (int t = wave; t < nt; t += NW) {
            const int r0 = 64 + 16 * t;
            const int first = c0 + r0 + l16 < ni ? r0 + l16 - q - bw : 64;  // first column slot in the band
            v4d e0, e1 = {0.0, 0.0, 0.0, 0.0};
            double a[16];
#pragma unroll
            for (int i = 0; i < 4; i++) e0[i] = b.z[i];
#pragma unroll
            for (int j = 0; j < 16; j++) a[j] = 4 * j >= first ? -b.a[j] : 0.0;
            if (t + NW < nt) band_tile_load(b, Lc, w, ni, c0, r0 + 16 * NW, off, z, K, lv, q);
#pragma unroll
            for (int j = 0; j < 16; j += 2) {
                e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j], u[(4 * j + q) * 16 + l16], e0, 0, 0, 0);
                e1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j + 1], u[(4 * j + 4 + q) * 16 + l16], e1, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = c0 + r0 + q + 4 * i;
                if (r < ni && l16 < K) z[(unsigned)(r * K + l16)] = e0[i] + e1[i];
            }
        }
        __syncthreads();
    }
    for (int c0 = ((ni - 1) / 64) * 64; c0 >= 0; c0 -= 64) {
        asm volatile("" : "+s"(w), "+v"(q), "+v"(l16));
        const double *Lc = L + (int64_t)c0 * w;
        const int nb = min(64, ni - c0);
        const int cl = 16 * rt + l16;  // column in the block
        const int last = min(ni - 1, c0 + 16 * rt + 15 + bw) - c0;
        const int nblk = last >= 64 ? ((last - 64) >> 4) + 1 : 0;
        const unsigned off = cl * (w - 1) + 4 * q;  // rows 16 blk + 4q .. + 3 of a column: 32 contiguous bytes
        v4d d0 = {0.0, 0.0, 0.0, 0.0}, d1 = {0.0, 0.0, 0.0, 0.0};
        constexpr int G = 2;
        double a[G][4], zb[E], inv[4][4];
        // the first blocks (read and not used when there are none), then what the diagonal block needs
#pragma unroll
        for (int g = 0; g < G; g++) band_load4(a[g], Lc + 64 + 16 * (h + H * g), off);
        if (h == 0)
#pragma unroll
            for (int g = 0; g < 4; g++) band_load4(inv[g], Lc + 16 * g, off);
#pragma unroll
        for (int e = 0; e < E; e++) zb[e] = z[(unsigned)((c0 + min((tid >> 4) + 4 * NW * e, nb - 1)) * K + lv)];
        for (int b0 = h; b0 < nblk; b0 += H * G) {
            double x[G][4], av[G][4];
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int r = 64 + 16 * (b0 + H * g) + 4 * q + j;
                    x[g][j] = z[(unsigned)(min(c0 + r, ni - 1) * K + lv)];
                    av[g][j] = r - cl <= bw && c0 + r < ni ? a[g][j] : 0.0;
                }
            if (b0 + H * G < nblk)
#pragma unroll
                for (int g = 0; g < G; g++) band_load4(a[g], Lc + 64 + 16 * (b0 + H * (G + g)), off);
#pragma unroll
            for (int g = 0; g < G; g++) {
                d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[g][0], x[g][0], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[g][1], x[g][1], d1, 0, 0, 0);
                d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[g][2], x[g][2], d0, 0, 0, 0);
                d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[g][3], x[g][3], d1, 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) part[h][(16 * rt + q + 4 * i) * 16 + l16] = d0[i] + d1[i];
        lds_barrier();
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int k = tid + 64 * NW * e;
            double v = part[0][k];
#pragma unroll
            for (int g = 1; g < H; g++) v += part[g][k];
            u[k] = zb[e] - v;
        }
        lds_barrier();
        if (h == 0) {
            v4d e0 = {0.0, 0.0, 0.0, 0.0}, e1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int g = 0; g < 4; g++) {
                double av[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int r = 16 * g + 4 * q + j;
                    av[j] = r >= cl && r < nb ? inv[g][j] : 0.0;
                }
                const double *x = u + (16 * g + 4 * q) * 16 + l16;
                e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[0], x[0], e0, 0, 0, 0);
                e1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[1], x[16], e1, 0, 0, 0);
                e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[2], x[32], e0, 0, 0, 0);
                e1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[3], x[48], e1, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = 16 * rt + q + 4 * i;
                if (r < nb && l16 < K) z[(unsigned)((c0 + r) * K + l16)] = e0[i] + e1[i];
            }
        }
        __syncthreads();
    }
}

// Coupling products with the CSR K_i, K cases at once, interleaved:
//   BOUNDARY: hf = f_b - K_bi z over the boundary rows (hf in lines of hk cases)
//   else:     z = K_ib u_b over the interior rows in factor order (u_b in lines of hk)
// Workgroup (g, s) takes 64 rows of subdomain s, 16 lanes per row: the lanes read 16
// entries at a time (one thread per row would chain three dependent loads per entry).
// One case: each lane adds its entries.  More: lane v adds case v of the entries that
// couple, handed round the group one by one; most interior rows have none (a lane per
// case walking all entries took 1.23 ms at 2000 heat subdomains and 16 cases, now 0.51).
constexpr int CROSS_ROWS = 64;
template <bool BOUNDARY, bool ONE>
__global__ void __launch_bounds__(256) k_cross(const PrimalDev P, int K, const double *f, int64_t fstr, double *hb,
                                               int hk, double *work) {
    const int s = blockIdx.y, g = blockIdx.x;
    const int ni = P.ni[s], nrow = BOUNDARY ? P.m[s] : ni;
    const int *perm = P.perm + P.perm_off[s];
    const int *iperm = P.iperm + P.perm_off[s];
    const int *rp = P.rowptr + P.rp_off[s];
    const int *ci = P.colidx + P.nz_off[s];
    const double *kv = P.vals + P.nz_off[s];
    double *h = hb + P.boff[s] * hk, *z = work + P.work_off[s] * K;
    const int grp = threadIdx.x >> 4, l = threadIdx.x & 15, v = min(l, K - 1);
    for (int k = 0; k < CROSS_ROWS / 16; k++) {
        const int r = g * CROSS_ROWS + 16 * k + grp;
        if (r >= nrow) break;  // uniform over the group
        const int lr = perm[BOUNDARY ? ni + r : r];
        const int end = rp[lr + 1];
        double acc = 0.0;
        for (int e0 = rp[lr]; e0 < end; e0 += 16) {
            const int e = min(e0 + l, end - 1);
            const int pc = iperm[ci[e]];
            const bool on = e0 + l < end && (pc < ni) == BOUNDARY;
            const int src = BOUNDARY ? pc * K : (pc - ni) * hk;
            if (ONE) {
                if (on) acc += kv[e] * (BOUNDARY ? z : h)[src];
            } else {
                const double val = on ? kv[e] : 0.0;
                unsigned left = (unsigned)(__ballot(on) >> (threadIdx.x & 48)) & 0xffff;
                while (left) {
                    const int j = __ffs(left) - 1;
                    left &= left - 1;
                    acc += __shfl(val, j, 16) * (BOUNDARY ? z : h)[__shfl(src, j, 16) + v];
                }
            }
        }
        if (ONE)
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 16);
        if (l < K) {
            if (BOUNDARY) h[(int64_t)r * hk + l] = f[l * fstr + P.perm_off[s] + lr] - acc;
            else z[(int64_t)r * K + l] = acc;
        }
    }
}

// u = [u_int; u_b] + R alpha in local DOF order, one thread per DOF
__global__ void __launch_bounds__(256) k_primal_write(const PrimalDev P, int K, const double *ub, int bk,
                                                      const double *alpha, int64_t astr, double *u, int64_t ustr,
                                                      const double *work) {
    const int s = blockIdx.y, n = P.n[s], ni = P.ni[s], k = P.kdim[s];
    const int lr = blockIdx.x * 256 + threadIdx.x;
    if (lr >= n) return;
    const int r = P.iperm[P.perm_off[s] + lr];
    const double *x = r < ni ? work + (P.work_off[s] + r) * K : ub + (P.boff[s] + r - ni) * bk;
    const double *R = P.R + P.r_off[s] + lr;
    for (int v = 0; v < K; v++) {
        const double *al = alpha + v * astr + P.asub[s];
        double t = x[v];
        for (int a = 0; a < k; a++) t += R[(int64_t)a * n] * al[a];
        u[v * ustr + P.perm_off[s] + lr] = t;
    }
}

template <bool BOUNDARY>
static void cross(const PrimalDev &P, int nsub, int K, const double *f, int64_t fstr, double *hb, int hk, double *work,
                  hipStream_t st) {
    const dim3 grid(((BOUNDARY ? P.max_m : P.max_ni) + CROSS_ROWS - 1) / CROSS_ROWS, nsub);
    hipLaunchKernelGGL(K == 1 ? (k_cross<BOUNDARY, true>) : (k_cross<BOUNDARY, false>), grid, dim3(256), 0, st, P, K, f,
                       fstr, hb, hk, work);
}

// nr vectors, up to 16 at a time; work holds min(nr, 16) values per interior row
void launch_rhs_prepare(const PrimalDev &P, int nsub, int nr, const double *f, int64_t fstr, double *hf, double *yf,
                        int64_t ystr, double *work, hipStream_t st) {
    for (int v0 = 0; v0 < nr; v0 += 16) {
        const int K = std::min(nr - v0, 16);
        const double *fv = f + v0 * fstr;
        hipLaunchKernelGGL(k_band_solves<false>, dim3(nsub), dim3(64 * BAND_WAVES), 0, st, P, K, fv, fstr,
                           yf + v0 * ystr, ystr, work);
        cross<true>(P, nsub, K, fv, fstr, hf + v0, nr, work, st);
    }
}

void launch_primal(const PrimalDev &P, int nsub, int nr, double *ub, double *yf, int64_t ystr, const double *alpha,
                   int64_t astr, double *u, int64_t ustr, double *work, hipStream_t st) {
    for (int v0 = 0; v0 < nr; v0 += 16) {
        const int K = std::min(nr - v0, 16);
        if (P.max_ni > 0) {
            cross<false>(P, nsub, K, nullptr, 0, ub + v0, nr, work, st);
            hipLaunchKernelGGL(k_band_solves<true>, dim3(nsub), dim3(64 * BAND_WAVES), 0, st, P, K,
                               (const double *)nullptr, (int64_t)0, yf + v0 * ystr, ystr, work);
        }
        hipLaunchKernelGGL(k_primal_write, dim3((P.max_n + 255) / 256, nsub), dim3(256), 0, st, P, K, ub + v0, nr,
                           alpha + v0 * astr, astr, u + v0 * ustr, ustr, work);
    }
}

// ---- structured grid on the device: K_i values (CSR of the grid builder)
// from the unit element matrix Ke and the element material scales.  One
// thread per CSR entry (row = local node x DOF, columns = the existing
// neighbours of the node in (z, y, x) offset order, DOFs inside); the entry
// sums scale_e * Ke over the elements holding both nodes in increasing (z, y,
// x) element order with separately rounded products and sums -- the order
// and rounding of the host builder's element loop, so the values agree bit
// for bit (structuralmechanics3d.cpp:353-509, physics.cpp:147-228).
__device__ __forceinline__ int hexa_corner(int cx, int cy, int cz) { return 4 * cz + (cy ? (cx ? 2 : 3) : (cx ? 1 : 0)); }

__global__ void __launch_bounds__(256) k_grid_stiffness(int nd, const int *box, int NE0, int NE1, const double *Ke,
                                                        const double *escale, const int *rowptr,
                                                        const int64_t *rp_off, const int64_t *nz_off, double *vals) {
    const int s = blockIdx.y;
    const int *bx = box + 6 * s;
    const int gx0 = bx[0], gy0 = bx[1], gz0 = bx[2], ex = bx[3], ey = bx[4], ez = bx[5];
    const int lx = ex + 1, ly = ey + 1, lz = ez + 1;
    const int n = lx * ly * lz * nd, ne = 8 * nd;
    const int *rp = rowptr + rp_off[s];
    const int nnz = rp[n];
    double *v = vals + nz_off[s];
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nnz; q += gridDim.x * blockDim.x) {
#pragma clang fp contract(off)
        int lo = 0, hi = n;  // row r with rp[r] <= q < rp[r + 1]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (rp[mid] <= q) lo = mid;
            else hi = mid;
        }
        const int r = lo, ln = r / nd, i = r % nd;
        const int pos = q - rp[r], slot = pos / nd, j = pos % nd;
        const int x = ln % lx, y = (ln / lx) % ly, z = ln / (lx * ly);
        const int nxo = 1 + (x > 0) + (x < lx - 1), nyo = 1 + (y > 0) + (y < ly - 1);
        const int x2 = x + slot % nxo - (x > 0), y2 = y + (slot / nxo) % nyo - (y > 0),
                  z2 = z + slot / (nxo * nyo) - (z > 0);
        double acc = 0.0;
        for (int e2 = max(max(z, z2) - 1, 0); e2 <= min(min(z, z2), ez - 1); e2++)
            for (int e1 = max(max(y, y2) - 1, 0); e1 <= min(min(y, y2), ey - 1); e1++)
                for (int e0 = max(max(x, x2) - 1, 0); e0 <= min(min(x, x2), ex - 1); e0++) {
                    const int a = hexa_corner(x - e0, y - e1, z - e2), b = hexa_corner(x2 - e0, y2 - e1, z2 - e2);
                    const double sc = escale[(gx0 + e0) + (int64_t)NE0 * ((gy0 + e1) + (int64_t)NE1 * (gz0 + e2))];
                    const double t = sc * Ke[(nd * a + i) * ne + nd * b + j];  // rounded product (no FMA)
                    acc = acc + t;
                }
        v[q] = acc;
    }
}

__global__ void k_gather_values(int64_t n, const int64_t *pos, const double *src, double *dst) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[pos[i]];
}

// ---- structured grid: element sensitivities sens_e = -w_e^T K_e0 u_e ----
__global__ void __launch_bounds__(256) k_element_sensitivity(int NE0, int NE1, int NE2, int nd, const double *Ke0,
                                                             const double *u, const double *w, double *sens) {
    extern __shared__ double K[];
    const int ne = 8 * nd;
    for (int q = threadIdx.x; q < ne * ne; q += 256) K[q] = Ke0[q];
    __syncthreads();
    const int NN0 = NE0 + 1, NN1 = NE1 + 1;
    const int64_t nel = (int64_t)NE0 * NE1 * NE2;
    const int cx[8] = {0, 1, 1, 0, 0, 1, 1, 0}, cy[8] = {0, 0, 1, 1, 0, 0, 1, 1}, cz[8] = {0, 0, 0, 0, 1, 1, 1, 1};
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nel; e += (int64_t)gridDim.x * blockDim.x) {
        const int ex = (int)(e % NE0), ey = (int)((e / NE0) % NE1), ez = (int)(e / ((int64_t)NE0 * NE1));
        double ue[24], we[24];
        for (int a = 0; a < 8; a++) {
            const int64_t node = (ex + cx[a]) + (int64_t)NN0 * ((ey + cy[a]) + (int64_t)NN1 * (ez + cz[a]));
            for (int c = 0; c < nd; c++) {
                ue[a * nd + c] = u[node * nd + c];
                we[a * nd + c] = w[node * nd + c];
            }
        }
        double v = 0.0;
        for (int i = 0; i < ne; i++) {
            double t = 0.0;
            for (int j = 0; j < ne; j++) t += K[i * ne + j] * ue[j];
            v += we[i] * t;
        }
        sens[e] = -v;
    }
}

void launch_element_sensitivity(const int *NE, int nd, const double *Ke0, const double *u, const double *w,
                                double *sens, hipStream_t st) {
    const int64_t nel = (int64_t)NE[0] * NE[1] * NE[2];
    const int ne = 8 * nd;
    hipLaunchKernelGGL(k_element_sensitivity, dim3(vgrid(nel)), dim3(256), (size_t)ne * ne * 8, st, NE[0], NE[1],
                       NE[2], nd, Ke0, u, w, sens);
}

void launch_grid_stiffness(int nsub, int nd, const int *box, const int *NE, const double *Ke, const double *escale,
                           const int *rowptr, const int64_t *rp_off, const int64_t *nz_off, int max_nnz, double *vals,
                           hipStream_t st) {
    const unsigned gx = (unsigned)std::max(1, std::min((max_nnz + 255) / 256, 2048));
    hipLaunchKernelGGL(k_grid_stiffness, dim3(gx, nsub), dim3(256), 0, st, nd, box, NE[0], NE[1], Ke, escale, rowptr,
                       rp_off, nz_off, vals);
}

void launch_gather_values(int64_t n, const int64_t *pos, const double *src, double *dst, hipStream_t st) {
    if (n > 0) hipLaunchKernelGGL(k_gather_values, dim3(vgrid(n)), dim3(256), 0, st, n, pos, src, dst);
}

// ---- KKT report (itersolver.cpp:199-251) ----
// r = K_i u_i - (f_i - B1_i^T lambda) + B0_i^T lambda0 over the local DOFs of
// every subdomain; out[2s] = sum r^2, out[2s+1] = sum (f_i - B1_i^T lambda)^2.
// bt1 = B1^T lambda and bt0 = B0^T lambda0 (may be null) are boundary vectors;
// the boundary values of u are copied to ub (for B1 u).  Workgroup (g, s)
// takes rows 64g..64g+63 of subdomain s, 16 lanes per CSR row (the lanes of
// a group read consecutive entries of the row, 16 groups read 16 consecutive
// rows), and writes its two sums to part[2 (s G + g)]; k_kkt_sums adds the G
// partials of a subdomain in order (deterministic).
constexpr int KKT_ROWS = 64;
__global__ void __launch_bounds__(256) k_kkt_primal(const PrimalDev P, const double *u, const double *f,
                                                    const double *bt1, const double *bt0, double *ub, double *part) {
    __shared__ double red[4];
    const int s = blockIdx.y, g = blockIdx.x, G = gridDim.x;
    const int n = P.n[s], ni = P.ni[s];
    const int64_t uo = P.perm_off[s], ro = P.rp_off[s], zo = P.nz_off[s], bo = P.boff[s];
    const int grp = threadIdx.x >> 4, l = threadIdx.x & 15;
    double a1 = 0.0, a2 = 0.0;
#pragma unroll
    for (int k = 0; k < KKT_ROWS / 16; k++) {
        const int i = g * KKT_ROWS + 16 * k + grp;
        if (i >= n) break;  // uniform over the group
        double ku = 0.0;
        const int q1 = P.rowptr[ro + i + 1];
        for (int q = P.rowptr[ro + i] + l; q < q1; q += 16) ku += P.vals[zo + q] * u[uo + P.colidx[zo + q]];
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) ku += __shfl_xor(ku, o, 16);
        if (l == 0) {
            double t = f[uo + i], c0 = 0.0;
            const int pi = P.iperm[uo + i];
            if (pi >= ni) {
                const int64_t j = bo + pi - ni;
                t -= bt1[j];
                if (bt0) c0 = bt0[j];
                ub[j] = u[uo + i];
            }
            const double r = ku - t + c0;
            a1 += r * r;
            a2 += t * t;
        }
    }
    a1 = block_sum(a1, red);
    a2 = block_sum(a2, red);
    if (threadIdx.x == 0) {
        part[2 * ((int64_t)s * G + g)] = a1;
        part[2 * ((int64_t)s * G + g) + 1] = a2;
    }
}

__global__ void k_kkt_sums(int nsub, int G, const double *part, double *out) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsub) return;
    double a1 = 0.0, a2 = 0.0;
    for (int g = 0; g < G; g++) {
        a1 += part[2 * ((int64_t)s * G + g)];
        a2 += part[2 * ((int64_t)s * G + g) + 1];
    }
    out[2 * s] = a1;
    out[2 * s + 1] = a2;
}

// bt0 = B0^T lambda0 on the boundary: one thread per subdomain walks its B0
// slots and their entries in order (a DOF may sit in several rows)
__global__ void k_b0t(int nsub, const int64_t *boff, const ClusterDev C, double *bt0) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsub) return;
    for (int64_t q = C.qoff[s]; q < C.qoff[s + 1]; q++) {
        const double l0 = C.lambda0[C.qrow[q]];
        for (int64_t e = C.qe_ptr[q]; e < C.qe_ptr[q + 1]; e++) bt0[boff[s] + C.qe_j[e]] += C.qe_c[e] * l0;
    }
}

int kkt_groups(int max_n) { return std::max(1, (max_n + KKT_ROWS - 1) / KKT_ROWS); }

void launch_kkt_primal(const PrimalDev &P, int nsub, int max_n, const double *u, const double *f, const double *bt1,
                       const double *bt0, double *ub, double *part, double *out, hipStream_t st) {
    const int G = kkt_groups(max_n);
    hipLaunchKernelGGL(k_kkt_primal, dim3(G, nsub), dim3(256), 0, st, P, u, f, bt1, bt0, ub, part);
    hipLaunchKernelGGL(k_kkt_sums, dim3((nsub + 255) / 256), dim3(256), 0, st, nsub, G, part, out);
}

void launch_b0t(const DualDev &D, const ClusterDev &C, double *bt0, hipStream_t st) {
    hipLaunchKernelGGL(k_b0t, dim3((D.nsub + 255) / 256), dim3(256), 0, st, D.nsub, D.boff, C, bt0);
}

// ---- output truncation (FETISolver.cpp:131-148) ----
__global__ void k_absmax_partial(const double *u, int64_t n, double *partial) {
    __shared__ double red[4];
    double m = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        m = fmax(m, fabs(u[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_down(m, o, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// D = 1 / precision / max(1, 10^ceil(log10(max|u|))); u <- trunc(D u) / D.
// The maximum starts at the smallest normal double, as the reference's does.
__global__ void k_truncate(double *u, int64_t n, const double *partial, int np, double precision) {
    __shared__ double dpl;
    if (threadIdx.x == 0) {
        double m = 2.2250738585072014e-308;
        for (int b = 0; b < np; b++) m = fmax(m, partial[b]);
        dpl = 1.0 / precision / fmax(1.0, pow(10.0, ceil(log10(m))));
    }
    __syncthreads();
    const double d = dpl;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        u[i] = trunc(d * u[i]) / d;
}

void launch_truncate(double *u, int64_t n, double precision, double *partial, hipStream_t st) {
    const int np = 256;
    hipLaunchKernelGGL(k_absmax_partial, dim3(np), dim3(256), 0, st, u, n, partial);
    hipLaunchKernelGGL(k_truncate, dim3(vgrid(n)), dim3(256), 0, st, u, n, (const double *)partial, np, precision);
}

}  // namespace esp
