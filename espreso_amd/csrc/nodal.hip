// Structured-grid fields on the device: nodal loads split over the subdomain
// copies of a node, subdomain fields summed or averaged over the copies, and the
// kernel dots R_s^T f_s of new loads.  Every pass reads and writes each value once
// (a few tens of MB at a million nodes), so the link to the host bounds what is
// left; the same loops on the host took 125 of 380 ms of a 16-case block at 2000
// heat subdomains.
#include <hip/hip_runtime.h>

#include "dual.h"

namespace esp {

static inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// f[q nd + c] = g[node(q) nd + c] / copies(node(q)) for the local nodes q of every
// subdomain; *bad is set when a value of g is not finite.  grid (chunks, subdomains, cases)
__global__ void __launch_bounds__(256) k_nodal_split(const GridDev G, const int64_t *__restrict__ uoff,
                                                     const double *__restrict__ g, int64_t gstr, double *__restrict__ f,
                                                     int64_t fstr, int *bad) {
    const int s = blockIdx.y, nd = G.nd;
    const int *b = G.box + 6 * s;
    const int lx = b[3] + 1, ly = b[4] + 1, n = lx * ly * (b[5] + 1) * nd;
    g += blockIdx.z * gstr;
    f += blockIdx.z * fstr + uoff[s];
    bool nan = false;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const int q = i / nd, c = i - q * nd;
        const int x = b[0] + q % lx, y = b[1] + q / lx % ly, z = b[2] + q / (lx * ly);
        const double v = g[(x + G.NN[0] * (y + (int64_t)G.NN[1] * z)) * nd + c];
        nan |= !isfinite(v);
        f[i] = v / (double)(G.cnt[0][x] * G.cnt[1][y] * G.cnt[2][z]);
    }
    if (nan) atomicOr(bad, 1);
}

// g[node nd + c] = sum over the copies of the node of u (average: divided by their
// number); a thread per value, cases along grid y
__global__ void __launch_bounds__(256) k_nodal_gather(const GridDev G, const int64_t *__restrict__ uoff,
                                                      const double *__restrict__ u, int64_t ustr,
                                                      double *__restrict__ g, int64_t gstr, int average) {
    const int nd = G.nd;
    const int64_t n = (int64_t)G.NN[0] * G.NN[1] * G.NN[2] * nd;
    u += blockIdx.y * ustr;
    g += blockIdx.y * gstr;
    for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t node = i / nd;
        const int c = (int)(i - node * nd), x = (int)(node % G.NN[0]);
        const int64_t yz = node / G.NN[0];
        const int y = (int)(yz % G.NN[1]), z = (int)(yz / G.NN[1]);
        const int cx = G.cnt[0][x], cy = G.cnt[1][y], cz = G.cnt[2][z];
        double v = 0.0;
        for (int k = G.hi[2][z] - cz + 1; k <= G.hi[2][z]; k++)
            for (int j = G.hi[1][y] - cy + 1; j <= G.hi[1][y]; j++)
                for (int l = G.hi[0][x] - cx + 1; l <= G.hi[0][x]; l++) {
                    const int s = G.subid[l + G.NS[0] * (j + G.NS[1] * k)];
                    const int *b = G.box + 6 * s;
                    const int q = (x - b[0]) + (b[3] + 1) * ((y - b[1]) + (b[4] + 1) * (z - b[2]));
                    v += u[uoff[s] + (int64_t)q * nd + c];
                }
        g[i] = average ? v / (double)(cx * cy * cz) : v;
    }
}

// e0f[(asub[s] + a) K + v] = -sum_i R_s(i, a) f_v(i): one workgroup per subdomain and case
__global__ void __launch_bounds__(256) k_rhs_dots(const PrimalDev P, const double *__restrict__ f, int64_t fstr, int K,
                                                  double *__restrict__ e0f) {
    __shared__ double red[4];
    const int s = blockIdx.x, v = blockIdx.y, n = P.n[s], k = P.kdim[s];
    const double *fs = f + v * fstr + P.perm_off[s], *R = P.R + P.r_off[s];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int a = 0; a < k; a++) {
        double t = 0.0;
#pragma unroll 4
        for (int i = threadIdx.x; i < n; i += 256) t += R[i + (int64_t)a * n] * fs[i];
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if (lane == 0) red[w] = t;
        __syncthreads();
        if (threadIdx.x == 0) e0f[(P.asub[s] + a) * K + v] = -((red[0] + red[1]) + (red[2] + red[3]));
        __syncthreads();
    }
}

// coarse right-hand side e[(coff + b) K + v] = sum over the block's subdomains of
// N_s^T e0f_s,v; a thread per (block, column, case)
__global__ void k_coarse_rhs(const DualDev D, int K, const double *__restrict__ e0f, double *__restrict__ e) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < D.nblk * 64 * K; t += gridDim.x * blockDim.x) {
        const int blk = t / (64 * K), b = t / K & 63, v = t % K;
        const int q0 = D.blk_ptr[blk], q1 = D.blk_ptr[blk + 1];
        if (b >= D.ck[D.blk_sub[q0]]) continue;  // blocks hold at most 64 columns
        double sum = 0.0;
        for (int q = q0; q < q1; q++) {
            const int s = D.blk_sub[q], k = D.kdim[s];
            const double *N = D.N + D.noff[s] + (int64_t)b * k;
            for (int a = 0; a < k; a++) sum += N[a] * e0f[(D.asub[s] + a) * K + v];
        }
        e[(int64_t)(D.coff[blk] + b) * K + v] = sum;
    }
}

void launch_nodal_split(const GridDev &G, int nsub, int max_n, int K, const int64_t *uoff, const double *g, int64_t gstr,
                        double *f, int64_t fstr, int *bad, hipStream_t st) {
    hipLaunchKernelGGL(k_nodal_split, dim3(std::max(1u, std::min(cdiv(max_n, 256), 64u)), nsub, K), dim3(256), 0, st, G,
                       uoff, g, gstr, f, fstr, bad);
}

void launch_nodal_gather(const GridDev &G, int K, const int64_t *uoff, const double *u, int64_t ustr, double *g,
                         int64_t gstr, bool average, hipStream_t st) {
    const int64_t n = (int64_t)G.NN[0] * G.NN[1] * G.NN[2] * G.nd;
    hipLaunchKernelGGL(k_nodal_gather, dim3(std::max(1u, std::min(cdiv(n, 256), 8192u)), K), dim3(256), 0, st, G, uoff,
                       u, ustr, g, gstr, average ? 1 : 0);
}

void launch_rhs_dots(const PrimalDev &P, const DualDev &D, int K, const double *f, int64_t fstr, double *e0f, double *e,
                     hipStream_t st) {
    hipLaunchKernelGGL(k_rhs_dots, dim3(D.nsub, K), dim3(256), 0, st, P, f, fstr, K, e0f);
    hipLaunchKernelGGL(k_coarse_rhs, dim3(std::max(1u, std::min(cdiv((int64_t)D.nblk * 64 * K, 256), 4096u))), dim3(256),
                       0, st, D, K, e0f, e);
}

}  // namespace esp
