// rte_adjoint.hip -- reverse mode of the truncated Neumann series: the
// vector-Jacobian product of the bottom-face exitance with respect to the
// per-voxel mu_a and mu_s (the reference differentiates by one extra forward
// Neumann solve per parameter, FisherInfo_IO/src/compute_grad_rte.cu:273-385;
// here one adjoint series serves all voxels).
//
// With W_0 = s0, W_{q+1} = D A W_q (q < n-1) and E = ball + e^T A sum_q W_q,
// for a cotangent c on the image (eps = sum_p c_p e_p):
//   xi_{n-1} = eps,  Lambda_q = A^T xi_q,  xi_{q-1} = eps + D Lambda_q,
//   dE.c = sum_q xi_q^T dA W_q + sum_{q>=1} Lambda_q^T dD (A W_{q-1})
//          + Lambda_0^T ds0 + c^T dball.
// A^T applies the off-diagonal part through reciprocity, A_off^T = P A_off P
// (tau and r symmetric, R(-u) = (-1)^l R(u)), and the self block S = S^T as is.
// The mu_t-derivative of A_off goes through k(d,s) = e^{-tau}/r^2:
//   d k / d mu_t(v) = -len_v(d,s) k, len_v the Siddon length of the ray in v,
// so the adjoint propagation also accumulates per pair
//   w(d,s) = sum_q k (xi_q(d).R) (R.W_q(s))
// which one back-projection along the rays turns into the gradient.
#include "rte_device.hpp"

namespace rte {

// Up to kMaxNC adjoint series (cotangents) share each propagation launch: the
// pair geometry, its z-power values and the projection of the forward term are
// formed once per pair for all of them.
template <typename T, typename TA>
struct AdjDev {
    const T *Xz[kMaxNC];  // [N][K] adjoint inputs n_a (-1)^l xi_a, in the z-power basis
    const T *Wqz;         // [N][K] forward term n_a W_a, in the z-power basis
    T *part[kMaxNC];      // [nchunk][N][K] (z-power basis; k_adj_combine turns the sum back)
    T *pairbuf[kMaxNC];   // [N][npad] pair weights w(d = source slot row, s = lane)
    const T *ktab;        // [N][npad]
};

template <int L>
__device__ __forceinline__ int l_of(int a)
{
    int l = 0;
#pragma unroll
    for (int ll = 1; ll <= L; ++ll) l += (a >= ll * ll) ? 1 : 0;
    return l;
}

// ---------------------------------------------------------------------------
// A_off applied to P xi_c (uniform input u, lane output o) for NC cotangents c,
// plus the pair weights pairbuf_c[u][slot(o)] += k (Z.P xi_c(u)) (Z.P W_q(o)).
// In the z-power basis Z(u) of the forward kernel: P acts on it as on the
// harmonics, (-1)^l on entry (l, m), since Z_l,m(-u) = (-1)^l Z_l,m(u), and the
// pair weight, a product of two projections, does not depend on the basis.
// grid = (nblk, nchunk), block = 64.
// ---------------------------------------------------------------------------
template <typename T, typename TA, int L, int NC>
__global__ __launch_bounds__(kWave) void k_prop_adj(PropArgs<T> A, AdjDev<T, TA> D)
{
#pragma clang fp contract(off)
    constexpr int K = (L + 1) * (L + 1);
    const GridDev<T> &g = A.g;
    const int lane = threadIdx.x, blk = blockIdx.x, chunk = blockIdx.y;
    int di, dj, dk;
    lane_dest(g, blk, lane, di, dj, dk);
    const bool valid = di < g.nx && dj < g.ny && dk < g.nz;
    const int cdi = min(di, g.nx - 1), cdj = min(dj, g.ny - 1), cdk = min(dk, g.nz - 1);
    const int vo = cdi + g.nx * (cdj + g.ny * cdk);
    const int slot = blk * kWave + lane;
    const int s0 = chunk * A.chunk_len;
    const int s1 = min(g.N, s0 + A.chunk_len);
    const int nxy = g.nx * g.ny;

    T acc[NC][K], wl[K];
#pragma unroll
    for (int a = 0; a < K; ++a) {
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c][a] = T(0);
        const T sgn = (l_of<L>(a) & 1) ? T(-1) : T(1);
        wl[a] = sgn * D.Wqz[(size_t)vo * K + a];
    }
    cptr<T> X[NC];
    T *pb[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        X[c] = as_const<T>(D.Xz[c]);
        pb[c] = D.pairbuf[c] + slot;
    }
    const gptr<T> ktab = as_global<T>(D.ktab);
    const T dxc = T(cdi) * g.dx, dyc = T(cdj) * g.dy, dzc = T(cdk) * g.dz;
    int si = s0 % g.nx, sj = (s0 / g.nx) % g.ny, sk = s0 / nxy;
    // the table entry and the pair weights of the next source are loaded one source
    // ahead (the last source's again at the chunk's end: in bounds, unused); a lane
    // outside the grid keeps its weights in registers and never stores them
    T kf_next = s0 < s1 ? __builtin_nontemporal_load(ktab + (size_t)s0 * g.npad + slot) : T(0), pw_next[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) pw_next[c] = s0 < s1 ? pb[c][(size_t)s0 * g.npad] : T(0);
    for (int s = s0; s < s1; ++s) {
        const T ddx = fmad(-T(si), g.dx, dxc), ddy = fmad(-T(sj), g.dy, dyc), ddz = fmad(-T(sk), g.dz, dzc);
        // the self pair's table entry is 0 and its direction (0, 0, 0): r^2 clamped as in k_prop
        const T r2 = max(fmad(ddx, ddx, fmad(ddy, ddy, ddz * ddz)), T(1e-30));
        const T kf = kf_next;
        T pw[NC];
        const int sn = (s + 1 < s1) ? s + 1 : s;
        kf_next = __builtin_nontemporal_load(ktab + (size_t)sn * g.npad + slot);  // read once, as in k_prop
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            pw[c] = pw_next[c];
            pw_next[c] = pb[c][(size_t)sn * g.npad];
        }
        const T rinv = dev_rsqrt<T>(r2);
        PairZ<T, L> G;
        pair_zpow<T, L>(G, ddx * rinv, ddy * rinv, ddz * rinv);
        const T dl = pair_dot_z<T, L>(wl, G);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            T w[K];
#pragma unroll
            for (int a = 0; a < K; ++a) w[a] = X[c][(size_t)s * K + a];
            const T t = kf * pair_dot_z<T, L>(w, G);
            pair_axpy_z<T, L>(acc[c], t, G);
            if (valid) pb[c][(size_t)s * g.npad] = fmad(t, dl, pw[c]);
        }
        if (++si == g.nx) {
            si = 0;
            if (++sj == g.ny) {
                sj = 0;
                ++sk;
            }
        }
    }
    if (valid) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            T *__restrict__ out = D.part[c] + ((size_t)chunk * g.N + vo) * K;
#pragma unroll
            for (int a = 0; a < K; ++a) out[a] = acc[c][a];
        }
    }
}

// [N][K] buffers into the z-power basis, out_i = M^T in_i (one thread per voxel
// and buffer; grid = (ceil(N / 256), n), block = 256)
template <typename T>
struct ZBufs {
    const T *in[kMaxNC + 1];
    T *out[kMaxNC + 1];
};

template <typename T, int L>
__global__ __launch_bounds__(256) void k_bufs_to_zpow(int N, ZBufs<T> B)
{
    constexpr int K = (L + 1) * (L + 1);
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= N) return;
    const T *__restrict__ w = B.in[blockIdx.y] + (size_t)v * K;
    T *__restrict__ o = B.out[blockIdx.y] + (size_t)v * K;
    double x[K], y[K];
#pragma unroll
    for (int a = 0; a < K; ++a) x[a] = double(w[a]);
    zpow_from_harmonic<double, L>(x, y);
#pragma unroll
    for (int j = 0; j < K; ++j) o[j] = T(y[j]);
}

// ---------------------------------------------------------------------------
// Per voxel: Lambda_q = A^T xi_q, the self-block and scatter gradient terms,
// and the next adjoint input xi_{q-1} = eps + D Lambda_q (written over X).
// Laid out as k_combine, and bound by the same partials: a thread per (voxel,
// coefficient) in place of one per voxel, 24^3, L = 5, FP32 143 -> 30 us; a 16^3
// gradient of 8 terms 4.87 -> 4.20 ms, 9^3 at L = 7 2.83 -> 1.71.
// The self block S(mu) = self_scale sum_k c_k M_k, c_k = (-mu)^{k-1}/k!, acts on xi
// (c_k), and on W_q for its mu-derivative (dc_k/dmu): two products with each moment.
// grid = ceil(N/VB), block = kCombThreads.
// ---------------------------------------------------------------------------
template <typename T, typename TA, int L>
__global__ __launch_bounds__(kCombThreads) void k_adj_combine(AdjCombArgs<T, TA> A)
{
    using Sh = CombShape<L>;
    constexpr int K = Sh::K, VP = Sh::VP, VPT = Sh::VPT, VB = Sh::VB, NJ = Sh::NJ, NZ = Sh::NZ;
    constexpr bool f32 = sizeof(T) == 4;
    __shared__ TA zs[VB * K];               // z-power sums
    __shared__ TA gp[VB * K], sp[VB * K];   // terms of the mu_t and mu_s gradients; FP64: the self block's sums first
    __shared__ T xs[VB * K], ws[VB * K];    // xi, W_q
    __shared__ T cf[2][kNMom][VB];          // c_k, dc_k/dmu
    __shared__ T ms[f32 ? kNMom * NJ * K : 1];
    const GridDev<T> &g = A.g;
    const CombTab<L> &tab = kCombTab<L>;
    const int tid = threadIdx.x, v0 = blockIdx.x * VB;
    const bool live = tid < VP * K;
    const int a = tid % K, q0 = tid / K;
    if constexpr (f32) {
        for (int q = tid; q < kNMom * NJ * K; q += kCombThreads) {
            const int aa = q % K, i = (q / K) % NJ, k = q / (K * NJ), b = tab.b[i][aa];
            ms[q] = b < 0 ? T(0) : A.momT[(size_t)k * K * K + aa * K + b];
        }
    }
    if (tid < VB) {
        // c = (-mu)^k/(k+1)!, dc/dmu = -k (-mu)^{k-1}/(k+1)! for moment index k+1; pw = (-mu)^{k-1}
        const T mu = A.mut[min(v0 + tid, g.N - 1)];
        T pw = T(1), fact = T(1);
        for (int k = 0; k < kNMom; ++k) {
            fact *= T(k + 1);
            cf[1][k][tid] = (k == 0) ? T(0) : -T(k) * pw / fact;
            pw = (k == 0) ? T(1) : pw * (-mu);
            cf[0][k][tid] = pw / fact;
        }
    }
    const TA na = A.nsc[live ? a : 0];
    const TA sgn = (l_of<L>(a) & 1) ? TA(-1) : TA(1);
    if (live) {
        const size_t cs = (size_t)g.N * K;
        size_t e[VPT];
        TA sum[VPT];
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int v = v0 + i * VP + q0;
            e[i] = v < g.N ? (size_t)v * K + a : a;  // beyond the grid: voxel 0's, not used
            xs[i * VP * K + tid] = T(sgn * TA(A.X[e[i]]) / na);
            ws[i * VP * K + tid] = T(TA(A.Wq[e[i]]) / na);
            sum[i] = TA(0);
        }
        const T *__restrict__ p = A.part;
#pragma unroll 8
        for (int c = 0; c < A.nchunk; ++c, p += cs) {
#pragma unroll
            for (int i = 0; i < VPT; ++i) sum[i] += TA(p[e[i]]);
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i) zs[i * VP * K + tid] = sum[i];
    }
    __syncthreads();
    if constexpr (!f32) {
        // the self block on the matrix instruction, as in k_combine
        typedef double d4 __attribute__((ext_vector_type(4)));
        constexpr int RT = (K + 15) / 16, CT = (VB + 15) / 16, KS = (K + 3) / 4;
        const int lane = tid & (kWave - 1), n = lane & 15, gr = lane >> 4;
        for (int u = tid / kWave; u < RT * CT; u += kCombThreads / kWave) {
            const int rt = u % RT, vv = (u / RT) * 16 + n, vc = min(vv, VB - 1), row = min(rt * 16 + n, K - 1);
            double x[2][KS], sum[2][4] = {};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int b = 4 * s + gr, o = vc * K + min(b, K - 1);
                const double xb = xs[o], wb = ws[o];
                x[0][s] = b < K ? xb : 0.0;
                x[1][s] = b < K ? wb : 0.0;
            }
            const gptr<double> M = as_global<double>(A.mom) + (size_t)row * K;
#pragma unroll 1
            for (int k = 0; k < kNMom; ++k) {
                d4 y[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const double m = M[(size_t)k * K * K + min(4 * s + gr, K - 1)];
                    y[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(m, x[0][s], y[0], 0, 0, 0);
                    y[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(m, x[1][s], y[1], 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum[0][r] += cf[0][k][vc] * y[0][r];
                    sum[1][r] += cf[1][k][vc] * y[1][r];
                }
            }
            // result r of a lane: row 4 r + gr, column n
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ra = rt * 16 + 4 * r + gr;
                if (vv < VB && ra < K) {
                    sp[vv * K + ra] = sum[0][r];
                    gp[vv * K + ra] = sum[1][r];
                }
            }
        }
        __syncthreads();
    }
    const int P = g.nx * g.ny;
    if (live) {
        const int l = l_of<L>(a);
        const bool m0 = a == l * l + l;
        TA gl = TA(1);
#pragma unroll
        for (int ll = 1; ll <= L; ++ll) gl = ll <= l ? gl * A.g_aniso : gl;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int v = v0 + i * VP + q0, o = (i * VP + q0) * K;
            TA acc = TA(0), st, gs;
#pragma unroll
            for (int t = 0; t < NZ; ++t) {  // back to the harmonic basis
                const int j = tab.j[t][a];
                if (j >= 0) acc = fmad(TA(tab.z[t][a]), zs[o + j], acc);
            }
            if constexpr (f32) {
                T x[NJ], w[NJ], s32 = T(0), g32 = T(0);
#pragma unroll
                for (int t = 0; t < NJ; ++t) {
                    const int b = tab.b[t][a];
                    const T xb = xs[o + (b < 0 ? a : b)], wb = ws[o + (b < 0 ? a : b)];
                    x[t] = b < 0 ? T(0) : xb;
                    w[t] = b < 0 ? T(0) : wb;
                }
#pragma unroll 2
                for (int k = 0; k < kNMom; ++k) {
                    T rx = T(0), rw = T(0);
#pragma unroll
                    for (int t = 0; t < NJ; ++t) {
                        const T m = ms[(k * NJ + t) * K + a];
                        rx = t ? fmad(m, x[t], rx) : m * x[t];
                        rw = t ? fmad(m, w[t], rw) : m * w[t];
                    }
                    s32 = fmad(cf[0][k][i * VP + q0], rx, s32);
                    g32 = fmad(cf[1][k][i * VP + q0], rw, g32);
                }
                st = TA(s32);
                gs = TA(xs[o + a] * g32);
            } else {
                st = sp[o + a];
                gs = xs[o + a] * gp[o + a];
            }
            acc = (sgn * acc * na + A.self_scale * st) * A.dV;  // Lambda_q
            gp[o + a] = gs;
            const bool in = v < g.N;
            const size_t e = (size_t)(in ? v : 0) * K + a;
            sp[o + a] = A.aw_prev ? acc * gl * A.aw_prev[e] : TA(0);
            if (!in) continue;
            if (A.lam0 && m0) A.lam0[(size_t)v * (L + 1) + l] = acc;
            TA xn = gl * TA(A.mus[v]) * acc;
            if (m0 && v >= g.N - P) xn += A.cot[v - (g.N - P)] * A.coefE[l];
            A.X[e] = T(sgn * xn * na);
        }
    }
    __syncthreads();
    if (tid < VB && v0 + tid < g.N) {
        TA gt = TA(0), gs = TA(0);
        for (int c = 0; c < K; ++c) {
            gt += gp[tid * K + c];
            gs += sp[tid * K + c];
        }
        A.gt[v0 + tid] += A.self_scale * A.dV * gt;
        if (A.aw_prev) A.gs[v0 + tid] += gs;
    }
}

// X <- n (-1)^l eps: the adjoint input of the last term.  grid = ceil(N/64).
template <typename T, typename TA, int L>
__global__ void k_adj_init(GridDev<T> g, const TA *cot, Scales sc, const TA *coefE, T *X)
{
    constexpr int K = (L + 1) * (L + 1);
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.N) return;
    const int zk = v / (g.nx * g.ny);
    const int pix = v - zk * g.nx * g.ny;
#pragma unroll
    for (int l = 0; l <= L; ++l) {
        const double sgn = (l & 1) ? -1.0 : 1.0;
#pragma unroll
        for (int m = -l; m <= l; ++m) {
            const int a = l * l + l + m;
            double x = 0.0;
            if (m == 0 && zk == g.nz - 1) x = (double)cot[pix] * (double)coefE[l];
            X[(size_t)v * K + a] = T(sgn * x * sc.n[a]);
        }
    }
}

// Wq <- n (g^l mu_s A W_{q-1}): the forward term W_q from the stored A W_{q-1}.
template <typename T, typename TA, int L>
__global__ void k_make_wq(GridDev<T> g, Scales sc, TA gan, const T *mus, const TA *aw_prev, T *Wq)
{
    constexpr int K = (L + 1) * (L + 1);
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.N) return;
    const TA ms = TA(mus[v]);
    TA gl = TA(1);
#pragma unroll
    for (int l = 0; l <= L; ++l) {
#pragma unroll
        for (int m = -l; m <= l; ++m) {
            const int a = l * l + l + m;
            Wq[(size_t)v * K + a] = T(gl * ms * aw_prev[(size_t)v * K + a] * TA(sc.n[a]));
        }
        gl *= gan;
    }
}

// ---------------------------------------------------------------------------
// Back-projection: gt(v) += scale * sum_pairs w(pair) len_v(pair), each pair's
// ray walked as the path table was built, accumulated in LDS when the grid fits
// and in global memory otherwise, over unordered pairs: the ray between two voxel
// centres crosses the same voxels with the same Siddon lengths both ways (the
// crossings alpha = (j + 1/2)/n mirror into each other; only zero-length
// segments at exact ties may fall in different voxels), so the pair weights of
// (d, s) and (s, d) are added and the ray is marched once.  As in the path table a
// brick pair is (bs, bs + D), D in the half space z, then y, then x >= 0; on D = 0
// only the pairs with slot(s) < slot(d).
// A wave takes M translations of a brick pair, lane = (translation, 64 / M of the
// destinations), and walks 16 sources of the brick with M steps over its
// destinations; what lies beyond the grid for all its translations is left out.  With
// M = 1 its rays leave the source through the same few voxels, and the atomics on
// one address are served one after the other, ~110 clocks of the LDS per crossing;
// translated rays are in different voxels throughout, but a small grid has few
// translations, and a ragged one leaves lanes without a voxel: see launch_backproject.
// A grid whose sums do not fit the LDS goes in slabs of z planes, a y-row of blocks each:
// a slab's rays (those that reach it) are walked whole and their voxels outside it left
// out.  (With atomics in memory a gradient at
// 28^3, L = 5, 8 terms took 506 ms, 32^3 1302, 40^3, L = 3, 5139; in slabs 55, 92 and 310.)  Only where that takes
// more than kBpSlabs slabs do the atomics go to memory.
// grid = (at most the resident blocks, slabs); of the units (translation group, D, 16 of
// the source brick's 64 voxels) a block takes one of each run of gridDim.x, its waves
// share them.  Which one moves on by rot from run to run where the z planes of a brick
// are not all in the grid: with the same one, 3 of 4 blocks of a grid of one plane had
// nothing to do (100x100x1: 18.6 -> 4.5 ms).
// ---------------------------------------------------------------------------
constexpr int kBpSlabs = 16;
struct BpPlan {
    int py, pz;      // pitches of y and z in the accumulator (elements)
    int zs;          // z planes of a slab
    int nD, nunits;
    int rot;
    int next;        // where in LDS the block's unit counter lies (bytes), -1: no room
};

// MEM 0: sums in memory; 1: in LDS; 2: in LDS by slabs
template <typename T, typename TA, int MEM, int M>
__global__ __launch_bounds__(1024) void k_backproject_sym(GridDev<T> g, BpPlan p, T thr2, const T *__restrict__ pairbuf,
                                                          TA scale, TA *gt)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    TA *sacc = reinterpret_cast<TA *>(smem_raw);
    int *next = reinterpret_cast<int *>(smem_raw + p.next);
    constexpr int ND = kWave / M;                   // destinations side by side
    const int tid = threadIdx.x, lane = tid & (kWave - 1), m = lane / ND, sub = lane % ND;
    const int nxy = g.nx * g.ny;
    constexpr bool LDS = MEM != 0;
    const int z0 = MEM == 2 ? blockIdx.y * p.zs : 0, z1 = MEM == 2 ? min(z0 + p.zs, g.nz) : g.nz;
    const int lo = z0 * p.pz, size = (z1 - z0) * p.pz;
    if constexpr (LDS)
        for (int i = tid; i < size; i += blockDim.x) sacc[i] = TA(0);
    if (p.next >= 0 && tid == 0) *next = 0;
    __syncthreads();
    const int ex = 2 * g.bx - 1, ey = 2 * g.by - 1;
    for (int own = tid / kWave;; own += blockDim.x / kWave) {
        // the block's next unit (in a fixed order where the accumulator leaves no room for a counter)
        if (p.next >= 0 && lane == 0) own = atomicAdd(next, 1);
        const unsigned run = __builtin_amdgcn_readfirstlane(own);
        const unsigned b = p.rot ? (blockIdx.x + run * (unsigned)p.rot) % gridDim.x : blockIdx.x;
        const int u = (int)(b + gridDim.x * run);
        if (gridDim.x * run >= (unsigned)p.nunits) break;
        if (u >= p.nunits) continue;
        const int slab = u & 3, f = (u >> 2) % p.nD + p.nD - 1, first = (u >> 2) / p.nD * M;
        const int Dx = f % ex - (g.bx - 1), Dy = (f / ex) % ey - (g.by - 1), Dz = f / (ex * ey) - (g.bz - 1);
        const int cx = g.bx - abs(Dx), cy = g.by - abs(Dy), cnt = cx * cy * (g.bz - abs(Dz));
        if (first >= cnt) continue;
        const bool other = (Dx | Dy | Dz) != 0, live = first + m < cnt;
        // this lane's source brick
        const int t = min(first + m, cnt - 1);
        const int bx0 = t % cx + max(0, -Dx), by0 = (t / cx) % cy + max(0, -Dy), bz0 = t / (cx * cy) + max(0, -Dz);
        const int bs = bx0 + g.bx * (by0 + g.by * bz0), bd = bs + Dx + g.bx * (Dy + g.by * Dz);
        // the nearest pair of the bricks is not coupled (thr2 is rounded, and r^2 below)
        const T nearx = T(max(0, kBrick * abs(Dx) - 3)) * g.dx, neary = T(max(0, kBrick * abs(Dy) - 3)) * g.dy,
                nearz = T(max(0, kBrick * abs(Dz) - 3)) * g.dz;
        if (sum_squares(nearx, neary, nearz) > thr2 * T(1.0001)) continue;
        // the lowest voxels of the wave's source bricks: a source (or the part of the destinations
        // that the step alone decides) that is beyond the grid there is so for all of them
        int lx = bx0, ly = by0, lz = bz0;
        if constexpr (M > 1) {
#pragma unroll
            for (int o = kWave / 2; o >= ND; o >>= 1) {
                lx = min(lx, __shfl_xor(lx, o));
                ly = min(ly, __shfl_xor(ly, o));
                lz = min(lz, __shfl_xor(lz, o));
            }
        }
        lx = __builtin_amdgcn_readfirstlane(lx) * kBrick;
        ly = __builtin_amdgcn_readfirstlane(ly) * kBrick;
        lz = __builtin_amdgcn_readfirstlane(lz) * kBrick;
        auto from = [&](int it) {  // the first step from it on with a pair in the grid
            for (; it < 16 * M; ++it) {
                const int q = slab * 16 + it / M, j = it % M * ND;
                if (lx + (q & 3) < g.nx && ly + ((q >> 2) & 3) < g.ny && lz + (q >> 4) < g.nz &&
                    (ND >= 16 || ly + Dy * kBrick + ((j >> 2) & 3) < g.ny) &&
                    (ND >= 64 || lz + Dz * kBrick + (j >> 4) < g.nz))
                    break;
            }
            return it;
        };
        // pair it = source 16 slab + it / M of the brick, destination slot (it % M) ND + sub
        struct Pair { int ix, iy, iz, v; T r2, w0, w1; };
        auto load = [&](int it) {
            const int q = slab * 16 + it / M, j = it % M * ND + sub;
            const int sx = q & 3, sy = (q >> 2) & 3, sz = q >> 4, lx = j & 3, ly = (j >> 2) & 3, lz = j >> 4;
            const int x = bx0 * kBrick + sx, y = by0 * kBrick + sy, z = bz0 * kBrick + sz;
            Pair P;
            P.ix = Dx * kBrick + lx - sx;
            P.iy = Dy * kBrick + ly - sy;
            P.iz = Dz * kBrick + lz - sz;
            const int X = x + P.ix, Y = y + P.iy, Z = z + P.iz;
            const T ddx = T(P.ix) * g.dx, ddy = T(P.iy) * g.dy, ddz = T(P.iz) * g.dz;
            P.r2 = sum_squares(ddx, ddy, ddz);
            const bool ok = live && x < g.nx && y < g.ny && z < g.nz && X < g.nx && Y < g.ny && Z < g.nz &&
                            (other || q < j) && P.r2 < thr2 && (MEM != 2 || (max(z, Z) >= z0 && min(z, Z) < z1));
            P.v = LDS ? x + p.py * y + p.pz * z : x + g.nx * y + nxy * z;
            P.w0 = P.w1 = T(0);
            if (ok) {
                P.w0 = pairbuf[(size_t)(x + g.nx * y + nxy * z) * g.npad + bd * kWave + j];
                P.w1 = pairbuf[(size_t)(X + g.nx * Y + nxy * Z) * g.npad + bs * kWave + q];
            }
            return P;
        };
        int it = from(0);
        if (it == 16 * M) continue;
        Pair nx = load(it);
        while (it < 16 * M) {
            const Pair P = nx;
            it = from(it + 1);
            if (it < 16 * M) nx = load(it);  // the next pair's weights under this one's march
            const TA w = TA(P.w0) + TA(P.w1);
            if (w == TA(0)) continue;
            const TA sw = scale * w;
            const T r = sqrt(P.r2);
            march_visit<T>(P.v, P.ix, P.iy, P.iz, LDS ? p.py : g.nx, LDS ? p.pz : nxy, r, [&](int v, T len) {
                if constexpr (MEM == 2) {
                    if ((unsigned)(v - lo) < (unsigned)size) atomicAdd(&sacc[v - lo], sw * TA(len));
                } else if constexpr (LDS) {
                    atomicAdd(&sacc[v], sw * TA(len));
                } else {
                    atomicAdd(&gt[v], sw * TA(len));
                }
            });
        }
    }
    if constexpr (LDS) {
        __syncthreads();
        for (int i = z0 * nxy + tid; i < z1 * nxy; i += blockDim.x) {
            const int x = i % g.nx, y = (i / g.nx) % g.ny, z = i / nxy;
            const TA a = sacc[x + p.py * y + p.pz * z - lo];
            if (a != TA(0)) atomicAdd(&gt[i], a);
        }
    }
}

// ---------------------------------------------------------------------------
// Back-projection onto parameter blocks (the exact Fisher information needs only
// sums of the mu_t gradient over each block, part[v] in [0, nparam) or -1): for
// NC backward passes at once, out_c[p] += scale * sum_pairs w_c(pair) len_p(pair),
// len_p the length of the pair's ray inside block p.  The tiling and the march are
// those of k_backproject_sym (unordered pairs, w_c = both directions' weights), one
// march for all NC passes; a lane adds the lengths of consecutive voxels of one
// block in a register and adds w_c times that run to the block's LDS accumulator
// when the ray leaves the block.  The part map is read from LDS.
// grid = ceil(ntiles / 16), block = 1024; LDS = N ints + NC nparam accumulators.
// ---------------------------------------------------------------------------
template <typename T, typename TA, int NC>
__global__ __launch_bounds__(1024) void k_backproject_blocks(GridDev<T> g, int ntiles, T thr2, BlockBp<T, TA> B)
{
    extern __shared__ unsigned char smem_raw[];
    int *spart = reinterpret_cast<int *>(smem_raw);
    TA *sacc = reinterpret_cast<TA *>(smem_raw + (((size_t)g.N * sizeof(int) + 15) & ~size_t(15)));
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    for (int i = tid; i < g.N; i += blockDim.x) spart[i] = B.part[i];
    for (int i = tid; i < NC * B.nparam; i += blockDim.x) sacc[i] = TA(0);
    __syncthreads();
    const int tile = blockIdx.x * (blockDim.x / kWave) + tid / kWave;
    if (tile < ntiles) {
        int bd = (int)((sqrtf(8.0f * (float)tile + 1.0f) - 1.0f) * 0.5f);
        while (bd > 0 && bd * (bd + 1) / 2 > tile) --bd;
        while ((bd + 1) * (bd + 2) / 2 <= tile) ++bd;
        const int bs = tile - bd * (bd + 1) / 2;
        int di, dj, dk;
        lane_dest(g, bd, lane, di, dj, dk);
        const bool dvalid = di < g.nx && dj < g.ny && dk < g.nz;
        const int cdi = min(di, g.nx - 1), cdj = min(dj, g.ny - 1), cdk = min(dk, g.nz - 1);
        const int nxy = g.nx * g.ny;
        const int dslot = bd * kWave + lane;
        const int dlin = cdi + g.nx * cdj + nxy * cdk;
        const int bxi = bs % g.bx, byi = (bs / g.bx) % g.by, bzi = bs / (g.bx * g.by);
        for (int q = 0; q < kWave; ++q) {
            const int si = bxi * kBrick + (q & 3), sj = byi * kBrick + ((q >> 2) & 3), sk = bzi * kBrick + (q >> 4);
            if (si >= g.nx || sj >= g.ny || sk >= g.nz) continue;  // wave-uniform
            const int sslot = bs * kWave + q;
            const int ix = cdi - si, iy = cdj - sj, iz = cdk - sk;
            const T ddx = T(ix) * g.dx, ddy = T(iy) * g.dy, ddz = T(iz) * g.dz;
            const T r2 = sum_squares(ddx, ddy, ddz);
            const bool self = (ix == 0) && (iy == 0) && (iz == 0);
            const bool once = bs != bd || sslot < dslot;
            if (!(dvalid && !self && once && r2 < thr2)) continue;
            const int slin = si + g.nx * sj + nxy * sk;
            TA sw[NC];
            bool any = false;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                sw[c] = B.scale * (TA(B.pairbuf[c][(size_t)slin * g.npad + dslot]) +
                                   TA(B.pairbuf[c][(size_t)dlin * g.npad + sslot]));
                any = any || sw[c] != TA(0);
            }
            if (!any) continue;
            int cur = -1;
            TA run = TA(0);
            auto flush = [&]() {
                if (cur >= 0) {
#pragma unroll
                    for (int c = 0; c < NC; ++c) atomicAdd(&sacc[c * B.nparam + cur], sw[c] * run);
                }
            };
            march_visit<T>(slin, ix, iy, iz, g.nx, nxy, sqrt(r2), [&](int v, T len) {
                const int p = spart[v];
                if (p != cur) {
                    flush();
                    cur = p;
                    run = TA(0);
                }
                run += TA(len);
            });
            flush();
        }
    }
    __syncthreads();
    for (int i = tid; i < NC * B.nparam; i += blockDim.x)
        if (sacc[i] != TA(0)) atomicAdd(&B.out[i / B.nparam][i % B.nparam], sacc[i]);
}

// ---------------------------------------------------------------------------
// Source and ballistic derivatives along each beam column (column products of
// k_source): s0_l0(k) = F_l h(k), h(k) = (mu_s/mu_t)(k) T(k) (1 - a_k),
// a_k = e^{-mu_t(k) dz}, T(k) = prod_{k'<k} a_k', ballistic = fact T(nz).
// ga/gs receive d(Lambda_0.s0 + c.ball)/d mu_a, d mu_s.  grid = ceil(P/64).
// ---------------------------------------------------------------------------
template <typename TA, int L>
__global__ void k_src_grad(int nx, int ny, int nz, double dxd, double dyd, double dzd, double xmin,
                           double ymin, double gan, BeamDev B, const TA *lam0, const TA *cot, TA *ga, TA *gs)
{
    const int pix = blockIdx.x * blockDim.x + threadIdx.x;
    const int P = nx * ny;
    if (pix >= P) return;
    const int i = pix % nx, j = pix / nx;
    const double xc = (double)i * dxd + xmin + dxd / 2.0;
    const double yc = (double)j * dyd + ymin + dyd / 2.0;
    const double rad = sqrt((xc - B.pos_x) * (xc - B.pos_x) + (yc - B.pos_y) * (yc - B.pos_y));
    if (!(rad <= B.half_diam)) return;
    const double dV = dxd * dyd * dzd;
    // F_l folded into Y(k) = sum_l Lambda0_l0(k) fact g^l sqrt((2l+1)/4pi) / dV
    double ball = 1.0;
    for (int k = 0; k < nz; ++k) ball *= exp(-(B.mua[pix + P * k] + B.mus[pix + P * k]) * dzd);
    ball *= B.fact;
    // suffix sum of Y(k) h(k) for k > k''
    double suffix = 0.0;
    for (int k = nz - 1; k >= 0; --k) {
        const int v = pix + P * k;
        double Tprod = 1.0;
        for (int kk = 0; kk < k; ++kk) Tprod *= exp(-(B.mua[pix + P * kk] + B.mus[pix + P * kk]) * dzd);
        const double ma = B.mua[v], ms = B.mus[v], mt = ma + ms;
        const double ak = exp(-mt * dzd);
        double Y = 0.0, gl = 1.0;
        for (int l = 0; l <= L; ++l) {
            Y += (double)lam0[(size_t)v * (L + 1) + l] * B.fact * gl * sqrt((2.0 * l + 1.0) / (4.0 * M_PI)) / dV;
            gl *= gan;
        }
        const double h = (ms / mt) * Tprod * (1.0 - ak);
        // d h / d mu_t(k) at fixed mu_s, and the mu_s/mu_t factor
        const double dh_dmt = ms * Tprod * (-(1.0 - ak) / (mt * mt) + dzd * ak / mt);
        const double dh_dms_extra = Tprod * (1.0 - ak) / mt;
        const double up = -dzd * suffix;                 // later voxels of the column
        const double bal = -dzd * (double)cot[pix] * ball;
        ga[v] += TA(up + Y * dh_dmt + bal);
        gs[v] += TA(up + Y * (dh_dmt + dh_dms_extra) + bal);
        suffix += Y * h;
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// The reference's forward-mode derivative (FisherInfo_IO/src/compute_grad_rte.cu:
// 273-301 mu_a, 341-371 mu_s): the first term of solve i is its parameter's
// region of the forward field phi = sum_q A W_q times -fs (mu_a) or
// fs (g^l - 1) (mu_s), in scaled coefficients; its pixel buffers start at zero
// (no ballistic term) with the bottom-layer stop-rule sums of that first term.
// fs = n: the reference scales its field out2 = phi / c_m by -1.0*C and
// (g^l - 1) C with C the vacuum speed (FisherInfo_IO/src/rte.h:15,
// compute_grad_rte.cu:292,350-353), which is phi times C / c_m = n here.
// wrt 2 with part == nullptr: phi itself, every voxel (a given first term,
// the reference's Neumann(src, out, 1), FisherInfo_IO/src/neumann.cu:23).
// grid = (ceil(N/64), nsolve), block = 64.
// ---------------------------------------------------------------------------
template <typename T, typename TA, int L>
__global__ __launch_bounds__(kWave) void k_ref_source(GridDev<T> g, Scales sc, const int *__restrict__ part,
                                                     const int *__restrict__ param, int wrt, TA gan, TA fs,
                                                     const TA *__restrict__ phi, const TA *__restrict__ wsum,
                                                     const SolveDev<T, TA> *__restrict__ sv)
{
    constexpr int K = (L + 1) * (L + 1);
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.N) return;
    const SolveDev<T, TA> S = sv[blockIdx.y];
    // part == nullptr: every voxel (a given first term, wrt 2)
    const bool in = part ? part[v] == param[blockIdx.y] : true;
    TA gl = TA(1), bs = TA(0);
#pragma unroll
    for (int l = 0; l <= L; ++l) {
        const TA f = wrt == 0 ? -fs : wrt == 1 ? fs * (gl - TA(1)) : TA(1);
#pragma unroll
        for (int m = -l; m <= l; ++m) {
            const int a = l * l + l + m;
            const T wt = in ? T(f * phi[(size_t)v * K + a] * TA(sc.n[a])) : T(0);
            S.W[(size_t)v * K + a] = wt;
            bs += wsum[a] * (TA(wt) / TA(sc.n[a]));
        }
        gl *= gan;
    }
    const int P = g.nx * g.ny;
    if (v >= (g.nz - 1) * P) {
        const int pix = v - (g.nz - 1) * P;
        S.E[pix] = TA(0);
        S.dE[pix] = TA(0);
        S.bsum[pix] = bs;
    }
    if (v < P) {
        S.R[v] = TA(0);
        S.dR[v] = TA(0);
    }
}

// y += x over n elements
template <typename TA>
__global__ void k_accumulate(size_t n, const TA *__restrict__ x, TA *__restrict__ y)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += x[i];
}

#define RTE_DISPATCH_L2(L, ...)                          \
    switch (L) {                                        \
    case 0: { constexpr int LL = 0; __VA_ARGS__; } break; \
    case 1: { constexpr int LL = 1; __VA_ARGS__; } break; \
    case 2: { constexpr int LL = 2; __VA_ARGS__; } break; \
    case 3: { constexpr int LL = 3; __VA_ARGS__; } break; \
    case 4: { constexpr int LL = 4; __VA_ARGS__; } break; \
    case 5: { constexpr int LL = 5; __VA_ARGS__; } break; \
    case 6: { constexpr int LL = 6; __VA_ARGS__; } break; \
    case 7: { constexpr int LL = 7; __VA_ARGS__; } break; \
    default: return hipErrorInvalidValue;                \
    }

template <typename T, typename TA>
hipError_t launch_adj_prop(int L, const PropArgs<T> &A, int nc, const T *const *X, T *const *Xz, const T *Wq, T *Wqz,
                           T *const *part, T *const *pairbuf, const T *ktab, hipStream_t st)
{
    if (nc < 1 || nc > kMaxNC) return hipErrorInvalidValue;
    // the inputs into the z-power basis: the forward term and each cotangent's xi
    ZBufs<T> B{};
    B.in[0] = Wq;
    B.out[0] = Wqz;
    AdjDev<T, TA> D{};
    D.Wqz = Wqz;
    D.ktab = ktab;
    for (int c = 0; c < nc; ++c) {
        B.in[1 + c] = X[c];
        B.out[1 + c] = Xz[c];
        D.Xz[c] = Xz[c];
        D.part[c] = part[c];
        D.pairbuf[c] = pairbuf[c];
    }
    RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_bufs_to_zpow<T, LL>), dim3((A.g.N + 255) / 256, 1 + nc), dim3(256), 0,
                                          st, A.g.N, B));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    dim3 grid(A.g.nblk, A.nchunk), block(kWave);
    if (nc == 1) {
        RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_prop_adj<T, TA, LL, 1>), grid, block, 0, st, A, D));
    } else {
        RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_prop_adj<T, TA, LL, 2>), grid, block, 0, st, A, D));
    }
    return hipGetLastError();
}

template <typename T, typename TA>
hipError_t launch_adj_combine(int L, const AdjCombArgs<T, TA> &A, hipStream_t st)
{
    RTE_DISPATCH_L2(L, {
        constexpr int VB = CombShape<LL>::VB;
        hipLaunchKernelGGL((k_adj_combine<T, TA, LL>), dim3((A.g.N + VB - 1) / VB), dim3(kCombThreads), 0, st, A);
    });
    return hipGetLastError();
}

template <typename T, typename TA>
hipError_t launch_adj_init(int L, const GridDev<T> &g, const TA *cot, const Scales &sc, const TA *coefE, T *X,
                           hipStream_t st)
{
    dim3 grid((g.N + 63) / 64), block(64);
    RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_adj_init<T, TA, LL>), grid, block, 0, st, g, cot, sc, coefE, X));
    return hipGetLastError();
}

template <typename T, typename TA>
hipError_t launch_make_wq(int L, const GridDev<T> &g, const Scales &sc, TA gan, const T *mus, const TA *aw_prev,
                          T *Wq, hipStream_t st)
{
    dim3 grid((g.N + 63) / 64), block(64);
    RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_make_wq<T, TA, LL>), grid, block, 0, st, g, sc, gan, mus, aw_prev, Wq));
    return hipGetLastError();
}

template <typename T, typename TA, int MEM, int M>
static hipError_t launch_bp_as(const GridDev<T> &g, BpPlan p, size_t lds, int cus, T thr2, const T *pairbuf, TA scale,
                               TA *gt, hipStream_t st)
{
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_backproject_sym<T, TA, MEM, M>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    // a large accumulator leaves room for one block per CU: make it 16 waves.  M = 1 takes as
    // many as fit (18^3, 47 KB: 24 waves a CU 1.10 ms, 12 1.36)
    const int threads = lds > 64 * 1024 ? 1024 : M == 1 ? 512 : 256, waves = threads / kWave;
    const int percu = M == 1 && threads == 512 ? min(4, (int)(160 * 1024 / lds)) : 1024 / threads;
    p.nunits = p.nD * ((g.nblk + M - 1) / M) * 4;
    const int blocks = min((p.nunits + waves - 1) / waves, cus * percu);
    p.rot = g.nz % kBrick ? (int)(0.618 * blocks) | 1 : 0;
    const int slabs = MEM == 2 ? (g.nz + p.zs - 1) / p.zs : 1;
    hipLaunchKernelGGL((k_backproject_sym<T, TA, MEM, M>), dim3(blocks, slabs), dim3(threads), lds, st, g, p, thr2, pairbuf,
                       scale, gt);
    return hipGetLastError();
}

template <typename T, typename TA>
hipError_t launch_backproject(const GridDev<T> &g, T thr2, const T *pairbuf, TA scale, TA *gt, hipStream_t st)
{
    DevLimits lim;
    const hipError_t le = device_limits(&lim);
    if (le != hipSuccess) return le;
    const int lds_max = lim.lds_max, cus = lim.cus;
    // odd pitches (the translations' voxels in different banks) where that fits
    BpPlan p{};
    size_t lds = 0;
    auto fits = [&](int py, int pz, int slabs) {
        p.py = py;
        p.pz = pz;
        p.zs = (g.nz + slabs - 1) / slabs;
        const size_t acc = ((size_t)pz * p.zs * sizeof(TA) + 15) / 16 * 16;
        p.next = acc + 16 <= (size_t)lds_max ? (int)acc : -1;
        lds = p.next >= 0 ? acc + 16 : acc;
        return lds <= (size_t)lds_max;
    };
    int mem = 0;
    for (int n = 1; n <= kBpSlabs && n <= g.nz && !mem; ++n)
        if (fits(g.nx | 1, (g.nx | 1) * g.ny | 1, n) || fits(g.nx, g.nx * g.ny, n)) mem = n == 1 ? 1 : 2;
    if (!mem) {
        p.next = 0;
        lds = 16;
    }
    p.nD = ((2 * g.bx - 1) * (2 * g.by - 1) * (2 * g.bz - 1) + 1) / 2;
    // 16 translations where the crossings are many enough for their units to fill the chip;
    // 1 on smaller grids, and on thin ones, whose translations meet in the same columns; 4 where a
    // coupling threshold leaves little of a large grid.  us with 1 / 4 / 16, FP32 table: 8^3 29 /
    // 127 / 567, 16^3 603 / 710 / 1043, 20^3 2300 / 2580 / 1640, 24^3 7430 / 7680 / 3760 (threshold
    // of 4.7 voxels 161 / 126 / 296, 10.3 806 / 815 / 667), 100x100x1 11900 / 11100 / 4500, 5x5x200
    // 2480 / 2740 / 4280; a wave per brick pair and source, as before the translations: 8^3 152,
    // 16^3 760, 20^3 2290, 24^3 8210, 100x100x1 12300, 5x5x200 3620
    double cross = 0.0;  // voxels crossed by the coupled pairs' rays
    const double fill = (double)g.N / g.npad;
    for (int Dz = 0; Dz < g.bz; ++Dz)
        for (int Dy = 0; Dy < g.by; ++Dy)
            for (int Dx = 0; Dx < g.bx; ++Dx) {
                const double x = (double)kBrick * Dx * g.dx, y = (double)kBrick * Dy * g.dy, z = (double)kBrick * Dz * g.dz;
                if (x * x + y * y + z * z >= (double)thr2) continue;
                const double signs = (Dx ? 2.0 : 1.0) * (Dy ? 2.0 : 1.0) * (Dz ? 2.0 : 1.0);
                cross += 0.5 * signs * (g.bx - Dx) * (g.by - Dy) * (g.bz - Dz) * kBrick * max(1, Dx + Dy + Dz);
            }
    cross *= fill * fill * kWave * kWave;
    const int top = max(g.bx, max(g.by, g.bz));
    const bool thin = g.nblk < 10 * top, big = g.nblk >= 200;  // 10 bricks a layer across the longest axis
    const int most = thin ? 1 : cross >= (big ? 1.8e8 : 6e8) ? 16 : big ? 4 : 1;
#define RTE_BP(MEM)                                                                                   \
    (most == 16  ? launch_bp_as<T, TA, MEM, 16>(g, p, lds, cus, thr2, pairbuf, scale, gt, st)         \
     : most == 4 ? launch_bp_as<T, TA, MEM, 4>(g, p, lds, cus, thr2, pairbuf, scale, gt, st)          \
                 : launch_bp_as<T, TA, MEM, 1>(g, p, lds, cus, thr2, pairbuf, scale, gt, st))
    return mem == 1 ? RTE_BP(1) : mem == 2 ? RTE_BP(2) : RTE_BP(0);
#undef RTE_BP
}

template <typename T, typename TA>
hipError_t launch_backproject_blocks(const GridDev<T> &g, T thr2, const BlockBp<T, TA> &B, int nc, hipStream_t st)
{
    DevLimits lim;
    const hipError_t le = device_limits(&lim);
    if (le != hipSuccess) return le;
    const int lds_max = lim.lds_max;
    if (nc < 1 || nc > kMaxNC || B.nparam < 1) return hipErrorInvalidValue;
    const size_t lds = (((size_t)g.N * sizeof(int) + 15) & ~size_t(15)) + (size_t)nc * B.nparam * sizeof(TA);
    if (lds > (size_t)lds_max) return hipErrorInvalidValue;  // the caller back-projects per voxel
    const int ntiles = g.nblk * (g.nblk + 1) / 2;
    constexpr int threads = 1024, waves = threads / kWave;
    const void *fn = nc == 1 ? reinterpret_cast<const void *>(&k_backproject_blocks<T, TA, 1>)
                             : reinterpret_cast<const void *>(&k_backproject_blocks<T, TA, 2>);
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    if (nc == 1)
        hipLaunchKernelGGL((k_backproject_blocks<T, TA, 1>), dim3((ntiles + waves - 1) / waves), dim3(threads), lds,
                           st, g, ntiles, thr2, B);
    else
        hipLaunchKernelGGL((k_backproject_blocks<T, TA, 2>), dim3((ntiles + waves - 1) / waves), dim3(threads), lds,
                           st, g, ntiles, thr2, B);
    return hipGetLastError();
}

template <typename TA>
hipError_t launch_src_grad(int L, int nx, int ny, int nz, double dx, double dy, double dz, double xmin, double ymin,
                           double gan, const BeamDev &B, const TA *lam0, const TA *cot, TA *ga, TA *gs, hipStream_t st)
{
    const int P = nx * ny;
    dim3 grid((P + 63) / 64), block(64);
    RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_src_grad<TA, LL>), grid, block, 0, st, nx, ny, nz, dx, dy, dz, xmin,
                                          ymin, gan, B, lam0, cot, ga, gs));
    return hipGetLastError();
}

template <typename T, typename TA>
hipError_t launch_ref_source(int L, const GridDev<T> &g, const Scales &sc, const int *part, const int *param, int wrt,
                             TA gan, TA fs, const TA *phi, const TA *wsum, const SolveDev<T, TA> *sv, int nsolve,
                             hipStream_t st)
{
    dim3 grid((g.N + kWave - 1) / kWave, nsolve), block(kWave);
    RTE_DISPATCH_L2(L, hipLaunchKernelGGL((k_ref_source<T, TA, LL>), grid, block, 0, st, g, sc, part, param, wrt,
                                          gan, fs, phi, wsum, sv));
    return hipGetLastError();
}

template <typename TA>
hipError_t launch_accumulate(size_t n, const TA *x, TA *y, hipStream_t st)
{
    hipLaunchKernelGGL(k_accumulate<TA>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, x, y);
    return hipGetLastError();
}

template hipError_t launch_ref_source<float, double>(int, const GridDev<float> &, const Scales &, const int *,
                                                     const int *, int, double, double, const double *, const double *,
                                                     const SolveDev<float, double> *, int, hipStream_t);
template hipError_t launch_ref_source<double, double>(int, const GridDev<double> &, const Scales &, const int *,
                                                      const int *, int, double, double, const double *, const double *,
                                                      const SolveDev<double, double> *, int, hipStream_t);
template hipError_t launch_accumulate<double>(size_t, const double *, double *, hipStream_t);
template hipError_t launch_adj_prop<float, double>(int, const PropArgs<float> &, int, const float *const *,
                                                   float *const *, const float *, float *, float *const *,
                                                   float *const *, const float *, hipStream_t);
template hipError_t launch_adj_prop<double, double>(int, const PropArgs<double> &, int, const double *const *,
                                                    double *const *, const double *, double *, double *const *,
                                                    double *const *, const double *, hipStream_t);
template hipError_t launch_adj_combine<float, double>(int, const AdjCombArgs<float, double> &, hipStream_t);
template hipError_t launch_adj_combine<double, double>(int, const AdjCombArgs<double, double> &, hipStream_t);
template hipError_t launch_adj_init<float, double>(int, const GridDev<float> &, const double *, const Scales &,
                                                   const double *, float *, hipStream_t);
template hipError_t launch_adj_init<double, double>(int, const GridDev<double> &, const double *, const Scales &,
                                                    const double *, double *, hipStream_t);
template hipError_t launch_make_wq<float, double>(int, const GridDev<float> &, const Scales &, double,
                                                  const float *, const double *, float *, hipStream_t);
template hipError_t launch_make_wq<double, double>(int, const GridDev<double> &, const Scales &, double,
                                                   const double *, const double *, double *, hipStream_t);
template hipError_t launch_backproject<float, double>(const GridDev<float> &, float, const float *,
                                                      double, double *, hipStream_t);
template hipError_t launch_backproject<double, double>(const GridDev<double> &, double, const double *,
                                                       double, double *, hipStream_t);
template hipError_t launch_backproject_blocks<float, double>(const GridDev<float> &, float,
                                                             const BlockBp<float, double> &, int, hipStream_t);
template hipError_t launch_backproject_blocks<double, double>(const GridDev<double> &, double,
                                                              const BlockBp<double, double> &, int, hipStream_t);
template hipError_t launch_src_grad<double>(int, int, int, int, double, double, double, double, double, double,
                                            const BeamDev &, const double *, const double *, double *, double *,
                                            hipStream_t);

}  // namespace rte
