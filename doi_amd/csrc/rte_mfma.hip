// rte_mfma.hip -- propagation A on the matrix cores (FP32 cached path, L = 4 and 5).
//
// The pair sums of k_prop,
//   acc(d) = sum_s kf(d,s) (Z(d-s) . W(s)) Z(d-s),
// are two contractions once the pairs are grouped by displacement: Z depends on d - s
// only, so a destination slab D (4x4x1 voxels) and a source tile S (4x4x2) moved by the
// same translations t (and every right-hand side) share all their Z.  With 16 columns
// c = (right-hand side, translation):
//   P(d, c)     = sum_j Z_j(d-s) W_j(s + t_c)            one product per source s: 16 d x 16 c
//   T(d, s, c)  = kf(d + t_c, s + t_c) P(d, c)            the only per-pair work left on the VALU
//   acc(j, c)  += sum_s Z_j(d-s) T(d, s, c)              one product per destination d: K x 16 c
// Z and W, and then Z and T, go through v_mfma_f32_16x16x32_f16 as two FP16 pieces each
// (x = h + l, Z and W to 24 bits, T to 22; products hh + hl + lh, sums in FP32); powers of two
// keep every piece in range and are taken out of each tile's sums: for W the largest of its
// source slab and right-hand side, for T the largest path-table entry of the source slab and
// destination (k_kexp).  Media where these leave a contribution fewer bits than FP32 run
// k_prop (even_medium).  Error of 32^3, L = 5 solves against FP64 2.8e-7 to 4.4e-7, on the FP32
// vector pipe 6.2e-7 to 6.4e-7.
//
// Measured per term at 32^3 (k_prop, all VALU, whose FMAs run at 94 % of the pipe's rate ->
// this): L = 5 one solve 3.28 -> 2.10 ms, 5 beams 9.4 -> 7.3, 15 on 3 media 27.5 -> 16.6;
// L = 4 2.71 -> 1.80, 7.5 -> 6.1, 19.7 -> 13.9.  Bound in the benchmark's launches: issue of a
// SIMD's two waves (VALU 40 %, MFMA 28 % of the clocks, mostly one after the other) and LDS
// (48 %, 9 % bank conflicts); the rest is waits at the tile's two barriers.
#include "rte_device.hpp"

namespace rte {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

// Layout of one displacement's (or source voxel's) pieces: NJ tiles of 16 coefficients,
// h then l, and for L = 5 the last 4 coefficients' h and l.
template <int L>
struct MLay {
    static constexpr int K = (L + 1) * (L + 1);
    static constexpr int NJ = 2;                      // whole 16-coefficient tiles
    static constexpr bool REM = L == 5;               // 4 coefficients beyond 32
    static constexpr int H = NJ * 32;                 // bytes of the h pieces
    static constexpr int WB = REM ? 144 : 2 * H;      // bytes of a W row
    static constexpr int U = WB / 16;                 // 16-byte pieces of a row
    // LDS pitches of a Z row, a y line of 7 rows, a plane of 7 lines, and a column of W rows:
    // in 16-byte units 10, 8 and 2 (mod 16), so that neither a 16-lane phase of a
    // b128 read (rows 4 x 4, of which the two middle y lines one piece further) nor a
    // 32-lane phase of a transposed read (4 rows x 2 pieces, two y lines) meets a bank twice
    static constexpr int XP = 160;
    static constexpr int YP = 1152;
    static constexpr int PP = 7 * YP;
    static constexpr int CP = 16 * WB + 32;
};

constexpr float kZScale = 1024.f;                     // Z pieces hold 2^10 Z

// split x = h + l, both rounded to nearest: |l| <= 2^-12 |x|, of either sign, so that the l l
// products that are left out are below 2^-24 and do not add up.  Error of A W against FP64,
// rms relative to k_prop's, mean over 24 media of 32^3: first term of a pencil beam 1.01
// (with h cut off, every l of x's sign, 1.47), the next four terms 0.3.
__device__ __forceinline__ void split2(float x, _Float16 &h, _Float16 &l)
{
    h = (_Float16)x;
    l = (_Float16)(x - (float)h);
}

template <int L>
__device__ __forceinline__ void store_row(unsigned char *row, const float (&v)[(L + 1) * (L + 1)])
{
    using M = MLay<L>;
    constexpr int J = M::NJ * 16;
    _Float16 h[J], l[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        h[j] = l[j] = (_Float16)0.f;
        if (j < M::K) split2(v[j < M::K ? j : 0], h[j], l[j]);
    }
#pragma unroll
    for (int q = 0; q < J / 8; ++q) {
        h8 a, b;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            a[e] = h[8 * q + e];
            b[e] = l[8 * q + e];
        }
        *reinterpret_cast<h8 *>(row + 16 * q) = a;
        *reinterpret_cast<h8 *>(row + M::H + 16 * q) = b;
    }
    if constexpr (M::REM) {
        h8 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            _Float16 x, y;
            split2(v[32 + e], x, y);
            a[e] = x;
            a[4 + e] = y;
        }
        *reinterpret_cast<h8 *>(row + 2 * M::H) = a;
    }
}

// ---------------------------------------------------------------------------
// The Z pieces of every displacement of a grid's bricks, once per grid and order:
// row (ix, iy, iz) = displacement (ix - (4 bx - 1), iy - (4 by - 1), iz - (nz - 1)).
// grid = ceil(rows / 256), block = 256.
// ---------------------------------------------------------------------------
template <int L>
__global__ __launch_bounds__(256) void k_ztab(int nxt, int nyt, int nzt, double dx, double dy, double dz,
                                              unsigned char *__restrict__ zt)
{
    using M = MLay<L>;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nxt * nyt * nzt) return;
    const int ix = (int)(i % nxt), iy = (int)((i / nxt) % nyt), iz = (int)(i / ((size_t)nxt * nyt));
    const double x = (ix - nxt / 2) * dx, y = (iy - nyt / 2) * dy, z = (iz - nzt / 2) * dz;
    const double r2 = x * x + y * y + z * z, ri = r2 > 0.0 ? 1.0 / sqrt(r2) : 0.0;
    PairZ<double, L> G;
    pair_zpow<double, L>(G, x * ri, y * ri, z * ri);
    float v[M::K];
#pragma unroll
    for (int a = 0; a < M::K; ++a) v[a] = (float)(G.R[a] * (double)kZScale);
    store_row<L>(zt + i * M::WB, v);
}

// ---------------------------------------------------------------------------
// W into its pieces: one lane per voxel of a slab (4x4x1 voxels, zero outside the
// grid), slab (bx, by, z) = (by nbx + bx) nz + z, and after the last one a slab of
// zeros.  The slab's largest |W'| is brought to [2^9, 2^10) by a power of two, kept
// (inverted) behind the rows.  grid = (ceil((nslab + 1) / 4), nsolve), block = 64.
// ---------------------------------------------------------------------------
template <typename TA, int L>
__global__ __launch_bounds__(kWave) void k_to_pieces(GridDev<float> g, const SolveDev<float, TA> *__restrict__ sv)
{
    using M = MLay<L>;
    constexpr int K = M::K;
    const int nslab = g.bx * g.by * g.nz;
    const int lane = threadIdx.x, slab = blockIdx.x * 4 + lane / 16, s = lane & 15;
    if (slab > nslab) return;  // whole 16-lane rows leave
    const SolveDev<float, TA> &S = sv[blockIdx.y];
    const int z = slab % g.nz, b = slab / g.nz;
    const int x = (b % g.bx) * kBrick + (s & 3), y = (b / g.bx) * kBrick + (s >> 2);
    float v[K];
#pragma unroll
    for (int a = 0; a < K; ++a) v[a] = 0.f;
    if (slab < nslab && x < g.nx && y < g.ny) {
        const float *__restrict__ w = S.W + (size_t)(x + g.nx * (y + g.ny * z)) * K;
        double t[K], q[K];
#pragma unroll
        for (int a = 0; a < K; ++a) t[a] = (double)w[a];
        zpow_from_harmonic<double, L>(t, q);
#pragma unroll
        for (int a = 0; a < K; ++a) v[a] = (float)q[a];
    }
    float m = 0.f;
#pragma unroll
    for (int a = 0; a < K; ++a) m = fmaxf(m, fabsf(v[a]));
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 16));
    // 2^k with m 2^k in [2^9, 2^10); within the exponents a float holds both ways
    int k = 0;
    if (m > 0.f) k = min(max(9 - ((int)(__float_as_uint(m) >> 23) - 127), -120), 120);
    const float up = __uint_as_float((unsigned)(127 + k) << 23), down = __uint_as_float((unsigned)(127 - k) << 23);
#pragma unroll
    for (int a = 0; a < K; ++a) v[a] *= up;
    unsigned char *base = reinterpret_cast<unsigned char *>(S.Wp);
    store_row<L>(base + ((size_t)slab * 16 + s) * M::WB, v);
    if (s == 0) reinterpret_cast<float *>(base + ((size_t)nslab + 1) * 16 * M::WB)[slab] = down;
}

// ---------------------------------------------------------------------------
// The exponents of the path table: byte [slab][slot] is the biased exponent of the
// largest kf of the slab's (up to 16) sources for that destination.  T is scaled with it.
// After the last slab the exponents of the slab of zeros, all 127: the entries read beside
// it are a neighbour's, of any size, and have to stay finite for T to be 0.
// grid = (ceil(npad / 1024), slabs + 1), block = 256: 4 slots per thread.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_kexp(GridDev<float> g, const float *__restrict__ ktab,
                                              unsigned *__restrict__ kexp)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= g.npad / 4) return;
    const int slab = blockIdx.y, z = slab % g.nz, b = slab / g.nz;
    if (slab == g.bx * g.by * g.nz) {
        kexp[(size_t)slab * (g.npad / 4) + q] = 0x7f7f7f7fu;
        return;
    }
    const int x0 = (b % g.bx) * kBrick, y0 = (b / g.bx) * kBrick;
    const f4 *__restrict__ row = reinterpret_cast<const f4 *>(ktab) + q;
    f4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        // sources beyond the grid: the last one's entries again
        const int x = min(x0 + (s & 3), g.nx - 1), y = min(y0 + (s >> 2), g.ny - 1);
        const f4 v = row[(size_t)(x + g.nx * (y + g.ny * z)) * (g.npad / 4)];
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], v[e]);
    }
    unsigned o = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) o |= (__float_as_uint(m[e]) >> 23) << (8 * e);
    kexp[(size_t)slab * (g.npad / 4) + q] = o;
}

// ---------------------------------------------------------------------------
// The propagation.  A workgroup of 8 waves (2 per SIMD) owns a unit: the destination
// bricks (bx + tx, by, zg ntz + tz), tx < ntx, tz < ntz, for the nr right-hand sides of a
// group: column c = r + nr (tx + ntx tz).  Waves 2 p and 2 p + 1 hold the bricks' slab
// p (16 destinations a column).  The sources come a slab at a time (16 voxels; the same
// translations: brick (xs + tx, ys), slab z + 4 tz): each wave of the pair forms P and T
// for 8 of them, T goes through LDS as pieces (there it is also transposed: a product
// wants 8 sources of one destination in a lane), and each wave sums 8 of the 16
// destinations, whose K x 16 sums stay in its registers over the unit's chunk of sources:
// brick rows ys in [y0, y1).  The chunk does not depend on the group, nor does the order of a
// destination's sources, and a column's arithmetic not on its neighbours: a solve's bits are
// the same in any group.
// Z planes (the 7 x 7 displacements of one z) come through a ring in LDS; a source
// slab uses 4 of them, one per pair of waves, and the next slab of the brick 3 of these
// again.  W's rows of the tile (16 columns x 16 sources) lie in LDS for the four pairs;
// the next tile's are requested when the products with this one's are done and written
// behind its sums.  The table entries are requested a tile ahead.  Z rows are read as they
// are for P (A operand: destinations x coefficients) and transposed by
// ds_read_b64_tr_b16 for the sums (A operand: coefficients x sources, h pieces in its
// first 16 sources and l pieces in the other 16, against (Th, Th) and (Tl, Tl)).
// grid = (units x chunks, groups), block = 512.
// ---------------------------------------------------------------------------
#define LDSP __attribute__((address_space(3)))
#define GLBP __attribute__((address_space(1)))

__device__ __forceinline__ f4 mm(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ h8 tr8(const LDSP unsigned char *p0, const LDSP unsigned char *p1)
{
    union { s4 s[2]; h8 h; } u;
    u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDSP s4 *)p0);
    u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDSP s4 *)p1);
    return u.h;
}

// the workgroup's LDS writes before it are seen by its reads after it; loads from global
// memory stay in flight across it
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int L>
struct MLds {
    static constexpr int RING = 7;                          // Z planes
    static constexpr int T = RING * MLay<L>::PP;            // T pieces: [slab 4][destination 16][column 16][64 bytes]
    static constexpr int W = T + 4 * 16384;                 // W rows: [column 16][source 16]
    static constexpr int PTR = W + 16 * MLay<L>::CP;        // per column: its path table, its W pieces, then the exponents
    static constexpr int ADDR = PTR + 384;                  // per half and lane: LDS addresses
    static constexpr int BYTES = ADDR + 2 * 64 * 32;
    static_assert(BYTES <= 163840, "LDS");
};

template <typename TA, int L>
__global__ __launch_bounds__(kMfmaThreads, 2) void k_prop_mfma(MfmaArgs A, const SolveDev<float, TA> *__restrict__ sv)
{
    using M = MLay<L>;
    using D = MLds<L>;
    constexpr int K = M::K, NJ = M::NJ, RING = D::RING;
    extern __shared__ __align__(16) unsigned char mfma_lds[];
    LDSP unsigned char *lds = (LDSP unsigned char *)mfma_lds;
    const GridDev<float> &g = A.g;
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int c = lane & 15, gq = lane >> 4, pr = wave >> 1, hf = wave & 1;
    // chunks vary fastest over the workgroups, which the 8 XCDs take in turn: an XCD's L2
    // holds few chunks' W rows
    const int chunk = blockIdx.x % A.nchunk, unit = blockIdx.x / A.nchunk;
    const int bx = unit % A.nxg * A.ntx, by = unit / A.nxg % g.by, bz = unit / (A.nxg * g.by) * A.ntz;
    const int y0 = g.by * chunk / A.nchunk, y1 = g.by * (chunk + 1) / A.nchunk;
    const int mtx = min(A.ntx, g.bx - bx), mtz = min(A.ntz, g.bz - bz);  // translations in use
    // source bricks x (of translation 0) and slabs z (relative to slab 4 bz)
    const int x0 = 1 - mtx, x1 = g.bx;
    const int d0 = -4 * (bz + mtz - 1), nd = g.nz - 4 * bz - d0;
    const int nslab = g.bx * g.by * g.nz;

    // this lane's column
    const int r = c % A.nr, t = c / A.nr, tx = t % A.ntx, tz = t / A.ntx;
    const int zd = 4 * (bz + tz) + pr;
    const bool act = tx < mtx && tz < mtz && zd < g.nz;
    const bool acol = tx < mtx && tz < mtz;  // the column has destinations
    const SolveDev<float, TA> *__restrict__ S = sv + (size_t)blockIdx.y * A.nr + (acol ? r : 0);
    const int zc = act ? zd : g.nz - 1, bxd = act ? bx + tx : bx;
    const int slot = ((bxd + g.bx * (by + g.by * (zc >> 2))) * kWave) + (zc & 3) * 16;
    if (threadIdx.x < 16) {
        *(LDSP unsigned long long *)(lds + D::PTR + c * 16) = (unsigned long long)S->ktab;
        *(LDSP unsigned long long *)(lds + D::PTR + c * 16 + 8) = (unsigned long long)S->Wp;
        *(LDSP unsigned long long *)(lds + D::PTR + 256 + c * 8) = (unsigned long long)S->kexp;
    }
    const unsigned long long row = (unsigned long long)g.npad * 4, rowx = row * g.nx, rowxy = rowx * g.ny;

    // the two columns whose W rows this wave brings
    struct WCol { const GLBP unsigned char *w; int tx, tz; bool act; } wc[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int cc = 2 * wave + e, t2 = cc / A.nr;
        wc[e].tx = t2 % A.ntx;
        wc[e].tz = t2 / A.ntx;
        wc[e].act = wc[e].tx < mtx && wc[e].tz < mtz;
        wc[e].w = (const GLBP unsigned char *)sv[(size_t)blockIdx.y * A.nr + (wc[e].act ? cc % A.nr : 0)].Wp;
    }

    // Lane parts of the addresses.  A wave's sources are sx = i % 4, sy = hf + 2 (i / 4).  Z
    // rows of a plane: displacement (lx - 3, ly - 3).  For P: row of destination c less source
    // (3, hf + 2), piece gq; for the sums: source sx = c / 4, sy = (gq & 1) + 2, the half's first
    // destination, 8-byte piece c & 3 of the h (gq < 2) or l pieces
    const int zrow = (c & 3) * M::XP + ((c >> 2) + 1 - hf) * M::YP;
    const int a1 = zrow + gq * 16, a1r = zrow + 2 * M::H + (gq & 1) * 8;
    const int zcol = (3 - (c >> 2) + 2 * hf) * M::XP + (1 - (gq & 1)) * M::YP + (c & 3) * 8;
    const int a2 = zcol + (gq >> 1) * M::H, a2r = zcol + 2 * M::H + (gq >> 1) * 8;
    // T pieces: (destination, column) rows of 64 bytes, h of the sources of half 0, of half 1,
    // then l; the quarters are permuted with the column (0, 2, 3, 1) against bank conflicts
    LDSP unsigned char *tb = lds + D::T + pr * 16384 + c * 64;
    const int sw = (0x1320 >> (4 * (c >> 2))) & 3;
    LDSP unsigned char *twh = tb + 4 * gq * 1024 + (hf ^ sw) * 16, *twl = tb + 4 * gq * 1024 + ((2 + hf) ^ sw) * 16;
    const LDSP unsigned char *trh = lds + D::T + c * 64 + 2 * hf * 1024 + ((gq & 1) ^ sw) * 16;
    const LDSP unsigned char *trl = lds + D::T + c * 64 + 2 * hf * 1024 + ((2 + (gq & 1)) ^ sw) * 16;
    // W rows of this lane's column: piece gq, the last coefficients
    const LDSP unsigned char *wp = lds + D::W + c * M::CP + 4 * hf * M::WB + gq * 16;
    const LDSP unsigned char *wpr = lds + D::W + c * M::CP + 4 * hf * M::WB + 2 * M::H;
    // what a lane needs of these for P, and for the sums, is kept in LDS and read at each phase:
    // the registers are full, and a spilled one comes back behind the table entries in flight
    LDSP u4 *ad = (LDSP u4 *)(lds + D::ADDR) + 2 * (hf * kWave + lane);
    if (pr == 0) {
        ad[0] = u4{(unsigned)a1, (unsigned)a1r, (unsigned)(wp - lds), (unsigned)(wpr - lds) + (gq >> 1) * 8};
        ad[1] = u4{(unsigned)a2, (unsigned)a2r, (unsigned)(trh - lds), (unsigned)(trl - lds)};
    }

    // destinations x = 2 hf + n / 4, y = n % 4; their last 4 coefficients in the lane rows
    // gq = y of one tile per x
    f4 acc[8][NJ], accr[2];
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[n][j] = f4{0.f, 0.f, 0.f, 0.f};
    accr[0] = accr[1] = f4{0.f, 0.f, 0.f, 0.f};

    // ---- the source brick columns, in order; those with every pair uncoupled (table
    // entries 0) are left out ---------------------------------------------------
    struct Col { int x, y; };
    auto far = [&](const Col &q) {
        const float mx = (float)max(0, 4 * abs(bx - q.x) - 3) * g.dx, my = (float)max(0, 4 * abs(by - q.y) - 3) * g.dy;
        return mx * mx + my * my > A.thr2 * 1.0001f;
    };
    auto settle = [&](Col &q) {
        while (q.y < y1) {
            if (q.x >= x1) {
                q.x = x0;
                ++q.y;
            } else if (far(q)) {
                ++q.x;
            } else {
                break;
            }
        }
    };
    Col at{x0, y0};
    settle(at);

    // the slab of W rows a column reads (one without a source there: the slab of zeros)
    auto slab_of = [&](const Col &q, int z, int txx, int tzz, bool a) {
        const int x = q.x + txx, zs = z + 4 * tzz;
        return a && x >= 0 && x < g.bx && zs >= 0 && zs < g.nz ? (q.y * g.bx + x) * g.nz + zs : nslab;
    };
    // the tile's W rows: 16-byte pieces of the wave's columns, column 0's whole 64s, then column
    // 1's and what is left of both; requested and written in these two parts
    constexpr int NF = 16 * M::U / 64, NL = 16 * M::U % 64;
    static_assert(NL <= 32);
    u4 wv[L == 5 ? NF + 1 : 2 * NF];
    auto wload = [&](const Col &cl, int z, auto part) {
        constexpr int e = part;
        const GLBP unsigned char *b = wc[e].w + (unsigned)slab_of(cl, z, wc[e].tx, wc[e].tz, wc[e].act) * (16ull * M::WB);
        unsigned o = lane;
        asm volatile("" : "+s"(b), "+v"(o));  // scalar base, 32-bit offset (not a kept pointer per lane)
        o *= 16;
#pragma unroll
        for (int k = 0; k < NF; ++k) wv[(L == 5 ? 0 : e * NF) + k] = *(const GLBP u4 *)(b + o + k * 1024);
        if constexpr (e == 1 && NL > 0) {
            const GLBP unsigned char *a =
                wc[0].w + (unsigned)slab_of(cl, z, wc[0].tx, wc[0].tz, wc[0].act) * (16ull * M::WB);
            wv[NF] = *(const GLBP u4 *)((lane & 16 ? b : a) + (o & 240) + NF * 1024);
        }
    };
    auto wstore = [&](auto part) {
        constexpr int e = part;
        unsigned o = lane;
        asm volatile("" : "+v"(o));
        o *= 16;
        LDSP unsigned char *w = lds + (D::W + 2 * wave * M::CP) + o;
#pragma unroll
        for (int k = 0; k < NF; ++k) *(LDSP u4 *)(w + e * M::CP + k * 1024) = wv[(L == 5 ? 0 : e * NF) + k];
        // the rest: lanes 0-15 column 0's, 16-31 column 1's (32-63 the same again: no branch, under
        // whose partial EXEC mask a spilled register of every lane could be saved)
        if constexpr (e == 1 && NL > 0) {
            const unsigned q = o & 496;
            *(LDSP u4 *)(lds + (D::W + 2 * wave * M::CP + NF * 1024) + q + (q >= 256 ? M::CP - 256 : 0)) = wv[NF];
        }
    };
    using Part0 = std::integral_constant<int, 0>;
    using Part1 = std::integral_constant<int, 1>;
    // path-table rows of a slab's sources, clamped to the grid (the W of a source outside is 0)
    // a kept register again, what is formed from it not kept
    auto now = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    struct KPtr { const GLBP unsigned char *y[2]; unsigned x[4]; };
    auto kptr = [&](const Col &q, int z) {
        KPtr k;
        const GLBP unsigned char *kt =
            *(const GLBP unsigned char * const LDSP *)(lds + D::PTR + (now(lane) & 15) * 16) + (unsigned)(now(slot) * 4 + (now(lane) & 48));
        const int xb = min(max(4 * (q.x + now(tx)), 0), g.nx - 1), zs = min(max(z + 4 * now(tz), 0), g.nz - 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) k.x[e] = (unsigned)(min(xb + e, g.nx - 1) - xb) * (unsigned)row;
#pragma unroll
        for (int e = 0; e < 2; ++e)
            k.y[e] = kt + ((unsigned)zs * rowxy + (unsigned)min(4 * q.y + hf + 2 * e, g.ny - 1) * rowx + (unsigned)xb * row);
        return k;
    };

    // ---- the stream of Z planes: of each brick column z = 3 + 4 bz - z0 - i for i = 0 ..
    // nd + 2, z0 its first slab; its tile j uses planes j .. j + 3, pair p the one 3 - p + j.
    // Wave w < 7 brings line w of a plane.
    const unsigned zline = A.nxt * M::WB, zplane = zline * g.by * 8 - zline;
    Col pc = at;                     // the next plane to request, of its brick column
    int pi = 0, ppos = 0, pslot = 0;  // in all; where the next one that arrives goes
    auto zload = [&]() {
        const int iz = min(max(g.nz - 1 + 3 - d0 - pi, 0), 2 * g.nz - 2);
        const GLBP unsigned char *z = (const GLBP unsigned char *)A.zt + (size_t)(unsigned)iz * zplane +
                                      ((unsigned)(4 * (by - pc.y) + 4 * g.by - 4 + min(wave, 6)) * zline +
                                       (unsigned)(4 * (bx - pc.x) + 4 * g.bx - 4) * M::WB);
        ++ppos;
        if (++pi == nd + 3) {
            pi = 0;
            ++pc.x;
            settle(pc);
        }
        unsigned o = lane;
        asm volatile("" : "+s"(z), "+v"(o));  // worked out again each time: one register less kept
        return *(const GLBP u4 *)(z + min(o, 7 * M::U - 1u) * 16);
    };
    auto zstore = [&](u4 v) {
        unsigned o = lane;
        asm volatile("" : "+v"(o));
        o = min(o, 7 * M::U - 1u);
        if (wave < 7) *(LDSP u4 *)(lds + pslot * M::PP + wave * M::YP + (o * 16 + o / M::U * (M::XP - M::WB))) = v;
        if (++pslot == RING) pslot = 0;
    };
    // up to ppos = n, at most 4 planes, together
    auto zfill = [&](int n) {
        u4 v[4];
        int k = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (ppos < n && pc.y < y1) {
                v[i] = zload();
                k = i + 1;
            }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < k) zstore(v[i]);
    };

    if (at.y < y1) {
        int z = 4 * bz + d0, win = 0, wslot = (3 - pr) % RING;  // the tile's slab, its first plane, this pair's plane
        lds_barrier();
        f4 tk[8];  // kf of the tile's sources, each replaced by the next tile's once used
        u4 en;     // kf exponents of the 16 destinations
        float sn;  // scale of the slab's W rows
        auto kload = [&](const KPtr &k, int i) { tk[i] = *(const GLBP f4 *)(k.y[i >> 2] + k.x[i & 3]); };
        auto eload = [&](const Col &q, int zz) {
            const int sl = slab_of(q, zz, tx, tz, acol);
            const int cc = now(lane) & 15;
            const GLBP unsigned char *w = *(const GLBP unsigned char * const LDSP *)(lds + D::PTR + cc * 16 + 8);
            const GLBP unsigned char *ke = *(const GLBP unsigned char * const LDSP *)(lds + D::PTR + 256 + cc * 8);
            sn = *(const GLBP float *)(w + ((unsigned long long)(unsigned)nslab + 1) * 16 * M::WB + (unsigned)sl * 4ull);
            en = *(const GLBP u4 *)(ke + (unsigned)sl * (unsigned long long)g.npad + (unsigned)slot);
        };
        {
            const KPtr k = kptr(at, z);
#pragma unroll
            for (int i = 0; i < 8; ++i) kload(k, i);
            eload(at, z);
        }
        wload(at, z, Part0{});
        wstore(Part0{});
        wload(at, z, Part1{});
        // the pads behind the Z rows are read into rows that are not used: finite
        if constexpr (M::REM) {
            for (int i = threadIdx.x * 16; i < D::T; i += kMfmaThreads * 16) *(LDSP u4 *)(lds + i) = u4{0, 0, 0, 0};
            lds_barrier();
        }
        zfill(4);
        zfill(RING);
        wstore(Part1{});
        lds_barrier();
        for (;;) {
            // the next tile (the current one again at the end: read, not used)
            Col nx = at;
            int nz = z + 1, nwin = win + 1;
            if (nz == 4 * bz + d0 + nd) {
                nz = 4 * bz + d0;
                nwin = win + 4;
                ++nx.x;
                settle(nx);
            }
            const bool last = nx.y >= y1;
            if (last) {
                nx = at;
                nz = z;
            }
            const u4 ex = en;
            const float sf = sn * 0x1p-9f;
            KPtr kn;
            // the plane that there is room for now
            const bool more = ppos < win + RING && pc.y < y1;
            u4 zn = {0, 0, 0, 0};

            // ---- P and T: a source's rows requested one source ahead, T of the source before
            // formed under its products ---------------------------------------------------
            const LDSP unsigned char *zp = lds + wslot * M::PP;
            h2 hh[4][2], ll[4][2];  // T's pieces: [destination 4 gq + e][pair of sources]
            {
                f4 a0, p0;
                h8 zh[2], wh[2], zq, wl;
                h4 zr, wr;
                f4 pp[2];
                const u4 ap = ad[0];
                const LDSP unsigned char *za = zp + ap.x, *zar = zp + ap.y, *wp = lds + ap.z, *wpr = lds + ap.w;
                asm("" : "+v"(za), "+v"(zar), "+v"(wp), "+v"(wpr));  // the rest is the instructions' offsets
                auto zoff = [](int i) { return (3 - (i & 3)) * M::XP + (2 - 2 * (i >> 2)) * M::YP; };
                auto woff = [](int i) { return ((i & 3) + 8 * (i >> 2)) * M::WB; };
                auto aload = [&](int i) {
                    zh[i & 1] = *(const LDSP h8 *)(za + zoff(i));
                    wh[i & 1] = *(const LDSP h8 *)(wp + woff(i));
                };
                // 2^(116 - e) of this lane's destinations 4 gq ..: |T| stays below 2^16
                const unsigned eb = gq < 2 ? (gq ? ex[1] : ex[0]) : (gq == 3 ? ex[3] : ex[2]);
                float ks[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) ks[e] = __uint_as_float((unsigned)max(243 - (int)((eb >> (8 * e)) & 255), 1) << 23);
                aload(0);
#pragma unroll
                for (int i = 0; i <= 8; ++i) {
                    const int u = i & 1;
                    if (i < 8) {
                        // the pieces used last are requested first
                        wl = *(const LDSP h8 *)(wp + woff(i) + M::H);
                        zq = *(const LDSP h8 *)(za + zoff(i) + M::H);
                        if constexpr (M::REM) {
                            zr = *(const LDSP h4 *)(zar + zoff(i));
                            wr = *(const LDSP h4 *)(wpr + woff(i));
                        }
                        if (i < 7) aload(i + 1);
                        f4 x = {0.f, 0.f, 0.f, 0.f};
                        x = mm(zh[u], wh[u], x);
                        x = mm(zh[u], wl, x);
                        x = mm(zq, wh[u], x);
                        // the last 4 coefficients: lane rows (Zh, Zl, Zh, Zl) against (Wh, Wh, Wl, Wl),
                        // half of each product's depth zero (on 16x16x16_f16, which has that depth, sums
                        // differed in their last bits from run to run)
                        if constexpr (M::REM) {
                            const u2 p = __builtin_bit_cast(u2, zr), q = __builtin_bit_cast(u2, wr);
                            x = mm(__builtin_bit_cast(h8, u4{p.x, p.y, 0u, 0u}), __builtin_bit_cast(h8, u4{q.x, q.y, 0u, 0u}), x);
                        }
                        pp[u] = x;
                    }
                    if (i == 1) {
                        eload(nx, nz);
                        kn = kptr(nx, nz);
                        if (more) zn = zload();
                    }
                    if (i > 0) {
                        // T = a p; h its leading 11 bits, l the rest of the exact product
                        f4 a;
#pragma unroll
                        for (int e = 0; e < 4; ++e) a[e] = tk[i - 1][e] * ks[e];
                        kload(kn, i - 1);
                        if (i & 1) {
                            a0 = a;
                            p0 = pp[0];
                        } else {  // two sources more; four make 8 bytes
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const h2 h = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(a0[e] * p0[e], a[e] * pp[1][e]));
                                hh[e][(i / 2 - 1) & 1] = h;
                                ll[e][(i / 2 - 1) & 1] = h2{(_Float16)__builtin_fmaf(a0[e], p0[e], -(float)h[0]),
                                                            (_Float16)__builtin_fmaf(a[e], pp[1][e], -(float)h[1])};
                                if (i == 4 || i == 8) {
                                    const int o = e * 1024 + (i == 8 ? 8 : 0);
                                    *(LDSP u2 *)(twh + o) = u2{__builtin_bit_cast(unsigned, hh[e][0]),
                                                               __builtin_bit_cast(unsigned, hh[e][1])};
                                    *(LDSP u2 *)(twl + o) = u2{__builtin_bit_cast(unsigned, ll[e][0]),
                                                               __builtin_bit_cast(unsigned, ll[e][1])};
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (more) zstore(zn);
            lds_barrier();  // T is whole; the tile's W rows have been read

            // ---- the sums; the next tile's W rows on their way ----------------------------
            wload(nx, nz, Part0{});
            if constexpr (L != 5) wload(nx, nz, Part1{});
            {
                const u4 ap = ad[1];
                const LDSP unsigned char *zc2 = zp + ap.x, *zcr = zp + ap.y, *trh = lds + pr * 16384 + ap.z,
                                         *trl = lds + pr * 16384 + ap.w;
                asm("" : "+v"(zc2), "+v"(zcr), "+v"(trh), "+v"(trl));
                h8 cf[2][NJ], cr, th[2], tl;
                auto cload = [&](int n) {
                    const int o = (n >> 2) * M::XP + (n & 3) * M::YP;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) cf[n & 1][j] = tr8(zc2 + o + 2 * M::YP + j * 32, zc2 + o + j * 32);
                    th[n & 1] = *(const LDSP h8 *)(trh + ((n >> 2) + 4 * (n & 3)) * 1024);
                };
                cload(0);
#pragma unroll
                for (int n = 0; n < 8; ++n) {
                    tl = *(const LDSP h8 *)(trl + ((n >> 2) + 4 * (n & 3)) * 1024);
                    // rows 4 y .. of the tile: the last coefficients (the others unused)
                    if constexpr (M::REM) {
                        const int o = (n >> 2) * M::XP + (n & 3) * (M::YP - 8);
                        cr = tr8(zcr + o + 2 * M::YP, zcr + o);
                    }
                    if (n < 7) cload(n + 1);
                    if (L == 5 && n == 3) {  // (for all of them the registers do not suffice)
                        wstore(Part0{});
                        wload(nx, nz, Part1{});
                    }
                    const int u = n & 1;
                    // T's scale and W's taken out again: 2^(e - 136) times the slab's
                    const unsigned eb = (ex[n & 3] >> (16 * hf + 8 * (n >> 2))) & 255;
                    const float f = sf * __uint_as_float(eb << 23);
                    f4 s[NJ], sr;
                    const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < NJ; ++j) s[j] = mm(cf[u][j], th[u], zero);
                    if constexpr (M::REM) sr = mm(cr, th[u], zero);
#pragma unroll
                    for (int j = 0; j < NJ; ++j) s[j] = mm(cf[u][j], tl, s[j]);
                    if constexpr (M::REM) sr = mm(cr, tl, sr);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
#pragma unroll
                        for (int j = 0; j < NJ; ++j) acc[n][j][e] = __builtin_fmaf(s[j][e], f, acc[n][j][e]);
                        if constexpr (M::REM)
                            accr[n >> 2][e] = __builtin_fmaf(sr[e], gq == (n & 3) ? f : 0.f, accr[n >> 2][e]);
                    }
                    
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (last) break;
            if constexpr (L != 5) wstore(Part0{});
            wstore(Part1{});
            lds_barrier();  // the next tile's W rows are there; T has been read
            if (nwin == win + 4 && ppos < nwin + 4) {  // a new brick column's first planes
                zfill(nwin + 4);
                lds_barrier();
            }
            wslot += nwin - win;
            if (wslot >= RING) wslot -= RING;
            at = nx;
            z = nz;
            win = nwin;
        }
    }

    // ---- the sums, in the Z basis (the lane's column worked out again) --------
    const int ln = now(lane), r2 = (ln & 15) % A.nr, t2 = (ln & 15) / A.nr, tx2 = t2 % A.ntx, z2 = 4 * (bz + t2 / A.ntx) + pr;
    const bool has = tx2 < mtx && t2 / A.ntx < mtz && z2 < g.nz;
    float *__restrict__ part =
        sv[(size_t)blockIdx.y * A.nr + (has ? r2 : 0)].part + (size_t)chunk * g.N * K + (unsigned)(has ? z2 : 0) * ((size_t)g.nx * g.ny * K);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        const int x = 4 * (bx + tx2) + 2 * hf + (n >> 2), y = 4 * by + (n & 3);
        const bool ok = has && x < g.nx && y < g.ny;
        float *o = part + (unsigned)(x + g.nx * y) * (unsigned)K;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int a = 16 * j + 4 * (ln >> 4);
            if constexpr (K % 4 == 0) {
                if (ok) *reinterpret_cast<f4 *>(o + a) = acc[n][j];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (ok && a + e < K) o[a + e] = acc[n][j][e];
            }
        }
        if constexpr (M::REM)
            if (ok && ln >> 4 == (n & 3)) *reinterpret_cast<f4 *>(o + 32) = accr[n >> 2];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
#define RTE_DISPATCH_M(L, ...)                              \
    switch (L) {                                            \
    case 4: { constexpr int LL = 4; __VA_ARGS__; } break;   \
    case 5: { constexpr int LL = 5; __VA_ARGS__; } break;   \
    default: return hipErrorInvalidValue;                   \
    }

size_t mfma_wp_bytes(int L, const GridDev<float> &g)
{
    const size_t slabs = (size_t)g.bx * g.by * g.nz + 1;  // and the slab of zeros
    const size_t row = L == 4 ? MLay<4>::WB : MLay<5>::WB;
    return (slabs * (16 * row + sizeof(float)) + 255) / 256 * 256;
}

size_t mfma_ztab_bytes(int L, const GridDev<float> &g)
{
    const size_t rows = (size_t)(8 * g.bx - 1) * (8 * g.by - 1) * (2 * g.nz - 1);
    return rows * (L == 4 ? MLay<4>::WB : MLay<5>::WB);
}

hipError_t launch_ztab(int L, const GridDev<float> &g, double dx, double dy, double dz, unsigned char *zt, hipStream_t st)
{
    const int nxt = 8 * g.bx - 1, nyt = 8 * g.by - 1, nzt = 2 * g.nz - 1;
    const size_t rows = (size_t)nxt * nyt * nzt;
    RTE_DISPATCH_M(L, hipLaunchKernelGGL((k_ztab<LL>), dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, st, nxt, nyt,
                                         nzt, dx, dy, dz, zt));
    return hipGetLastError();
}

// The translations of a group of nr solves: of the splits of its 16 / nr columns per solve
// into x and z the one with the least tiles (units times the source slabs of each: every
// translation adds the bricks, or slabs, at which not all columns have a source).
double mfma_translations(const GridDev<float> &g, int nr, int *ntx, int *ntz)
{
    double best = 0;
    for (int x = 1; x * nr <= kMfmaCols; ++x)
        for (int z = 1; x * z * nr <= kMfmaCols; ++z) {
            if ((x > 1 && x > g.bx) || (z > 1 && z > g.bz)) continue;
            const double units = (double)((g.bx + x - 1) / x) * g.by * ((g.bz + z - 1) / z);
            const double cost = units * g.by * (g.bx + x - 1) * (g.nz + 4.0 * (z - 1));
            if (best == 0 || cost < best) {
                best = cost;
                *ntx = x;
                *ntz = z;
            }
        }
    return best;
}

size_t kexp_bytes(const GridDev<float> &g) { return ((size_t)g.bx * g.by * g.nz + 1) * g.npad; }

hipError_t launch_kexp(const GridDev<float> &g, const float *ktab, unsigned char *kexp, hipStream_t st)
{
    const dim3 grid((g.npad + 1023) / 1024, g.bx * g.by * g.nz + 1);
    hipLaunchKernelGGL(k_kexp, grid, dim3(256), 0, st, g, ktab, reinterpret_cast<unsigned *>(kexp));
    return hipGetLastError();
}

template <typename TA>
hipError_t launch_to_pieces(int L, const GridDev<float> &g, const SolveDev<float, TA> *sv, int nsolve, hipStream_t st)
{
    if (nsolve < 1 || nsolve > 65535) return hipErrorInvalidValue;
    const int nslab = g.bx * g.by * g.nz;
    const dim3 grid((nslab + 1 + 3) / 4, nsolve);
    RTE_DISPATCH_M(L, hipLaunchKernelGGL((k_to_pieces<TA, LL>), grid, dim3(kWave), 0, st, g, sv));
    return hipGetLastError();
}

template <typename TA>
hipError_t launch_prop_mfma(int L, int nr, const PropArgs<float> &P, const SolveDev<float, TA> *sv, int ngroups,
                            hipStream_t st)
{
    if (!P.zt || nr < 1 || nr > kMfmaCols || ngroups < 1 || ngroups > 65535) return hipErrorInvalidValue;
    MfmaArgs A;
    A.g = P.g;
    A.zt = P.zt;
    A.thr2 = P.thr2;
    A.nr = nr;
    mfma_translations(P.g, nr, &A.ntx, &A.ntz);
    A.nxg = (P.g.bx + A.ntx - 1) / A.ntx;
    const long long units = (long long)A.nxg * P.g.by * ((P.g.bz + A.ntz - 1) / A.ntz);
    A.nchunk = P.nchunk;
    A.nxt = 8 * P.g.bx - 1;
    const dim3 grid((unsigned)(units * P.nchunk), ngroups), block(kMfmaThreads);
    RTE_DISPATCH_M(L, {
        constexpr int lds = MLds<LL>::BYTES;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_prop_mfma<TA, LL>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_prop_mfma<TA, LL>), grid, block, lds, st, A, sv);
    });
    return hipGetLastError();
}

template hipError_t launch_to_pieces<double>(int, const GridDev<float> &, const SolveDev<float, double> *, int, hipStream_t);
template hipError_t launch_to_pieces<float>(int, const GridDev<float> &, const SolveDev<float, float> *, int, hipStream_t);
template hipError_t launch_prop_mfma<double>(int, int, const PropArgs<float> &, const SolveDev<float, double> *, int,
                                             hipStream_t);
template hipError_t launch_prop_mfma<float>(int, int, const PropArgs<float> &, const SolveDev<float, float> *, int,
                                            hipStream_t);

}  // namespace rte
