// One stage of the fused RBC2D step (navier/rbc2d.py:396-434) in eight phases, a launch
// each (the first takes two when its right-hand side is large).
//
// The dense operators of the step act on one axis at a time, and every banded
// solve runs along one axis, so the work falls into phases that each need whole
// lines of one axis: a block that holds some lines can run an operator product
// and the line solve that follows (or precedes) it without a launch in between.
//
//   1  values and x-derivatives on the dealiased x grid | banded right-hand side
//   2  values and y-derivatives on the y grid, convective products
//   3  forward transform along y (with truncation and the pseudo-inverse)
//   4  forward transform along x onto the right-hand side, Helmholtz solve along x
//   5  Helmholtz solve along y; Poisson right-hand side and divergence along y
//   6  Poisson right-hand side along x, eigen-split line solves | divergence along x
//   7  Poisson back transform, pressure-gradient projections along y
//   8  velocity correction | pressure update
//
// Single instances are bound by the latency of these dependent launches (each
// about 2 us before its first load returns, whatever its work), so the number of
// launches and the serial chain inside each are what counts; batches are bound by
// the FP64 matrix cores, so there it is the products' operations.  Both gain from
// the operators' structure: collocation operators are mirror-symmetric and the
// modal ones keep (or flip) the parity of a mode, so products run on halves; the
// derivative operators are triangular (their zero chunks are skipped); stencils
// and B D S are banded and applied in the loads and epilogues of other phases.
//
// Products: operators are stored in the order in which the FP64 MFMA consumes
// them (fragments of 16 outputs x 16 terms, 4 doubles per lane, zero-padded), so
// a wave reads them straight into registers as contiguous 2 KB pieces, with no
// bounds checks; the field operand is read at clamped, valid addresses (terms past
// the end meet zeros of the operator).  Products along x read it from global memory
// too (16 lanes walk a row); products along y, whose fragments hold 16 rows, pass
// it through a wave's own LDS tile: 16 neighbouring lanes on 16 different rows make
// a load four times as slow as 16 lanes along a row (the convective products at
// 256 x 256 took 1840 cycles per chunk that way, 1024 of them on the matrix cores).
// Step s of lane group g holds term 8 (s / 2) + 2 g + s % 2 of a chunk, so that one
// 16-byte load per lane reads pairs of neighbouring terms and the four lane groups
// read 64 contiguous bytes of a row.
#include "common.h"
#include "line_scan.h"
#include "rhs_impl.h"
#include "../../include/pypde_amd.h"

#include <algorithm>
#include <cstdint>

namespace pypde {

// rhs_impl.h switches contraction off for its sums; the kernels here may fuse
#pragma clang fp contract(fast)

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2u __attribute__((ext_vector_type(2), aligned(8)));  // pair at any 8-byte address
typedef double v2a __attribute__((ext_vector_type(2)));

constexpr int kCus = 256;   // of the device
constexpr int kFrag = 256;  // doubles per operator fragment (16 outputs x 16 terms)

// term of chunk k that lane group g takes at step s
__device__ __forceinline__ int term(int k, int g, int s) { return 16 * k + 8 * (s >> 1) + 2 * g + (s & 1); }

__device__ __forceinline__ v4d mfma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Fragment (tile, chunk) of a packed operator with kc chunks, this lane's part.
__device__ __forceinline__ v4d op_frag(const double* __restrict__ op, int tile, int kc, int chunk, int lane)
{
    return *reinterpret_cast<const v4d*>(op + ((long long)tile * kc + chunk) * kFrag + lane * 4);
}

// Software pipeline over the chunks [kb, ke): D chunks of loads in flight.
template <int D, class Load, class Compute>
__device__ __forceinline__ void pipeline(int kb, int ke, Load load, Compute compute)
{
#pragma unroll
    for (int st = 0; st < D; ++st)
        if (kb + st < ke) load(st, kb + st);
    for (int k0 = kb; k0 < ke; k0 += D) {
#pragma unroll
        for (int st = 0; st < D; ++st) {
            if (k0 + st >= ke) break;
            compute(st, k0 + st);
            if (k0 + st + D < ke) load(st, k0 + st + D);
        }
    }
}

// Pairs of neighbouring entries of a row of n >= 2, read 16 bytes at a time at
// valid addresses: the pair at `at`, or past the row's end its last pair.  In a row
// of odd length the last entry alone (at = n - 1) is the second of that pair;
// pair_first picks it when the value is used, not when it is loaded, so that no
// use of a load makes the wave wait for it early.
__device__ __forceinline__ v2u row_pair(const double* __restrict__ row, int at, int n)
{
    return *reinterpret_cast<const v2u*>(row + min(at, n - 2));
}

// 16 rows x 16 columns of a field through a wave's LDS tile: row(i) is row i of the
// tile, the loads run along rows (8 lanes each), frag reads row n's pair of terms
// (k, g, 2 h) and (k, g, 2 h + 1).
constexpr int kTilePitch = 18;  // 16 rows' pairs in distinct banks
struct RowTile {
    v2u t[2];
    template <class Row>
    __device__ __forceinline__ void load(Row row, int k, int ncol, int lane)
    {
#pragma unroll
        for (int i = 0; i < 2; ++i) t[i] = row_pair(row((lane >> 3) + 8 * i), 16 * k + 2 * (lane & 7), ncol);
    }
    __device__ __forceinline__ void store(double* xs, int lane) const
    {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *reinterpret_cast<v2a*>(xs + ((lane >> 3) + 8 * i) * kTilePitch + 2 * (lane & 7)) = v2a{t[i].x, t[i].y};
    }
    static __device__ __forceinline__ v2a frag(const double* xs, int h, int n, int g)
    {
        return *reinterpret_cast<const v2a*>(xs + n * kTilePitch + 8 * h + 2 * g);
    }
};

template <class V>
__device__ __forceinline__ double pair_first(V p, int at, int n) { return at == n - 1 ? p.y : p.x; }

__device__ __forceinline__ int div_up(int a, int b) { return (a + b - 1) / b; }

using Stage = pypde_rbc_stage;

// chunks in flight where a wave runs one tile (4 MFMAs, 256 cycles per chunk)
constexpr int kDeep = 6;

// ---------------------------------------------------------------------------
// Banded line solve of one parity chain of a line on a row of 16 lanes, C
// positions per lane: y_i = v_i + LM_i y_{i-1}, z_i = R_i y_i + MU_i z_{i+1} +
// NU_i z_{i+2} (chain positions).  Entries past the chain's end have zero tables
// and values.  t: [LM | R | MU | NU][C] of this lane's positions.
template <int C>
__device__ __forceinline__ void chain_solve(double (&v)[C], const double (&t)[4][C], int lane)
{
    double A = 1.0, B = 0.0;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        B = v[k] + t[0][k] * B;
        A = t[0][k] * A;
    }
    fwd_row_step<1>(A, B, lane);
    fwd_row_step<2>(A, B, lane);
    fwd_row_step<4>(A, B, lane);
    fwd_row_step<8>(A, B, lane);
    double y = dpp_f64<0x111>(0.0, B);
#pragma unroll
    for (int k = 0; k < C; ++k) {
        y = v[k] + t[0][k] * y;
        v[k] = y;
    }
    BwdMap m{0.0, 0.0, 1.0, 0.0, 0.0, 1.0};
#pragma unroll
    for (int k = C - 1; k >= 0; --k) {
        const double s = t[1][k] * v[k] + t[2][k] * m.s1 + t[3][k] * m.s2;
        const double a = t[2][k] * m.a1 + t[3][k] * m.a2;
        const double b = t[2][k] * m.b1 + t[3][k] * m.b2;
        m.s2 = m.s1; m.a2 = m.a1; m.b2 = m.b1;
        m.s1 = s; m.a1 = a; m.b1 = b;
    }
    bwd_row_step<1>(m, lane);
    bwd_row_step<2>(m, lane);
    bwd_row_step<4>(m, lane);
    bwd_row_step<8>(m, lane);
    double Z1 = dpp_f64<0x101>(0.0, m.s1), Z2 = dpp_f64<0x101>(0.0, m.s2);
#pragma unroll
    for (int k = C - 1; k >= 0; --k) {
        const double z = t[1][k] * v[k] + t[2][k] * Z1 + t[3][k] * Z2;
        v[k] = z;
        Z2 = Z1;
        Z1 = z;
    }
}

// Tables of chain positions [c C, c C + C): tab[slot][stride], chains padded with
// zeros to 16 C positions, position c C + k at [k / 2][c][k % 2], so that the 16 lanes
// of a chain read 256 contiguous bytes.  With the positions in order, 16 bytes of a
// cache line each at C = 16, phase 5 took 15.6 us at 16 x 300.
template <int C>
__device__ __forceinline__ void chain_tables(double (&t)[4][C], const double* __restrict__ tab, long long stride,
                                             int c)
{
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int k = 0; k < C; k += 2) {
            const v2u x = *reinterpret_cast<const v2u*>(tab + s * stride + k * 16 + 2 * c);
            t[s][k] = x.x;
            t[s][k + 1] = x.y;
        }
}

// ---------------------------------------------------------------------------
// Phase 1: Y1[e][value | x-derivative][L0][M1] from X, E and O over the even and
// odd modes of the first half of the x grid, both mirrored rows written; merged
// with the banded right-hand side (blocks [0, nbr)), which reads the same state.
template <int RT, int NT, int D>
__global__ void __launch_bounds__(256) stage_xpass(Stage a, pypde_rbc_rhs r, unsigned nbr, int ntask)
{
    if (blockIdx.x < nbr) {
        const long long total = 3LL * r.M0 * r.M1 * r.batch;
        for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < total; t += (long long)nbr * 256)
            rhs_banded_at(r.X, r.pres, r.cst, r.R, r.mdta, r.dta, r.fdiff, r.tx, r.ty, r.M0, r.M1, r.N0, r.N1, t);
        return;
    }
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int blk0 = xcd_remap(blockIdx.x - nbr, gridDim.x - nbr);
    const int task = blk0 * 4 + (threadIdx.x >> 6);
    if (task >= ntask) return;
    const int M0 = a.M0, M1 = a.M1, L0 = a.L0;
    const int H0 = (L0 + 1) / 2, HT = div_up(H0, 16), HTG = div_up(HT, RT);
    const int kc = div_up((M0 + 1) / 2, 16);
    const int CT = div_up(M1, 16 * NT);
    const int w = task % (2 * HTG), ec = task / (2 * HTG);
    const int blk = w / HTG, t0 = (w % HTG) * RT;
    const int c0 = (ec % CT) * 16 * NT, e = ec / CT;
    const double* __restrict__ X = a.X + (long long)e * M0 * M1;
    // packed [field set][value | derivative][even | odd][HT][kc]
    const double* __restrict__ op = a.gx + ((long long)((e % 3 == 2) * 2 + blk) * 2 * HT) * kc * kFrag;
    v4d acc[2][RT][NT] = {};
    v4d f[D][2][RT];
    double x[D][2][NT][4];
    auto load = [&](int st, int k) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
#pragma unroll
            for (int i = 0; i < RT; ++i) f[st][q][i] = op_frag(op, q * HT + min(t0 + i, HT - 1), kc, k, lane);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const double* row = X + (long long)min(2 * term(k, g, s) + q, M0 - 1) * M1;
#pragma unroll
                for (int j = 0; j < NT; ++j) x[st][q][j][s] = row[min(c0 + 16 * j + n, M1 - 1)];
            }
        }
    };
    auto compute = [&](int st, int k) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[q][i][j] = mfma(f[st][q][i][s], x[st][q][j][s], acc[q][i][j]);
    };
    pipeline<D>(0, kc, load, compute);
    double* __restrict__ Y = a.Y1 + ((long long)e * 2 + blk) * L0 * M1;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int row = (t0 + i) * 16 + g + 4 * u, col = c0 + 16 * j + n;
                if (row >= H0 || col >= M1) continue;
                const double E = acc[0][i][j][u], O = acc[1][i][j][u];
                Y[(long long)row * M1 + col] = E + O;
                const int mr = L0 - 1 - row;
                if (mr != row) Y[(long long)mr * M1 + col] = blk ? O - E : E - O;
            }
}

// ---------------------------------------------------------------------------
// Phase 2: the eight dealiased fields (u, v, and both derivatives of u, v, T) at
// 16 x-rows and 16 NY mirrored pairs of y points, one field per wave, and the
// convective products of rbc_products (pointwise.hip), folded for the forward
// transform: Pr[e][sum | difference][L0][H1].  The fields never reach memory;
// with the c-term (ratio != 0) the previous stage's velocities come from uv and
// this stage's go there ([b][u | v][point | mirror][L0][H1], each entry read and
// written by one thread).
constexpr int kYPitch = 34;  // a wave's 16 x 32 tile of its rows: the rows' pairs in distinct banks

template <int NY>  // tiles of 16 point pairs per block
__global__ void __launch_bounds__(512) stage_yprod(Stage a)
{
    __shared__ union {
        double x[8][16 * kYPitch];
        double field[8][2][NY][16][17];
    } sh;
    auto& buf = sh.field;
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int M1 = a.M1, L0 = a.L0, L1 = a.L1, H1 = (L1 + 1) / 2;
    const int HT = div_up(H1, 16), YG = div_up(HT, NY), RG = div_up(L0, 16);
    const int kc = div_up((M1 + 1) / 2, 16);
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    const int yg = id % YG, rr = id / YG;
    const int r0 = (rr % RG) * 16, b = rr / RG;
    // waves 0, 1: u, v; 2, 3, 4: d/dx of u, v, T; 5, 6, 7: d/dy of u, v, T
    const int fld = wave < 2 ? wave : (wave < 5 ? wave - 2 : wave - 5);
    const int dx = wave >= 2 && wave < 5, dy = wave >= 5;
    const double* __restrict__ Y = a.Y1 + ((long long)(3 * b + fld) * 2 + dx) * L0 * M1;
    const double* __restrict__ op = a.gy + (long long)dy * 2 * HT * kc * kFrag;  // [q][HT][kc]
    double* xs = sh.x[wave];
    {
        v4d acc[2][NY] = {};
        v4d f[2][2][NY];
        v2u x[2][4];
        auto load = [&](int st, int k) {
            // rows g, g + 4, ..., 16 lanes along each
#pragma unroll
            for (int i = 0; i < 4; ++i)
                x[st][i] = row_pair(Y + (long long)min(r0 + g + 4 * i, L0 - 1) * M1, 32 * k + 2 * n, M1);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < NY; ++j)
                    f[st][q][j] = op_frag(op, q * HT + min(yg * NY + j, HT - 1), kc, k, lane);
        };
        auto compute = [&](int st, int k) {
            wave_lds_sync();  // the previous chunk is read
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<v2a*>(xs + (g + 4 * i) * kYPitch + 2 * n) = v2a{x[st][i].x, x[st][i].y};
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const v2a p = *reinterpret_cast<const v2a*>(xs + n * kYPitch + 2 * term(0, g, s));
                const double ev = pair_first(p, 2 * term(k, g, s), M1);
#pragma unroll
                for (int j = 0; j < NY; ++j) {
                    acc[0][j] = mfma(ev, f[st][0][j][s], acc[0][j]);
                    acc[1][j] = mfma(p.y, f[st][1][j][s], acc[1][j]);
                }
            }
        };
        pipeline<2>(0, kc, load, compute);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int j = 0; j < NY; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u) buf[wave][q][j][g + 4 * u][n] = acc[q][j][u];
    }
    __syncthreads();
    const int t = threadIdx.x;
    {
#pragma clang fp contract(off)
        const int j = t >> 8, ri = (t >> 4) & 15, ln = t & 15;
        const int i = r0 + ri, l = (yg * NY + j) * 16 + ln;
        if (j >= NY || i >= L0 || l >= H1) return;
        double E[8], O[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            E[w] = buf[w][0][j][ri][ln];
            O[w] = buf[w][1][j][ri][ln];
        }
        const double* tb = a.dtbc + (long long)i * L1;
        const double tb1 = tb[l], tb2 = tb[L1 - 1 - l];
        const double ux1 = E[0] + O[0], ux2 = E[0] - O[0], uz1 = E[1] + O[1], uz2 = E[1] - O[1];
        const double xu1 = E[2] + O[2], xu2 = E[2] - O[2], xv1 = E[3] + O[3], xv2 = E[3] - O[3];
        const double xt1 = E[4] + O[4], xt2 = E[4] - O[4];
        const double yu1 = E[5] + O[5], yu2 = O[5] - E[5], yv1 = E[6] + O[6], yv2 = O[6] - E[6];
        const double yt1 = E[7] + O[7], yt2 = O[7] - E[7];
        double pu1 = xu1 * ux1 + yu1 * uz1, pu2 = xu2 * ux2 + yu2 * uz2;
        double pv1 = xv1 * ux1 + yv1 * uz1, pv2 = xv2 * ux2 + yv2 * uz2;
        double pt1 = (xt1 * ux1 + yt1 * uz1) + uz1 * tb1, pt2 = (xt2 * ux2 + yt2 * uz2) + uz2 * tb2;
        const long long per = (long long)L0 * H1, at = (long long)i * H1 + l;
        if (a.uv) {
            double* uv = a.uv + (long long)b * 4 * per + at;
            if (a.ratio != 0.0) {
                const double r = a.ratio;
                const double ox1 = uv[0], ox2 = uv[per], oz1 = uv[2 * per], oz2 = uv[3 * per];
                pu1 = pu1 + r * (xu1 * ox1 + yu1 * oz1);
                pv1 = pv1 + r * (xv1 * ox1 + yv1 * oz1);
                pt1 = pt1 + r * ((xt1 * ox1 + yt1 * oz1) + oz1 * tb1);
                pu2 = pu2 + r * (xu2 * ox2 + yu2 * oz2);
                pv2 = pv2 + r * (xv2 * ox2 + yv2 * oz2);
                pt2 = pt2 + r * ((xt2 * ox2 + yt2 * oz2) + oz2 * tb2);
            }
            uv[0] = ux1;
            uv[per] = ux2;
            uv[2 * per] = uz1;
            uv[3 * per] = uz2;
        }
        // the middle point of an odd grid is its own mirror: counted once
        const bool mid = L1 - 1 - l == l;
        double* P = a.Pr + (long long)b * 6 * per + at;
        P[0] = mid ? pu1 : pu1 + pu2;
        P[per] = mid ? 0.0 : pu1 - pu2;
        P[2 * per] = mid ? pv1 : pv1 + pv2;
        P[3 * per] = mid ? 0.0 : pv1 - pv2;
        P[4 * per] = mid ? pt1 : pt1 + pt2;
        P[5 * per] = mid ? 0.0 : pt1 - pt2;
    }
}

// ---------------------------------------------------------------------------
// Phase 3: Z[e][L0][M1] = -dt b (products) BF_y^T: even output modes from the
// sums, odd ones from the differences; a lane holds neighbouring modes and
// stores them as a pair.
template <int RT, int NT, int D>
__global__ void __launch_bounds__(256) stage_zconv(Stage a, int ntask)
{
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int task = xcd_remap(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    if (task >= ntask) return;
    const int M1 = a.M1, L0 = a.L0, H1 = (a.L1 + 1) / 2;
    const int MT = div_up((M1 + 1) / 2, 16), MG = div_up(MT, NT), RG = div_up(L0, 16 * RT);
    const int kc = div_up(H1, 16);
    const int t0 = (task % MG) * NT, rr = task / MG;
    const int r0 = (rr % RG) * 16 * RT, e = rr / RG;
    const double* __restrict__ P = a.Pr + (long long)e * 2 * L0 * H1;
    const double* __restrict__ op = a.bfy;  // [q][MT][kc]
    const double al = a.mdtb[e / 3];
    v4d acc[2][RT][NT] = {};
    v4d f[D][2][NT];
    RowTile x[D][2][RT];
    __shared__ double tiles[4][2][RT][16 * kTilePitch];
    auto& xs = tiles[threadIdx.x >> 6];
    auto load = [&](int st, int k) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
                x[st][q][i].load([&](int r) { return P + ((long long)q * L0 + min(r0 + 16 * i + r, L0 - 1)) * H1; }, k, H1,
                                 lane);
#pragma unroll
            for (int j = 0; j < NT; ++j) f[st][q][j] = op_frag(op, q * MT + min(t0 + j, MT - 1), kc, k, lane);
        }
    };
    auto compute = [&](int st, int k) {
        wave_lds_sync();  // the previous chunk is read
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < RT; ++i) x[st][q][i].store(xs[q][i], lane);
        wave_lds_sync();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const v2a p = RowTile::frag(xs[q][i], h, n, g);
                    const double v = pair_first(p, term(k, g, 2 * h), H1);
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[q][i][j] = mfma(v, f[st][q][j][2 * h], acc[q][i][j]);
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[q][i][j] = mfma(p.y, f[st][q][j][2 * h + 1], acc[q][i][j]);
                }
    };
    pipeline<D>(0, kc, load, compute);
    // every value is formed before the first conditional store (a use of a load
    // between stores would wait for the stores too)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[q][i][j] *= al;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int row = r0 + 16 * i + g + 4 * u, col = 2 * ((t0 + j) * 16 + n);
                if (row >= L0 || col >= M1 || t0 + j >= MT) continue;
                double* z = a.Z + ((long long)e * L0 + row) * M1 + col;
                if (col + 1 < M1) *reinterpret_cast<v2u*>(z) = v2u{acc[0][i][j][u], acc[1][i][j][u]};
                else *z = acc[0][i][j][u];
            }
}

// ---------------------------------------------------------------------------
// Phase 4: for 16 NT columns and the x modes of one parity, R += BF_x Z (the input
// folded over the mirrored x rows while it is staged into LDS) and the Helmholtz
// solve along x of those chains, in place on R.  One instance takes NT = 1 (96
// blocks at 256 x 256) and everything early; batches NT = 2, which halves the
// operator traffic from L2 (32 bytes per cycle and CU with 16 columns) and keeps two
// blocks per CU: the right-hand side then reuses the LDS of the staged input and the
// tables are read after the product.
template <int C, int NT>
__global__ void __launch_bounds__(512, NT == 1 ? 1 : 4) stage_rhs_hx(Stage a)
{
    extern __shared__ double lds[];
    // two rows apart = 128 bytes past a multiple of 256: neighbouring lane groups
    // read distinct banks
    constexpr int W = 16 * NT, XP = W + 8, YP = W + 1;
    const int M0 = a.M0, M1 = a.M1, L0 = a.L0, H0 = (L0 + 1) / 2;
    const int kc = div_up(H0, 16), CT = div_up(M1, W);
    double* Xs = lds;
    double* Ys = NT == 1 ? lds + kc * 16 * XP : lds;  // [16 C][YP]
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4, wave = tid >> 6;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    const int q = id & 1, c0 = ((id >> 1) % CT) * W, e = (id >> 1) / CT;
    const int rows = (M0 + 1 - q) / 2, RT = div_up((M0 + 1) / 2, 16);  // packed tiles of either parity
    const double* __restrict__ Z = a.Z + (long long)e * L0 * M1;
    double* __restrict__ R = a.R + (long long)e * M0 * M1;
    const int tc = tid % W, tr = tid / W;
    {
        constexpr int RP = 512 / W;  // rows per pass
        const int col = min(c0 + tc, M1 - 1);
        for (int k0 = tr; k0 < kc * 16; k0 += 8 * RP) {
            double u[8], d[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int k = min(k0 + RP * s, H0 - 1);
                u[s] = Z[(long long)k * M1 + col];
                d[s] = Z[(long long)(L0 - 1 - k) * M1 + col];
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int k = k0 + RP * s;
                if (k >= kc * 16) break;
                const double sum = k == L0 - 1 - k ? u[s] : (q ? u[s] - d[s] : u[s] + d[s]);
                Xs[k * XP + tc] = k < H0 ? sum : 0.0;
            }
        }
    }
    // tiles of this wave: wave, wave + 8 (at most C tiles)
    constexpr int TW = (C + 7) / 8;
    double add[TW][NT][4];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = (wave + 8 * t) * 16 + g + 4 * u;
                add[t][j][u] = R[(long long)min(2 * i + q, M0 - 1) * M1 + min(c0 + 16 * j + n, M1 - 1)];
            }
    double tab[4][C];   // of the chain this thread solves below
    const double* __restrict__ hx = a.hx + ((long long)e * 2 + q) * 4 * 16 * C;
    if (NT == 1 && tid < 256) chain_tables<C>(tab, hx, 16 * C, tid & 15);
    __syncthreads();
    const double* __restrict__ op = a.bfx + (long long)q * RT * kc * kFrag;
    v4d acc[TW][NT] = {};
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        if (wave + 8 * t < RT) {
            constexpr int D = NT == 1 ? kDeep : 3;
            v4d f[D];
            auto load = [&](int st, int k) { f[st] = op_frag(op, wave + 8 * t, kc, k, lane); };
            auto compute = [&](int st, int k) {
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[t][j] = mfma(f[st][s], Xs[term(k, g, s) * XP + 16 * j + n], acc[t][j]);
            };
            pipeline<D>(0, kc, load, compute);
        }
    }
    if (NT > 1) {
        chain_tables<C>(tab, hx, 16 * C, tid & 15);
        __syncthreads();  // every wave is done with Xs
    }
#pragma unroll
    for (int t = 0; t < TW; ++t)
        if (wave + 8 * t < C)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int i = (wave + 8 * t) * 16 + g + 4 * u;
                    Ys[i * YP + 16 * j + n] = i < rows ? add[t][j][u] + acc[t][j][u] : 0.0;
                }
    __syncthreads();
    if (tid < 256 * NT) {
        const int line = tid >> 4, c = tid & 15;
        double v[C];
#pragma unroll
        for (int k = 0; k < C; ++k) v[k] = Ys[(c * C + k) * YP + line];
        chain_solve<C>(v, tab, lane);
#pragma unroll
        for (int k = 0; k < C; ++k) Ys[(c * C + k) * YP + line] = v[k];
    }
    __syncthreads();
    if (c0 + tc < M1)
        for (int i = tr; i < rows; i += 512 / W) R[(long long)(2 * i + q) * M1 + c0 + tc] = Ys[i * YP + tc];
}

// ---------------------------------------------------------------------------
// Phase 5: for 16 rows of a field, the Helmholtz solve along y (both parity
// chains of each row, 16 lanes each), the solved rows to X, and products of them
// along y: U with H S (Poisson right-hand side), V with H D S and with D S (the
// divergence).  `per` operator tiles per block; blocks of one row group beyond
// the first repeat the solve instead of waiting for another launch, and only the
// first writes X.  With four tiles per block two waves share a tile, each half of
// its terms.
template <int C>
__global__ void __launch_bounds__(512) stage_hy(Stage a, int parts0, int parts1, int per)
{
    extern __shared__ double Ys[];
    __shared__ double half[4][4][64];
    const int M0 = a.M0, M1 = a.M1, N1 = a.N1;
    const int kc = div_up(M1, 16), T1 = kc, TN = div_up(N1, 16), RG = div_up(M0, 16);
    // row pitch and the position of entry i: one gap of two per 2 C entries, so
    // that the 16 lanes of a chain read distinct banks
    auto pos = [](int i) { return i + 2 * (i / (2 * C)); };
    const int pitch = pos(16 * kc) | 1;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4, wave = tid >> 6;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    const int np = parts0 + parts1 + 1;  // blocks per (instance, row group): U, V, T
    int part = id % np;
    const int r0 = ((id / np) % RG) * 16, b = id / np / RG;
    const int f = part < parts0 ? 0 : (part < parts0 + parts1 ? 1 : 2);
    part -= f == 0 ? 0 : (f == 1 ? parts0 : parts0 + parts1);
    const int e = 3 * b + f;
    const double* __restrict__ R = a.R + (long long)e * M0 * M1;
    // rows into LDS, two per wave, 8 loads in flight
    for (int c0 = lane; c0 < 16 * kc; c0 += 64 * 4) {
        double v[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                v[i][s] = R[(long long)min(r0 + wave * 2 + i, M0 - 1) * M1 + min(c0 + 64 * s, M1 - 1)];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c = c0 + 64 * s;
                if (c < 16 * kc) Ys[(wave * 2 + i) * pitch + pos(c)] = c < M1 ? v[i][s] : 0.0;
            }
    }
    {
        // a wave's chains are two rows, both parities
        const int line = tid >> 5, q = (tid >> 4) & 1, c = tid & 15;
        double* y = Ys + line * pitch;
        double tab[4][C], v[C];
        chain_tables<C>(tab, a.hy + ((long long)e * 2 + q) * 4 * 16 * C, 16 * C, c);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < C; ++k) {
            const int i = 2 * (c * C + k) + q;
            v[k] = i < 16 * kc ? y[pos(i)] : 0.0;
        }
        chain_solve<C>(v, tab, lane);
#pragma unroll
        for (int k = 0; k < C; ++k) {
            const int i = 2 * (c * C + k) + q;
            if (i < 16 * kc) y[pos(i)] = v[k];
        }
    }
    __syncthreads();
    if (part == 0) {
        double* __restrict__ X = a.X + (long long)e * M0 * M1;
        for (int i = 0; i < 2; ++i) {
            const int rr = wave * 2 + i;
            if (r0 + rr < M0)
                for (int c = lane; c < M1; c += 64) X[(long long)(r0 + rr) * M1 + c] = Ys[rr * pitch + pos(c)];
        }
    }
    if (f == 2) return;
    const int ntile = f == 0 ? T1 : T1 + TN;
    const int tend = min(ntile, (part + 1) * per);
    const double* yr = Ys + n * pitch;
    const bool split = per == 4;
    for (int t = part * per + (split ? wave & 3 : wave); t < part * per + per; t += 8) {
        const bool live = t < tend;
        const bool dv = t >= T1;  // divergence tile: triangular, terms from 16 t - 1 on
        // packed [H S : T1 tiles][H D S : T1 tiles][D S : TN tiles]
        const int tile = (f == 0 ? 0 : T1) + t;
        int kb = dv ? max(t - T1 - 1, 0) : 0, ke = live ? kc : kb;
        if (split) {
            const int mid = (kb + ke + 1) / 2;
            if (wave < 4) ke = mid;
            else kb = mid;
        }
        v4d acc = {};
        v4d fr[kDeep];
        auto load = [&](int st, int k) { fr[st] = op_frag(a.wy, tile, kc, k, lane); };
        auto compute = [&](int st, int k) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc = mfma(yr[pos(term(k, g, s & 2)) + (s & 1)], fr[st][s], acc);
        };
        pipeline<kDeep>(kb, ke, load, compute);
        v4d sum = acc;
        if (split) {
            if (wave >= 4)
#pragma unroll
                for (int u = 0; u < 4; ++u) half[wave & 3][u][lane] = sum[u];
            __syncthreads();
            if (wave >= 4) return;
#pragma unroll
            for (int u = 0; u < 4; ++u) sum[u] += half[wave][u][lane];
        }
        if (!live) continue;
        const int ncol = dv ? N1 : M1;
        double* out = dv ? a.W2v + (long long)b * M0 * N1 : a.W2 + ((long long)2 * b + f) * M0 * M1;
        const int col = (dv ? t - T1 : t) * 16 + n;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = r0 + g + 4 * u;
            if (row < M0 && col < ncol) out[(long long)row * ncol + col] = sum[u];
        }
    }
}

// ---------------------------------------------------------------------------
// Phase 6: blocks [0, nbp): for 16 y modes and the x modes of one parity, the
// Poisson right-hand side (B D S)_x W_U + (B S)_x W_V summed over its diagonals
// and the per-line solves along x, to RP.  Other blocks: the divergence
// div = (D S)_x (U S_y^T) + S_x (V (D S)_y^T), one output tile per wave, the first
// product over the opposite parity's modes from the first nonzero chunk on.
template <int C>
__global__ void __launch_bounds__(256) stage_poisson(Stage a, unsigned nbp, int ntask)
{
    extern __shared__ double lds[];
    double (*Ys)[17] = reinterpret_cast<double(*)[17]>(lds);                           // [16 C]
    double (*Ws)[16 * C + 4][16] = reinterpret_cast<double(*)[16 * C + 4][16]>(lds + 16 * C * 17);  // [2]
    double* Bs = lds + 16 * C * 17 + 2 * (16 * C + 4) * 16;                            // [8][16 C]
    const int M0 = a.M0, M1 = a.M1, N0 = a.N0, N1 = a.N1;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    if (blockIdx.x < nbp) {
        const int CT = div_up(M1, 16);
        const int id = xcd_remap(blockIdx.x, nbp);
        const int p = id & 1, c0 = ((id >> 1) % CT) * 16, b = (id >> 1) / CT;
        const int rows = (M0 + 1 - p) / 2;
        const double* __restrict__ WU = a.W2 + (long long)2 * b * M0 * M1;
        const double* __restrict__ WV = WU + (long long)M0 * M1;
        const int ln = tid & 15, col = min(c0 + ln, M1 - 1), r = tid >> 4;
        const int line = tid >> 4, c = tid & 15;
        // the rows that the diagonals reach: of the other parity for U, of this one
        // for V; Ws[f][j] holds chain row j - 1 (U: 2 (j - 1) + 1 - p, V: 2 (j - 1) + p)
        double x[2][C + 1];
#pragma unroll
        for (int k = 0; k <= C; ++k) {
            const int j = r + 16 * k - 1;
            x[0][k] = WU[(long long)min(max(2 * j + 1 - p, 0), M0 - 1) * M1 + col];
            x[1][k] = WV[(long long)min(max(2 * j + p, 0), M0 - 1) * M1 + col];
        }
        double cf[(C + 1) / 2];   // this thread's share of the coefficients, [8][16 C]
#pragma unroll
        for (int k = 0; k < C / 2; ++k) {
            const int i = tid + 256 * k, d = i / (16 * C);
            cf[k] = a.bds[d * M0 + min(2 * (i - d * 16 * C) + p, M0 - 1)];
        }
        double tab[4][C];
        chain_tables<C>(tab, a.prec + ((long long)p * 4 * M1 + min(c0 + line, M1 - 1)) * 16 * C, (long long)M1 * 16 * C, c);
#pragma unroll
        for (int k = 0; k <= C; ++k)
            if (r + 16 * k < 16 * C + 4) {
                Ws[0][r + 16 * k][ln] = x[0][k];
                Ws[1][r + 16 * k][ln] = x[1][k];
            }
#pragma unroll
        for (int k = 0; k < C / 2; ++k) Bs[tid + 256 * k] = cf[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < C; ++k) {
            // chain row i: V rows i - 1 .. i + 2; U rows from i - 1 (even i) or i (odd)
            const int i = r + 16 * k, u0 = p ? i + 1 : i;
            double u = 0.0;
#pragma unroll
            for (int d = 0; d < 4; ++d) u += Bs[d * 16 * C + i] * Ws[0][u0 + d][ln];
#pragma unroll
            for (int d = 0; d < 4; ++d) u += Bs[(4 + d) * 16 * C + i] * Ws[1][i + d][ln];
            Ys[i][ln] = i < rows ? u : 0.0;
        }
        __syncthreads();
        {
            double v[C];
#pragma unroll
            for (int k = 0; k < C; ++k) v[k] = Ys[c * C + k][line];
            chain_solve<C>(v, tab, lane);
#pragma unroll
            for (int k = 0; k < C; ++k) Ys[c * C + k][line] = v[k];
        }
        __syncthreads();
        double* __restrict__ RP = a.RP + (long long)b * M0 * M1;
        if (c0 + ln < M1)
            for (int i = tid >> 4; i < rows; i += 16) RP[(long long)(2 * i + p) * M1 + c0 + ln] = Ys[i][ln];
        return;
    }
    const int task = xcd_remap(blockIdx.x - nbp, gridDim.x - nbp) * 4 + (tid >> 6);
    if (task >= ntask) return;
    const int RT = div_up((N0 + 1) / 2, 16), CT = div_up(N1, 16), kc = div_up((M0 + 1) / 2, 16);
    const int t = task % RT, q = (task / RT) & 1, cb = task / (2 * RT);
    const int c0 = (cb % CT) * 16, b = cb / CT;
    const int col = c0 + n;
    const double* __restrict__ U = a.X + (long long)3 * b * M0 * M1;
    const int ca = min(col, M1 - 1), cz = min(max(col - 2, 0), M1 - 1);
    const double* __restrict__ V = a.W2v + (long long)b * M0 * N1;
    double va[4], vz[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int row = 2 * (t * 16 + g + 4 * u) + q;
        va[u] = V[(long long)min(row, M0 - 1) * N1 + min(col, N1 - 1)];
        vz[u] = V[(long long)min(max(row - 2, 0), M0 - 1) * N1 + min(col, N1 - 1)];
        if (row >= M0) va[u] = 0.0;
        if (row < 2) vz[u] = 0.0;
    }
    const double* __restrict__ op = a.cdx + (long long)q * RT * kc * kFrag;
    v4d acc = {};
    v4d f[4];
    double x[4][4], z[4][4];
    auto load = [&](int st, int k) {
        f[st] = op_frag(op, t, kc, k, lane);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double* row = U + (long long)min(2 * term(k, g, s) + 1 - q, M0 - 1) * M1;
            x[st][s] = row[ca];
            z[st][s] = row[cz];
        }
    };
    auto compute = [&](int st, int k) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double v = (col < M1 ? x[st][s] : 0.0) - (col >= 2 ? z[st][s] : 0.0);
            acc = mfma(f[st][s], v, acc);
        }
    };
    pipeline<4>(max(t - 1, 0), kc, load, compute);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int row = 2 * (t * 16 + g + 4 * u) + q;
        if (row < N0 && col < N1)
            a.div[((long long)b * N0 + row) * N1 + col] = acc[u] + (va[u] - vz[u]);
    }
}

// ---------------------------------------------------------------------------
// Phase 7: P = RP Q^T (with the gauge P[0,0] = 0) and the y factors of the
// velocity correction, W1 = RP [T S Q ; T D S Q]^T.  The gauge does not reach W1:
// the constant mode's derivatives vanish.
template <int RT, int NT, int D>
__global__ void __launch_bounds__(256) stage_qy(Stage a, int ntask)
{
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int task = xcd_remap(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    if (task >= ntask) return;
    const int M0 = a.M0, M1 = a.M1;
    const int kc = div_up(M1, 16), T1 = kc, TG = div_up(3 * T1, NT), RG = div_up(M0, 16 * RT);
    const int t0 = (task % TG) * NT, rr = task / TG;
    const int r0 = (rr % RG) * 16 * RT, b = rr / RG;
    const double* __restrict__ RP = a.RP + (long long)b * M0 * M1;
    v4d acc[RT][NT] = {};
    v4d f[D][NT];
    RowTile x[D][RT];
    __shared__ double tiles[4][RT][16 * kTilePitch];
    auto& xs = tiles[threadIdx.x >> 6];
    auto load = [&](int st, int k) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
            x[st][i].load([&](int r) { return RP + (long long)min(r0 + 16 * i + r, M0 - 1) * M1; }, k, M1, lane);
#pragma unroll
        for (int j = 0; j < NT; ++j) f[st][j] = op_frag(a.qy, min(t0 + j, 3 * T1 - 1), kc, k, lane);
    };
    auto compute = [&](int st, int k) {
        wave_lds_sync();  // the previous chunk is read
#pragma unroll
        for (int i = 0; i < RT; ++i) x[st][i].store(xs[i], lane);
        wave_lds_sync();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const v2a p = RowTile::frag(xs[i], h, n, g);
                const double v = pair_first(p, term(k, g, 2 * h), M1);
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma(v, f[st][j][2 * h], acc[i][j]);
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma(p.y, f[st][j][2 * h + 1], acc[i][j]);
            }
    };
    pipeline<D>(0, kc, load, compute);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        if (t0 + j >= 3 * T1) break;
        const int sel = (t0 + j) / T1, col = (t0 + j - sel * T1) * 16 + n;
        double* __restrict__ out = sel == 0 ? a.P + (long long)b * M0 * M1
                                            : a.W1 + ((long long)2 * b + sel - 1) * M0 * M1;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int row = r0 + 16 * i + g + 4 * u;
                if (row >= M0 || col >= M1) continue;
                out[(long long)row * M1 + col] = (sel == 0 && row == 0 && col == 0) ? 0.0 : acc[i][j][u];
            }
    }
}

// ---------------------------------------------------------------------------
// Phase 8: blocks [0, nbr): pres = (pres - nu div beta) + S_x P S_y^T / (dt a), the
// stencils as four terms.  Other blocks: U -= (T D S)_x W1[0] (opposite parity),
// V -= (T S)_x W1[1], one wave per 16 NT columns, 16 modes of one parity.
template <int NT, int D>
__global__ void __launch_bounds__(256) stage_correct(Stage a, unsigned nbr, int ntask)
{
    const int M0 = a.M0, M1 = a.M1, N0 = a.N0, N1 = a.N1;
    if (blockIdx.x < nbr) {
#pragma clang fp contract(off)
        const long long per = (long long)N0 * N1, total = per * a.batch;
        for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < total; t += (long long)nbr * 256) {
            const int b = (int)(t / per);
            const int r = (int)(t - b * per), i = r / N1, j = r - i * N1;
            const double* __restrict__ P = a.P + (long long)b * M0 * M1;
            const int i0 = min(i, M0 - 1), i2 = max(i - 2, 0), j0 = min(j, M1 - 1), j2 = max(j - 2, 0);
            const double p00 = P[(long long)i0 * M1 + j0], p02 = P[(long long)i0 * M1 + j2];
            const double p20 = P[(long long)i2 * M1 + j0], p22 = P[(long long)i2 * M1 + j2];
            const double sx = i >= 2 ? a.sn[i2] : 0.0, sy = j >= 2 ? a.sn[M0 + j2] : 0.0;
            const double ux = i < M0 ? 1.0 : 0.0, uy = j < M1 ? 1.0 : 0.0;
            const double s = ux * (uy * p00 + sy * p02) + sx * (uy * p20 + sy * p22);
            const double add = __builtin_fma(-(a.nu[b] * a.div[t]), a.beta, a.pres[t]);
            a.pres[t] = add + a.idta[b] * s;
        }
        return;
    }
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int task = xcd_remap(blockIdx.x - nbr, gridDim.x - nbr) * 4 + (threadIdx.x >> 6);
    if (task >= ntask) return;
    const int RT = div_up((M0 + 1) / 2, 16), CT = div_up(M1, 16 * NT), kc = RT;
    const int t = task % RT, q = (task / RT) & 1, cb = task / (2 * RT);
    const int c0 = (cb % CT) * 16 * NT, bf = cb / CT, f = bf & 1, b = bf >> 1;
    const int par = f == 0 ? 1 - q : q;
    const double* __restrict__ W = a.W1 + (long long)bf * M0 * M1;
    const double* __restrict__ op = a.corr + (long long)(2 * f + q) * RT * kc * kFrag;
    double* __restrict__ X = a.X + (long long)(3 * b + f) * M0 * M1;
    double old[NT][4];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = 2 * (t * 16 + g + 4 * u) + q;
            old[j][u] = X[(long long)min(i, M0 - 1) * M1 + min(c0 + 16 * j + n, M1 - 1)];
        }
    v4d acc[NT] = {};
    v4d fr[D];
    double x[D][NT][4];
    auto load = [&](int st, int k) {
        fr[st] = op_frag(op, t, kc, k, lane);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double* row = W + (long long)min(2 * term(k, g, s) + par, M0 - 1) * M1;
#pragma unroll
            for (int j = 0; j < NT; ++j) x[st][j][s] = row[min(c0 + 16 * j + n, M1 - 1)];
        }
    };
    auto compute = [&](int st, int k) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = mfma(fr[st][s], x[st][j][s], acc[j]);
    };
    pipeline<D>(0, kc, load, compute);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) old[j][u] -= acc[j][u];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = 2 * (t * 16 + g + 4 * u) + q, col = c0 + 16 * j + n;
            if (i < M0 && col < M1) X[(long long)i * M1 + col] = old[j][u];
        }
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
static int up(int a, int b) { return (a + b - 1) / b; }
static unsigned blocks4(long long tasks) { return (unsigned)((tasks + 3) / 4); }

// chain positions per lane for lines of m entries (two parity chains on 16 lanes)
static int chain_len(int m)
{
    const int c = up((m + 1) / 2, 16);
    return c <= 2 ? 2 : c <= 4 ? 4 : c <= 8 ? 8 : 16;
}

// Outputs from which the right-hand side leaves the x-pass's launch for one of its
// own, whose tiles share each row's y sums in LDS.  Below, a launch costs more than
// they save.  Phase 1 merged against alone: 256 x 256 (194 K outputs) 16.5 us against
// 21.4, 400 x 400 (475 K) 35.6 against 38.4; 64 x 64^2 (738 K) 31.4 against 27.9, 512 x
// 512 (780 K) 58.0 against 53.8, 16 x 256^2 (3.1 M) 151 against 108.
constexpr long long kRhsAlone = 700000;

// Waves from which a wave takes 2 x 2 or 2 x 1 tiles: two for every SIMD, all that
// their registers leave room for.  Half the operand traffic, but half the waves.
constexpr long long kWideTasks = 2048;

static int phase1(const Stage& a, const pypde_rbc_rhs* r, hipStream_t s)
{
    pypde_rbc_rhs rhs{};
    unsigned nbr = 0;
    if (r) {
        rhs = *r;
        const long long outs = 3LL * rhs.M0 * rhs.M1 * rhs.batch;
        if (outs >= kRhsAlone) {
            rhs.rows_per_thread = 16;   // the tile form
            const int rc = pypde_rbc_rhs_banded(&rhs, s);
            if (rc != OK) return rc;
        } else {
            nbr = (unsigned)std::min<long long>((outs + 255) / 256, 16384);
        }
    }
    const int HT = up((a.L0 + 1) / 2, 16);
    // with the right-hand side, 2 x 2 / 2 x 1 / 1 x 1 tiles: 512 x 512 (1152 and 2304
    // wide tasks) 58.9 / 52.6 / 55.0 us, 400 x 400 (780 and 1500) 49.8 / 41.4 / 34.3,
    // 4 x 512^2 (4608 and 9216) 143 / 143 / 170
    const long long big = 3LL * a.batch * up(a.M1, 32) * 2 * up(HT, 2);
    if (big >= kWideTasks) {
        hipLaunchKernelGGL((stage_xpass<2, 2, 2>), dim3(nbr + blocks4(big)), dim3(256), 0, s, a, rhs, nbr, (int)big);
    } else if (3LL * a.batch * up(a.M1, 16) * 2 * up(HT, 2) >= kWideTasks) {
        const long long t = 3LL * a.batch * up(a.M1, 16) * 2 * up(HT, 2);
        hipLaunchKernelGGL((stage_xpass<2, 1, 2>), dim3(nbr + blocks4(t)), dim3(256), 0, s, a, rhs, nbr, (int)t);
    } else {
        const long long t = 3LL * a.batch * up(a.M1, 16) * 2 * HT;
        hipLaunchKernelGGL((stage_xpass<1, 1, 4>), dim3(nbr + blocks4(t)), dim3(256), 0, s, a, rhs, nbr, (int)t);
    }
    return check_launch("pypde_rbc_phase 1");
}

static int phase2(const Stage& a, hipStream_t s)
{
    const int HT = up((a.L1 + 1) / 2, 16), rows = a.batch * up(a.L0, 16);
    // two tiles per block halve the traffic of the rows; while single tiles find a CU
    // each, they are done in two thirds of the time (224 x 224: 9.4 us against 13.3,
    // 16 x 300: 10.7 against 16.4; 240 x 240 with 276 blocks: 15.4 against 14.8)
    if (rows * HT <= kCus) hipLaunchKernelGGL(stage_yprod<1>, dim3((unsigned)(rows * HT)), dim3(512), 0, s, a);
    else hipLaunchKernelGGL(stage_yprod<2>, dim3((unsigned)(rows * up(HT, 2))), dim3(512), 0, s, a);
    return check_launch("pypde_rbc_phase 2");
}

static int phase3(const Stage& a, hipStream_t s)
{
    const int MT = up((a.M1 + 1) / 2, 16);
    // 2 x 2 tiles against single ones: 576 tasks (512 x 512) 36.7 us against 32.4, 1152
    // (8 x 256^2) 34.3 against 29.8, 2304 (16 x 256^2) 50.0 against 49.1
    const long long big = 3LL * a.batch * up(a.L0, 32) * up(MT, 2);
    if (big >= kWideTasks) {
        hipLaunchKernelGGL((stage_zconv<2, 2, 2>), dim3(blocks4(big)), dim3(256), 0, s, a, (int)big);
    } else {
        const long long t = 3LL * a.batch * up(a.L0, 16) * MT;
        hipLaunchKernelGGL((stage_zconv<1, 1, 4>), dim3(blocks4(t)), dim3(256), 0, s, a, (int)t);
    }
    return check_launch("pypde_rbc_phase 3");
}

template <int C, int NT>
static int phase4_n(const Stage& a, hipStream_t s)
{
    const size_t x = (size_t)up((a.L0 + 1) / 2, 16) * 16 * (16 * NT + 8), y = (size_t)16 * C * (16 * NT + 1);
    const size_t lds = (NT == 1 ? x + y : std::max(x, y)) * sizeof(double);
    if (const int rc = allow_lds<stage_rhs_hx<C, NT>>(lds)) return rc;
    const long long blocks = 2LL * 3 * a.batch * up(a.M1, 16 * NT);
    hipLaunchKernelGGL((stage_rhs_hx<C, NT>), dim3((unsigned)blocks), dim3(512), lds, s, a);
    return check_launch("pypde_rbc_phase 4");
}

template <int C>
static int phase4_c(const Stage& a, hipStream_t s)
{
    // 32 columns per block once that still gives every CU two blocks (16 x 256^2, 768
    // blocks: 39.0 us against 52.3 with 16; 256 x 256, 48: 15.4 against 10.0); the
    // longest chains would spill registers in that form
    if constexpr (C < 16)
        if (6LL * a.batch * up(a.M1, 32) >= 512) return phase4_n<C, 2>(a, s);
    return phase4_n<C, 1>(a, s);
}

template <int C>
static int phase5_c(const Stage& a, hipStream_t s)
{
    const int kc = up(a.M1, 16), TN = up(a.N1, 16), rows = a.batch * up(a.M0, 16);
    const int len = 16 * kc;
    const size_t lds = 16 * (size_t)((len + 2 * (len / (2 * C))) | 1) * sizeof(double);
    if (const int rc = allow_lds<stage_hy<C>>(lds)) return rc;
    // four operator tiles per block while the blocks run side by side (two per CU,
    // one with the longest chains), else more, so that the solve is repeated less
    // often (4, 8, 16 tiles: 256 x 256 10.1, 12.4, 18.3 us; 4 x 256^2 24.2, 20.3, 19.8;
    // 512 x 512 45.4, 40.7, 33.9)
    int per = 4;
    while (per < 16 && (long long)rows * (up(kc, per) + up(kc + TN, per) + 1) > (C == 16 ? 256 : 512)) per *= 2;
    const int p0 = up(kc, per), p1 = up(kc + TN, per);
    hipLaunchKernelGGL(stage_hy<C>, dim3((unsigned)(rows * (p0 + p1 + 1))), dim3(512), lds, s, a, p0, p1, per);
    return check_launch("pypde_rbc_phase 5");
}

template <int C>
static int phase6_c(const Stage& a, hipStream_t s)
{
    const unsigned nbp = 2u * a.batch * up(a.M1, 16);
    const long long t = 2LL * a.batch * up((a.N0 + 1) / 2, 16) * up(a.N1, 16);
    const size_t lds = (16 * C * 17 + 2 * (16 * C + 4) * 16 + 8 * 16 * C) * sizeof(double);
    if (const int rc = allow_lds<stage_poisson<C>>(lds)) return rc;
    hipLaunchKernelGGL(stage_poisson<C>, dim3(nbp + blocks4(t)), dim3(256), lds, s, a, nbp, (int)t);
    return check_launch("pypde_rbc_phase 6");
}

static int phase7(const Stage& a, hipStream_t s)
{
    const int T = 3 * up(a.M1, 16);
    // 2 x 2 tiles against single ones: 768 tasks (512 x 512) 27.6 us against 24.1, 1536
    // (8 x 256^2) 23.4 against 22.1, 3072 (16 x 256^2) 32.6 against 41.2
    const long long big = (long long)a.batch * up(a.M0, 32) * up(T, 2);
    if (big >= kWideTasks) {
        hipLaunchKernelGGL((stage_qy<2, 2, 2>), dim3(blocks4(big)), dim3(256), 0, s, a, (int)big);
    } else {
        const long long t = (long long)a.batch * up(a.M0, 16) * T;
        hipLaunchKernelGGL((stage_qy<1, 1, kDeep>), dim3(blocks4(t)), dim3(256), 0, s, a, (int)t);
    }
    return check_launch("pypde_rbc_phase 7");
}

static int phase8(const Stage& a, hipStream_t s)
{
    const long long pr = ((long long)a.N0 * a.N1 * a.batch + 255) / 256;
    const unsigned nbr = (unsigned)std::min<long long>(pr, 16384);
    const long long per = 4LL * a.batch * up((a.M0 + 1) / 2, 16);
    // 32 columns per wave against 16: 1024 tasks (512 x 512) 12.6 us against 13.3, 2048
    // (8 x 256^2) 17.5 against 15.9, 4096 (16 x 256^2) 25.6 against 27.4
    const long long big = per * up(a.M1, 32);
    if (big >= kWideTasks) {
        hipLaunchKernelGGL((stage_correct<2, 3>), dim3(nbr + blocks4(big)), dim3(256), 0, s, a, nbr, (int)big);
    } else {
        const long long t = per * up(a.M1, 16);
        hipLaunchKernelGGL((stage_correct<1, kDeep>), dim3(nbr + blocks4(t)), dim3(256), 0, s, a, nbr, (int)t);
    }
    return check_launch("pypde_rbc_phase 8");
}

}  // namespace pypde

using namespace pypde;

extern "C" int pypde_rbc_phase(const pypde_rbc_stage* st, const pypde_rbc_rhs* rhs, int phase, void* stream)
{
    PYPDE_REQUIRE(st, "null stage");
    const Stage& a = *st;
    PYPDE_REQUIRE(phase >= 1 && phase <= 8, "phase %d not in 1..8", phase);
    PYPDE_REQUIRE(a.M0 >= 6 && a.M1 >= 6 && a.N0 == a.M0 + 2 && a.N1 == a.M1 + 2 && a.L0 >= a.N0 &&
                      a.L1 >= a.N1 && a.batch >= 0,
                  "invalid stage geometry: M0 %d M1 %d N0 %d N1 %d L0 %d L1 %d batch %d", a.M0, a.M1, a.N0, a.N1,
                  a.L0, a.L1, a.batch);
    PYPDE_REQUIRE(a.M0 <= PYPDE_STAGE_MAX_MODES && a.M1 <= PYPDE_STAGE_MAX_MODES &&
                      a.L0 <= 2 * PYPDE_STAGE_MAX_MODES && a.L1 <= 2 * PYPDE_STAGE_MAX_MODES,
                  "stage: at most %d modes per axis", PYPDE_STAGE_MAX_MODES);
    PYPDE_REQUIRE(a.X && a.pres && a.P && a.Y1 && a.Pr && a.Z && a.R && a.W2 && a.W2v && a.RP && a.W1 && a.div &&
                      a.gx && a.gy && a.bfy && a.bfx && a.wy && a.qy && a.cdx && a.corr && a.bds && a.sn &&
                      a.dtbc && a.hx && a.hy && a.prec && a.mdtb && a.idta && a.nu,
                  "null stage pointer");
    for (const double* op : {a.gx, a.gy, a.bfy, a.bfx, a.wy, a.qy, a.cdx, a.corr})
        PYPDE_REQUIRE(reinterpret_cast<uintptr_t>(op) % sizeof(v4d) == 0,
                      "stage: packed operators are read 32 bytes at a time and must be 32-byte aligned");
    PYPDE_REQUIRE(a.ratio == 0.0 || a.uv, "the c-term needs the previous stage's velocities");
    PYPDE_REQUIRE((long long)a.batch * (a.L0 / 16 + 1) * (a.L1 / 16 + 1) * 6 < (1LL << 30), "stage: batch too large");
    if (rhs) {
        PYPDE_REQUIRE(phase == 1, "the banded right-hand side belongs to phase 1");
        PYPDE_REQUIRE(rhs->X && rhs->pres && rhs->R && rhs->mdta && rhs->dta && rhs->tx && rhs->ty,
                      "null right-hand-side pointer (X, pres, R, mdta, dta, tx and ty are required)");
        PYPDE_REQUIRE(rhs->M0 >= 1 && rhs->M1 >= 1 && rhs->N0 == rhs->M0 + 2 && rhs->N1 == rhs->M1 + 2 &&
                          rhs->batch >= 0,
                      "invalid right-hand-side geometry: M0 %d M1 %d N0 %d N1 %d batch %d", rhs->M0, rhs->M1,
                      rhs->N0, rhs->N1, rhs->batch);
        PYPDE_REQUIRE(rhs->R != rhs->X, "R must not alias X (neighbouring entries are read)");
        PYPDE_REQUIRE(rhs->rows_per_thread == 1,
                      "the merged launch computes one right-hand-side output per thread (rows_per_thread must "
                      "be 1, got %d)", rhs->rows_per_thread);
    }
    if (a.batch == 0) return OK;
    hipStream_t s = as_stream(stream);
    switch (phase) {
    case 1: return phase1(a, rhs, s);
    case 2: return phase2(a, s);
    case 3: return phase3(a, s);
    case 4:
        switch (chain_len(a.M0)) {
        case 2: return phase4_c<2>(a, s);
        case 4: return phase4_c<4>(a, s);
        case 8: return phase4_c<8>(a, s);
        default: return phase4_c<16>(a, s);
        }
    case 5:
        switch (chain_len(a.M1)) {
        case 2: return phase5_c<2>(a, s);
        case 4: return phase5_c<4>(a, s);
        case 8: return phase5_c<8>(a, s);
        default: return phase5_c<16>(a, s);
        }
    case 6:
        switch (chain_len(a.M0)) {
        case 2: return phase6_c<2>(a, s);
        case 4: return phase6_c<4>(a, s);
        case 8: return phase6_c<8>(a, s);
        default: return phase6_c<16>(a, s);
        }
    case 7: return phase7(a, s);
    default: return phase8(a, s);
    }
}
