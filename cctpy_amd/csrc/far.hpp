// Far field of segment clusters, shared by the tracking kernels (cctamd.hip) and the
// kernels that build the clusters (far.hip).
//
// The tracking kernels need the field of S segments at P points per RK4 stage.  Segments
// that lie close together act on a distant point block through a short series instead
// of one by one.  A design's segments are ordered in space (far.hip) and cut into clusters of
// kSmallTiles tiles of 32 rows (512 segments), and four of those make a large cluster
// (2,048).  With c a cluster's centre, E its radius, x = (q - c) / E, r = |x|,
// (X, Y, Z) = x / r^2 and rho = 1 / r^2, each component of its field is a harmonic function
// outside the ball, a sum of exterior solid harmonics
//     B(q) = sum over m <= n <= N of t_n^m (beta_c Re(X + iY)^m + beta_s Im(X + iY)^m),
//     t_m^m = 1 / r,   t_{n+1} = Z t_n - kappa rho t_{n-1},  kappa = (n^2 - m^2) / (4 n^2 - 1)
// (the recurrence of the associated Legendre functions in n, with the double factorial
// (2n - 1)!! taken into beta).  The coefficients are the curl of the multipole series of the
// vector potential sum kl / |q - m| (addition theorem of 1 / |x - y| in regular and exterior
// solid harmonics), built once per segment set.  A block takes a large cluster's
// series where the large one is far enough, else the series of those of its four parts that
// are, and sums the other parts' segments one by one.
//
// Orders per distance (FarOrders), for the worst cluster: one element with all the current on
// the rim, towards the point.  Relative to that element's term the cut is at most
// (N + 1) (E / |q - c|)^N or so: below 4e-16 at every distance of the FP64 table (a term of the
// full sum is rounded by as much), 2e-9 of the FP32 one (terms rounded at 6e-8); other clusters'
// cuts are smaller against their sum of |terms| (random elements in a ball: by 100 or more).  With the
// rounding of the series, which are evaluated in FP64 on both paths, worst of elements on the rim,
// bars, rings and balls at every distance of the tables, against extended precision: 1.1e-15 and
// 1.0e-9.  FP64 from 3.55 radii on with order 31 at the most keeps the same bound but sums more
// segments one by one: 512 protons in the AG-CCT section 52 us per stage, with order 35 48.
#pragma once

#include "common.hpp"

namespace cctamd_detail {

constexpr int kSmallTiles = 16;           // tiles of a small cluster
constexpr int kParts = 4;                 // small clusters of a large one
constexpr int kFarGeo = 8;                // doubles per cluster: centre, 1 / E, E, 0, 0, 0
constexpr int kFarRec = 8;                // doubles per record: beta_c xyz, beta_s xyz, -kappa, 0
constexpr int kFarQ64 = 9, kFarQ32 = 5;   // highest order + 1 = 4 Q: 36 on the FP64 path, 20 on the FP32 path

// Record (m, n) of a cluster is at far_row(Q, m) + (n - m); rows hold a multiple of four
// records (zero beyond the highest order), so that the row loops need no remainder.
__host__ __device__ constexpr int far_row(int q, int m) {
    return 4 * (m * q - 2 * (m >> 2) * ((m >> 2) - 1) - (m >> 2) * (m & 3));
}
__host__ __device__ constexpr int far_records(int q) { return far_row(q, 4 * q); }

template <bool F64>
struct FarOrders;
template <>
struct FarOrders<true> {
    static constexpr int n = 10;
    static constexpr double ratio[n] = {3.1, 3.55, 4.05, 5.1, 7.05, 9.85, 13.3, 25.0, 47.0, 120.0};
    static constexpr int order[n] = {35, 31, 28, 24, 20, 17, 15, 12, 10, 8};
};
template <>
struct FarOrders<false> {
    static constexpr int n = 7;
    static constexpr double ratio[n] = {4.0, 4.5, 6.0, 8.0, 12.0, 20.0, 40.0};
    static constexpr int order[n] = {18, 16, 14, 12, 10, 8, 6};
};

// A ball around the points of a block (held by the lanes of every one of its waves alike).
// Its centre is the middle of the bounding box in FP32, any point would do; the radius
// covers every point; a point that is not finite gives an infinite radius (no cluster is far).
struct Ball {
    double x, y, z, r;
};

// Largest of v over the wave (a NaN loses), by DPP: neighbours within the 16-lane rows, then the
// rows' last lanes into the next rows; lane 63 has it.  Shuffles go through LDS and cost
// several times as much.
__device__ __forceinline__ float wave_max(float v) {
    const auto with = [&](int moved) { v = fmaxf(v, __builtin_bit_cast(float, moved)); };
    // the lanes without a source keep their own value (old = v)
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, false));
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, false));
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, false));
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, false));
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
    with(__builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

template <int PL>
__device__ __forceinline__ Ball block_ball(const double (&px)[PL], const double (&py)[PL], const double (&pz)[PL]) {
    float lo[3], hi[3];
    lo[0] = hi[0] = (float)px[0];
    lo[1] = hi[1] = (float)py[0];
    lo[2] = hi[2] = (float)pz[0];
#pragma unroll
    for (int j = 1; j < PL; ++j) {
        const float v[3] = {(float)px[j], (float)py[j], (float)pz[j]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lo[c] = fminf(lo[c], v[c]);
            hi[c] = fmaxf(hi[c], v[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        hi[c] = wave_max(hi[c]);
        lo[c] = -wave_max(-lo[c]);
    }
    Ball b{0.5 * ((double)lo[0] + hi[0]), 0.5 * ((double)lo[1] + hi[1]), 0.5 * ((double)lo[2] + hi[2]), 0.0};
    float r2 = 0.0f;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const double dx = px[j] - b.x, dy = py[j] - b.y, dz = pz[j] - b.z;
        const double d2 = dx * dx + dy * dy + dz * dz;
        bad = bad || !(d2 < 1.0e30);
        r2 = fmaxf(r2, (float)d2);
    }
    // 1.00001: FP32 rounding of d2 and of the root
    b.r = __any(bad) ? __builtin_huge_val() : 1.00001 * (double)__builtin_sqrtf(wave_max(r2));
    return b;
}

// Cost of a series in quarters of a block of four terms, for dealing it out.  A wave of one point
// set takes row after row (LR = 1), one whose four rows of lanes hold the same points takes four
// rows m at a time (LR = 4), a unit either way.  A unit's start: the blocks of those before it, a
// row's own start and end (kFarRowCost each) and what a series needs before its first row.
constexpr int kFarRowCost = 3, kFarSeriesCost = 12;
template <int LR>
__host__ __device__ constexpr int far_units(int N) { return LR == 1 ? N + 1 : (N >> 2) + 1; }
template <int LR>
__host__ __device__ constexpr int far_unit_blocks(int N, int u) {
    return LR == 1 ? (N - u + 4) >> 2 : (N >> 2) - u + 1;
}
__host__ __device__ constexpr int far_blocks_upto(int l) {  // sum of ceil(k / 4) over k = 1 .. l
    return ((l >> 2) + 1) * (2 * (l >> 2) + (l & 3));
}
template <int LR>
__host__ __device__ constexpr int far_unit_start(int N, int u) {  // 0 for u = 0
    const int blocks = LR == 1 ? far_blocks_upto(N + 1) - far_blocks_upto(N + 1 - u)
                               : u * far_units<4>(N) - u * (u - 1) / 2;
    return u == 0 ? 0 : kFarSeriesCost + kFarRowCost * u + 4 * blocks;
}
// Order and cost of a series in one value, as the lists carry them about; the order takes as many
// bits as the path's highest one needs (6 on the FP32 path too: its gantry stage 4 % slower).
constexpr int far_order_bits(int q) { return q > 8 ? 6 : 5; }
template <bool F64, int LR>
__host__ __device__ constexpr int far_pack(int N) {
    return far_unit_start<LR>(N, far_units<LR>(N)) << far_order_bits(F64 ? kFarQ64 : kFarQ32) | N;
}

// Order and cost (far_pack) of the series that serves a cluster for a block, 0 if the cluster is too
// close (its segments are then summed one by one).  Every wave and workgroup of a block gets the
// same answer: the same operations on the same values, each rounded by itself.
#pragma clang fp contract(off)
template <bool F64, int LR>
__device__ __forceinline__ int far_order(const double* __restrict__ geo, const Ball& b) {
    const double dx = geo[0] - b.x, dy = geo[1] - b.y, dz = geo[2] - b.z;
    const float d = __builtin_amdgcn_sqrtf((float)(dx * dx + dy * dy + dz * dz));
    const float ratio = (d - (float)b.r) * (float)geo[3];
    using T = FarOrders<F64>;
    int n = 0;
#pragma unroll
    for (int k = 0; k < T::n; ++k) n = ratio >= (float)T::ratio[k] ? far_pack<F64, LR>(T::order[k]) : n;
    return n;
}
#pragma clang fp contract(fast)

// Sum of v over the lanes of the wave up to and with this one: within the 16-lane rows, then the
// rows' last lanes into the next rows.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

__device__ __forceinline__ int lane_rank(uint64_t mask) {  // set bits below this lane
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Work lists of a workgroup for its point block, in LDS: the small clusters whose segments are
// summed one by one, and the clusters, small or large, that act through their series.  Every
// workgroup of a block makes the same lists; each takes its share of them (the segments of the
// near clusters and the rows of the series are dealt out over all waves of the block's work
// items, so that neither falls to a few of them).
template <int NW>
struct FarLists {
    static constexpr int kRound = kWave * NW;  // large clusters per round
    int near[kParts * kRound];                 // small cluster
    int far[kParts * kRound];                  // cluster | order (far_order_bits) | large (1 bit)
    int start[kParts * kRound];                // cost of the series before this one in the list
    unsigned short close[kRound];              // large clusters of the round that are not far
    int tally[2][(kParts + 1) * NW];           // of a wave: series | other clusters << 16, cost of the series
};

struct FarCounts {
    int near, far, cost;
};

// Lists of the large clusters [base, base + kRound) of a work item's design (w.tile_start: its
// first small cluster, w.tile_count: its small clusters).  All waves of all workgroups run through
// this at once, so its instructions count: with FP64 roots, orders and costs of four rounds kept in
// registers and every tally added up by every lane it took 2.5 us, a tenth of a stage of the AG-CCT
// section; now 1.5.
template <bool F64, int LR, int NW>
__device__ __forceinline__ FarCounts far_lists(FarLists<NW>& L, const FarSet& fs, const Work& w, const Ball& ball,
                                               int base, int wave, int lane) {
    constexpr int bits = far_order_bits(F64 ? kFarQ64 : kFarQ32);
    FarCounts n{0, 0, 0};
    // a cluster per lane: it joins the series, or put(its place among the others) takes it
    const auto round = [&](int slot, bool valid, int cl, const double* geo, int large, auto&& put) {
        int order = 0, upto = 0;
        uint64_t far = 0, other = 0;
        if (__any(valid)) {  // wave-uniform
            order = valid ? far_order<F64, LR>(geo + (int64_t)cl * kFarGeo, ball) : 0;
            far = __ballot(order != 0);
            other = __ballot(valid && order == 0);
            upto = wave_scan(order >> bits);
        }
        const int own = __popcll(far) | __popcll(other) << 16;
        if (lane == kWave - 1) {
            L.tally[0][slot * NW + wave] = own;
            L.tally[1][slot * NW + wave] = upto;
        }
        __syncthreads();
        // sums up to each wave in lanes 0 .. NW - 1
        int count = L.tally[0][slot * NW + (lane & (NW - 1))], cost = L.tally[1][slot * NW + (lane & (NW - 1))];
        // one block, with the two wait states between a write and its read by lane moves written out
#define CCTAMD_SCAN(N)                                                                           \
    "s_nop 0\n\t"                                                                                \
    "v_add_u32_dpp %0, %0, %0 row_shr:" #N " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"         \
    "v_add_u32_dpp %1, %1, %1 row_shr:" #N " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
        asm volatile("s_nop 0\n\t" CCTAMD_SCAN(1) CCTAMD_SCAN(2) CCTAMD_SCAN(4) "s_nop 1" : "+v"(count), "+v"(cost));
#undef CCTAMD_SCAN
        static_assert(NW <= 8, "tallies of a round within a scan of eight lanes");
        const int before = __builtin_amdgcn_readlane(count, wave) - own;
        if (order != 0) {
            const int at = n.far + (before & 0xffff) + lane_rank(far);
            L.far[at] = cl << (bits + 1) | (order & ((1 << bits) - 1)) << 1 | large;
            L.start[at] = n.cost + __builtin_amdgcn_readlane(cost, wave) - __builtin_amdgcn_readlane(upto, kWave - 1) +
                          upto - (order >> bits);
        } else if (valid) {
            put(n.near + (before >> 16) + lane_rank(other));
        }
        const int all = __builtin_amdgcn_readlane(count, NW - 1);
        n.far += all & 0xffff;
        n.near += all >> 16;
        n.cost += __builtin_amdgcn_readlane(cost, NW - 1);
    };
    const int nlarge = (w.tile_count + kParts - 1) / kParts;
    const int l = base + wave * kWave + lane;
    round(0, l < nlarge, w.tile_start / kParts + l, fs.geo_large, 1,
          [&](int at) { L.close[at] = (unsigned short)(l - base); });
    __syncthreads();
    const int parts = kParts * n.near;
    n.near = 0;
#pragma unroll 1
    for (int r = 0; r * FarLists<NW>::kRound < parts; ++r) {
        const int j = (r * NW + wave) * kWave + lane;
        const int part = j < parts ? (base + L.close[j / kParts]) * kParts + j % kParts : w.tile_count;
        const int cl = w.tile_start + part;
        round(r + 1, part < w.tile_count, cl, fs.geo, 0, [&](int at) { L.near[at] = cl; });
    }
    __syncthreads();
    return n;
}

// Read-only memory: wave-uniform addresses are read by scalar loads.
typedef const __attribute__((address_space(4))) double* ConstDoubles;

__device__ __forceinline__ ConstDoubles const_doubles(const double* p) { return (ConstDoubles)p; }

// Waits for this wave's scalar (and LDS) loads; what follows stays behind it.
__device__ __forceinline__ void loads_done() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
}

// An address whose scalar loads are not joined with those at others (a joined load would be
// waited for with the part that is used first).
__device__ __forceinline__ ConstDoubles apart(ConstDoubles p) {
    asm volatile("" : "+s"(p));
    return p;
}

// One (n, m) of the series at one point.  Record I (0 or 1) of the two that a 16-lane row
// holds, lane i with double i of them; each coefficient reaches the row's lanes through the
// row-broadcast DPP control of the FP64 multiply-add that uses it.  `rec` is only ever
// written by loads (the DPP hazard, see row_bcast).
template <int I>
__device__ __forceinline__ void far_term(double rec, double Z, double rho, double& t, double& u, double& c0, double& c1,
                                         double& c2, double& s0, double& s1, double& s2) {
    double tn;
    asm volatile(
        "v_mul_f64 %0, %10, %7\n\t"
        "v_fmac_f64_dpp %1, %9, %7 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %9, %7 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %9, %7 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %9, %8 row_newbcast:%18 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %4, %9, %7 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %5, %9, %7 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %6, %9, %7 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
        "v_mul_f64 %8, %11, %7"
        : "=&v"(tn), "+v"(c0), "+v"(c1), "+v"(c2), "+v"(s0), "+v"(s1), "+v"(s2), "+v"(t), "+v"(u)
        : "v"(rec), "v"(Z), "v"(rho), "i"(8 * I), "i"(8 * I + 1), "i"(8 * I + 2), "i"(8 * I + 3), "i"(8 * I + 4),
          "i"(8 * I + 5), "i"(8 * I + 6));
    t = tn;
}

// Adds units u0 .. u1 - 1 of the series of a cluster (wave-uniform) at the lane's PL points: rows m
// of the unit's number (LR = 1), or row 4 u + i in the wave's row i of lanes (LR = 4).  9 FP64
// instructions per (n, m) and point.
// The coefficients of a cluster (up to 46 KB) are read once per block and stage, from L2 at
// best, and a term uses them up quickly: with scalar loads, which a wave can only wait for all
// at once, the AG-CCT section's FP64 stage spent two thirds of its time waiting.  Vector loads
// of 16 doubles (two records) return in order; those of the two blocks after the one in use are on
// their way, across the ends of rows too.
template <int Q, int PL, int LR>
__device__ __forceinline__ void far_rows(ConstDoubles geo, const double* __restrict__ coef, int N, int u0, int u1,
                                         const double (&px)[PL], const double (&py)[PL], const double (&pz)[PL],
                                         double (&ax)[PL], double (&ay)[PL], double (&az)[PL]) {
    const int lrow = LR == 1 ? 0 : (int)(threadIdx.x >> 4) & 3;
    const double* lanes = coef + (threadIdx.x & 15);
    const auto unit = [&](int u) {  // this lane's first record of a unit
        return LR == 1 ? lanes + far_row(Q, u) * kFarRec
                       : lanes + (far_row(Q, 4 * u) + lrow * 4 * (Q - u)) * kFarRec;
    };
    // loads of the next block in the order of use; past the last one it is loaded again
    int fu = u0, fk = far_unit_blocks<LR>(N, u0);
    const double* next = unit(u0);
    const auto fetch = [&](double& p, double& q) {
        p = next[0];
        q = next[16];
        if (--fk > 0) {
            next += 32;
        } else if (fu + 1 < u1) {
            next = unit(++fu);
            fk = far_unit_blocks<LR>(N, fu);
        }
    };
    double a0, a1, b0, b1, d0, d1;
    fetch(a0, a1);
    fetch(b0, b1);

    double Z[PL], rho[PL], ri[PL], wc[PL], ws[PL], sc[PL], ss[PL];
    {
        const double gx = geo[0], gy = geo[1], gz = geo[2], inv = geo[3];
        double bc[PL], bs[PL];
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const double x = (px[j] - gx) * inv, y = (py[j] - gy) * inv, z = (pz[j] - gz) * inv;
            const double r2 = x * x + y * y + z * z;
            const double h = __builtin_amdgcn_rsq(r2);  // refined as in rsqrt_f64
            const double e = __builtin_fma(-r2 * h, h, 1.0);
            ri[j] = __builtin_fma(h * e, __builtin_fma(e, 0.375, 0.5), h);
            rho[j] = ri[j] * ri[j];
            Z[j] = z * rho[j];
            sc[j] = bc[j] = x * rho[j];
            ss[j] = bs[j] = y * rho[j];
            wc[j] = 1.0;
            ws[j] = 0.0;
        }
        const auto times = [](double& c, double& s, double bc, double bs) {
            const double t = c * bc - s * bs;
            s = c * bs + s * bc;
            c = t;
        };
        if constexpr (LR == 4) {  // (X + iY)^lrow, and the step (X + iY)^4
#pragma unroll
            for (int j = 0; j < PL; ++j) {
                double c2 = sc[j], s2 = ss[j];
                times(c2, s2, sc[j], ss[j]);
                wc[j] = lrow & 1 ? sc[j] : 1.0;
                ws[j] = lrow & 1 ? ss[j] : 0.0;
                double c = wc[j], s = ws[j];
                times(c, s, c2, s2);
                wc[j] = lrow & 2 ? c : wc[j];
                ws[j] = lrow & 2 ? s : ws[j];
                times(c2, s2, c2, s2);
                sc[j] = bc[j] = c2;
                ss[j] = bs[j] = s2;
            }
        }
#pragma unroll 1
        for (int bits = u0; bits; bits >>= 1) {  // times the step's power u0
            if (bits & 1) {
#pragma unroll
                for (int j = 0; j < PL; ++j) times(wc[j], ws[j], bc[j], bs[j]);
            }
#pragma unroll
            for (int j = 0; j < PL; ++j) {
                const double c = bc[j], s = bs[j];
                bc[j] = c * c - s * s;
                bs[j] = 2.0 * c * s;
            }
        }
    }
    double t[PL], u[PL], c0[PL], c1[PL], c2[PL], s0[PL], s1[PL], s2[PL];
    const auto begin = [&]() {
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            t[j] = ri[j];
            u[j] = c0[j] = c1[j] = c2[j] = s0[j] = s1[j] = s2[j] = 0.0;
        }
    };
    begin();
    int at = u0, left = far_unit_blocks<LR>(N, u0);
    const auto block = [&](double p, double q) {  // four records, two per register; true after the last row
#pragma unroll
        for (int j = 0; j < PL; ++j)
            far_term<0>(p, Z[j], rho[j], t[j], u[j], c0[j], c1[j], c2[j], s0[j], s1[j], s2[j]);
#pragma unroll
        for (int j = 0; j < PL; ++j)
            far_term<1>(p, Z[j], rho[j], t[j], u[j], c0[j], c1[j], c2[j], s0[j], s1[j], s2[j]);
#pragma unroll
        for (int j = 0; j < PL; ++j)
            far_term<0>(q, Z[j], rho[j], t[j], u[j], c0[j], c1[j], c2[j], s0[j], s1[j], s2[j]);
#pragma unroll
        for (int j = 0; j < PL; ++j)
            far_term<1>(q, Z[j], rho[j], t[j], u[j], c0[j], c1[j], c2[j], s0[j], s1[j], s2[j]);
        if (--left > 0) return false;
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            ax[j] = __builtin_fma(wc[j], c0[j], __builtin_fma(ws[j], s0[j], ax[j]));
            ay[j] = __builtin_fma(wc[j], c1[j], __builtin_fma(ws[j], s1[j], ay[j]));
            az[j] = __builtin_fma(wc[j], c2[j], __builtin_fma(ws[j], s2[j], az[j]));
            const double c = wc[j] * sc[j] - ws[j] * ss[j];
            ws[j] = wc[j] * ss[j] + ws[j] * sc[j];
            wc[j] = c;
        }
        if (++at == u1) return true;
        left = far_unit_blocks<LR>(N, at);
        begin();
        return false;
    };
#pragma unroll 1
    for (;;) {
        fetch(d0, d1);
        if (block(a0, a1)) break;
        fetch(a0, a1);
        if (block(b0, b1)) break;
        fetch(b0, b1);
        if (block(d0, d1)) break;
    }
}

// Share `me` of `all` equal shares of a block's series, by cost: a wave takes a stretch of the
// rows of the whole list, so that every wave of the block has as much to do to within a row, and
// starts few series (those of its stretch).  Dealt out by series, or by eighths of one where there
// were few, waves had two or three pieces of very different lengths, and each piece began with
// powers of X + iY: 4,096 protons in the gantry spent 37 us of a stage here, now 18; a stage of 512
// in the AG-CCT section (FP64, orders up to 31) took 49.8 us, now 44.5.
template <int Q, int LR, int NW, int PL>
__device__ __forceinline__ void far_share(const FarLists<NW>& L, const FarCounts& n, const FarSet& fs, int me, int all, int lane,
                                          const double (&px)[PL], const double (&py)[PL], const double (&pz)[PL],
                                          double (&ax)[PL], double (&ay)[PL], double (&az)[PL]) {
    constexpr int bits = far_order_bits(Q);
    const int nfar = n.far;
    const int from = (int)((int64_t)n.cost * me / all), to = (int)((int64_t)n.cost * (me + 1) / all);
    if (from == to) return;
    int e = -1;  // the last series that starts at or before `from`
    for (int k = 0; k < nfar; k += kWave) {
        const bool before = k + lane < nfar && L.start[k + lane] <= from;
        e += __popcll(__ballot(before));
    }
    for (; e < nfar; ++e) {
        const int at = __builtin_amdgcn_readfirstlane(L.start[e]);
        if (at >= to) break;
        const int entry = __builtin_amdgcn_readfirstlane(L.far[e]);
        const int N = entry >> 1 & ((1 << bits) - 1);
        const bool is = lane < far_units<LR>(N);
        const int start = far_unit_start<LR>(N, lane);
        const int u0 = __popcll(__ballot(is && start < from - at)), u1 = __popcll(__ballot(is && start < to - at));
        if (u0 == u1) continue;
        const bool large = entry & 1;
        const int64_t cl = entry >> (bits + 1);
        far_rows<Q, PL, LR>(const_doubles((large ? fs.geo_large : fs.geo) + cl * kFarGeo),
                            (large ? fs.coef_large : fs.coef) + cl * far_records(Q) * kFarRec, N, u0, u1, px, py, pz,
                            ax, ay, az);
    }
}

}  // namespace cctamd_detail
