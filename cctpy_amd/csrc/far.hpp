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
// solid harmonics), built once per segment set.  Cut at order N the series is off by about
// (E / |q - c|)^N of the cluster's sum of |terms|.  A block takes a large cluster's
// series where the large one is far enough, else the series of those of its four parts that
// are, and sums the other parts' segments one by one.
//
// Orders per distance (FarOrders): the smallest N whose cut lies below the rounding of the
// sum it replaces.  Measured against an extended-precision sum over random segments in a
// ball, relative to the sum of |terms|: ratio 3.0, N = 31: 8e-17; 3.3, 28: 1.2e-16; 4.0, 24:
// 2.2e-16; 6.0, 20: 1e-17; 10, 15: 5e-17.  The FP32 path cuts at 1e-10 to 1e-11 (its own
// terms are rounded at 6e-8) and evaluates the series in FP64.
#pragma once

#include "common.hpp"

namespace cctamd_detail {

constexpr int kSmallTiles = 16;           // tiles of a small cluster
constexpr int kParts = 4;                 // small clusters of a large one
constexpr int kFarGeo = 8;                // doubles per cluster: centre, 1 / E, E, 0, 0, 0
constexpr int kFarRec = 8;                // doubles per record: beta_c xyz, beta_s xyz, -kappa, 0
constexpr int kFarQ64 = 8, kFarQ32 = 5;   // highest order + 1 = 4 Q: 32 on the FP64 path, 20 on the FP32 path

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
    static constexpr int n = 9;
    static constexpr double ratio[n] = {3.0, 3.4, 4.2, 6.0, 8.0, 12.0, 20.0, 40.0, 100.0};
    static constexpr int order[n] = {31, 28, 24, 19, 17, 14, 12, 10, 8};
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

// Order of the series that serves a cluster for a block, 0 if the cluster is too close (its
// segments are then summed one by one).  Every wave and workgroup of a block gets the same
// answer: the same operations on the same values, each rounded by itself.
#pragma clang fp contract(off)
template <bool F64>
__device__ __forceinline__ int far_order(const double* __restrict__ geo, const Ball& b) {
    const double dx = geo[0] - b.x, dy = geo[1] - b.y, dz = geo[2] - b.z;
    const double ratio = (__builtin_sqrt(dx * dx + dy * dy + dz * dz) - b.r) * geo[3];
    using T = FarOrders<F64>;
    int n = 0;
#pragma unroll
    for (int k = 0; k < T::n; ++k) n = ratio >= T::ratio[k] ? T::order[k] : n;
    return n;
}
#pragma clang fp contract(fast)

// Work lists of a workgroup for its point block, in LDS: the small clusters whose segments are
// summed one by one, and the clusters, small or large, that act through their series.  Every
// workgroup of a block makes the same lists; each takes its share of them (the tiles of the
// near clusters and the series are dealt out over all waves of the block's work items, so
// that the near part, a few percent of the segments, does not fall to a few of them).
template <int NW>
struct FarLists {
    static constexpr int kRound = kWave * NW;  // large clusters per round
    int near[kParts * kRound];                 // small cluster
    int far[kParts * kRound];                  // cluster << 6 | order << 1 | large
    unsigned short close[kRound];              // large clusters of the round that are not far
    alignas(16) int count[2][kParts * NW];
    int nnear, nfar;
};

__device__ __forceinline__ int lane_rank(uint64_t mask) {  // set bits below this lane
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Lists of the large clusters [base, base + kRound) of a work item's design (w.tile_start: its
// first small cluster, w.tile_count: its small clusters).
template <bool F64, int NW>
__device__ __forceinline__ void far_lists(FarLists<NW>& L, const FarSet& fs, const Work& w, const Ball& ball, int base,
                                          int wave, int lane) {
    const int nlarge = (w.tile_count + kParts - 1) / kParts;
    // sum of the counts of round r, all and those of the waves before this one
    const auto add = [&](int which, int r, int& mine, int& all) {
        const int4* c = reinterpret_cast<const int4*>(&L.count[which][r * NW]);
#pragma unroll
        for (int i = 0; i < NW / 4; ++i) {
            const int4 v = c[i];
            mine += (4 * i < wave ? v.x : 0) + (4 * i + 1 < wave ? v.y : 0) + (4 * i + 2 < wave ? v.z : 0) +
                    (4 * i + 3 < wave ? v.w : 0);
            all += v.x + v.y + v.z + v.w;
        }
    };
    int nfar, nclose;
    {
        const int l = base + wave * kWave + lane;
        const bool valid = l < nlarge;
        const int cl = w.tile_start / kParts + (valid ? l : 0);
        const int order = far_order<F64>(fs.geo_large + (int64_t)cl * kFarGeo, ball);
        const uint64_t far = __ballot(valid && order != 0), close = __ballot(valid && order == 0);
        if (lane == 0) {
            L.count[0][wave] = __popcll(far);
            L.count[1][wave] = __popcll(close);
        }
        __syncthreads();
        int f = 0, c = 0;
        nfar = nclose = 0;
        add(0, 0, f, nfar);
        add(1, 0, c, nclose);
        if (valid && order != 0) L.far[f + lane_rank(far)] = cl << 6 | order << 1 | 1;
        if (valid && order == 0) L.close[c + lane_rank(close)] = (unsigned short)(l - base);
        __syncthreads();
    }
    int order[kParts], cl[kParts];
    uint64_t far[kParts], near[kParts];
    const int rounds = (kParts * nclose + FarLists<NW>::kRound - 1) / FarLists<NW>::kRound;
#pragma unroll
    for (int r = 0; r < kParts; ++r) {
        far[r] = near[r] = 0;
        if (r >= rounds) continue;
        const int j = (r * NW + wave) * kWave + lane;
        const int part = j < kParts * nclose ? (base + L.close[j / kParts]) * kParts + j % kParts : 0;
        const bool valid = j < kParts * nclose && part < w.tile_count;
        cl[r] = w.tile_start + (valid ? part : 0);
        order[r] = far_order<F64>(fs.geo + (int64_t)cl[r] * kFarGeo, ball);
        far[r] = __ballot(valid && order[r] != 0);
        near[r] = __ballot(valid && order[r] == 0);
        if (lane == 0) {
            L.count[0][r * NW + wave] = __popcll(far[r]);
            L.count[1][r * NW + wave] = __popcll(near[r]);
        }
    }
    __syncthreads();
    int nnear = 0;
    const uint64_t me = 1ull << lane;
#pragma unroll
    for (int r = 0; r < kParts; ++r) {
        if (r >= rounds) continue;
        int f = nfar, n = nnear;
        add(0, r, f, nfar);
        add(1, r, n, nnear);
        if (far[r] & me) L.far[f + lane_rank(far[r])] = cl[r] << 6 | order[r] << 1;
        if (near[r] & me) L.near[n + lane_rank(near[r])] = cl[r];
    }
    if (wave == 0 && lane == 0) {
        L.nnear = nnear;
        L.nfar = nfar;
    }
    __syncthreads();
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

constexpr int kFarPad = 16;  // records that may be read past the last one

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

// Adds the series of a cluster (wave-uniform) at the lane's PL points: rows m = a0, a0 + step, ...
// and b0, b0 + step, ... up to order N (a0, b0 < step, step a power of two), which may differ
// between the 16-lane rows of the wave.  Waves or rows of lanes share a cluster by their a0
// and b0; pairing row w with row step - 1 - w gives all of them about as many terms (row m has
// N - m + 1).  9 FP64 instructions per (n, m) and point.
// The coefficients of a cluster (up to 35 KB) are read once per block and stage, from L2 at
// best, and a term uses them up quickly: with scalar loads, which a wave can only wait for all
// at once, the AG-CCT section's FP64 stage spent two thirds of its time waiting.  Vector loads
// of 16 doubles (two records) return in order, and three pairs of them are on their way.
template <int Q, int PL>
__device__ __forceinline__ void far_series(ConstDoubles geo, const double* __restrict__ coef, int N, int a0, int b0,
                                           int step, const double (&px)[PL], const double (&py)[PL],
                                           const double (&pz)[PL], double (&ax)[PL], double (&ay)[PL],
                                           double (&az)[PL]) {
    double X[PL], Y[PL], Z[PL], rho[PL], ri[PL], ac[PL], as[PL], bc[PL], bs[PL], sc[PL], ss[PL];
    const double gx = geo[0], gy = geo[1], gz = geo[2], inv = geo[3];
    coef += threadIdx.x & 15;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const double x = (px[j] - gx) * inv, y = (py[j] - gy) * inv, z = (pz[j] - gz) * inv;
        const double r2 = x * x + y * y + z * z;
        const double h = __builtin_amdgcn_rsq(r2);  // refined as in rsqrt_f64
        const double e = __builtin_fma(-r2 * h, h, 1.0);
        ri[j] = __builtin_fma(h * e, __builtin_fma(e, 0.375, 0.5), h);
        rho[j] = ri[j] * ri[j];
        X[j] = x * rho[j];
        Y[j] = y * rho[j];
        Z[j] = z * rho[j];
        ac[j] = bc[j] = 1.0;
        as[j] = bs[j] = 0.0;
        sc[j] = X[j];
        ss[j] = Y[j];
    }
#pragma unroll 1
    for (int bit = 1; bit < step; bit <<= 1) {  // (X + iY)^a0, ^b0 and, at the end, ^step
        const bool ua = (a0 & bit) != 0, ub = (b0 & bit) != 0;
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const double c = sc[j], s = ss[j];
            if (ua) {
                const double t = ac[j] * c - as[j] * s;
                as[j] = ac[j] * s + as[j] * c;
                ac[j] = t;
            }
            if (ub) {
                const double t = bc[j] * c - bs[j] * s;
                bs[j] = bc[j] * s + bs[j] * c;
                bc[j] = t;
            }
            sc[j] = c * c - s * s;
            ss[j] = 2.0 * c * s;
        }
    }
    const auto row = [&](int m, const double (&wc)[PL], const double (&ws)[PL]) {
        const double* rec = coef + (int64_t)far_row(Q, m) * kFarRec;
        double t[PL], u[PL], c0[PL], c1[PL], c2[PL], s0[PL], s1[PL], s2[PL];
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            t[j] = ri[j];
            u[j] = c0[j] = c1[j] = c2[j] = s0[j] = s1[j] = s2[j] = 0.0;
        }
        const auto four = [&](double p, double q) {  // four records, two per register
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
        };
        // past the row's end the next row's records are loaded and not used (kFarPad follow the array)
        double p0 = rec[0], p1 = rec[16], q0 = rec[32], q1 = rec[48], r0, r1;
#pragma unroll 1
        for (int n = m;;) {
            r0 = rec[64];
            r1 = rec[80];
            four(p0, p1);
            if ((n += 4) > N) break;
            p0 = rec[96];
            p1 = rec[112];
            four(q0, q1);
            if ((n += 4) > N) break;
            q0 = rec[128];
            q1 = rec[144];
            four(r0, r1);
            if ((n += 4) > N) break;
            rec += 96;
        }
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            ax[j] = __builtin_fma(wc[j], c0[j], __builtin_fma(ws[j], s0[j], ax[j]));
            ay[j] = __builtin_fma(wc[j], c1[j], __builtin_fma(ws[j], s1[j], ay[j]));
            az[j] = __builtin_fma(wc[j], c2[j], __builtin_fma(ws[j], s2[j], az[j]));
        }
    };
    const auto ahead = [&](double (&wc)[PL], double (&ws)[PL]) {
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const double t = wc[j] * sc[j] - ws[j] * ss[j];
            ws[j] = wc[j] * ss[j] + ws[j] * sc[j];
            wc[j] = t;
        }
    };
#pragma unroll 1
    for (int m = a0, m2 = b0; m <= N || m2 <= N; m += step, m2 += step) {
        if (m <= N) row(m, ac, as);
        if (m2 <= N) row(m2, bc, bs);
        ahead(ac, as);
        ahead(bc, bs);
    }
}

// The series of entry e of a block's list.
template <int Q, int NW, int PL>
__device__ __forceinline__ void far_entry(const FarLists<NW>& L, const FarSet& fs, int e, int a0, int b0, int step,
                                          const double (&px)[PL], const double (&py)[PL], const double (&pz)[PL],
                                          double (&ax)[PL], double (&ay)[PL], double (&az)[PL]) {
    const int entry = __builtin_amdgcn_readfirstlane(L.far[e]);
    const bool large = entry & 1;
    const int64_t cl = entry >> 6;
    far_series<Q, PL>(const_doubles((large ? fs.geo_large : fs.geo) + cl * kFarGeo),
                      (large ? fs.coef_large : fs.coef) + cl * far_records(Q) * kFarRec, entry >> 1 & 31, a0, b0, step,
                      px, py, pz, ax, ay, az);
}

}  // namespace cctamd_detail
