// Segment clusters and the coefficients of their far field (see far.hpp), built on the device
// once per segment set.  The segments of a design are ordered in units (consecutive rows: 1
// to 8 of them on the FP64 path, a 32-row tile on the FP32 path, whose near tiles keep their
// terms and their order): first along a Hilbert curve (keys here, sorted by the caller), then
// each stretch of kChunk units is split in halves across its longest side down to the small
// clusters (k_far_split).  The curve alone leaves clusters that straddle gaps between the
// windings: on the AG-CCT section its 512-segment clusters have a median radius of 42 mm and
// a 95th percentile of 82 mm, the splits 36 and 50 mm, and a block sums a third fewer terms.
// Then cluster balls, multipole moments of the vector potential and the coefficients of its
// curl.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "far.hpp"

namespace cctamd_detail {
namespace {

// Place of a cell along the 3-d Hilbert curve of 2^16 cells per side, by J. Skilling's
// transpose method (Programming the Hilbert curve, 2004).
__device__ inline uint64_t hilbert48(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t v[3] = {x, y, z};
    for (uint32_t q = 1u << 15; q > 1; q >>= 1) {
        const uint32_t p = q - 1;
        for (int i = 0; i < 3; ++i) {
            if (v[i] & q) {
                v[0] ^= p;
            } else {
                const uint32_t t = (v[0] ^ v[i]) & p;
                v[0] ^= t;
                v[i] ^= t;
            }
        }
    }
    v[1] ^= v[0];
    v[2] ^= v[1];
    uint32_t t = 0;
    for (uint32_t q = 1u << 15; q > 1; q >>= 1)
        if (v[2] & q) t ^= q - 1;
    uint64_t h = 0;
    for (int b = 15; b >= 0; --b)
        for (int i = 0; i < 3; ++i) h = (h << 1) | (((v[i] ^ t) >> b) & 1u);
    return h;
}

// Cells of 2^-10 m around the origin (+- 32 m): they only order the segments, farther ones
// share the outermost cells and just cluster worse.
__device__ inline uint32_t cell_of(double v) {
    const double c = __builtin_floor(v * 1024.0) + 32768.0;
    return c >= 0.0 ? (c <= 65535.0 ? (uint32_t)c : 65535u) : 0u;
}

__device__ inline bool carries(const double* __restrict__ row) {
    return row[0] != 0.0 || row[1] != 0.0 || row[2] != 0.0;
}

// Key of each unit: its design, then its place along the curve; units without current come
// last.  centre: the mean of the unit's current-carrying midpoints, FLT_MAX without any.
__global__ void k_far_keys(const double* __restrict__ seg64, int unit, const int64_t* __restrict__ unit_off,
                           int64_t nd, int64_t nunit, int64_t* __restrict__ key, float4* __restrict__ centre) {
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nunit) return;
    const double* r = seg64 + u * unit * 8;
    double c[3] = {0.0, 0.0, 0.0};
    int n = 0;
    for (int k = 0; k < unit; ++k, r += 8) {
        if (!carries(r)) continue;
        ++n;
        for (int i = 0; i < 3; ++i) c[i] += r[4 + i];
    }
    for (int i = 0; i < 3; ++i) c[i] /= n > 0 ? n : 1;
    const uint64_t h = n > 0 ? hilbert48(cell_of(c[0]), cell_of(c[1]), cell_of(c[2])) : 0xffffffffffffull;
    key[u] = (int64_t)(((uint64_t)find_design(unit_off, nd, u) << 48) | h);
    const auto f = [&](double v) {  // not above FLT_MAX, not a NaN
        return n > 0 && v < 3.0e38 ? (float)v : 3.402823466e38f;
    };
    centre[u] = make_float4(f(c[0]), f(c[1]), f(c[2]), 0.0f);
}

// Splits a stretch of kChunk units of one design into halves across the longest side of their
// bounding box, then each half, down to groups of `group` units (a power of two): every level
// finds the median of each group bit by bit on 16-bit places along the side (all groups at
// once) and moves the units to their half, in LDS.  Places past the design's units come last in
// every group.  One workgroup per stretch; sorting the groups instead took eight times as long.
constexpr int kChunk = 16384;
constexpr int kSplitWG = 1024;
constexpr int kPer = kChunk / kSplitWG;

__device__ inline unsigned ordered_bits(float v) {
    const unsigned b = __float_as_uint(v);
    return b & 0x80000000u ? ~b : b | 0x80000000u;
}
__device__ inline float from_ordered_bits(unsigned b) {
    return __uint_as_float(b & 0x80000000u ? b & 0x7fffffffu : ~b);
}

__global__ __launch_bounds__(kSplitWG) void k_far_split(int64_t* __restrict__ perm, const float4* __restrict__ centre,
                                                        const int64_t* __restrict__ unit_off,
                                                        const int64_t* __restrict__ chunk_off, int64_t nd, int group) {
    constexpr int kMaxGroups = kChunk / 32;  // groups of a level: of 32 units at least
    __shared__ uint16_t id[2][kChunk];
    __shared__ unsigned box[6][kMaxGroups];
    __shared__ int count[kMaxGroups], less[kMaxGroups], same[kMaxGroups];  // less, same: by run of `width` places
    const int64_t d = find_design(chunk_off, nd, blockIdx.x);
    const int64_t first = unit_off[d] + ((int64_t)blockIdx.x - chunk_off[d]) * kChunk;
    const int64_t left = unit_off[d + 1] - first;
    const int n = left < kChunk ? (int)left : kChunk;
    const int lane = threadIdx.x & (kWave - 1);
    int from = 0;
    for (int e = threadIdx.x; e < kChunk; e += kSplitWG) id[0][e] = (uint16_t)e;
    __syncthreads();
    for (int size = kChunk; size > group; size >>= 1) {
        if (size / 2 >= n) continue;  // uniform: nothing in the second half
        const int ng = kChunk / size;
        // place e = threadIdx.x + i kSplitWG: a wave's 64 places are `kWave / width` runs of one group each
        const int width = size < kWave ? size : kWave;
        const uint64_t run = (width == kWave ? ~0ull : ((1ull << width) - 1)) << (lane / width * width);
        for (int i = threadIdx.x; i < 6 * ng; i += kSplitWG) box[i / ng][i % ng] = i / ng < 3 ? 0xffffffffu : 0u;
        __syncthreads();
        float4 c[kPer];
        int what[kPer];  // 0: with current, 1: without, 2: no unit
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int e = threadIdx.x + i * kSplitWG, u = id[from][e];
            what[i] = 2;
            unsigned lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
            if (u < n) {
                c[i] = centre[perm[first + u]];
                what[i] = c[i].x < 3.0e38f && c[i].y < 3.0e38f && c[i].z < 3.0e38f ? 0 : 1;
                if (what[i] == 0) {
                    lo[0] = hi[0] = ordered_bits(c[i].x);
                    lo[1] = hi[1] = ordered_bits(c[i].y);
                    lo[2] = hi[2] = ordered_bits(c[i].z);
                }
            }
            for (int off = 1; off < width; off <<= 1)
                for (int k = 0; k < 3; ++k) {
                    const unsigned a = __shfl_xor(lo[k], off), b = __shfl_xor(hi[k], off);
                    lo[k] = a < lo[k] ? a : lo[k];
                    hi[k] = b > hi[k] ? b : hi[k];
                }
            if (lane % width == 0)
                for (int k = 0; k < 3; ++k) {
                    atomicMin(&box[k][e / size], lo[k]);
                    atomicMax(&box[3 + k][e / size], hi[k]);
                }
        }
        __syncthreads();
        unsigned key[kPer], cut[kPer];
        int want[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int g = (threadIdx.x + i * kSplitWG) / size;
            float base = 0.0f, side = 0.0f, v = 0.0f;
            for (int k = 0; k < 3; ++k) {
                const unsigned lo = box[k][g], hi = box[3 + k][g];
                const float l = from_ordered_bits(lo), w = hi >= lo ? from_ordered_bits(hi) - l : 0.0f;
                if (w > side) {
                    side = w;
                    base = l;
                    v = k == 0 ? c[i].x : k == 1 ? c[i].y : c[i].z;
                }
            }
            key[i] = what[i] == 2 ? 65535u : what[i] == 1 ? 65534u : side > 0.0f ? (unsigned)((v - base) / side * 65533.0f) : 0u;
            cut[i] = 0;
            want[i] = size / 2;  // the want-th smallest of those that agree with `cut` so far
        }
        for (int bit = 15; bit >= 0; --bit) {
            for (int g = threadIdx.x; g < ng; g += kSplitWG) count[g] = 0;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const uint64_t m = __ballot((key[i] ^ cut[i]) >> bit == 0) & run;
                if (lane % width == 0) atomicAdd(&count[(threadIdx.x + i * kSplitWG) / size], __popcll(m));
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const int below = count[(threadIdx.x + i * kSplitWG) / size];
                if (below < want[i]) {
                    want[i] -= below;
                    cut[i] |= 1u << bit;
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const uint64_t ml = __ballot(key[i] < cut[i]) & run, ms = __ballot(key[i] == cut[i]) & run;
            if (lane % width == 0) {
                less[(threadIdx.x + i * kSplitWG) / width] = __popcll(ml);
                same[(threadIdx.x + i * kSplitWG) / width] = __popcll(ms);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int e = threadIdx.x + i * kSplitWG, r0 = e / size * (size / width);
            int l = 0, s = 0;  // smaller and equal ones before this place in its group
            for (int r = r0; r < e / width; ++r) {
                l += less[r];
                s += same[r];
            }
            const uint64_t low = run & ((1ull << lane) - 1);
            l += __popcll(__ballot(key[i] < cut[i]) & low);
            s += __popcll(__ballot(key[i] == cut[i]) & low);
            const int taken = s < want[i] ? s : want[i];  // equal ones that go to the first half
            int to;
            if (key[i] < cut[i])
                to = l;
            else if (key[i] == cut[i] && s < want[i])
                to = size / 2 - want[i] + s;
            else
                to = size / 2 + (e % size - l - taken);
            id[from ^ 1][e / size * size + to] = id[from][e];
        }
        __syncthreads();
        from ^= 1;
    }
    int64_t to[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kSplitWG;
        to[i] = e < n ? perm[first + id[from][e]] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kSplitWG;
        if (e < n) perm[first + e] = to[i];
    }
}

// The unit at each place of the clusters, -1 for none.
__device__ inline int64_t unit_at(const int64_t* __restrict__ perm, const int64_t* __restrict__ unit_off,
                                  const int64_t* __restrict__ cluster_off, int64_t nd, int64_t per_cluster,
                                  int64_t place) {
    const int64_t d = find_design(cluster_off, nd, place / per_cluster);
    const int64_t rank = place - cluster_off[d] * per_cluster;
    return rank < unit_off[d + 1] - unit_off[d] ? perm[unit_off[d] + rank] : -1;
}

// FP64 path: the rows in cluster order, packed to {kl, m} (48 bytes: a quarter less to read
// than seg64, three scalar loads for two rows instead of eight); pad rows in the places left over.
__global__ void k_far_rows(const double* __restrict__ seg64, const int64_t* __restrict__ perm, int unit,
                           const int64_t* __restrict__ unit_off, const int64_t* __restrict__ cluster_off, int64_t nd,
                           int64_t per_cluster, int64_t nrow, double* __restrict__ rows) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrow * 2) return;
    const int64_t row = i >> 1, half = i & 1;  // kl or m
    const int64_t u = unit_at(perm, unit_off, cluster_off, nd, per_cluster, row / unit);
    const double pad = half ? 1.0e3 : 0.0;
    double v[3] = {pad, pad, pad};
    if (u >= 0)
        for (int c = 0; c < 3; ++c) v[c] = seg64[(u * unit + row % unit) * 8 + 4 * half + c];
    for (int c = 0; c < 3; ++c) rows[i * 3 + c] = v[c];
}

// FP32 path: the tile at each place.
__global__ void k_far_tiles(const int64_t* __restrict__ perm, const int64_t* __restrict__ unit_off,
                            const int64_t* __restrict__ cluster_off, int64_t nd, int64_t per_cluster, int64_t nplace,
                            int32_t* __restrict__ tiles) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nplace) tiles[i] = (int32_t)unit_at(perm, unit_off, cluster_off, nd, per_cluster, i);
}

// Row i of cluster cl of ntile tiles, kl and m.
struct ClusterRow {
    const double *kl, *m;
};

__device__ inline bool cluster_row(const double* __restrict__ rows, const int32_t* __restrict__ tiles, int64_t cl,
                                   int ntile, int i, ClusterRow& r) {
    if (!tiles) {
        r.kl = rows + (cl * ntile * kTile + i) * 6;
        r.m = r.kl + 3;
    } else {
        const int32_t t = tiles[cl * ntile + i / kTile];
        if (t < 0) return false;
        r.kl = rows + ((int64_t)t * kTile + i % kTile) * 8;
        r.m = r.kl + 4;
    }
    return carries(r.kl);
}

constexpr int kFarWG = 256;

__device__ inline double wg_reduce(double v, double* lds, bool largest) {
    lds[threadIdx.x] = v;
    __syncthreads();
    for (int s = kFarWG / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            const double a = lds[threadIdx.x], b = lds[threadIdx.x + s];
            // a NaN stays: the comparison that fails keeps it
            lds[threadIdx.x] = largest ? (a >= b || a != a ? a : b) : (a <= b || a != a ? a : b);
        }
        __syncthreads();
    }
    const double r = lds[0];
    __syncthreads();
    return r;
}

// Centre (middle of the bounding box) and radius of each cluster's current-carrying midpoints.
// A cluster of one point gets a radius of 1 nm, one without current too (its series is zero).
__global__ __launch_bounds__(kFarWG) void k_far_balls(const double* __restrict__ rows, const int32_t* __restrict__ tiles,
                                                      int ntile, double* __restrict__ geo) {
    __shared__ double lds[kFarWG];
    const int64_t cl = blockIdx.x;
    const double inf = __builtin_huge_val();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    for (int i = threadIdx.x; i < ntile * kTile; i += kFarWG) {
        ClusterRow r;
        if (!cluster_row(rows, tiles, cl, ntile, i, r)) continue;
        for (int c = 0; c < 3; ++c) {
            const double v = r.m[c];
            lo[c] = v <= lo[c] || v != v ? v : lo[c];
            hi[c] = v >= hi[c] || v != v ? v : hi[c];
        }
    }
    double ctr[3];
    for (int c = 0; c < 3; ++c) {
        const double a = wg_reduce(lo[c], lds, false), b = wg_reduce(hi[c], lds, true);
        ctr[c] = a > b ? 0.0 : 0.5 * (a + b);
    }
    double far2 = 0.0;
    for (int i = threadIdx.x; i < ntile * kTile; i += kFarWG) {
        ClusterRow r;
        if (!cluster_row(rows, tiles, cl, ntile, i, r)) continue;
        const double dx = r.m[0] - ctr[0], dy = r.m[1] - ctr[1], dz = r.m[2] - ctr[2];
        const double d2 = dx * dx + dy * dy + dz * dz;
        far2 = d2 >= far2 || d2 != d2 ? d2 : far2;
    }
    far2 = wg_reduce(far2, lds, true);
    if (threadIdx.x == 0) {
        double e = __builtin_sqrt(far2);
        e = e < 1.0e-9 ? 1.0e-9 : e;
        double* g = geo + cl * kFarGeo;
        g[0] = ctr[0];
        g[1] = ctr[1];
        g[2] = ctr[2];
        g[3] = 1.0 / e;  // 0 or NaN for a cluster that is not finite: never far
        g[4] = e;
        g[5] = g[6] = g[7] = 0.0;
    }
}

// Moments of the vector potential, sum over the cluster's rows of kl R_n^m((m - c) / E) with
// the regular solid harmonics R_n^m = r^n P_n^m e^{i m phi} / (n + m)!:
//   R_m^m = (x + iy)^m / (2^m m!),  (n + 1 - m)(n + 1 + m) R_{n+1} = (2n + 1) z R_n - r^2 R_{n-1}.
// One wave per (cluster, m): its lanes stride the rows, kFarChunk orders at a time in
// registers; the lanes' sums are added in a fixed order through LDS (kFarHalf orders at a
// time), which costs 150 instructions per chunk where shuffles cost 1,400.
constexpr int kFarChunk = 8, kFarHalf = 4;
constexpr int kMomWaves = 4;

// The recurrence's factors (2n + 1) / q and 1 / q, q = (n + 1 - m)(n + 1 + m), by n - m, for every m.
struct RegularFactors {
    static constexpr int kTop = 4 * kFarQ64, kLen = kTop + kFarChunk;
    double f[kTop][kLen][2];
};
constexpr RegularFactors regular_factors() {
    RegularFactors t{};
    for (int m = 0; m < RegularFactors::kTop; ++m)
        for (int k = 0; k < RegularFactors::kLen; ++k) {
            t.f[m][k][1] = 1.0 / ((double)(k + 1) * (double)(k + 1 + 2 * m));
            t.f[m][k][0] = (2 * (m + k) + 1) * t.f[m][k][1];
        }
    return t;
}
__constant__ RegularFactors kRegular = regular_factors();

__global__ __launch_bounds__(kWave * kMomWaves) void k_far_moments(const double* __restrict__ rows,
                                                                   const int32_t* __restrict__ tiles, int ntile, int q,
                                                                   const double* __restrict__ geo,
                                                                   double* __restrict__ mom) {
    __shared__ double lds[kMomWaves][kFarHalf * 6][kWave + 1];
    const int64_t cl = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int top = 4 * q - 2;  // highest order of the potential
    const int m = __builtin_amdgcn_readfirstlane(blockIdx.y * kMomWaves + wave);
    if (m > top) return;  // whole waves; no barrier below
    double(*mine)[kWave + 1] = lds[wave];
    const double* g = geo + cl * kFarGeo;
    const double inv = g[3];
    double f = 1.0;
    for (int k = 1; k <= m; ++k) f /= 2.0 * k;
    double* out = mom + (cl * far_records(q) + far_row(q, m)) * 6;
    const double(*fac)[2] = kRegular.f[m];  // wave-uniform: scalar loads
#pragma unroll 1
    for (int n0 = m; n0 <= top; n0 += kFarChunk) {
        double acc[kFarChunk][6];
#pragma unroll
        for (int k = 0; k < kFarChunk; ++k)
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[k][c] = 0.0;
#pragma unroll 1
        for (int i = lane; i < ntile * kTile; i += kWave) {  // the same number of rounds in every lane
            ClusterRow r;
            const bool live = cluster_row(rows, tiles, cl, ntile, i, r);
            const double x = live ? (r.m[0] - g[0]) * inv : 0.0, y = live ? (r.m[1] - g[1]) * inv : 0.0;
            const double z = live ? (r.m[2] - g[2]) * inv : 0.0;
            const double r2 = x * x + y * y + z * z;
            double pc = live ? f : 0.0, ps = 0.0, bc = x, bs = y;  // f (x + iy)^m by squares
            for (int k = m; k != 0; k >>= 1) {
                if (k & 1) {
                    const double t = pc * bc - ps * bs;
                    ps = pc * bs + ps * bc;
                    pc = t;
                }
                const double t = bc * bc - bs * bs;
                bs = 2.0 * bc * bs;
                bc = t;
            }
            double cur = 1.0, old = 0.0;  // R_n over R_m^m
            for (int n = m; n < n0; ++n) {
                const double nx = fac[n - m][0] * (z * cur) - fac[n - m][1] * (r2 * old);
                old = cur;
                cur = nx;
            }
            const double k0 = live ? r.kl[0] : 0.0, k1 = live ? r.kl[1] : 0.0, k2 = live ? r.kl[2] : 0.0;
            const double kc[3] = {k0 * pc, k1 * pc, k2 * pc}, ks[3] = {k0 * ps, k1 * ps, k2 * ps};
#pragma unroll
            for (int k = 0; k < kFarChunk; ++k) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    acc[k][c] = __builtin_fma(kc[c], cur, acc[k][c]);
                    acc[k][3 + c] = __builtin_fma(ks[c], cur, acc[k][3 + c]);
                }
                const double nx = fac[n0 + k - m][0] * (z * cur) - fac[n0 + k - m][1] * (r2 * old);
                old = cur;
                cur = nx;
            }
        }
#pragma unroll
        for (int h = 0; h < kFarChunk; h += kFarHalf) {
#pragma unroll
            for (int k = 0; k < kFarHalf; ++k)
#pragma unroll
                for (int c = 0; c < 6; ++c) mine[k * 6 + c][lane] = acc[h + k][c];
            __builtin_amdgcn_wave_barrier();
            const int v = lane >> 1;  // two lanes per value
            double s = 0.0;
            if (v < kFarHalf * 6)
                for (int i = 0; i < kWave / 2; ++i) s += mine[v][(lane & 1) * (kWave / 2) + i];
            s += __shfl_xor(s, 1);
            if (v < kFarHalf * 6 && (lane & 1) == 0 && n0 + h + v / 6 <= top) out[(n0 - m + h) * 6 + v] = s;
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// Coefficients of the field, B = curl A, order n from the potential's order n - 1:
//   d/dx, d/dy and d/dz of the exterior harmonic I_n^m are (I_{n+1}^{m-1} - I_{n+1}^{m+1}) / 2,
//   i (I_{n+1}^{m-1} + I_{n+1}^{m+1}) / 2 and -I_{n+1}^m  (I^{-1} = -conj I^1).
__global__ void k_far_coef(int q, int64_t nrec, const double* __restrict__ geo, const double* __restrict__ mom,
                           double* __restrict__ coef) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrec) return;
    const int per = far_records(q);
    const int64_t cl = i / per;
    const int rec = (int)(i % per), top = 4 * q - 1;
    int m = 0;
    while (m < top && far_row(q, m + 1) <= rec) ++m;
    const int n = m + rec - far_row(q, m);
    double* o = coef + i * kFarRec;
    for (int c = 0; c < kFarRec; ++c) o[c] = 0.0;
    if (n > top) return;
    if (n > 0) o[6] = -(double)(n * n - m * m) / (double)((2 * n + 1) * (2 * n - 1));
    if (n == 0) return;
    // a(k, c): coefficient of the potential's Re I_{n-1}^k (c < 3) or Im I_{n-1}^k (c >= 3)
    const double* base = mom + cl * per * 6;
    const auto a = [&](int k, int c) {
        if (k < 0 || k > n - 1 || (c >= 3 && k == 0)) return 0.0;
        const double v = base[(far_row(q, k) + (n - 1 - k)) * 6 + c];
        return k == 0 ? v : 2.0 * v;
    };
    const double lowc = m == 1 ? 1.0 : 0.5;  // Re I^0 has only its I^1 neighbour
    double dxc[3], dxs[3], dyc[3], dys[3], dzc[3], dzs[3];
    for (int c = 0; c < 3; ++c) {
        dxc[c] = -lowc * a(m - 1, c) + 0.5 * a(m + 1, c);
        dyc[c] = 0.5 * a(m - 1, 3 + c) + 0.5 * a(m + 1, 3 + c);
        dzc[c] = -a(m, c);
        dxs[c] = m == 0 ? 0.0 : -0.5 * a(m - 1, 3 + c) + 0.5 * a(m + 1, 3 + c);
        dys[c] = m == 0 ? 0.0 : -lowc * a(m - 1, c) - 0.5 * a(m + 1, c);
        dzs[c] = -a(m, 3 + c);
    }
    double s = geo[cl * kFarGeo + 3] * geo[cl * kFarGeo + 3];
    for (int k = 1; k <= n; ++k) s *= 2 * k - 1;
    o[0] = s * (dyc[2] - dzc[1]);
    o[1] = s * (dzc[0] - dxc[2]);
    o[2] = s * (dxc[1] - dyc[0]);
    o[3] = s * (dys[2] - dzs[1]);
    o[4] = s * (dzs[0] - dxs[2]);
    o[5] = s * (dxs[1] - dys[0]);
}

}  // namespace
}  // namespace cctamd_detail

using namespace cctamd_detail;

extern "C" {

int64_t cctamd_far_coef_doubles(int precision) {
    if (precision != 33 && precision != 64) return CCTAMD_EINVAL;
    return (int64_t)far_records(precision == 64 ? kFarQ64 : kFarQ32) * kFarRec;
}

int cctamd_far_keys(const double* seg64, int unit, const int64_t* unit_off, int64_t ndesign, int64_t nunit,
                    int64_t* key, float* centre, void* stream) {
    if (unit < 1 || unit > kTile || (unit & (unit - 1)) || ndesign <= 0 || ndesign > 0x7fff || nunit < 0)
        return CCTAMD_EINVAL;
    if (nunit == 0) return CCTAMD_OK;
    if (!seg64 || !unit_off || !key || !centre) return CCTAMD_EINVAL;
    const int64_t blocks = ceil_div(nunit, 256);
    if (blocks > 0x7fffffff) return CCTAMD_ERANGE;
    hipLaunchKernelGGL(k_far_keys, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, seg64, unit, unit_off,
                       ndesign, nunit, key, (float4*)centre);
    return hip_status(hipGetLastError());
}

int cctamd_far_build(int precision, const double* seg64, int unit, const float* centre, const int64_t* unit_off,
                     const int64_t* chunk_off, int64_t nchunk, const int64_t* cluster_off, int64_t ndesign,
                     int64_t ncluster, int64_t* perm, double* rows, int32_t* tiles, double* geo, double* geo_large,
                     double* mom, double* coef, double* coef_large, void* stream) {
    if ((precision != 33 && precision != 64) || ndesign <= 0 || ncluster < 0 || ncluster % kParts || nchunk < 0)
        return CCTAMD_EINVAL;
    if (precision == 33 ? unit != kTile : (unit < 1 || unit > 8 || (unit & (unit - 1)))) return CCTAMD_EINVAL;
    if (ncluster == 0) return CCTAMD_OK;
    if (!seg64 || !centre || !unit_off || !chunk_off || !cluster_off || !perm || !geo || !geo_large || !mom || !coef ||
        !coef_large || nchunk == 0)
        return CCTAMD_EINVAL;
    if (precision == 64 ? !rows : !tiles) return CCTAMD_EINVAL;
    const int q = precision == 64 ? kFarQ64 : kFarQ32;
    const int ntile = kSmallTiles;
    const int64_t places = ncluster * ntile, nrec = ncluster * far_records(q);
    if (places > 0x7fffffff || ceil_div(places * kTile * 2, 256) > 0x7fffffff || ceil_div(nrec, 256) > 0x7fffffff ||
        nchunk > 0x7fffffff)
        return CCTAMD_ERANGE;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_far_split, dim3((unsigned)nchunk), dim3(kSplitWG), 0, st, perm, (const float4*)centre,
                       unit_off, chunk_off, ndesign, ntile * kTile / unit);
    if (precision == 64)
        hipLaunchKernelGGL(k_far_rows, dim3((unsigned)ceil_div(places * kTile * 2, 256)), dim3(256), 0, st, seg64, perm,
                           unit, unit_off, cluster_off, ndesign, (int64_t)ntile * kTile / unit, places * kTile, rows);
    else
        hipLaunchKernelGGL(k_far_tiles, dim3((unsigned)ceil_div(places, 256)), dim3(256), 0, st, perm, unit_off,
                           cluster_off, ndesign, (int64_t)ntile, places, tiles);
    const double* src = precision == 64 ? rows : seg64;
    const int32_t* ids = precision == 64 ? nullptr : tiles;
    for (int large = 0; large < 2; ++large) {
        const int64_t nc = large ? ncluster / kParts : ncluster;
        const int nt = large ? kParts * kSmallTiles : ntile;
        double* g = large ? geo_large : geo;
        const int64_t nr = nc * far_records(q);
        hipLaunchKernelGGL(k_far_balls, dim3((unsigned)nc), dim3(kFarWG), 0, st, src, ids, nt, g);
        hipLaunchKernelGGL(k_far_moments, dim3((unsigned)nc, (unsigned)((4 * q - 1 + kMomWaves - 1) / kMomWaves)),
                           dim3(kWave * kMomWaves), 0, st, src, ids, nt, q, g, mom);
        hipLaunchKernelGGL(k_far_coef, dim3((unsigned)ceil_div(nr, 256)), dim3(256), 0, st, q, nr, g, mom,
                           large ? coef_large : coef);
    }
    return hip_status(hipGetLastError());
}

int64_t cctamd_far_plan(int64_t ndesign, const int64_t* design_ntile, const int64_t* design_npt,
                        const int64_t* design_cluster_off, const int64_t* design_pt_off, int ppl,
                        int64_t target_items, int32_t* work, int64_t* design_wbase, int32_t* design_nchunk) {
    if (ndesign <= 0 || !design_ntile || !design_npt || target_items <= 0) return CCTAMD_EINVAL;
    if (!valid_ppl(ppl)) return CCTAMD_EINVAL;
    const int64_t pb = pb_of(ppl);
    int64_t total = 0;
    for (int64_t d = 0; d < ndesign; ++d) {
        if (design_ntile[d] < 0 || design_npt[d] < 0) return CCTAMD_EINVAL;
        total += ceil_div(design_npt[d], pb) * ceil_div(design_ntile[d], kSmallTiles);
    }
    int64_t n = 0;
    for (int64_t d = 0; d < ndesign; ++d) {
        const int64_t nb = ceil_div(design_npt[d], pb), ns = ceil_div(design_ntile[d], kSmallTiles);
        // items in proportion to the clusters, at least one per point block and at most one per
        // tile (what an item deals in)
        int64_t nc = nb > 0 ? std::max<int64_t>(1, ns * target_items / std::max<int64_t>(total, 1)) : 0;
        nc = std::min(nc, std::max<int64_t>(design_ntile[d], nb > 0 ? 1 : 0));
        if (nc > kXcds) nc -= nc % kXcds;  // items that read the same rows share an XCD (as in cctamd_plan)
        if (work) {
            if (!design_cluster_off || !design_pt_off || !design_wbase || !design_nchunk) return CCTAMD_EINVAL;
            if (nc > 0x7fffffff) return CCTAMD_ERANGE;
            design_wbase[d] = n;
            design_nchunk[d] = (int32_t)nc;
            for (int64_t b = 0; b < nb && nc > 0; ++b) {
                for (int64_t c = 0; c < nc; ++c) {
                    const int64_t ps = design_pt_off[d] + b * pb;
                    const int64_t pc = std::min(pb, design_npt[d] - b * pb);
                    // cluster numbers are kept shifted by 6 bits (FarLists), their tiles in 31
                    if (ps + pc > 0x7fffffff || (design_cluster_off[d] + ns) > (0x7fffffff >> 6)) return CCTAMD_ERANGE;
                    int32_t* w = work + CCTAMD_WORK_INTS * (n + b * nc + c);
                    w[0] = (int32_t)d;
                    w[1] = (int32_t)ps;
                    w[2] = (int32_t)pc;
                    w[3] = (int32_t)design_cluster_off[d];
                    w[4] = (int32_t)ns;
                    w[5] = (int32_t)c;
                    w[6] = (int32_t)nc;
                    w[7] = (int32_t)b;
                }
            }
        }
        n += nb * nc;
    }
    return n;
}

}  // extern "C"
