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
// bounding box, then each half, down to groups of `group` units (a power of two).  Every level
// finds the median of each group bit by bit and moves the units to their half, in LDS, all
// groups at once; a thread holds kPer places of one group, so that a level of groups of up to
// 1,024 units needs no barrier for its counts.  Places past the design's units come last in
// every group.  One workgroup per stretch (0.23 ms; stretches of half the size take half of it but
// cost the design search 8 % of its tracking, their clusters being rounder only within them).
constexpr int kChunk = 16384;
constexpr int kSplitWG = 1024;
constexpr int kPer = kChunk / kSplitWG;
constexpr int kSplitBits = 11;  // resolution of a split along its side
constexpr unsigned kNoCurrent = 65534, kNoUnit = 65535;

__device__ inline unsigned ordered_bits(float v) {
    const unsigned b = __float_as_uint(v);
    return b & 0x80000000u ? ~b : b | 0x80000000u;
}
__device__ inline float from_ordered_bits(unsigned b) {
    return __uint_as_float(b & 0x80000000u ? b & 0x7fffffffu : ~b);
}

// Smallest and largest of three values over the `width` neighbouring lanes (a power of two).
__device__ inline void box_lanes(unsigned (&lo)[3], unsigned (&hi)[3], int width) {
    for (int off = 1; off < width; off <<= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const unsigned a = __shfl_xor(lo[k], off), b = __shfl_xor(hi[k], off);
            lo[k] = a < lo[k] ? a : lo[k];
            hi[k] = b > hi[k] ? b : hi[k];
        }
}

__global__ __launch_bounds__(kSplitWG) void k_far_split(int64_t* __restrict__ perm, const float4* __restrict__ centre,
                                                        const int64_t* __restrict__ unit_off,
                                                        const int64_t* __restrict__ chunk_off, int64_t nd, int group) {
    constexpr int kGroups = kChunk / (kWave * kPer);  // groups of more than a wave's places, at most
    __shared__ uint16_t xyz[3][kChunk];               // places in the stretch's box, by unit
    __shared__ uint16_t id[kChunk];
    __shared__ unsigned box[6][kGroups];
    __shared__ int count[2][kGroups], tot[2][kSplitWG / kWave];
    const int64_t d = find_design(chunk_off, nd, blockIdx.x);
    const int64_t first = unit_off[d] + ((int64_t)blockIdx.x - chunk_off[d]) * kChunk;
    const int64_t left = unit_off[d + 1] - first;
    const int n = left < kChunk ? (int)left : kChunk;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, e0 = tid * kPer;
    // the stretch's box (units with current), then every unit's place in it
    if (tid < 6) box[tid][0] = tid < 3 ? 0xffffffffu : 0u;
    __syncthreads();
    {
        unsigned lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
        for (int i = 0; i < kPer; ++i) {
            if (e0 + i >= n) break;
            const float4 c = centre[perm[first + e0 + i]];
            if (!(c.x < 3.0e38f && c.y < 3.0e38f && c.z < 3.0e38f)) continue;
            const unsigned v[3] = {ordered_bits(c.x), ordered_bits(c.y), ordered_bits(c.z)};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] = v[k] < lo[k] ? v[k] : lo[k];
                hi[k] = v[k] > hi[k] ? v[k] : hi[k];
            }
        }
        box_lanes(lo, hi, kWave);
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                atomicMin(&box[k][0], lo[k]);
                atomicMax(&box[3 + k][0], hi[k]);
            }
    }
    __syncthreads();
    {
        float base[3], side = 0.0f;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            base[k] = from_ordered_bits(box[k][0]);
            const float w = box[3 + k][0] >= box[k][0] ? from_ordered_bits(box[3 + k][0]) - base[k] : 0.0f;
            side = w > side ? w : side;
        }
        const float scale = side > 0.0f ? 65533.0f / side : 0.0f;
        for (int i = 0; i < kPer; ++i) {
            const int e = e0 + i;
            unsigned q[3] = {kNoUnit, kNoUnit, kNoUnit};
            if (e < n) {
                const float4 c = centre[perm[first + e]];
                const bool with = c.x < 3.0e38f && c.y < 3.0e38f && c.z < 3.0e38f;
                const float v[3] = {c.x, c.y, c.z};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const float f = (v[k] - base[k]) * scale;
                    q[k] = !with ? kNoCurrent : f > 0.0f ? (f < 65533.0f ? (unsigned)f : 65533u) : 0u;
                }
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) xyz[k][e] = (uint16_t)q[k];
            id[e] = (uint16_t)e;
        }
    }
    __syncthreads();
    for (int size = kChunk; size > group; size >>= 1) {
        if (size / 2 >= n) continue;  // uniform: nothing in the second half
        const int threads = size / kPer, width = threads < kWave ? threads : kWave, g = e0 / size;
        const bool wide = threads > kWave;  // uniform
        unsigned what[kPer], lo[3] = {kNoUnit, kNoUnit, kNoUnit}, hi[3] = {0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            what[i] = id[e0 + i];
            if (xyz[0][what[i]] >= kNoCurrent) continue;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const unsigned v = xyz[k][what[i]];
                lo[k] = v < lo[k] ? v : lo[k];
                hi[k] = v > hi[k] ? v : hi[k];
            }
        }
        box_lanes(lo, hi, width);
        if (wide) {
            if (tid < 6 * kGroups) box[tid / kGroups][tid % kGroups] = tid / kGroups < 3 ? kNoUnit : 0u;
            __syncthreads();
            if (lane == 0)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    atomicMin(&box[k][g], lo[k]);
                    atomicMax(&box[3 + k][g], hi[k]);
                }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] = box[k][g];
                hi[k] = box[3 + k][g];
            }
        }
        int axis = 0;
        unsigned side = 0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const unsigned w = hi[k] >= lo[k] ? hi[k] - lo[k] : 0u;
            if (w > side) {
                side = w;
                axis = k;
            }
        }
        const unsigned base = axis == 0 ? lo[0] : axis == 1 ? lo[1] : lo[2];
        const int bits = side ? 32 - __builtin_clz(side) : 0, shift = bits > kSplitBits ? bits - kSplitBits : 0;
        unsigned key[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const unsigned v = xyz[axis][what[i]];
            key[i] = v == kNoUnit ? (2u << kSplitBits) - 1 : v == kNoCurrent ? 1u << kSplitBits : (v - base) >> shift;
        }
        // the median: the want-th smallest key is `cut`
        unsigned cut = 0;
        int want = size / 2;
        for (int bit = kSplitBits; bit >= 0; --bit) {
            if (wide && tid < kGroups) count[bit & 1][tid] = 0;
            int below = 0;
#pragma unroll
            for (int i = 0; i < kPer; ++i) below += (key[i] ^ cut) >> bit == 0;
            for (int off = 1; off < width; off <<= 1) below += __shfl_xor(below, off);
            if (wide) {
                __syncthreads();
                if (lane == 0) atomicAdd(&count[bit & 1][g], below);
                __syncthreads();
                below = count[bit & 1][g];
            }
            if (below < want) {
                want -= below;
                cut |= 1u << bit;
            }
        }
        // smaller and equal ones before this thread's places in its group
        int l = 0, s = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            l += key[i] < cut;
            s += key[i] == cut;
        }
        const int ownl = l, owns = s;
        for (int off = 1; off < width; off <<= 1) {
            const int a = __shfl_up(l, off), b = __shfl_up(s, off);
            if ((lane & (width - 1)) >= off) {
                l += a;
                s += b;
            }
        }
        if (wide) {
            if (lane == kWave - 1) {
                tot[0][wave] = l;
                tot[1][wave] = s;
            }
            __syncthreads();
            for (int v = g * (threads / kWave); v < wave; ++v) {
                l += tot[0][v];
                s += tot[1][v];
            }
        }
        l -= ownl;
        s -= owns;
        __syncthreads();  // every id has been read
        int k = e0 - g * size;  // places before this one
#pragma unroll
        for (int i = 0; i < kPer; ++i, ++k) {
            int to;
            if (key[i] < cut)
                to = l++;
            else if (key[i] == cut && s < want)
                to = size / 2 - want + s++;
            else {
                to = size / 2 + (k - l - (s < want ? s : want));
                s += key[i] == cut;
            }
            id[g * size + to] = (uint16_t)what[i];
        }
        __syncthreads();
    }
    int64_t to[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) to[i] = e0 + i < n ? perm[first + id[e0 + i]] : 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i)
        if (e0 + i < n) perm[first + e0 + i] = to[i];
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
// Small clusters first, then the large ones (workgroups from nsmall on).
__global__ __launch_bounds__(kFarWG) void k_far_balls(const double* __restrict__ rows, const int32_t* __restrict__ tiles,
                                                      int64_t nsmall, double* __restrict__ geo_small,
                                                      double* __restrict__ geo_large) {
    __shared__ double lds[kFarWG];
    const bool large = blockIdx.x >= nsmall;
    const int64_t cl = large ? blockIdx.x - nsmall : blockIdx.x;
    const int ntile = large ? kParts * kSmallTiles : kSmallTiles;
    double* geo = large ? geo_large : geo_small;
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
// One workgroup per small cluster's 512 rows, staged in LDS; a large cluster's moments are
// the sum of its parts' about its own centre (k_far_coef adds them).  A wave takes one m at a
// time, eight rows per lane whose recurrences stay in registers, kFarChunk orders per round;
// the lanes' sums are added in a fixed order through LDS.  10 FP64 instructions per row and
// order: 0.45 ms for the AG-CCT section's 368,640 rows on the FP64 path (orders up to 34 of the
// potential), 0.16 ms on the FP32 path (both sizes of cluster), at 2 waves per SIMD and half of the issue slots.  Held to 168
// VGPRs for a third wave it spills and takes 4 times as long; adding the wave's halves in
// registers before LDS gained nothing.
constexpr int kFarChunk = 4;
constexpr int kMomWaves = 4;
constexpr int kMomRows = kSmallTiles * kTile, kMomPer = kMomRows / kWave;

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
                                                                   const int32_t* __restrict__ tiles, int q, int64_t nsmall,
                                                                   const double* __restrict__ geo_small,
                                                                   const double* __restrict__ geo_large,
                                                                   double* __restrict__ mom) {
    __shared__ double row[6][kMomRows];  // (m - c) / E and kl; zeros for a row without current
    __shared__ double lds[kMomWaves][kFarChunk * 6][kWave + 1];
    const bool large = blockIdx.x >= nsmall;  // about the large cluster's centre: the second half of the sets
    const int64_t cl = large ? blockIdx.x - nsmall : blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int top = 4 * q - 2;  // highest order of the potential
    const double* g = large ? geo_large + cl / kParts * kFarGeo : geo_small + cl * kFarGeo;
    const double inv = g[3];
    for (int i = threadIdx.x; i < kMomRows; i += kWave * kMomWaves) {
        ClusterRow r;
        const bool live = cluster_row(rows, tiles, cl, kSmallTiles, i, r);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            row[c][i] = live ? (r.m[c] - g[c]) * inv : 0.0;
            row[3 + c][i] = live ? r.kl[c] : 0.0;
        }
    }
    __syncthreads();
    double(*mine)[kWave + 1] = lds[wave];
#pragma unroll 1
    for (int turn = 0; turn * kMomWaves <= top; ++turn) {
        // m in turns, there and back: row m has top - m + 1 orders
        const int m = turn * kMomWaves + (turn & 1 ? kMomWaves - 1 - wave : wave);
        if (m > top) continue;
        const double(*fac)[2] = kRegular.f[m];  // wave-uniform: scalar loads
        double f = 1.0;
        for (int k = 1; k <= m; ++k) f /= 2.0 * k;
        double* out = mom + ((int64_t)blockIdx.x * far_records(q) + far_row(q, m)) * 6;
        double pc[kMomPer], ps[kMomPer], cur[kMomPer], old[kMomPer];
#pragma unroll
        for (int j = 0; j < kMomPer; ++j) {
            const double x = row[0][lane + j * kWave], y = row[1][lane + j * kWave];
            pc[j] = f;  // f (x + iy)^m by squares
            ps[j] = 0.0;
            double bc = x, bs = y;
            for (int k = m; k != 0; k >>= 1) {
                if (k & 1) {
                    const double t = pc[j] * bc - ps[j] * bs;
                    ps[j] = pc[j] * bs + ps[j] * bc;
                    pc[j] = t;
                }
                const double t = bc * bc - bs * bs;
                bs = 2.0 * bc * bs;
                bc = t;
            }
            cur[j] = 1.0;  // R_n over R_m^m
            old[j] = 0.0;
        }
#pragma unroll 1
        for (int n0 = m; n0 <= top; n0 += kFarChunk) {
            double acc[kFarChunk][6];
#pragma unroll
            for (int k = 0; k < kFarChunk; ++k)
#pragma unroll
                for (int c = 0; c < 6; ++c) acc[k][c] = 0.0;
#pragma unroll
            for (int j = 0; j < kMomPer; ++j) {
                const int i = lane + j * kWave;
                const double x = row[0][i], y = row[1][i], z = row[2][i];
                const double r2 = x * x + y * y + z * z;
                const double kc[3] = {row[3][i] * pc[j], row[4][i] * pc[j], row[5][i] * pc[j]};
                const double ks[3] = {row[3][i] * ps[j], row[4][i] * ps[j], row[5][i] * ps[j]};
#pragma unroll
                for (int k = 0; k < kFarChunk; ++k) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        acc[k][c] = __builtin_fma(kc[c], cur[j], acc[k][c]);
                        acc[k][3 + c] = __builtin_fma(ks[c], cur[j], acc[k][3 + c]);
                    }
                    const double nx = fac[n0 + k - m][0] * (z * cur[j]) - fac[n0 + k - m][1] * (r2 * old[j]);
                    old[j] = cur[j];
                    cur[j] = nx;
                }
            }
#pragma unroll
            for (int k = 0; k < kFarChunk; ++k)
#pragma unroll
                for (int c = 0; c < 6; ++c) mine[k * 6 + c][lane] = acc[k][c];
            __builtin_amdgcn_wave_barrier();
            const int v = lane >> 1;  // two lanes per value
            double s = 0.0;
            if (v < kFarChunk * 6)
#pragma unroll
                for (int i = 0; i < kWave / 2; ++i) s += mine[v][(lane & 1) * (kWave / 2) + i];
            s += __shfl_xor(s, 1);
            if (v < kFarChunk * 6 && (lane & 1) == 0 && n0 + v / 6 <= top) out[(n0 - m) * 6 + v] = s;
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// Coefficients of the field, B = curl A, order n from the potential's order n - 1:
//   d/dx, d/dy and d/dz of the exterior harmonic I_n^m are (I_{n+1}^{m-1} - I_{n+1}^{m+1}) / 2,
//   i (I_{n+1}^{m-1} + I_{n+1}^{m+1}) / 2 and -I_{n+1}^m  (I^{-1} = -conj I^1).
// A large cluster's moments are the sum of its parts' (records from nsmall * far_records on).
__global__ void k_far_coef(int q, int64_t nsmall, int64_t nrec, const double* __restrict__ geo_small,
                           const double* __restrict__ geo_large, const double* __restrict__ mom,
                           double* __restrict__ coef_small, double* __restrict__ coef_large) {
    const int64_t at = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (at >= nrec) return;
    const int per = far_records(q);
    const bool large = at >= nsmall * per;
    const int64_t i = large ? at - nsmall * per : at;
    const int parts = large ? kParts : 1;
    const double* geo = large ? geo_large : geo_small;
    double* coef = large ? coef_large : coef_small;
    if (large) mom += nsmall * per * 6;
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
    const double* base = mom + cl * parts * per * 6;
    const auto a = [&](int k, int c) {
        if (k < 0 || k > n - 1 || (c >= 3 && k == 0)) return 0.0;
        const double* at = base + (far_row(q, k) + (n - 1 - k)) * 6 + c;
        double v = at[0];
        for (int p = 1; p < parts; ++p) v += at[(int64_t)p * per * 6];
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

// How far the blocks of a point set reach across the segments: route[0] / route[1] is the share of a block's
// segments inside the block's ball, by 256 of them, in the mean over the blocks (weighed by their tiles).  With
// points in no order along the magnet, or in rows across it, most segments are, and hardly any cluster is far
// from a block.  FP64 maps of 3,000 to 20,000 points in the AG-CCT section, a single CCT, a population's design
// and the gantry, time through the clusters over that of the full sum by the share: below 0.06 0.15-0.73, 0.3
// 0.61-0.87, 0.56 0.78-0.95, 0.7 0.92-1.13, 1.0 (shuffled) 1.00-1.11: the full sum from 2/3 on (spread_out).
// One wave per block; 5 us with the launch that clears the counts.
__global__ __launch_bounds__(kWave) void k_point_spread(const double* __restrict__ seg64, const Work* __restrict__ work,
                                                        const double* __restrict__ pts, int64_t ptot,
                                                        unsigned long long* __restrict__ route) {
    constexpr int kMost = 4, kSamples = 256;  // points per lane, segments looked at
    const Work w = work[blockIdx.x];
    if (w.chunk != 0) return;  // a block's first item
    const Work last = work[blockIdx.x + w.nchunk - 1];
    const int64_t row0 = (int64_t)w.tile_start * kTile;
    const int64_t nrow = (int64_t)(last.tile_start + last.tile_count) * kTile - row0;
    if (nrow <= 0) return;
    const int lane = threadIdx.x;
    double px[kMost], py[kMost], pz[kMost];
#pragma unroll
    for (int j = 0; j < kMost; ++j) {
        const int at = lane + j * kWave;
        const int64_t g = w.pt_start + (at < w.pt_count ? at : w.pt_count - 1);
        px[j] = pts[g];
        py[j] = pts[ptot + g];
        pz[j] = pts[2 * ptot + g];
    }
    const Ball b = block_ball<kMost>(px, py, pz);
    const double reach = b.r * b.r;
    int live = 0, near = 0;
    for (int j = 0; j < kSamples / kWave; ++j) {
        const double* r = seg64 + (row0 + (lane + j * kWave) * nrow / kSamples) * 8;
        const double dx = r[4] - b.x, dy = r[5] - b.y, dz = r[6] - b.z;
        const bool is = carries(r);
        live += __popcll(__ballot(is));
        near += __popcll(__ballot(is && !(dx * dx + dy * dy + dz * dz >= reach)));
    }
    if (lane != 0) return;
    const unsigned long long tiles = (unsigned long long)(nrow / kTile);
    atomicAdd(route, near * tiles);
    atomicAdd(route + 1, live * tiles);
}

__global__ void k_clear_counts(unsigned long long* __restrict__ route) { route[threadIdx.x] = 0; }

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
    const int64_t places = ncluster * ntile, nrec = 2 * ncluster * far_records(q);
    // k_bs_partial_f64 counts the packed rows in 31 bits
    if (precision == 64 && places * kTile > 0x7fffffff) return CCTAMD_ERANGE;
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
    const int64_t nlarge = ncluster / kParts, nr = (ncluster + nlarge) * far_records(q);
    hipLaunchKernelGGL(k_far_balls, dim3((unsigned)(ncluster + nlarge)), dim3(kFarWG), 0, st, src, ids, ncluster, geo,
                       geo_large);
    hipLaunchKernelGGL(k_far_moments, dim3((unsigned)(2 * ncluster)), dim3(kWave * kMomWaves), 0, st, src, ids, q,
                       ncluster, geo, geo_large, mom);
    hipLaunchKernelGGL(k_far_coef, dim3((unsigned)ceil_div(nr, 256)), dim3(256), 0, st, q, ncluster, nr, geo, geo_large,
                       mom, coef, coef_large);
    return hip_status(hipGetLastError());
}

int cctamd_point_spread(int ppl, const double* seg64, const int32_t* work, int64_t nwork, const double* points,
                        int64_t npoints, int64_t* spread, void* stream) {
    if (!valid_ppl(ppl) || nwork < 0 || npoints < 0 || !spread) return CCTAMD_EINVAL;
    if (nwork > 0 && (!seg64 || !work || !points || npoints == 0)) return CCTAMD_EINVAL;
    if (nwork > 0x7fffffff) return CCTAMD_ERANGE;
    hipStream_t st = (hipStream_t)stream;
    unsigned long long* route = (unsigned long long*)spread;
    hipLaunchKernelGGL(k_clear_counts, dim3(1), dim3(2), 0, st, route);
    if (nwork > 0)
        hipLaunchKernelGGL(k_point_spread, dim3((unsigned)nwork), dim3(kWave), 0, st, seg64, (const Work*)work, points,
                           npoints, route);
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
        // the blocks' items that read the same rows share an XCD (as in cctamd_plan)
        if (nb > 1 && nc > kXcds) nc -= nc % kXcds;
        if (work) {
            if (!design_cluster_off || !design_pt_off || !design_wbase || !design_nchunk) return CCTAMD_EINVAL;
            if (nc > 0x7fffffff) return CCTAMD_ERANGE;
            design_wbase[d] = n;
            design_nchunk[d] = (int32_t)nc;
            for (int64_t b = 0; b < nb && nc > 0; ++b) {
                for (int64_t c = 0; c < nc; ++c) {
                    const int64_t ps = design_pt_off[d] + b * pb;
                    const int64_t pc = std::min(pb, design_npt[d] - b * pb);
                    // cluster numbers are kept shifted by up to 7 bits (FarLists), their tiles in 31
                    if (ps + pc > 0x7fffffff || design_cluster_off[d] + ns > 0x7fffffff >> (far_order_bits(kFarQ64) + 1))
                        return CCTAMD_ERANGE;
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
