// k_optim.hip -- Adam, int32 inclusive scans, and the GPU-resident
// densification cycle (classify -> scans -> keep flags of the old and
// appended rows -> one gather of every surviving row of the 18 parameter /
// optimizer buffers, in place past the old rows' end and through a workspace
// below it -> the staged rows' copy back).
#include <algorithm>

#include "kernels.h"
#include "ms_device.h"

using namespace msd;

namespace {

// fused_adam_kernel (msplat_metal.metal:1383-1406).
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m_, float *__restrict__ v_, int64_t n,
                                              float step, float b1, float b2, float bc2_sqrt, float eps) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float gi = g[i];
        const float m = __builtin_fmaf(b1, m_[i], (1.0f - b1) * gi);
        const float v = __builtin_fmaf(b2, v_[i], (1.0f - b2) * gi * gi);
        p[i] -= step * m / (__builtin_sqrtf(v) / bc2_sqrt + eps);
        m_[i] = m;
        v_[i] = v;
    }
}

// p[i] = min(p[i], value): the opacity reset of Model::afterTrain
// (model.cpp:290-296), which the reference runs as a host loop on unified
// memory.
__global__ void k_clamp_max(float *__restrict__ p, int64_t n, float value) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        if (p[i] > value) p[i] = value;
}

// Zeroes n float4s, one 16-byte store per thread in a single pass.  It
// clears the raster backward's per-splat gradient rows before each step:
// 192 MB at 3M splats, which hipMemsetAsync wrote at about 2.3 TB/s.
__global__ __launch_bounds__(256) void k_zero16(float4 *__restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// RGBA8 of an [n,3] float image: (uint8)(clamp(x, 0, 1) * 255) per channel
// (truncation, the host loop of renderFromPoseToBuffer, msplat_api.mm:207-236)
// and alpha 255, one 4-byte store per pixel.
__global__ void k_rgba8(const float *__restrict__ img, int64_t n, uint32_t *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float *p = img + 3 * i;
        uint32_t v = 0xff000000u;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float x = __builtin_fminf(__builtin_fmaxf(p[c], 0.0f), 1.0f) * 255.0f;
            v |= (uint32_t)x << (8 * c);
        }
        out[i] = v;
    }
}

// ---- inclusive scans of int32 in tiles of kScanTile ----------------------
// A scan's first kernel leaves each element's prefix inside its tile and the
// tile's total; k_scan_totals turns the totals into the tiles' offsets, and
// whoever reads a prefix adds its tile's offset.  Adding them in a pass of its
// own, and scanning the split and dup flags apart from each other and from
// their classification, took nine launches and 28 us of a densification of
// 300k splats; the three there are now take 10.
constexpr int kScanBlock = 256, kScanItems = 4, kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ int block_incl_scan(int v, int *s_w) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    if (lane == 63) s_w[wave] = v;
    __syncthreads();
    int off = 0;
    for (int w = 0; w < wave; ++w) off += s_w[w];
    __syncthreads();
    return v + off;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_local(const int *__restrict__ in, int *__restrict__ out,
                                                           int n, int *__restrict__ totals) {
    __shared__ int s_w[kScanBlock / 64];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        sum += v[k];
    }
    const int incl = block_incl_scan(sum, s_w);
    int run = incl - sum;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        run += v[k];
        if (base + k < n) out[base + k] = run;
    }
    if (threadIdx.x == kScanBlock - 1) totals[blockIdx.x] = incl;
}

// Workgroup b: the nb tile totals at totals + b (nb + 1) become the tiles'
// exclusive offsets, with the sum of all of them after the last.
__global__ __launch_bounds__(1024) void k_scan_totals(int *__restrict__ totals, int nb) {
    __shared__ int s_w[16];
    totals += (size_t)blockIdx.x * (nb + 1);
    const int chunk = (nb + 1023) / 1024;
    const int b = min(nb, (int)threadIdx.x * chunk), e = min(nb, b + chunk);
    int sum = 0;
    for (int i = b; i < e; ++i) sum += totals[i];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (lane == 63) s_w[wave] = incl;
    __syncthreads();
    int off = 0;
    for (int w = 0; w < wave; ++w) off += s_w[w];
    int run = off + incl - sum;  // exclusive offset of this thread's chunk
    for (int i = b; i < e; ++i) {
        const int t = totals[i];
        totals[i] = run;  // becomes the exclusive block offset
        run += t;
    }
    if (b < e && e == nb) totals[nb] = run;
}

// The inclusive prefix of element i, from its tile's prefix and offset.
__device__ __forceinline__ int prefix_at(const int *__restrict__ pre, const int *__restrict__ offs, int i) {
    return pre[i] + offs[i / kScanTile];
}

// ---- densification (msplat_metal.metal:3231-3491) ------------------------

// The largest of a splat's SD scales (kScaleDim, :3253-3255).
__device__ __forceinline__ float max_scale(const float *__restrict__ scales, size_t i, int SD) {
    float ms = ms_expf(scales[(size_t)SD * i]);
    for (int k = 1; k < SD; ++k) ms = __builtin_fmaxf(ms, ms_expf(scales[(size_t)SD * i + k]));
    return ms;
}

// densify_classify_kernel (:3231-3266) for splat i; SD floats of scale per
// splat.
__device__ __forceinline__ void classify(int i, int SD, const float *__restrict__ gnorm,
                                         const float *__restrict__ vis, const float *__restrict__ scales,
                                         const float *__restrict__ max2d, float half_max_dim, float grad_th,
                                         float size_th, float screen_th, int check_screen, bool &split, bool &dup) {
    split = dup = false;
    const float vc = vis[i];
    if (vc <= 0.0f) return;
    const float avg = (gnorm[i] / vc) * half_max_dim;
    const bool high = avg > grad_th;
    const bool large = max_scale(scales, i, SD) > size_th;
    bool sp = large;
    if (check_screen && max2d[i] > screen_th) sp = true;
    split = sp && high;
    dup = !large && high;
}

// The flags of kScanTile splats per workgroup with their prefixes inside the
// tile; the tiles' totals go to totals (split) and totals + gridDim.x + 1
// (dup).  Splat k 256 + t of the tile is thread t's in round k, so the loads
// stay coalesced and a prefix is the counts of the (round, wave) pairs before
// it plus a popcount.
__global__ __launch_bounds__(kScanBlock) void k_classify(
    int N, int SD, const float *__restrict__ gnorm, const float *__restrict__ vis, const float *__restrict__ scales,
    const float *__restrict__ max2d, float half_max_dim, float grad_th, float size_th, float screen_th,
    int check_screen, int *__restrict__ split, int *__restrict__ dup, int *__restrict__ split_pre,
    int *__restrict__ dup_pre, int *__restrict__ totals) {
    constexpr int kWaves = kScanBlock / 64;
    __shared__ int s_split[kScanItems * kWaves], s_dup[kScanItems * kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t upto = ~0ull >> (63 - lane);
    uint64_t bs[kScanItems], bd[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = blockIdx.x * kScanTile + k * kScanBlock + threadIdx.x;
        bool sp = false, dp = false;
        if (i < N)
            classify(i, SD, gnorm, vis, scales, max2d, half_max_dim, grad_th, size_th, screen_th, check_screen, sp, dp);
        bs[k] = __ballot(sp);
        bd[k] = __ballot(dp);
        if (lane == 0) {
            s_split[k * kWaves + wave] = __popcll(bs[k]);
            s_dup[k * kWaves + wave] = __popcll(bd[k]);
        }
    }
    __syncthreads();
    int before_s = 0, before_d = 0, seen = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        for (; seen < k * kWaves + wave; ++seen) {
            before_s += s_split[seen];
            before_d += s_dup[seen];
        }
        const int i = blockIdx.x * kScanTile + k * kScanBlock + threadIdx.x;
        if (i < N) {
            split[i] = (int)((bs[k] >> lane) & 1);
            dup[i] = (int)((bd[k] >> lane) & 1);
            split_pre[i] = before_s + __popcll(bs[k] & upto);
            dup_pre[i] = before_d + __popcll(bd[k] & upto);
        }
    }
    if (threadIdx.x == kScanBlock - 1) {  // the last wave's last round ends the tile
        totals[blockIdx.x] = before_s + __popcll(bs[kScanItems - 1]);
        totals[gridDim.x + 1 + blockIdx.x] = before_d + __popcll(bd[kScanItems - 1]);
    }
}

// The rows after the compaction are a stable selection from the virtual
// list [old rows 0..N) ++ [two children per split splat, in split order]
// ++ [one copy per dup splat, in dup order] (msplat_metal.metal:3271-3412
// append these rows, :3417-3491 cull and compact them).  Nothing is
// appended here: every virtual row is a function of its parent's row, so
// k_densify_keep decides each virtual row's fate from the parent alone,
// and k_densify_gather writes each output row once, in output order.

// The split offset of child k of parent i (the rotated, scaled normal
// sample of :3285-3313), in the reference's operation order.
__device__ __forceinline__ float3 split_offset(const float *__restrict__ quats, const float *__restrict__ scales,
                                               const float *__restrict__ rs, int SD, int i, int ri) {
    float qw = quats[(size_t)i * 4], qx = quats[(size_t)i * 4 + 1], qy = quats[(size_t)i * 4 + 2],
          qz = quats[(size_t)i * 4 + 3];
    const float qlen = __builtin_sqrtf(qw * qw + qx * qx + qy * qy + qz * qz);
    qw /= qlen;
    qx /= qlen;
    qy /= qlen;
    qz /= qlen;
    const size_t si = (size_t)i * SD;
    const float sx = ms_expf(scales[si]), sy = ms_expf(scales[si + 1]);
    const float sz = SD > 2 ? ms_expf(scales[si + 2]) : 0.0f;
    const float r0 = rs[(size_t)ri * 3] * sx, r1 = rs[(size_t)ri * 3 + 1] * sy, r2 = rs[(size_t)ri * 3 + 2] * sz;
    float3 v;
    v.x = (1 - 2 * (qy * qy + qz * qz)) * r0 + 2 * (qx * qy - qw * qz) * r1 + 2 * (qx * qz + qw * qy) * r2;
    v.y = 2 * (qx * qy + qw * qz) * r0 + (1 - 2 * (qx * qx + qz * qz)) * r1 + 2 * (qy * qz - qw * qx) * r2;
    v.z = 2 * (qx * qz - qw * qy) * r0 + 2 * (qy * qz + qw * qx) * r1 + (1 - 2 * (qx * qx + qy * qy)) * r2;
    return v;
}

// The reference's cull test (densify_cull_classify_kernel, :3417-3456) for
// a row with opacity logit `opac` and scales `sc` (already reduced by
// log 1.6 where the row is a child or the copy of a split splat).
__device__ __forceinline__ bool culled(float opac, const float *sc, int SD, float alpha_th, float scale_th,
                                       bool check_huge) {
    const float os = 1.0f / (1.0f + ms_expf(-opac));
    bool cull = os < alpha_th;
    if (check_huge) {
        float ms = ms_expf(sc[0]);
        for (int k = 1; k < SD; ++k) ms = __builtin_fmaxf(ms, ms_expf(sc[k]));
        if (ms > scale_th) cull = true;
    }
    return cull;
}

// One thread per old row i: keep[] of row i and of the rows it appends
// (children at N + 2 ord + k, the copy at N + 2 nS + dup ord), and the
// parent of every appended row.  The appended rows carry the parent's
// opacity; a child's scales are the parent's minus log 1.6, and so are a
// copy's when its parent is also split (the reference appends the copy
// after reducing the split parent's scales in place, :3358-3360).
__global__ __launch_bounds__(256) void k_densify_keep(int N, int nS, int SD, const int *__restrict__ split,
                                                      const int *__restrict__ dup,
                                                      const int *__restrict__ split_pre,
                                                      const int *__restrict__ dup_pre,
                                                      const int *__restrict__ split_offs,
                                                      const int *__restrict__ dup_offs,
                                                      const float *__restrict__ opac,
                                                      const float *__restrict__ scales,
                                                      const float *__restrict__ max2d, float log_size_fac,
                                                      float alpha_th, float scale_th, float screen_size,
                                                      int check_huge, int check_screen, int *__restrict__ keep,
                                                      int *__restrict__ parent) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float op = opac[i];
    float sc[3], sc_dec[3];
    for (int k = 0; k < SD; ++k) {
        sc[k] = scales[(size_t)i * SD + k];
        sc_dec[k] = sc[k] - log_size_fac;
    }
    const bool sp = split[i] != 0;
    bool cull = sp || culled(op, sc, SD, alpha_th, scale_th, check_huge);
    if (check_huge && check_screen && max2d[i] > screen_size) cull = true;
    keep[i] = cull ? 0 : 1;
    if (sp) {
        const int a = 2 * (prefix_at(split_pre, split_offs, i) - 1);
        const int kc = culled(op, sc_dec, SD, alpha_th, scale_th, check_huge) ? 0 : 1;
        keep[N + a] = kc;
        keep[N + a + 1] = kc;
        parent[a] = i;
        parent[a + 1] = i;
    }
    if (dup[i]) {
        const int a = 2 * nS + prefix_at(dup_pre, dup_offs, i) - 1;
        keep[N + a] = culled(op, sp ? sc_dec : sc, SD, alpha_th, scale_th, check_huge) ? 0 : 1;
        parent[a] = i;
    }
}

// src_of[output row] = virtual row, from the inclusive scan of keep[].
__global__ __launch_bounds__(256) void k_densify_src(int n_virt, const int *__restrict__ keep,
                                                     const int *__restrict__ keep_pre,
                                                     const int *__restrict__ keep_offs, int *__restrict__ src_of) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n_virt && keep[v]) src_of[prefix_at(keep_pre, keep_offs, v) - 1] = v;
}

// Output rows are written in blocks of kGatherRows rows.
constexpr int kGatherRows = 256, kMaxDensBufs = 18;

struct GatherBuf {
    float *own;      // the caller's buffer: the old rows, and the output rows from N on
    float *ws;       // the output rows below N (workspace)
    int stride;      // floats per row
    uint32_t magic;  // ceil(2^24 / stride): j / stride = (j * magic) >> 24 for j < 2^15
    int group;       // 0 means, 1 scales, 2.. others
};
struct GatherArgs {
    GatherBuf b[kMaxDensBufs];  // the parameters, then the first and the second moments
    int per_set;                // buffers in each of the three
    int row_blocks, N, nS, SD;
    float log_size_fac;
    const int *split, *parent, *src_of, *new_count;
    const float *quats, *scales, *rs;  // the parent rows of the children
};

// Every output row of every buffer, once: workgroup = (parameters, first or
// second moments; block of kGatherRows output rows).  The rows of a block are
// contiguous in each output buffer, so each store instruction writes 1 KB of
// consecutive floats; reads follow the kept rows, which are contiguous runs
// of old rows.  An old row is copied, an appended row is derived from its
// parent (moments zero).  Only old rows, those below N, are read, so output
// rows from N on go straight to the caller's buffer; those below wait in the
// workspace until every row has been read (k_densify_copy_back).  Bound by
// HBM.  A workgroup takes all six buffers of its rows, with the row to read
// and what becomes of it worked out once per row in LDS, so that an element
// is one load: with one buffer per workgroup, whose few elements each looked
// their parent up, 300k splats (488k rows before the cull) took 150 us
// and now take 111; whole rows without the LDS map took 185.  The copy back of
// all rows took 99 us, of those below N 67.
__global__ __launch_bounds__(256) void k_densify_gather(GatherArgs g) {
    __shared__ int s_row[kGatherRows], s_app[kGatherRows];  // row to read; appended row's number or -1
    __shared__ uint8_t s_reduced[kGatherRows];              // its scales are the parent's less log 1.6
    const int set = (int)blockIdx.x / g.row_blocks;
    const int new_count = *g.new_count;
    const int r0 = ((int)blockIdx.x - set * g.row_blocks) * kGatherRows;
    const int rows = min(kGatherRows, new_count - r0);
    if (rows <= 0) return;
    if ((int)threadIdx.x < rows) {
        const int v = g.src_of[r0 + threadIdx.x], a = v - g.N;
        const int p = a < 0 ? v : g.parent[a];
        s_row[threadIdx.x] = p;
        s_app[threadIdx.x] = a < 0 ? -1 : a;
        s_reduced[threadIdx.x] = a >= 0 && set == 0 && (a < 2 * g.nS || g.split[p]);
    }
    __syncthreads();
    for (int bi = set * g.per_set; bi < (set + 1) * g.per_set; ++bi) {
        const GatherBuf B = g.b[bi];
        const int S = B.stride, total = rows * S;
        // the block's elements below output row N are staged
        const int staged = (int)min<int64_t>(total, max<int64_t>(0, ((int64_t)g.N - r0) * S));
        const float *__restrict__ src = B.own;
        float *ws = B.ws + (size_t)r0 * S, *own = B.own + (size_t)r0 * S;
        constexpr int U = 8;
        for (int j0 = threadIdx.x; j0 < total; j0 += 256 * U) {
            float out[U];
            int row[U];
            bool app[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = min(j0 + u * 256, total - 1);
                row[u] = (int)(((uint64_t)(uint32_t)j * B.magic) >> 24);
                app[u] = s_app[row[u]] >= 0;
                out[u] = 0.0f;
                // (a moment's appended rows are zero)
                if (!(set && app[u])) out[u] = src[(size_t)s_row[row[u]] * S + (j - row[u] * S)];
            }
            if (set == 0 && B.group < 2) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int a = s_app[row[u]];
                    if (B.group == 1) {
                        if (s_reduced[row[u]]) out[u] = out[u] - g.log_size_fac;
                    } else if (app[u] && a < 2 * g.nS) {
                        const int c = min(j0 + u * 256, total - 1) - row[u] * S;
                        const float3 o = split_offset(g.quats, g.scales, g.rs, g.SD, s_row[row[u]], a);
                        out[u] = out[u] + (c == 0 ? o.x : c == 1 ? o.y : o.z);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = j0 + u * 256;
                // (the copy back writes the staged moments' zeros itself)
                if (j < total && !(set && app[u] && j < staged)) (j < staged ? ws : own)[j] = out[u];
            }
        }
    }
}

// The staged output rows (those below N) back into the caller's buffers, in
// 4096-float blocks; in a moment buffer the appended ones, which follow the
// kept old rows, are zeros that were never staged.
constexpr int kCopyFloats = 4096;
struct CopyArgs {
    const float *src[kMaxDensBufs];
    float *dst[kMaxDensBufs];
    int stride[kMaxDensBufs], block0[kMaxDensBufs + 1];
    int nbuf, moment0;  // buffers from moment0 on hold moments
    int N;
    const int *new_count, *keep_pre, *keep_offs;
};
__global__ __launch_bounds__(256) void k_densify_copy_back(CopyArgs a) {
    int bi = 0;
    while (bi + 1 < a.nbuf && (int)blockIdx.x >= a.block0[bi + 1]) ++bi;
    const int64_t total = (int64_t)min(*a.new_count, a.N) * a.stride[bi];
    const int64_t base = (int64_t)((int)blockIdx.x - a.block0[bi]) * kCopyFloats;
    if (base >= total) return;
    const int64_t held =
        bi < a.moment0 ? total : min<int64_t>(total, (int64_t)prefix_at(a.keep_pre, a.keep_offs, a.N - 1) * a.stride[bi]);
    const float *__restrict__ s = a.src[bi] + base;
    float *__restrict__ d = a.dst[bi] + base;
    const int n = (int)min<int64_t>(kCopyFloats, total - base);
    const int n_held = (int)max<int64_t>(0, min<int64_t>(n, held - base));
    constexpr int U = kCopyFloats / 256;
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int j = threadIdx.x + u * 256;
        v[u] = j < n_held ? s[j] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int j = threadIdx.x + u * 256;
        if (j < n) d[j] = v[u];
    }
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

__global__ void k_zero_counters(int *__restrict__ a, int na, int *__restrict__ b, int nb) {
    for (int i = threadIdx.x; i < na; i += blockDim.x) a[i] = 0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) b[i] = 0;
}

__global__ void k_step_report(const double *__restrict__ loss, const int *__restrict__ ctr, int n_ctr,
                              mskern::Publish out) {
    double *d = reinterpret_cast<double *>(out.data);
    if (threadIdx.x < 2) d[threadIdx.x] = loss[threadIdx.x];
    for (int i = threadIdx.x; i < n_ctr; i += blockDim.x) out.data[4 + i] = ctr[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(out.flag, out.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

namespace mskern {

void launch_adam(hipStream_t s, float *p, const float *g, float *m, float *v, int64_t n, float step, float b1,
                 float b2, float bc2_sqrt, float eps) {
    if (n <= 0) return;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)blocks), dim3(256), 0, s, p, g, m, v, n, step, b1, b2, bc2_sqrt, eps);
}

void launch_clamp_max(hipStream_t s, float *p, int64_t n, float value) {
    if (n <= 0) return;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_clamp_max, dim3((unsigned)blocks), dim3(256), 0, s, p, n, value);
}

void launch_zero16(hipStream_t s, float *p, int64_t n_float4) {
    if (n_float4 <= 0) return;
    const int64_t blocks = (n_float4 + 255) / 256;
    hipLaunchKernelGGL(k_zero16, dim3((unsigned)blocks), dim3(256), 0, s, reinterpret_cast<float4 *>(p), n_float4);
}

void launch_zero_counters(hipStream_t s, int *a, int na, int *b, int nb) {
    hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(256), 0, s, a, na, b, nb);
}

void launch_step_report(hipStream_t s, const double *loss, const int *ctr, int n_ctr, const Publish &out) {
    hipLaunchKernelGGL(k_step_report, dim3(1), dim3(256), 0, s, loss, ctr, n_ctr, out);
}

void launch_rgba8(hipStream_t s, const float *img, int64_t n, uint32_t *out) {
    if (n <= 0) return;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_rgba8, dim3((unsigned)blocks), dim3(256), 0, s, img, n, out);
}

static int scan_tiles(int64_t n) { return (int)((n + kScanTile - 1) / kScanTile); }

// the split and dup totals of n splats, then the keep totals of the at most
// 4n virtual rows, each with its sum after it
int64_t densify_scan_ints(int64_t n) { return std::max<int64_t>(2 * (scan_tiles(n) + 1), scan_tiles(4 * n) + 1); }

void launch_densify_classify(hipStream_t s, const DensifyArgs &a, const int *&n_split, const int *&n_dup) {
    const int N = a.n, nb = scan_tiles(N);
    hipLaunchKernelGGL(k_classify, dim3(nb), dim3(kScanBlock), 0, s, N, a.scale_dim, a.grad_norm, a.vis, a.params[1],
                       a.max2d, a.half_max_dim, a.grad_th, a.size_th, a.screen_th, a.check_screen, a.split, a.dup,
                       a.split_pre, a.dup_pre, a.scan_temp);
    hipLaunchKernelGGL(k_scan_totals, dim3(2), dim3(1024), 0, s, a.scan_temp, nb);
    n_split = a.scan_temp + nb;
    n_dup = a.scan_temp + 2 * nb + 1;
}

int64_t densify_workspace_floats(int n_virt, int scale_dim, int fr_stride) {
    // 18 compacted buffers of n_virt rows, each padded to 64 floats
    const int strides[6] = {3, scale_dim, 4, 3, fr_stride, 1};
    int64_t f = 0;
    for (int gi = 0; gi < 6; ++gi) f += 3 * (((int64_t)n_virt * strides[gi] + 63) / 64 * 64);
    return f;
}

const int *launch_densify_apply(hipStream_t s, const DensifyArgs &a, int nS, int n_virt) {
    const int N = a.n, nb_n = scan_tiles(N), nb = scan_tiles(n_virt);
    hipLaunchKernelGGL(k_densify_keep, dim3(nblk(N, 256)), dim3(256), 0, s, N, nS, a.scale_dim, a.split, a.dup,
                       a.split_pre, a.dup_pre, a.scan_temp, a.scan_temp + nb_n + 1, a.params[5], a.params[1], a.max2d,
                       a.log_size_fac, a.cull_alpha, a.cull_scale, a.cull_screen, a.check_huge, a.check_screen, a.keep,
                       a.parent);
    hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(kScanBlock), 0, s, a.keep, a.keep_pre, n_virt, a.scan_temp);
    hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(1024), 0, s, a.scan_temp, nb);
    const int *new_count = a.scan_temp + nb;
    hipLaunchKernelGGL(k_densify_src, dim3(nblk(n_virt, 256)), dim3(256), 0, s, n_virt, a.keep, a.keep_pre,
                       a.scan_temp, a.src_of);
    const int strides[6] = {3, a.scale_dim, 4, 3, a.fr_stride, 1};
    GatherArgs g{};
    CopyArgs c{};
    g.N = c.N = N;
    g.nS = nS;
    g.SD = a.scale_dim;
    g.log_size_fac = a.log_size_fac;
    g.split = a.split;
    g.parent = a.parent;
    g.src_of = a.src_of;
    g.new_count = c.new_count = new_count;
    g.quats = a.params[2];
    g.scales = a.params[1];
    g.rs = a.random;
    g.row_blocks = (int)nblk(n_virt, kGatherRows);
    c.keep_pre = a.keep_pre;
    c.keep_offs = a.scan_temp;
    float *ws = a.workspace;
    int cb = 0, nbuf = 0;
    for (int r = 0; r < 3; ++r) {
        if (r == 1) g.per_set = c.moment0 = nbuf;
        for (int gi = 0; gi < 6; ++gi) {
            if (strides[gi] <= 0) continue;
            float *buf = r == 0 ? a.params[gi] : r == 1 ? a.exp_avg[gi] : a.exp_avg_sq[gi];
            GatherBuf &B = g.b[nbuf];
            B.own = buf;
            B.ws = ws;
            B.stride = strides[gi];
            B.magic = (uint32_t)(((1u << 24) + strides[gi] - 1) / strides[gi]);
            B.group = gi;
            c.src[nbuf] = ws;
            c.dst[nbuf] = buf;
            c.stride[nbuf] = strides[gi];
            c.block0[nbuf] = cb;
            cb += (int)nblk((int64_t)std::min(N, n_virt) * strides[gi], kCopyFloats);
            ws += ((int64_t)n_virt * strides[gi] + 63) / 64 * 64;
            ++nbuf;
        }
    }
    c.nbuf = nbuf;
    c.block0[nbuf] = cb;
    hipLaunchKernelGGL(k_densify_gather, dim3(3 * g.row_blocks), dim3(256), 0, s, g);
    hipLaunchKernelGGL(k_densify_copy_back, dim3(cb), dim3(256), 0, s, c);
    return new_count;
}

}  // namespace mskern
