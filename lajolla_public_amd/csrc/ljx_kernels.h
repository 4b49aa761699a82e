// Wavefront path-tracing kernels (surface transport).
//
// One bounce of lajolla's path_tracing (src/path_tracing.h:7-325) is split
// into stages that each run over a compacted SoA queue of path ids:
//
//   k_raygen      sample_primary + the two screen-jitter draws
//   k_extend      closest-hit traversal, 64 rays per wave fetch; keys each
//                 queue entry by the hit material's type or MISS
//   k_sort_*      orders the queue's paths by key (material sort)
//   k_shade<MT>   one kernel per material type: emission + MIS of the hit
//                 reached by the previous BSDF sample, Russian roulette,
//                 throughput update, then NEE (light pick, point, shadow ray
//                 with its pending contribution) and BSDF sampling
//   k_miss        environment term of escaped paths
//   k_shadow      any-hit traversal; an occlusion byte per shadow ray
//   k_shadow_resolve  adds the pending NEE contributions of unoccluded rays
//   k_accumulate  per-pixel sum of the pass's samples in sample order
//
// Each path draws from its own PCG stream (stream = sample * W * H + pixel)
// in the reference's per-path order, so results do not depend on launch
// shape or queue order.
#pragma once

#include "ljx_feed.h"
#include "ljx_guide.h"
#include "ljx_shade.h"

namespace ljx {

constexpr int kNumMatTypes = 9;
constexpr int kBucketAny = 9;  // unsorted hits (below the sort threshold), shaded by runtime dispatch
constexpr int kBucketScatter = 10;  // volumetric paths that scatter in their medium
constexpr int kBucketMiss = 11;     // buckets from here on cast no shadow rays
constexpr int kBucketNoMat = 12;
constexpr int kNumBuckets = 13;
// counter slots
constexpr int C_EXT = 0;      // C_EXT + (0|1): extension queues
constexpr int C_BUCKET = 4;   // C_BUCKET + bucket: its paths
constexpr int C_HOST = C_BUCKET + kNumBuckets;  // the counters the host reads back
// ticket counters (Feed), in sets: two for the closest-hit launches, used in
// turn by the bounces, and one each for the bounce's other launches
constexpr int C_FEED = 32;
static_assert(C_HOST <= C_FEED && C_FEED % kFeedLine == 0, "queue counters share no line with tickets");
constexpr int C_FEED_SHADOW = C_FEED + 2 * kFeedSet;
constexpr int C_FEED_WALK = C_FEED + 3 * kFeedSet;
constexpr int C_FEED_FLIGHT = C_FEED + 4 * kFeedSet;
constexpr int C_ALLOC = C_FEED + 5 * kFeedSet;

// One job of a batched render: its camera, image and place in the batch's
// global work index space (sample-major over its 8x8-tiled pixel grid).
struct BatchJob {
    CameraRec camera;
    long long work_base;
    long long valid_base;  // pixels' samples (W * H * spp) of the jobs before it
    int W, H, ntx8, npix8;
    int spp, pad;
    uint64_t seed;
    double *accum;    // W * H * 3
    float *out;       // W * H * 3
};
// 64-bit statistics slots
constexpr int S_EXT_RAYS = 0, S_SH_RAYS = 1, S_NODES = 2, S_PRIMS = 3, S_SH_NODES = 4, S_SH_PRIMS = 5,
              S_GUIDE_Q = 6, S_NUM = 8;

struct PathBufs {
    uint64_t *rng;
    float4 *tp;       // throughput rgb, eta_scale
    float4 *rad;      // radiance rgb
    float4 *prev;     // f (with cosine) of the last BSDF sample, its solid-angle pdf
    int *depth;       // index b of the vertex a path's current ray will hit (0: primary)
    float4 *ray_o;    // origin, tnear
    float4 *ray_d;    // direction, tfar
    float4 *hit;      // t, u, v, slot (int bits; -1: miss)
    uint32_t *extq0, *extq1;
    uint8_t *key;     // per extension-queue entry: its hit's bucket
    uint32_t *order;  // the extension queue's paths by bucket, each bucket in queue order
    int *sort_blk;    // per bucket, per kScanBlock queue entries: paths, then their exclusive prefix
    float4 *sh_o, *sh_d, *sh_c;
    uint8_t *sh_occ;  // per shadow ray: 0 unoccluded (or not traced yet), 1 occluded, kShNone where there is none
    unsigned long long *wave_stat;  // per wave of the traversal grid: shadow rays traced
    int waves;                      // its length
    uint8_t *alive;   // per path slot: 1 when shading gave it another ray (cleared as the queue is built)
    int *alive_blk;   // per kScanBlock slots: live paths, then their exclusive prefix
    // volumetric path state
    int *medium;      // current medium id
    float4 *nee_c;    // nee_p_cache xyz, dir_pdf
    float4 *mtp;      // multi_trans_pdf rgb, never_scatter (1/0)
    float4 *sh_x;     // shadow walk: pdf_nee, pdf_dir, NEE stream state (lo, hi bits)
    double4 *vf_t;    // free flight: transmittance rgb, distance travelled
    double4 *vf_p;    // free flight: transmittance pdf rgb, 1 if it ended in a real collision
    int *ctr;
    unsigned long long *stat;
    int *spill;
    double *accum;    // W * H * 3
    int capacity;
    // image / pass
    int W, H, ntx8;
    int pass_s0, pass_ns, pass_q0, pass_nq;
    int spp, max_depth, rr_depth;
    int volpath;
    int vol_flight;  // free flight runs in k_vol_flight (scenes with grid media), else in k_vol_event and k_vol_shade
    int vol_grey;    // every medium is a grid of one density channel
    int max_null;
    uint64_t seed;
    // learned guiding (path integrator)
    float4 *glob;      // capacity x 8 lobes: kappa * mean xyz, log constant (pdf = exp(dot + c))
    float4 *gdir;      // guide-sampled direction xyz; w: 1 from the guide, 0 from the BSDF, -1 not guided
    float4 *rec_feat;  // rec_depth x capacity x 2: network features of each vertex
    float4 *rec_dir;   // rec_depth x capacity: sampled direction xyz; w: 1 if a training sample
    float4 *rec_beta;  // rec_depth x capacity: throughput at the vertex
    float4 *rec_c;     // rec_depth x capacity: radiance the vertex adds (emission, NEE, environment)
    int rec_depth;     // vertices recorded per path (0: not recording)
    int rec_stride;    // record arrays are [vertex][slot]: the pass's slot count
    uint32_t guide_mask;  // material types sampled from the mixture
    float guide_mix;   // probability of the guide in the mixture
    float box_lo[3], box_scale[3];  // position features: (p - lo) * scale
    // batched rendering: slot i of a pass holds global work item work0 + i
    const BatchJob *jobs;  // null for a single render
    int njobs;
    int sort_threshold;    // bounces with fewer extension rays skip the material sort
    long long work0;
    // slots of the pass that hold a pixel (the others pad 8x8 tiles), and how
    // many such slots lie before the pass (batch: before work0; single render:
    // in the tiles before pass_q0)
    int pass_valid;
    long long valid0;
};

// A vertex's shadow ray is written at its path's place in P.order; places
// without one carry this mark in sh_occ.
constexpr uint8_t kShNone = 3;
// Shadow-queue entries carry the path slot in the low kSlotBits bits and the
// vertex index in the rest (clamped there: only the guiding record, a few
// vertices deep, reads it).
constexpr int kSlotBits = 26;
constexpr uint32_t kSlotMask = (1u << kSlotBits) - 1;
// Material types never guided: their lobes are near-specular transmission.
__host__ __device__ constexpr bool guidable(int mt) { return mt != 2 && mt != 5; }

// The camera path held by slot i: its job (0 for a single render), sample
// index, pixel, and its PCG stream, path_stream(s * W * H + y * W + x).
struct SlotInfo {
    int job, s, x, y, W, H;
    bool valid;
    __device__ uint64_t stream() const {
        return path_stream(uint64_t(s) * uint64_t(W) * uint64_t(H) + uint64_t(y) * W + x);
    }
};
__device__ __forceinline__ SlotInfo slot_info(const PathBufs &P, int i) {
    SlotInfo r;
    int q, ntx8;
    if (P.jobs) {
        long long w = P.work0 + i;
        int lo = 0, hi = P.njobs - 1;  // last job with work_base <= w
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (P.jobs[mid].work_base <= w) lo = mid;
            else hi = mid - 1;
        }
        const BatchJob &J = P.jobs[lo];
        long long local = w - J.work_base;
        r.job = lo;
        r.s = int(local / J.npix8);
        q = int(local % J.npix8);
        ntx8 = J.ntx8;
        r.W = J.W;
        r.H = J.H;
    } else {
        r.job = 0;
        r.s = P.pass_s0 + i / P.pass_nq;
        q = P.pass_q0 + i % P.pass_nq;
        ntx8 = P.ntx8;
        r.W = P.W;
        r.H = P.H;
    }
    int tile = q >> 6, w = q & 63;
    r.x = (tile % ntx8) * 8 + (w & 7);
    r.y = (tile / ntx8) * 8 + (w >> 3);
    r.valid = r.x < r.W && r.y < r.H;
    return r;
}

// Pixels of the 8x8-tiled index space before tiled pixel (x, y) of a W x H
// image: whole tile rows, whole tiles of this row, rows and pixels within the
// tile (the last tile row and column may be narrower than 8).
__host__ __device__ inline long long tiled_rank(int x, int y, int W, int H) {
    const int x0 = x & ~7, y0 = y & ~7;
    const int tw = W - x0 < 8 ? W - x0 : 8, th = H - y0 < 8 ? H - y0 : 8;
    return (long long)y0 * W + (long long)x0 * th + (y - y0) * tw + (x - x0);
}
// The same for a tiled pixel index q of any slot, padding included.
__host__ __device__ inline long long tiled_rank_q(long long q, int ntx8, int W, int H) {
    const long long tile = q >> 6;
    const int w = int(q & 63), ty = int(tile / ntx8), tx = int(tile % ntx8);
    if (8 * ty >= H) return (long long)W * H;
    const int tw = W - 8 * tx < 8 ? W - 8 * tx : 8, th = H - 8 * ty < 8 ? H - 8 * ty : 8;
    const int r = w >> 3, c = w & 7;
    return 8ll * ty * W + 8ll * tx * th + (r < th ? r * tw + (c < tw ? c : tw) : th * tw);
}

// Counter resets folded into kernels that do not read those counters.
__global__ void k_reset_counters(int *ctr, int first, int count) {
    for (int i = threadIdx.x; i < count; i += blockDim.x) ctr[first + i] = 0;
}

// The next bounce's extension queue: the slots shading marked alive, in slot
// order (a stable compaction), so that neighbouring lanes of the next
// bounce's kernels read neighbouring path state and trace rays from
// neighbouring pixels.  Three launches over the pass's n slots: counts per
// kScanBlock slots, their exclusive scan (which also sets the queue's
// length), and the scatter, which clears the flags it read.
constexpr int kScanBlock = 4096;  // 256 threads x 16 slots
__device__ __forceinline__ int alive_in(uint4 f) {
    // flags are 0 or 1 bytes
    return __popc(f.x) + __popc(f.y) + __popc(f.z) + __popc(f.w);
}
__device__ __forceinline__ int block_excl_scan(int v, int &total) {
    __shared__ int wsum[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int before = 0;
    total = 0;
    for (int k = 0; k < 4; k++) {
        if (k < w) before += wsum[k];
        total += wsum[k];
    }
    __syncthreads();
    return before + x - v;
}
// Clears the flags of a pass's n slots (rounded up to 16); the scatter keeps
// them clear from then on.
__global__ __launch_bounds__(256) void k_alive_clear(PathBufs P, int n) {
    const int n16 = (n + 15) / 16;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += gridDim.x * blockDim.x)
        reinterpret_cast<uint4 *>(P.alive)[i] = make_uint4(0, 0, 0, 0);
}
__global__ __launch_bounds__(256) void k_alive_count(PathBufs P, int n) {
    const int s0 = blockIdx.x * kScanBlock + threadIdx.x * 16;
    const int c = s0 < n ? alive_in(*reinterpret_cast<const uint4 *>(P.alive + s0)) : 0;
    int total;
    block_excl_scan(c, total);
    if (threadIdx.x == 0) P.alive_blk[blockIdx.x] = total;
}
// Exclusive scan in place of n <= 16384 counts by one block of 1,024 threads
// x 16 counts; returns the total in the last thread.
__device__ __forceinline__ int scan_blocks(int *blk, int n) {
    __shared__ int part[1024];
    const int b0 = threadIdx.x * 16;
    int v[16], sum = 0;
    for (int k = 0; k < 16; k++) {
        v[k] = b0 + k < n ? blk[b0 + k] : 0;
        sum += v[k];
    }
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int y = threadIdx.x >= o ? part[threadIdx.x - o] : 0;
        __syncthreads();
        part[threadIdx.x] += y;
        __syncthreads();
    }
    int run = part[threadIdx.x] - sum;
    for (int k = 0; k < 16; k++) {
        if (b0 + k < n) blk[b0 + k] = run;
        run += v[k];
    }
    return part[threadIdx.x];
}
__global__ __launch_bounds__(1024) void k_alive_scan(PathBufs P, int nblk, int cur) {
    const int total = scan_blocks(P.alive_blk, nblk);
    if (threadIdx.x == 1023) P.ctr[C_EXT + (cur ^ 1)] = total;
}
__global__ __launch_bounds__(256) void k_alive_scatter(PathBufs P, int n, int cur) {
    uint32_t *next = cur ? P.extq0 : P.extq1;
    const int s0 = blockIdx.x * kScanBlock + threadIdx.x * 16;
    uint4 f = make_uint4(0, 0, 0, 0);
    if (s0 < n) f = *reinterpret_cast<const uint4 *>(P.alive + s0);
    int total;
    int k = P.alive_blk[blockIdx.x] + block_excl_scan(alive_in(f), total);
    if (s0 < n && (f.x | f.y | f.z | f.w)) {
        const uint32_t w[4] = {f.x, f.y, f.z, f.w};
        for (int j = 0; j < 16; j++)
            if ((w[j >> 2] >> (8 * (j & 3))) & 0xffu) next[k++] = uint32_t(s0 + j);
        *reinterpret_cast<uint4 *>(P.alive + s0) = make_uint4(0, 0, 0, 0);
    }
}

// The material sort of a bounce: a stable counting sort of the extension
// queue's n entries by the keys k_extend wrote.  Appending each path to its
// bucket's queue inside the traversal costs one atomic instruction per wave
// on a counter line that every wave of the chip shares; such instructions run
// one every 11.3 ns whatever their lanes, so 67M paths spent 12 ms there
// (with Feed's counters: closest hits of a 1,048,576-path Cornell render 1.40
// -> 0.34 ms, of the 1080p 64-sample terrain 70.4 -> 56.8 ms; the sort adds
// 0.14 and 1.3 ms).
// Three launches: counts per kScanBlock entries and bucket, their exclusive
// scans (one block per bucket, which also sets the bucket's length), and the
// scatter.  Buckets end up in queue order, so their paths' state stays near
// coalesced.
constexpr int kSortRows = kScanBlock / 256;  // a wave's 1,024 entries: 16 rows of 64
// Wave-level ranks of a wave's rows of keys: rank[r] is the entry's place
// among the wave's entries of its key; lane b returns the count of key b.
__device__ __forceinline__ int sort_ranks(const int (&key)[kSortRows], int (&rank)[kSortRows]) {
    const int lane = __lane_id();
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < kSortRows; r++) {
        uint64_t pending = __ballot(key[r] >= 0);
        rank[r] = 0;
        while (pending) {
            const int k = __builtin_amdgcn_readlane(key[r], __ffsll((unsigned long long)pending) - 1);
            const uint64_t m = __ballot(key[r] == k);
            const int before = __builtin_amdgcn_readlane(cnt, k);
            if (key[r] == k)
                rank[r] = before + int(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0)));
            if (lane == k) cnt += __popcll(m);
            pending &= ~m;
        }
    }
    return cnt;
}
__device__ __forceinline__ int sort_load(const PathBufs &P, int n, int (&key)[kSortRows]) {
    const int i0 = blockIdx.x * kScanBlock + (threadIdx.x >> 6) * (64 * kSortRows) + (threadIdx.x & 63);
#pragma unroll
    for (int r = 0; r < kSortRows; r++) key[r] = i0 + 64 * r < n ? P.key[i0 + 64 * r] : -1;
    return i0;
}
__global__ __launch_bounds__(256) void k_sort_count(PathBufs P, int cur, int nblk) {
    __shared__ int wcnt[4][kNumBuckets];
    const int n = P.ctr[C_EXT + cur];
    if (blockIdx.x * kScanBlock >= n) return;
    int key[kSortRows], rank[kSortRows];
    sort_load(P, n, key);
    const int cnt = sort_ranks(key, rank), lane = threadIdx.x & 63;
    if (lane < kNumBuckets) wcnt[threadIdx.x >> 6][lane] = cnt;
    __syncthreads();
    const int b = threadIdx.x;
    if (b < kNumBuckets) P.sort_blk[size_t(b) * nblk + blockIdx.x] = wcnt[0][b] + wcnt[1][b] + wcnt[2][b] + wcnt[3][b];
}
__global__ __launch_bounds__(1024) void k_sort_scan(PathBufs P, int cur, int nblk) {
    // 1024 threads x 16 blocks each: at most 16384 blocks (n <= 2^26)
    const int live = (P.ctr[C_EXT + cur] + kScanBlock - 1) / kScanBlock;
    const int total = scan_blocks(P.sort_blk + size_t(blockIdx.x) * nblk, live);
    if (threadIdx.x == 1023) P.ctr[C_BUCKET + blockIdx.x] = total;
}
// Where bucket b starts in P.order.
__device__ __forceinline__ int bucket_start(const PathBufs &P, int b) {
    int s = 0;
    for (int k = 0; k < b; k++) s += P.ctr[C_BUCKET + k];
    return s;
}
__global__ __launch_bounds__(256) void k_sort_scatter(PathBufs P, int cur, int nblk) {
    __shared__ int wcnt[4][kNumBuckets], place[4][kNumBuckets];
    const int n = P.ctr[C_EXT + cur];
    if (blockIdx.x * kScanBlock >= n) return;
    const uint32_t *q = cur ? P.extq1 : P.extq0;
    int key[kSortRows], rank[kSortRows];
    const int i0 = sort_load(P, n, key);
    const int cnt = sort_ranks(key, rank), lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane < kNumBuckets) wcnt[w][lane] = cnt;
    __syncthreads();
    if (threadIdx.x < 4 * kNumBuckets) {
        const int ww = threadIdx.x / kNumBuckets, b = threadIdx.x % kNumBuckets;
        int at = bucket_start(P, b) + P.sort_blk[size_t(b) * nblk + blockIdx.x];
        for (int k = 0; k < ww; k++) at += wcnt[k][b];
        place[ww][b] = at;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; r++)
        if (key[r] >= 0) P.order[place[w][key[r]] + rank[r]] = q[i0 + 64 * r];
}

__global__ void k_fill_f64(double *p, size_t n) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    size_t stride = size_t(gridDim.x) * blockDim.x;
    for (; i < n; i += stride) p[i] = 0.0;
}

// Camera rays of the pass.  The first extension queue lists the slots that
// hold a pixel, in slot order: a slot's place in it has a closed form
// (tiled_rank), so padded tiles cost no atomics (appending them with one
// atomic per wave ran at 11 ns an atomic, all waves on one counter: 4.9 ms of
// 28 for 19.5M paths at 637x479, where this takes 0.7 ms).
__global__ void k_raygen(DeviceScene S, PathBufs P) {
    int n = P.pass_ns * P.pass_nq;
    int stride = gridDim.x * blockDim.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) P.ctr[C_EXT + 0] = P.pass_valid;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        P.rad[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        const SlotInfo si = slot_info(P, i);
        if (!si.valid) continue;
        uint64_t stream = si.stream();
        uint64_t inc = pcg_inc(stream);
        uint64_t st = pcg_init_state(stream, P.jobs ? P.jobs[si.job].seed : P.seed);
        double r0 = pcg_double(st, inc), r1 = pcg_double(st, inc);
        D3 o, d;
        const CameraRec &cam = P.jobs ? P.jobs[si.job].camera : S.camera;
        sample_primary(cam, (si.x + r0) / si.W, (si.y + r1) / si.H, o, d);
        P.rng[i] = st;
        P.ray_o[i] = make_float4(float(o.x), float(o.y), float(o.z), 0.0f);
        P.ray_d[i] = make_float4(float(d.x), float(d.y), float(d.z), __builtin_huge_valf());
        P.tp[i] = make_float4(1.f, 1.f, 1.f, 1.f);
        P.prev[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        P.depth[i] = 0;
        const long long rank = tiled_rank(si.x, si.y, si.W, si.H);
        const long long k = P.jobs ? P.jobs[si.job].valid_base + (long long)si.s * si.W * si.H + rank - P.valid0
                                   : (long long)(si.s - P.pass_s0) * (P.pass_valid / P.pass_ns) + rank - P.valid0;
        P.extq0[k] = uint32_t(i);
    }
}

// Closest-hit traversal of the extension queue: a wave walks 64 rays (Feed)
// until the last one ends; each hit's distance is refined while its triangle
// is in cache, and each queue entry gets the key of the material it hit.
// (Refilling lanes as their rays end, as k_shadow does, measured slower here:
// the refill points run the finishing work divergently.)
// The feed counters of a launch start at zero: k_reset_counters clears every
// counter at a pass's start and each launch clears the set the next launch
// uses.
template <bool STATS, bool SPH>
__device__ __forceinline__ int extend_finish(const DeviceScene &S, const PathBufs &P, uint32_t pid,
                                             const Tracer<false, STATS, SPH> &tr, bool sorted) {
    int bucket;
    if (tr.found) {
        TraceHit h = tr.hit;
        // the direction again for the FP64 distance (kept out of the
        // traversal's registers when no spheres need it there)
        const float4 d2 = SPH ? make_float4(tr.dx, tr.dy, tr.dz, 0.f) : P.ray_d[pid];
        h.t = refine_t<SPH>(S.prims, h.slot, h.t, tr.r.ox, tr.r.oy, tr.r.oz, d2.x, d2.y, d2.z);
        P.hit[pid] = make_float4(h.t, h.u, h.v, __int_as_float(h.slot));
        const int sb = S.slot_bucket[h.slot];
        // textured materials are shaded by the runtime-dispatch kernel
        bucket = (sorted || sb >= kNumMatTypes) ? sb : kBucketAny;
    } else {
        P.hit[pid] = make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
        bucket = kBucketMiss;
    }
    return bucket;
}

// Triangle-only scenes: capped at 64 registers, eight waves per SIMD (the
// LDS stacks allow eight), at the cost of a 16-byte spill; scenes with
// spheres need the FP64 root solve's registers and keep their own count.
template <bool STATS, bool SPH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPH ? 1 : 8))) void k_extend(DeviceScene S, PathBufs P, int cur) {
    __shared__ int stack[kStackLds * 256];
    const uint32_t *q = cur ? P.extq1 : P.extq0;
    const int n = P.ctr[C_EXT + cur];
    const bool sorted = n >= P.sort_threshold;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(&P.stat[S_EXT_RAYS], (unsigned long long)n);
    }
    int *feeds = P.ctr + C_FEED;
    if (blockIdx.x == 0 && threadIdx.x < kFeeds) {
        feeds[(cur ^ 1) * kFeedSet + threadIdx.x * kFeedLine] = 0;
        P.ctr[C_FEED_SHADOW + threadIdx.x * kFeedLine] = 0;
        P.ctr[C_FEED_WALK + threadIdx.x * kFeedLine] = 0;
        P.ctr[C_FEED_FLIGHT + threadIdx.x * kFeedLine] = 0;
    }
    const TraceScene ts{S.qnodes, S.prims, S.spheres};
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int sstride = gridDim.x * blockDim.x;
    int *spill = P.spill + gtid;
    const int lane = __lane_id();
    uint32_t nn = 0, np = 0;
    Feed feed;
    feed.start(feeds + cur * kFeedSet, n);
    for (int base = feed.base(); base < n; feed.next(), base = feed.base()) {
        const int i = base + lane;
        if (i < n) {
            const uint32_t pid = q[i];
            const float4 o = P.ray_o[pid], d = P.ray_d[pid];
            Tracer<false, STATS, SPH> tr;
            tr.start(o.x, o.y, o.z, d.x, d.y, d.z, o.w, d.w);
            if (S.num_nodes > 0)
                while (!tr.step(ts, stack + threadIdx.x, blockDim.x, spill, sstride, nn, np)) {
                }
            const int bucket = extend_finish<STATS, SPH>(S, P, pid, tr, sorted);
            if (!P.volpath) P.key[i] = uint8_t(bucket);
        }
    }
    if (STATS) {
        atomicAdd(&P.stat[S_NODES], (unsigned long long)nn);
        atomicAdd(&P.stat[S_PRIMS], (unsigned long long)np);
    }
}

// Pending NEE contribution and the next ray of one path vertex.
template <int MT, bool SPH, bool GUIDE>
__device__ __forceinline__ void shade_surface(const DeviceScene &S, const PathBufs &P, uint32_t pid, bool &push_ext,
                                              bool &push_sh, float4 &sh_o, float4 &sh_d, float4 &sh_c) {
    float4 h = P.hit[pid];
    float4 ro = P.ray_o[pid], rd = P.ray_d[pid];
    D3 org = f3d(ro), dir = f3d(rd);
    int b = P.depth[pid];
    uint64_t st = P.rng[pid];
    const uint64_t inc = pcg_inc(slot_info(P, int(pid)).stream());
    float4 tp4 = P.tp[pid];
    D3 tp{tp4.x, tp4.y, tp4.z};
    double eta_scale = tp4.w;
    float4 rad4 = P.rad[pid];
    D3 rad{rad4.x, rad4.y, rad4.z};
    Vertex v = make_vertex<SPH>(S, __float_as_int(h.w), h.x, h.y, h.z, org, dir);
    // constant materials are read in place; the runtime-dispatch kernel, which
    // also takes textured ones, works on a copy with the textures evaluated
    // (the footprint is nonzero on camera rays only, path_tracing.h:14-16)
    MatRec mat_tex;
    if constexpr (MT < 0) {
        mat_tex = S.materials[v.material_id];
        if (mat_tex.textured) {
            double fp = 0;
            if (b == 0) {
                const SlotInfo si = slot_info(P, int(pid));
                fp = (0.25 / double(max(si.W, si.H))) * sqrt(dist2(org, v.pos)) / v.inv_uv;
            }
            resolve_textures(S, mat_tex, v.tu, v.tv, fp);
        }
    }
    const MatRec &mat = MT < 0 ? mat_tex : S.materials[v.material_id];
    bool alive = true;
    push_ext = false;
    push_sh = false;
    // guided vertex: directions come from the mixture (1 - a) BSDF + a guide
    bool guided = false;
    float4 gd = make_float4(0.f, 0.f, 0.f, -1.f);
    const float4 *lobes = nullptr;
    const double alpha = GUIDE ? double(P.guide_mix) : 0.0;
    if (GUIDE && guidable(MT >= 0 ? MT : int(mat.type))) {
        gd = P.gdir[pid];
        guided = gd.w >= 0.f;
        lobes = P.glob + size_t(pid) * guide::kLobes;
    }
    const bool rec = GUIDE && b < P.rec_depth;
    const size_t rix = size_t(b) * P.rec_stride + pid;
    D3 rad_in = rad;
    if (b == 0) {
        // path_tracing.h:58-61
        if (v.area_light_id >= 0)
            rad = rad + tp * light_emission<MT == kMtEnv>(S.lights[v.area_light_id], -dir, LightPoint{v.pos, v.g.ng});
    } else {
        // path_tracing.h:243-322 for the vertex reached by the previous sample
        float4 pv = P.prev[pid];
        D3 f{pv.x, pv.y, pv.z};
        double pdf = pv.w;
        double G = fabs(dot(dir, v.g.ng)) / dist2(v.pos, org);
        double p2 = pdf * G;
        if (v.area_light_id >= 0) {
            const LightRec &l = S.lights[v.area_light_id];
            LightPoint lp{v.pos, v.g.ng};
            D3 L = light_emission<MT == kMtEnv>(l, -dir, lp);
            D3 C2 = G * f * L;
            double p1 = S.light_pmf[v.area_light_id] * pdf_light_point<SPH, MT == kMtEnv>(S, l, lp, org);
            double w2 = (p2 * p2) / (p1 * p1 + p2 * p2);
            C2 = C2 / p2;
            rad = rad + tp * C2 * w2;
        }
        double rr = 1;
        if (b + 1 >= P.rr_depth) {
            rr = fmin(maxc((1 / eta_scale) * tp), 0.95);
            if (pcg_double(st, inc) > rr) alive = false;
        }
        if (alive) tp = tp * (G * f) / (p2 * rr);
    }
    if (rec) {
        D3 add = rad - rad_in;
        P.rec_c[rix] = make_float4(float(add.x), float(add.y), float(add.z), 0.f);
    }
    if (alive && !(P.max_depth == -1 || b + 3 <= P.max_depth + 1)) alive = false;
    if (alive && S.num_lights == 0) {
        // the reference asserts on an empty light table (src/table_dist.cpp:29); end the path
        alive = false;
    }
    if (alive) {
        // next-event estimation (path_tracing.h:96-207)
        double lu0 = pcg_double(st, inc), lu1 = pcg_double(st, inc);
        double lw = pcg_double(st, inc), sw = pcg_double(st, inc);
        int lid = sample_cdf_guided(S.light_cdf, S.num_lights, lw, S.light_guide, S.light_guide_m);
        const LightRec &l = S.lights[lid];
        D3 dir_light, L;
        double G = 0, tfar, lpdf;
        if (l.type == 0) {
            LightPoint lp = sample_shape<SPH>(S, S.shapes[l.shape_id], v.pos, lu0, lu1, sw);
            dir_light = normalize(lp.pos - v.pos);
            double dl = sqrt(dist2(lp.pos, v.pos));
            tfar = (1 - S.eps) * dl;
            G = fmax(-dot(dir_light, lp.n), 0.0) / dist2(lp.pos, v.pos);
            lpdf = pdf_shape<SPH>(S.shapes[l.shape_id], lp, v.pos);
            L = dot(lp.n, -dir_light) > 0 ? l.intensity : D3{0, 0, 0};
        } else {
            env_nee(l, lu0, lu1, dir_light, lpdf, L);
            tfar = __builtin_huge_val();
            G = 1;
        }
        double p1 = S.light_pmf[lid] * lpdf;
        D3 dir_view = -dir;
        if (G > 0 && p1 > 0) {
            D3 f = bsdf_eval<MT>(mat, dir_view, dir_light, v.g);
            D3 C1 = G * f * L;
            double pb = bsdf_pdf<MT>(mat, dir_view, dir_light, v.g);
            if (guided)
                pb = (1 - alpha) * pb +
                     alpha * double(guide::mixture_pdf(lobes, float(dir_light.x), float(dir_light.y), float(dir_light.z)));
            double p2 = pb * G;
            double w1 = (p1 * p1) / (p1 * p1 + p2 * p2);
            C1 = C1 / p1;
            D3 c = tp * C1 * w1;
            if (c.x != 0 || c.y != 0 || c.z != 0) {
                push_sh = true;
                sh_o = make_float4(float(v.pos.x), float(v.pos.y), float(v.pos.z), float(S.eps));
                sh_d = make_float4(float(dir_light.x), float(dir_light.y), float(dir_light.z), float(tfar));
                sh_c = make_float4(float(c.x), float(c.y), float(c.z),
                                   __int_as_float(int(pid | (uint32_t(min(b, (1 << (32 - kSlotBits)) - 1)) << kSlotBits))));
            }
        }
        // BSDF sampling (path_tracing.h:209-259)
        double bu0 = pcg_double(st, inc), bu1 = pcg_double(st, inc), bw = pcg_double(st, inc);
        BsdfSample bs;
        if (guided && gd.w > 0.5f) {
            // drawn from the guide by k_guide_infer; the BSDF draws above keep
            // the path's stream aligned with the unguided tracer
            bs.valid = true;
            bs.dir = normalize(D3{double(gd.x), double(gd.y), double(gd.z)});
            bs.eta = 0;
        } else {
            bs = bsdf_sample<MT>(mat, dir_view, v.g, bu0, bu1, bw);
        }
        if (!bs.valid) {
            alive = false;
        } else {
            if (bs.eta != 0) eta_scale /= (bs.eta * bs.eta);
            D3 f = bsdf_eval<MT>(mat, dir_view, bs.dir, v.g);
            double pdf = bsdf_pdf<MT>(mat, dir_view, bs.dir, v.g);
            if (guided) {
                // one-sample MIS over the two strategies (balance heuristic):
                // the path weight is f / mixture pdf
                pdf = (1 - alpha) * pdf +
                      alpha * double(guide::mixture_pdf(lobes, float(bs.dir.x), float(bs.dir.y), float(bs.dir.z)));
                if (f.x == 0 && f.y == 0 && f.z == 0) pdf = 0;  // nothing more can be added
            }
            if (pdf <= 0) {
                alive = false;
            } else {
                P.prev[pid] = make_float4(float(f.x), float(f.y), float(f.z), float(pdf));
                P.ray_o[pid] = make_float4(float(v.pos.x), float(v.pos.y), float(v.pos.z), float(S.eps));
                P.ray_d[pid] = make_float4(float(bs.dir.x), float(bs.dir.y), float(bs.dir.z), __builtin_huge_valf());
                P.depth[pid] = b + 1;
                push_ext = true;
                if (rec && guided) {
                    P.rec_dir[rix] = make_float4(float(bs.dir.x), float(bs.dir.y), float(bs.dir.z), 1.f);
                    P.rec_beta[rix] = make_float4(float(tp.x), float(tp.y), float(tp.z), 0.f);
                }
            }
        }
    }
    P.rng[pid] = st;
    P.tp[pid] = make_float4(float(tp.x), float(tp.y), float(tp.z), float(eta_scale));
    P.rad[pid] = make_float4(float(rad.x), float(rad.y), float(rad.z), 0.f);
}

// MT = -1: the unsorted bucket, with the material type dispatched per path;
// kMtEnv: so for every bucket of hits.
template <int MT, bool SPH, bool GUIDE>
__device__ __forceinline__ void shade_queue(const DeviceScene &S, const PathBufs &P, int cur) {
    constexpr int B = MT >= 0 ? MT : MT == kMtEnv ? 0 : kBucketAny;
    const int start = bucket_start(P, B);
    const int n = MT == kMtEnv ? bucket_start(P, kBucketAny + 1) : P.ctr[C_BUCKET + B];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int j = start + i;
        const uint32_t pid = P.order[j];
        bool pe = false, ps = false;
        float4 so, sd, sc;
        shade_surface<MT, SPH, GUIDE>(S, P, pid, pe, ps, so, sd, sc);
        if (pe) P.alive[pid] = 1;
        // the shadow ray takes its path's place in the order: appending it to
        // a queue costs an atomic per wave on one counter (11.3 ns each, one
        // after the other: 38 of 122 ms for the 1080p terrain at 64 samples)
        P.sh_occ[j] = ps ? uint8_t(0) : kShNone;
        if (ps) {
            P.sh_o[j] = so;
            P.sh_d[j] = sd;
            P.sh_c[j] = sc;
        }
    }
}

// The shading kernel of one material type (or, MT < 0, of run-time dispatch).
// Occupancy of these FP64-heavy kernels is set by their register count:
// 185-204 for Lambertian, RoughPlastic, DisneyDiffuse, DisneyMetal and
// DisneySheen without spheres in the scene, 255 or 256 with them (up to 22
// spilled), hence two waves per SIMD; DisneyBSDF spills at two, but running
// beside the other types' kernels is faster there than at one (shading of the
// 1080p large-mesh render 42.1 -> 40.6 ms).  Three waves, which the first five reach with
// little spilling, are slower, 43.0 against 35.4 ms for the same shading: the
// kernels keep the vector-memory data unit 0.9 busy, and more waves beside
// DisneyBSDF's only take its share of it.
// RoughDielectric, DisneyGlass and DisneyClearcoat fit two waves without
// spheres (241-254 registers) and keep one with them (304-322).
constexpr int shade_waves(int mt, bool sph) { return mt < 0 || (sph && (mt == 2 || mt == 5 || mt == 6)) ? 1 : 2; }
template <int MT, bool SPH, bool GUIDE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(shade_waves(MT, SPH)))) void k_shade(
    DeviceScene S, PathBufs P, int cur) {
    shade_queue<MT, SPH, GUIDE>(S, P, cur);
}

// Escaped paths: environment emission with MIS (path_tracing.h:17-28, 284-302).
__global__ __launch_bounds__(256) void k_miss(DeviceScene S, PathBufs P) {
    int n = P.ctr[C_BUCKET + kBucketMiss];
    const uint32_t *q = P.order + bucket_start(P, kBucketMiss);
    if (S.envmap_light_id < 0) return;
    const LightRec &env = S.lights[S.envmap_light_id];
    int stride = gridDim.x * blockDim.x;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint32_t pid = q[i];
        float4 rd = P.ray_d[pid];
        D3 dir = f3d(rd);
        float4 tp4 = P.tp[pid];
        D3 tp{tp4.x, tp4.y, tp4.z};
        float4 r4 = P.rad[pid];
        D3 rad{r4.x, r4.y, r4.z};
        // the direction's lat-long coordinates serve the radiance and the pdf
        // (src/lights/envmap.inl:22-72)
        const D3 ld = xform3(env.to_local, dir);
        double eu, ev;
        env_uv(ld, eu, ev);
        D3 L = env_texel_bilinear(env, eu, ev) * env.scale;
        D3 rad_in = rad;
        int b = P.depth[pid];
        if (b == 0) {
            rad = rad + tp * L;
        } else {
            float4 pv = P.prev[pid];
            D3 f{pv.x, pv.y, pv.z};
            double p2 = pv.w;  // G = 1
            D3 C2 = f * L;
            const double se = sqrt(clampd(1 - ld.y * ld.y, 0, 1));
            const double epdf = se > 0 ? pdf_env_uv(env, eu, ev) / (2 * kPi * kPi * se) : 0.0;
            double p1 = S.light_pmf[S.envmap_light_id] * epdf;
            double w2 = (p2 * p2) / (p1 * p1 + p2 * p2);
            C2 = C2 / p2;
            rad = rad + tp * C2 * w2;
        }
        P.rad[pid] = make_float4(float(rad.x), float(rad.y), float(rad.z), 0.f);
        if (b < P.rec_depth) {
            D3 add = rad - rad_in;
            P.rec_c[size_t(b) * P.rec_stride + pid] = make_float4(float(add.x), float(add.y), float(add.z), 0.f);
        }
    }
}

// Hands a wave's lanes the entries of a queue one by one, passing over those
// that need no work: chunks of 64 entries from a Feed, the entries of a chunk
// to work on gathered in `list` (lane k holds the k-th of them).
struct FeedRange {
    Feed feed;
    int n, list, at, count;
    bool fresh;  // the feed's current chunk has not been opened
    bool done;   // no entries are left
    __device__ __forceinline__ void start(int *counters, int n_, int tickets = 0) {
        n = n_;
        feed.start(counters, n, tickets);
        at = count = 0;
        fresh = true;
        done = false;
    }
    // One entry with valid(entry) for every lane that wants one, or -1 once
    // none are left.  All lanes of the wave must call it.
    template <class F>
    __device__ __forceinline__ int take(bool want, F &&valid) {
        int got = -1;
        uint64_t w = __ballot(want);
        auto below = [](uint64_t m) {
            return int(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0)));
        };
        while (w && !done) {
            if (at == count) {
                if (!fresh) feed.next();
                fresh = false;
                const int base = feed.base();
                if (base >= n) {
                    done = true;
                    break;
                }
                const int lane = __lane_id(), i = base + lane;
                const bool v = i < n && valid(i);
                const uint64_t m = __ballot(v);
                const int r = below(m);
                at = 0;
                count = __popcll(m);
                list = __builtin_amdgcn_ds_permute(4 * (v ? r : count + lane - r), i);
            }
            const int k = at + below(w);
            const int e = __shfl(list, k < 63 ? k : 63);
            if (want && got < 0 && k < count) got = e;
            at = min(count, at + __popcll(w));
            w = __ballot(want && got < 0);
        }
        return got;
    }
};

// Any-hit traversal of the bounce's shadow rays (the places of P.order up to
// the misses); writes whether each is occluded (k_shadow_resolve adds the
// contributions).  A lane whose ray ended takes its next one as soon as
// kShadowRefill lanes of its wave are idle, instead of waiting for the
// wave's longest ray (3.6% faster on the 1080p large-mesh render than
// starting the lanes' rays together).
constexpr int kShadowRefill = 16;
template <bool STATS, bool SPH>
__global__ __launch_bounds__(256) void k_shadow(DeviceScene S, PathBufs P) {
    __shared__ int stack[kStackLds * 256];
    const int n = bucket_start(P, kBucketMiss);
    const TraceScene ts{S.qnodes, S.prims, S.spheres};
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    int *spill = P.spill + gtid;
    uint32_t nn = 0, np = 0;
    Tracer<true, STATS, SPH> tr;
    bool busy = false, fin = false;
    FeedRange range;
    range.start(P.ctr + C_FEED_SHADOW, n);
    int i = 0, rays = 0;
    while (true) {
        const uint64_t idle = __ballot(!busy);
        const int nidle = __popcll(idle);
        if ((nidle >= kShadowRefill && !range.done) || nidle == 64) {
            if (fin) P.sh_occ[i] = tr.found ? 1 : 0;
            fin = false;
            const int k = range.take(!busy, [&](int j) { return P.sh_occ[j] != kShNone; });
            if (k >= 0) {
                i = k;
                const float4 o = P.sh_o[i], d = P.sh_d[i];
                tr.start(o.x, o.y, o.z, d.x, d.y, d.z, o.w, d.w);
                busy = true;
            }
            const int now = __popcll(__ballot(busy));
            rays += now - (64 - nidle);
            if (now == 0) break;
        }
        if (busy) {
            if (S.num_nodes == 0 || tr.step(ts, stack + threadIdx.x, blockDim.x, spill, stride, nn, np)) {
                busy = false;
                fin = true;
            }
        }
    }
    // (one slot per wave: an atomic per wave on a shared total takes 93 us a launch)
    if (__lane_id() == 0) P.wave_stat[gtid >> 6] += (unsigned long long)rays;
    if (STATS) {
        atomicAdd(&P.stat[S_SH_NODES], (unsigned long long)nn);
        atomicAdd(&P.stat[S_SH_PRIMS], (unsigned long long)np);
    }
}

// After k_shadow: an unoccluded shadow ray adds its pending NEE contribution
// to its path (and to the recorded radiance of its vertex when guiding
// records the pass).
__global__ __launch_bounds__(256) void k_shadow_resolve(PathBufs P) {
    const int n = bucket_start(P, kBucketMiss);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (P.sh_occ[i] != 0) continue;
        const float4 c = P.sh_c[i];
        const uint32_t bits = uint32_t(__float_as_int(c.w));
        const uint32_t pid = bits & kSlotMask;
        const float4 r = P.rad[pid];
        P.rad[pid] = make_float4(r.x + c.x, r.y + c.y, r.z + c.z, 0.f);
        const int b = int(bits >> kSlotBits);
        if (b < P.rec_depth) {
            float4 *rc = &P.rec_c[size_t(b) * P.rec_stride + pid];
            const float4 o = *rc;
            *rc = make_float4(o.x + c.x, o.y + c.y, o.z + c.z, 0.f);
        }
    }
}

// Render statistics: cleared at a render's start, and the waves' shadow rays
// added up at its end.
__global__ __launch_bounds__(1024) void k_reset_stats(PathBufs P) {
    if (threadIdx.x < S_NUM) P.stat[threadIdx.x] = 0;
    for (int i = threadIdx.x; i < P.waves; i += 1024) P.wave_stat[i] = 0;
}
__global__ __launch_bounds__(1024) void k_sum_stats(PathBufs P) {
    unsigned long long s = 0;
    for (int i = threadIdx.x; i < P.waves; i += 1024) s += P.wave_stat[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) atomicAdd(&P.stat[S_SH_RAYS], s);
}

// render.cpp:89-94 (path) and :136-145 (volpath drops non-finite samples).
__global__ void k_accumulate(PathBufs P) {
    int nq = P.pass_nq;
    int stride = gridDim.x * blockDim.x;
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < nq; j += stride) {
        SlotInfo si = slot_info(P, j);
        if (!si.valid) continue;
        const int x = si.x, y = si.y;
        double r = 0, g = 0, b = 0;
        for (int k = 0; k < P.pass_ns; k++) {
            float4 v = P.rad[k * nq + j];
            if (P.volpath && !(isfinite(v.x) && isfinite(v.y) && isfinite(v.z))) continue;
            r += v.x;
            g += v.y;
            b += v.z;
        }
        size_t o = (size_t(y) * P.W + x) * 3;
        P.accum[o] += r;
        P.accum[o + 1] += g;
        P.accum[o + 2] += b;
    }
}

// Batched renders: per-slot atomic sums into each job's image.
__global__ void k_accumulate_batch(PathBufs P, int n) {
    int stride = gridDim.x * blockDim.x;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        SlotInfo si = slot_info(P, i);
        if (!si.valid) continue;
        float4 v = P.rad[i];
        if (P.volpath && !(isfinite(v.x) && isfinite(v.y) && isfinite(v.z))) continue;
        double *a = P.jobs[si.job].accum + (size_t(si.y) * si.W + si.x) * 3;
        atomicAdd(a, double(v.x));
        atomicAdd(a + 1, double(v.y));
        atomicAdd(a + 2, double(v.z));
    }
}

__global__ void k_job_clear(const BatchJob *jobs, int j) {
    const BatchJob &J = jobs[j];
    size_t n = size_t(J.W) * J.H * 3;
    size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) J.accum[i] = 0.0;
}

__global__ void k_job_resolve(const BatchJob *jobs, int j) {
    const BatchJob &J = jobs[j];
    size_t n = size_t(J.W) * J.H * 3;
    double inv = 1.0 / double(J.spp);
    size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) J.out[i] = float(J.accum[i] * inv);
}

// Auxiliary integrators (src/render.cpp:12-69): one ray through each pixel
// centre; depth, shading normal, mean curvature, the camera ray
// differential (radius, spread) or the mipmap level (none with constant
// textures: black).  Misses are black.
template <bool SPH>
__global__ __launch_bounds__(256) void k_aux(DeviceScene S, PathBufs P, int mode, float *out) {
    __shared__ int stack[kStackLds * 256];
    const int n = P.W * P.H;
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    int *spill = P.spill + gtid;
    uint32_t nn = 0, np = 0;
    for (int i = gtid; i < n; i += stride) {
        int x = i % P.W, y = i / P.W;
        D3 o, d;
        sample_primary(S.camera, (x + 0.5) / P.W, (y + 0.5) / P.H, o, d);
        TraceHit h;
        bool hit = S.num_nodes > 0 &&
                   trace_ray<false, false, SPH>(TraceScene{S.qnodes, S.prims, S.spheres}, float(o.x), float(o.y),
                                                float(o.z), float(d.x), float(d.y), float(d.z), 0.f,
                                                __builtin_huge_valf(), stack + threadIdx.x, blockDim.x, spill, stride,
                                                h, nn, np);
        D3 c{0, 0, 0};
        if (hit) {
            Vertex v = make_vertex<SPH>(S, h.slot, h.t, h.u, h.v, o, d);
            if (mode == 0) {
                double dist = sqrt(dist2(v.pos, o));
                c = D3{dist, dist, dist};
            } else if (mode == 1) {
                c = v.g.sf.n;
            } else if (mode == 2) {
                double k = vertex_mean_curvature(S, h.slot, double(h.u), double(h.v), v);
                c = D3{k, k, k};
            } else if (mode == 3) {
                c = D3{0, 0.25 / double(max(P.W, P.H)), 0};  // init_ray_differential (src/ray.h:35-37)
            } else if (mode == 4 && v.material_id >= 0) {
                // the level the camera ray's footprint selects in the material's first colour
                // texture when it is an image (render.cpp:44-60; get_texture, material.cpp:121-123)
                const MatRec &m = S.materials[v.material_id];
                if (m.type != 6 && m.tex[0] && S.textures[m.tex[0] - 1].type == 1) {
                    const TexRec &t = S.textures[m.tex[0] - 1];
                    double fp = (0.25 / double(max(P.W, P.H))) * sqrt(dist2(v.pos, o)) / v.inv_uv;
                    double sf = max(t.w[0], t.h[0]) * fmax(t.uscale, t.vscale) * fp;
                    double level = log2(sf < double(1e-8f) ? double(1e-8f) : sf);
                    c = D3{level, level, level};
                }
            }
        }
        out[3 * size_t(i)] = float(c.x);
        out[3 * size_t(i) + 1] = float(c.y);
        out[3 * size_t(i) + 2] = float(c.z);
    }
}

__global__ void k_resolve(const double *accum, float *out, size_t n, double inv_spp) {
    size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = float(accum[i] * inv_spp);
}

}  // namespace ljx
