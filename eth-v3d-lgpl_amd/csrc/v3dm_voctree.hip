// Vocabulary-tree quantisation on gfx950: the greedy descent of
// VocabularyTree::findBestLeafIndex (V3D/Base/v3d_voctree.h:63-99) for many keys at once,
// level by level.
//
// Per level the keys are bucketed by their current node (a counting sort into buckets
// padded to 32 keys), so that a wave takes 32 keys with the same parent and scores them
// against the parent's children with v_mfma_f32_32x32x16_f16 on two FP16 parts of every
// component, as the matcher's split pass does (v3dm_split.h): the children are the A operand
// (32 per block, split once per tree, read straight from L2), the keys the resident B operand,
// split as they are loaded.  Keys are scaled by the power of two that puts their norm in
// [1, 2), nodes by the one that puts the largest node norm there.  The reference's choice is
// the first child of maximal sequential-FP32 score, which differs from the exact product by
// at most 128 * 2^-24 ||key|| ||node|| = 2^-17 ||key|| ||node||; the split score differs from it
// by at most (3 * 2^-22 + 24 * 2^-23) ||key|| ||node|| + 2^-39 sqrt(128) * 2 ||key|| max||node||
// < 2^-18 ||key|| max||node||; together less than eps = 2^-16 * ||key|| * max||node||, so a key
// whose best approximate score leads the second by more than 2 eps has the reference's child.
// The other keys (near ties, non-finite values, norms outside [2^-60, 2^60], scores near the
// -1e30 floor) are decided exactly: sequential FP32 sums with IEEE products, the scan's strict
// '>' (first index on ties, NaN never wins).
#include <algorithm>

#include "v3dm_device.h"
#include "v3dm_voctree.h"

namespace v3dm {

constexpr float kVtEpsRel = 1.52587890625e-05f;  // 2^-16
constexpr float kVtNormMin = 8.673617379884035e-19f, kVtNormMax = 1.152921504606847e18f;  // 2^-60, 2^60

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// x * scale = hi + lo (8 components)
__device__ __forceinline__ void vt_split8(float4 a, float4 b, float scale, v8h& hi, v8h& lo)
{
    float const f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float const x = f[k] * scale;
        hi[k] = (_Float16)x;
        lo[k] = (_Float16)(x - (float)hi[k]);
    }
}

// Node rows -> FP16 parts in the order in which the score kernel's lanes read them: tiles of 32
// rows, in a tile [matrix step s][part][half h][row] of 8 components, the dims
// 32 (s / 2) + 16 h + 8 (s % 2) + v.  One load of a wave is then one run of 1 KiB (two when the
// children straddle tiles).
__global__ __launch_bounds__(256) void k_vt_split_nodes(float const* __restrict__ nodes, long long rows, float scale,
                                                        unsigned char* __restrict__ split)
{
    int const c = threadIdx.x >> 4;  // dims [8 c, 8 c + 8)
    for (long long row = (long long)blockIdx.x * 16 + (threadIdx.x & 15); row < rows;
         row += (long long)gridDim.x * 16) {
        float4 const* x = reinterpret_cast<float4 const*>(nodes + (size_t)row * kDim) + 2 * c;
        v8h hi, lo;
        vt_split8(x[0], x[1], scale, hi, lo);
        int const s = 2 * (c >> 2) + (c & 1), h = (c >> 1) & 1;
        unsigned char* const o = split + (size_t)(row >> 5) * kVtTileBytes + s * 2048 + h * 512 + (row & 31) * 16;
        *reinterpret_cast<v8h*>(o) = hi;
        *reinterpret_cast<v8h*>(o + 1024) = lo;
    }
}

void launch_vt_split_nodes(float const* nodes, long long rows, float scale, unsigned char* split, hipStream_t st)
{
    hipLaunchKernelGGL(k_vt_split_nodes, dim3((unsigned)std::min((rows + 15) / 16, 65536LL)), dim3(256), 0, st, nodes, rows, scale,
                       split);
}

__global__ void k_vt_reset(int* counters)
{
    if (threadIdx.x < kVtCounters) counters[threadIdx.x] = 0;
}

void launch_vt_reset(int* counters, hipStream_t st)
{
    hipLaunchKernelGGL(k_vt_reset, dim3(1), dim3(64), 0, st, counters);
}

// ------------------------------------------------------------------------------ bucketing
// Bucket counts and the level's counters to zero, the order to "no key": one launch (three took
// 15 us a level).
__global__ __launch_bounds__(256) void k_vt_clear(int* __restrict__ cnt, int nCnt, int* __restrict__ order,
                                                  int nOrder, int* __restrict__ counters)
{
    int const t0 = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
    if (t0 < kVtCounters && t0 != kVtCntFlagged) counters[t0] = 0;
    for (int i = t0; i < nCnt; i += step) cnt[i] = 0;
    for (int i = t0; i < nOrder; i += step) order[i] = -1;
}

// Bucket counts live kVtBinStride ints apart (one L2 line per bucket): the global atomics
// of different buckets then never share a line.  For up to kVtLdsBins parents every
// work-group first counts its kVtKeysPerGroup keys in LDS and adds one total per bucket it
// saw; the scatter reserves each bucket's range for the work-group with one atomic and
// places the keys by their LDS rank.  Wider parent levels use one global atomic per key.
// What bounds both is the groups' atomics and latency: 1024 threads load their 8 keys together
// (count and scatter of 10^6 keys over 2500 parents 14 and 23 us); with 4 keys a thread, so
// twice the atomics, 21 and 31 us, with 256 threads taking 16 keys in turn 25 and 31 us.
constexpr int kVtGroup = 1024;
constexpr int kVtKeysPerThread = 8;
constexpr int kVtKeysPerGroup = kVtGroup * kVtKeysPerThread;

__device__ __forceinline__ int vt_bucket(int nd, int k, long long parentStart, int nParents,
                                         int* __restrict__ exactList, int* __restrict__ counters)
{
    if (nd == kVtNone) return -1;
    long long const b = (long long)nd - parentStart;
    if (b >= 0 && b < nParents) return (int)b;
    exactList[atomicAdd(&counters[kVtCntExact], 1)] = k;  // not a node of the parent level
    return -1;
}

__global__ __launch_bounds__(kVtGroup) void k_vt_count_lds(int const* __restrict__ node, int n,
                                                           long long parentStart, int nParents,
                                                           int* __restrict__ cnt, int* __restrict__ exactList,
                                                           int* __restrict__ counters)
{
    extern __shared__ int hist[];
    int const tid = threadIdx.x;
    for (int b = tid; b < nParents; b += kVtGroup) hist[b] = 0;
    __syncthreads();
    int const k0 = blockIdx.x * kVtKeysPerGroup;
    int nd[kVtKeysPerThread];
#pragma unroll
    for (int i = 0; i < kVtKeysPerThread; ++i) {
        int const k = k0 + i * kVtGroup + tid;
        nd[i] = k < n ? node[k] : kVtNone;
    }
#pragma unroll
    for (int i = 0; i < kVtKeysPerThread; ++i) {
        int const b = vt_bucket(nd[i], k0 + i * kVtGroup + tid, parentStart, nParents, exactList, counters);
        if (b >= 0) atomicAdd(&hist[b], 1);
    }
    __syncthreads();
    for (int b = tid; b < nParents; b += kVtGroup) {
        int const c = hist[b];
        if (c) atomicAdd(&cnt[(size_t)b * kVtBinStride], c);
    }
}

__global__ __launch_bounds__(kVtGroup) void k_vt_scatter_lds(int const* __restrict__ node, int n,
                                                             long long parentStart, int nParents,
                                                             int* __restrict__ cursor, int* __restrict__ order)
{
    extern __shared__ int hist[];
    int const tid = threadIdx.x;
    for (int b = tid; b < nParents; b += kVtGroup) hist[b] = 0;
    __syncthreads();
    int const k0 = blockIdx.x * kVtKeysPerGroup;
    int bin[kVtKeysPerThread], rank[kVtKeysPerThread];
#pragma unroll
    for (int i = 0; i < kVtKeysPerThread; ++i) {
        int const k = k0 + i * kVtGroup + tid;
        int const nd = k < n ? node[k] : kVtNone;
        long long const b = (long long)nd - parentStart;
        bin[i] = (nd != kVtNone && b >= 0 && b < nParents) ? (int)b : -1;
    }
#pragma unroll
    for (int i = 0; i < kVtKeysPerThread; ++i)
        if (bin[i] >= 0) rank[i] = atomicAdd(&hist[bin[i]], 1);
    __syncthreads();
    for (int b = tid; b < nParents; b += kVtGroup) {
        int const c = hist[b];
        if (c) hist[b] = atomicAdd(&cursor[(size_t)b * kVtBinStride], c);  // the group's range in the bucket
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kVtKeysPerThread; ++i)
        if (bin[i] >= 0) order[hist[bin[i]] + rank[i]] = k0 + i * kVtGroup + tid;
}

__global__ __launch_bounds__(256) void k_vt_count(int const* __restrict__ node, int n, long long parentStart,
                                                  int nParents, int* __restrict__ cnt, int* __restrict__ exactList,
                                                  int* __restrict__ counters)
{
    int const k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    int const b = vt_bucket(node[k], k, parentStart, nParents, exactList, counters);
    if (b >= 0) atomicAdd(&cnt[(size_t)b * kVtBinStride], 1);
}

// One work-group: exclusive prefix of the bucket sizes rounded up to 32 (so that no slot of
// 32 keys spans two buckets), slot count for the score kernel.
__global__ __launch_bounds__(1024) void k_vt_scan(int const* __restrict__ cnt, int nParents, int* __restrict__ cursor,
                                                  int* __restrict__ counters)
{
    __shared__ int part[1024];
    int const t = threadIdx.x;
    int const per = (nParents + 1023) / 1024;
    int const b0 = t * per, b1 = min(b0 + per, nParents);
    int s = 0;
    for (int b = b0; b < b1; ++b) s += (cnt[(size_t)b * kVtBinStride] + 31) & ~31;
    part[t] = s;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {  // Hillis-Steele inclusive scan
        int const v = (t >= o) ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - s;
    for (int b = b0; b < b1; ++b) {
        cursor[(size_t)b * kVtBinStride] = run;
        run += (cnt[(size_t)b * kVtBinStride] + 31) & ~31;
    }
    if (t == 1023) counters[kVtCntSlots] = part[1023] / 32;
}

__global__ __launch_bounds__(256) void k_vt_scatter(int const* __restrict__ node, int n, long long parentStart,
                                                    int nParents, int* __restrict__ cursor, int* __restrict__ order)
{
    int const k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    int const nd = node[k];
    if (nd == kVtNone) return;
    long long const b = (long long)nd - parentStart;
    if (b >= 0 && b < nParents) order[atomicAdd(&cursor[(size_t)b * kVtBinStride], 1)] = k;
}

void launch_vt_bucket(int const* node, int n, VtLevel const& lv, int* cnt, int* cursor, int* order, int orderCap,
                      int* exactList, int* counters, hipStream_t st)
{
    int const binInts = lv.nParents * kVtBinStride;
    hipLaunchKernelGGL(k_vt_clear, dim3(std::min((std::max(orderCap, binInts) + 255) / 256, 4096)), dim3(256), 0, st,
                       cnt, binInts, order, orderCap, counters);
    if (lv.nParents <= kVtLdsBins) {
        int const g = (n + kVtKeysPerGroup - 1) / kVtKeysPerGroup;
        size_t const lds = (size_t)lv.nParents * sizeof(int);
        hipLaunchKernelGGL(k_vt_count_lds, dim3(g), dim3(kVtGroup), lds, st, node, n, lv.parentStart, lv.nParents, cnt,
                           exactList, counters);
        hipLaunchKernelGGL(k_vt_scan, dim3(1), dim3(1024), 0, st, cnt, lv.nParents, cursor, counters);
        hipLaunchKernelGGL(k_vt_scatter_lds, dim3(g), dim3(kVtGroup), lds, st, node, n, lv.parentStart, lv.nParents,
                           cursor, order);
    } else {
        int const g = (n + 255) / 256;
        hipLaunchKernelGGL(k_vt_count, dim3(g), dim3(256), 0, st, node, n, lv.parentStart, lv.nParents, cnt,
                           exactList, counters);
        hipLaunchKernelGGL(k_vt_scan, dim3(1), dim3(1024), 0, st, cnt, lv.nParents, cursor, counters);
        hipLaunchKernelGGL(k_vt_scatter, dim3(g), dim3(256), 0, st, node, n, lv.parentStart, lv.nParents, cursor,
                           order);
    }
}

// ------------------------------------------------------------------------------ certified scores
// One block of 32 children as the A operand: a[2 s] the low, a[2 s + 1] the high parts.
__device__ __forceinline__ void vt_load_block(v8h (&a)[16], unsigned char const* __restrict__ nodes, long long row,
                                              int h)
{
    unsigned char const* const ap = nodes + (size_t)(row >> 5) * kVtTileBytes + h * 512 + (row & 31) * 16;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        a[2 * q] = *reinterpret_cast<v8h const*>(ap + q * 2048 + 1024);
        a[2 * q + 1] = *reinterpret_cast<v8h const*>(ap + q * 2048);
    }
}

// Wave = one slot of 32 keys with the same parent.  Lane l holds key l % 32 as the B operand;
// element v of matrix step s is dim 32 (s / 2) + 16 h + 8 (s % 2) + v (h = l / 32) on both
// sides.  Accumulator element r of lane l: child 8 (r / 4) + 4 h + r % 4 of the block, key
// l % 32.  Level 0 (identity) also forms the keys' norms.
//
// What bounds it: the keys' rows (512 bytes each, gathered in bucket order: 100 us for 10^6 at
// the card's copy rate).  The keys are loaded whole lines at a time and turned into operands
// through the wave's own LDS, a quarter of their dims at a time; the children come in operand
// order.  With every lane loading from its own row, for keys and children, the same kernel
// took 264-306 us a level (64 lines an instruction, each line fetched eight times), and the FP32
// matrix instructions 281-305 us besides a pass of 213 us for the norms; 121-150 us so.
__global__ __launch_bounds__(256, 3) void k_vt_score(float const* __restrict__ keys, float* __restrict__ keyNorm,
                                                     int n, unsigned char const* __restrict__ nodes,
                                                     float maxNodeNorm, int nodeExp, int usable, int branch,
                                                     int identity, int const* __restrict__ order,
                                                     int* __restrict__ node, int* __restrict__ exactList,
                                                     int* __restrict__ counters, float inf)
{
    __shared__ __attribute__((aligned(16))) float stages[4][32 * kExactRow];
    int const lane = threadIdx.x & 63;
    int const h = lane >> 5;
    int const c32 = lane & 31;
    int const slot = blockIdx.x * 4 + (threadIdx.x >> 6);
    int const nSlots = identity ? (n + 31) / 32 : counters[kVtCntSlots];
    if (slot >= nSlots) return;  // uniform per wave; the waves of a group share nothing
    float* const stage = stages[threadIdx.x >> 6];
    int kk;
    if (identity) kk = (slot * 32 + c32 < n) ? slot * 32 + c32 : -1;
    else kk = order[slot * 32 + c32];
    // an absent key repeats the slot's first one (read with all lanes active: lane 0 holds a key)
    int const first = __builtin_amdgcn_readfirstlane(kk);
    int const kr = kk >= 0 ? kk : first;
    // load u of a quarter: rows 8 u + l / 8, 16 bytes at column l % 8
    v4f in[16];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float const* const row = keys + (size_t)__shfl(kr, 8 * u + (lane >> 3)) * kDim + 4 * (lane & 7);
#pragma unroll
        for (int p = 0; p < 4; ++p) in[4 * p + u] = *reinterpret_cast<v4f const*>(row + 32 * p);
    }
    long long const c0 = identity ? 0 : ((long long)node[first] + 1) * branch;
    float norm = identity ? 0.0f : keyNorm[kr];
    int const nb = usable ? (branch + 31) / 32 : 0;  // an unusable tree may have no split rows
    // rows past the last child exist (the tiles have 32 rows of padding)
    v8h a[16] = {};
    if (nb > 0) vt_load_block(a, nodes, c0 + c32, h);
    float4 raw[16];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        // LDS operations of one wave are in order: the fences only keep the compiler's order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *reinterpret_cast<v4f*>(stage + (8 * u + (lane >> 3)) * kExactRow + 4 * (lane & 7)) = in[4 * p + u];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int q = 0; q < 4; ++q)
            raw[4 * p + q] = *reinterpret_cast<float4 const*>(stage + c32 * kExactRow + 16 * h + 4 * q);
    }
    if (identity) {
        float s = 0.0f;
#pragma unroll
        for (int q = 0; q < 16; ++q)
            s += raw[q].x * raw[q].x + raw[q].y * raw[q].y + raw[q].z * raw[q].z + raw[q].w * raw[q].w;
        norm = sqrtf(s + __shfl_xor(s, 32));
        if (h == 0 && kk >= 0) keyNorm[kk] = norm;
    }
    bool const inRange = usable && norm >= kVtNormMin && norm <= kVtNormMax;
    int const keyExp = inRange ? (int)(__float_as_uint(norm) >> 23) - 127 : 0;
    float const scale = __uint_as_float((unsigned)(127 + 14 - keyExp) << 23);  // 2^(14 - keyExp)
    v8h bh[8], bl[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) vt_split8(raw[2 * s], raw[2 * s + 1], scale, bh[s], bl[s]);
    Top2 s = top2_init();
    for (int cb = 0; cb < nb; ++cb) {
        v16f acc = {};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[2 * q], bh[q], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[2 * q + 1], bl[q], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[2 * q + 1], bh[q], acc, 0, 0, 0);
        }
        // the next block's loads are in flight during the selection
        if (cb + 1 < nb) vt_load_block(a, nodes, c0 + (cb + 1) * 32 + c32, h);
        __builtin_amdgcn_sched_barrier(0);
        if (cb * 32 + 32 <= branch) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                top2_push_fast(s, acc[r], cb * 32 + 8 * (r >> 2) + 4 * h + (r & 3), inf);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                int const j = cb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                top2_push_fast(s, (j < branch) ? acc[r] : -INFINITY, j, inf);
            }
        }
    }
    s = top2_merge(s, top2_shfl_xor(s, 32));
    if (h != 0 || kk < 0) return;
    float const b1 = ldexpf(s.b1, keyExp + nodeExp - 28);
    float const b2 = s.b2 > -1e29f ? ldexpf(s.b2, keyExp + nodeExp - 28) : kInit;
    float const eps = kVtEpsRel * norm * maxNodeNorm + 1e-30f;
    bool const settled = inRange && (eps < 3.0e38f) && s.a1 >= 0 && (b1 - b2 > 2.0f * eps) && (b1 - eps > -1e30f);
    if (settled) node[kk] = (int)(c0 + s.a1);
    else exactList[atomicAdd(&counters[kVtCntExact], 1)] = kk;
}

void launch_vt_score(float const* keys, float* keyNorm, int n, unsigned char const* nodes, float maxNodeNorm,
                     int nodeExp, bool usable, VtLevel const& lv, int const* order, bool identity, int maxSlots,
                     int* node, int* exactList, int* counters, hipStream_t st)
{
    if (n <= 0 || maxSlots <= 0) return;
    hipLaunchKernelGGL(k_vt_score, dim3((maxSlots + 3) / 4), dim3(256), 0, st, keys, keyNorm, n, nodes, maxNodeNorm,
                       nodeExp, usable ? 1 : 0, lv.branch, identity ? 1 : 0, order, node, exactList, counters,
                       INFINITY);
}

// ------------------------------------------------------------------------------ exact decisions
// One wave per listed key: lane j scans children j, j + 64, ... with the reference's
// sequential FP32 score (IEEE product, then IEEE sum, ascending dims) and strict '>'
// against its running best (start: the -1e30 floor); the lanes' bests combine to the
// first child of maximal score.  No valid child gives -1, so the key moves to node
// c0 - 1, as the reference's leafId = nextLeafId + bestNode does.
//
// The 64 children of a step are loaded whole lines at a time and pass through the wave's own
// LDS a quarter of their dims at a time (exact_chunk, v3dm_device.h); the key is read from LDS
// by broadcast.  With every lane loading its own child's row, each line was fetched eight
// times: 180-205 us a level for 10^6 keys of a <50,3> tree, 70-76 us so; counting the keys with
// one atomic instead of one a wave left 6-27 us.
__global__ __launch_bounds__(256) void k_vt_exact(float const* __restrict__ keys, float const* __restrict__ nodes,
                                                  long long nNodes, int branch, int level,
                                                  int const* __restrict__ exactList, int* __restrict__ node,
                                                  int* __restrict__ counters)
{
    __shared__ __attribute__((aligned(16))) float keyRows[4][kDim];
    __shared__ __attribute__((aligned(16))) float stages[4][kExactLds];
    int const lane = threadIdx.x & 63;
    int const wave = threadIdx.x >> 6;
    int const cnt = counters[kVtCntExact];
    float* const kw = keyRows[wave];
    float* const stage = stages[wave];
    float const* const mine = stage + lane * kExactRow;
    // atomics of one address take about 10 ns each: the whole list is counted by one
    if (blockIdx.x == 0 && threadIdx.x == 0 && cnt > 0) atomicAdd(&counters[kVtCntFlagged], cnt);
    for (int e = blockIdx.x * 4 + wave; e < cnt; e += gridDim.x * 4) {
        int const kk = exactList[e];
        long long const c0 = (level == 0) ? 0 : ((long long)node[kk] + 1) * branch;
        if (c0 < 0 || c0 + branch > nNodes) {
            if (lane == 0) {
                node[kk] = kVtNone;
                atomicSub(&counters[kVtCntFlagged], 1);
            }
            continue;
        }
        // LDS operations of one wave are in order: the fences only keep the compiler's order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        reinterpret_cast<float2*>(kw)[lane] = reinterpret_cast<float2 const*>(keys + (size_t)kk * kDim)[lane];
        float bestS = -INFINITY;
        int bestJ = -1;
        for (int j0 = 0; j0 < branch; j0 += 64) {
            float const* const c = nodes + (size_t)(c0 + j0) * kDim;
            int const nRows = branch - j0;  // of which this step takes 64; the rest repeat the last
            float score = 0.0f;
            v4f v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = exact_chunk(c, min(8 * u + (lane >> 3), nRows - 1), lane & 7);
#pragma unroll 1
            for (int p = 0; p < 4; ++p) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    *reinterpret_cast<v4f*>(stage + (8 * u + (lane >> 3)) * kExactRow + 4 * (lane & 7)) = v[u];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                int const next = min(p + 1, 3);  // (the last quarter once more, unused)
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    v[u] = exact_chunk(c, min(8 * u + (lane >> 3), nRows - 1), 8 * next + (lane & 7));
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    float4 const x = *reinterpret_cast<float4 const*>(mine + 4 * k);
                    float4 const y = *reinterpret_cast<float4 const*>(kw + 32 * p + 4 * k);
                    score = add_nc(score, mul_nc(y.x, x.x));
                    score = add_nc(score, mul_nc(y.y, x.y));
                    score = add_nc(score, mul_nc(y.z, x.z));
                    score = add_nc(score, mul_nc(y.w, x.w));
                }
            }
            if (lane < nRows && score > -1e30f && score > bestS) {
                bestS = score;
                bestJ = j0 + lane;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            float const os = __shfl_xor(bestS, o);
            int const oj = __shfl_xor(bestJ, o);
            bool const take = oj >= 0 && (bestJ < 0 || os > bestS || (os == bestS && oj < bestJ));
            bestS = take ? os : bestS;
            bestJ = take ? oj : bestJ;
        }
        if (lane == 0) node[kk] = (int)(c0 + bestJ);
    }
}

void launch_vt_exact(float const* keys, float const* nodes, VtLevel const& lv, int const* exactList, int* node,
                     int* counters, hipStream_t st)
{
    hipLaunchKernelGGL(k_vt_exact, dim3(1024), dim3(256), 0, st, keys, nodes, lv.nNodes, lv.branch, lv.level,
                       exactList, node, counters);
}

__global__ __launch_bounds__(256) void k_vt_finish(int const* __restrict__ node, int n, long long leafStart,
                                                   int globalIds, int32_t* __restrict__ out)
{
    int const k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    int const nd = node[k];
    out[k] = (nd == kVtNone || globalIds) ? nd : (int32_t)((long long)nd - leafStart);
}

void launch_vt_finish(int const* node, int n, long long leafStart, bool globalIds, int32_t* out, hipStream_t st)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_vt_finish, dim3((n + 255) / 256), dim3(256), 0, st, node, n, leafStart, globalIds ? 1 : 0,
                       out);
}

}  // namespace v3dm
