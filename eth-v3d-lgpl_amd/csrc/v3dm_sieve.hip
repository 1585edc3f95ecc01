// The sieve of plain putative matching (gfx950): int8 score pass, exact scores of its
// candidates, decisions.
//
// Reference path: V3D_CUDA::SIFT_Matching::findPutativeMatches
// (V3D/CUDA/v3d_cudamatching.cu:522-552); best and second best are those of the exact scores
// fl32(sum of the FP64 products), as the exact re-check decides open queries of the other passes.
#include <algorithm>
#include <cmath>

#include "v3dm_batch.h"
#include "v3dm_device.h"
#include "v3dm_sieve.h"

namespace v3dm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

bool sieve_bound(float minScore, float minRatio, float* T)
{
    double t = minScore;
    // the rule's own roundings (2 - 2 b, the quotient) are below 2^-21 of its values
    if (minRatio >= 0.0f) t = std::min(t, 1.0 - (1.0 - (double)minScore) * (1.0 + 1e-5) / (double)minRatio);
    t -= 1e-5;
    *T = (float)t;
    return t >= kSieveMin && t < 1e6;  // NaN, and a ratio of zero, are out
}

// ------------------------------------------------------------------------------ score pass
// Wave = 128 left features (four 32-column blocks, their int8 rows the resident B operands, 64
// VGPRs) against a run of 32-row tiles of right features, four v_mfma_i32_32x32x32_i8 a block
// and tile.  The rows lie in operand order, so a tile is four loads of 1 KiB straight from L1 /
// L2 (the four waves of a group take the same tiles), two tiles ahead; there is no LDS staging
// and no barrier.  Per block the 16 scores of a lane are reduced by 8 max3 and compared with
// the lane's bound; only a block with a score above it looks at single scores and lists them
// (LDS, at most the limit per wave; sets hold less than 2^24 rows).  After its last tile the wave
// scores its list exactly, a pair per lane, and enters each score for both features: an atomic
// maximum of (score, ~index) returns the smaller of two keys, which goes to the second best's
// maximum; so every key but the largest reaches it, and equal scores keep the smallest index.
// A wave with more candidates than its limit stops and marks all its features for the exact re-check
// instead, within the call's bound (SieveBest).
//
// What bounds it: the int8 matrix instructions (16384 x 16384: 2^20 of them, 20 us of the 37),
// then the tail, where each wave waits for the rows and the atomics of its few candidates
// (512 x 512, nothing but tail: 9 us).  16384 x 16384: 37 us for the pass and 5 for the decisions
// against 182 + 6 + 14 of the FP16 split pass, its merge and its re-check (605 of the FP32
// instruction); 4096 x 4096: 12 + 3 against 24 + 5 + 4; 480 x 512: 9 + 2 against 8 + 5 + 4.
constexpr int kSieveBlocks = 4;
constexpr int kSieveLook = 32;  // candidates of a wave above which entries are read before the atomics

__device__ __forceinline__ int max3i(int a, int b, int c) { return max(max(a, b), c); }

__device__ __forceinline__ int max16(v16i const& a)
{
    int const x = max3i(a[0], a[1], a[2]), y = max3i(a[3], a[4], a[5]), z = max3i(a[6], a[7], a[8]);
    int const u = max3i(a[9], a[10], a[11]), v = max3i(a[12], a[13], a[14]);
    return max3i(max3i(x, y, z), max(u, v), a[15]);
}

__device__ __forceinline__ void sieve_tile(v4i (&a)[4], signed char const* __restrict__ q, int t, int lane)
{
    v4i const* const p = reinterpret_cast<v4i const*>(q + (size_t)t * kSieveTileBytes) + lane;
#pragma unroll
    for (int s = 0; s < 4; ++s) a[s] = p[64 * s];
}

// fl32 of the FP64 sum in ascending order, as exact_scores (v3dm_device.h).
__device__ __forceinline__ float sieve_exact(float const* __restrict__ x, float const* __restrict__ y)
{
    float4 const* const a = reinterpret_cast<float4 const*>(x);
    float4 const* const b = reinterpret_cast<float4 const*>(y);
    double acc = 0.0;
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
        float4 u[8], v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            u[k] = a[8 * p + k];
            v[k] = b[8 * p + k];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            acc += (double)u[k].x * (double)v[k].x;
            acc += (double)u[k].y * (double)v[k].y;
            acc += (double)u[k].z * (double)v[k].z;
            acc += (double)u[k].w * (double)v[k].w;
        }
    }
    return (float)acc;
}

// look: the entries are read first (they only grow, so an older value is as good), and a key that
// changes neither is dropped: with many candidates a feature, most are.
__device__ __forceinline__ void sieve_enter(unsigned long long* best, unsigned* second, unsigned long long key,
                                            bool look)
{
    if (look) {
        unsigned const s2 = __hip_atomic_load(second, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((unsigned)(key >> 32) <= s2 && key < __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return;
    }
    unsigned long long const old = atomicMax(best, key);
    unsigned const loser = (unsigned)((old < key ? old : key) >> 32);
    if (loser) atomicMax(second, loser);
}

// Features [at, end) marked as flooded and, the first time, listed (one count a step of the wave);
// nOther: the other side's count.
__device__ __forceinline__ void sieve_mark(unsigned long long* __restrict__ best, int at, int end, int* flags,
                                           int* count, int nOther, SieveBest const& out, int lane)
{
    for (; at < end; at += 64) {
        int const i = at + lane;
        bool const fresh = i < end && atomicMax(best + i, kSieveFlood) != kSieveFlood;
        unsigned long long const m = __builtin_amdgcn_ballot_w64(fresh);
        if (!flags || m == 0) continue;
        int const n = __builtin_popcountll(m);
        int slot = 0;
        if (lane == 0) {
            slot = atomicAdd(count, n);
            if (out.gate && (long long)(slot + n) * nOther > out.mostListed)
                __hip_atomic_store(out.gate, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        slot = __builtin_amdgcn_readfirstlane(slot);
        if (fresh)
            flags[slot + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = i;
    }
}

// One wave: left features [i0, i0 + 128) against right tiles [t0, t1); list: out.limit entries.  ML, MR: the sets' largest
// norms; bestL / secondL, bestR / secondR: the features' entries.
__device__ __forceinline__ void sieve_wave(SieveSet const& L, SieveSet const& R, int i0, int t0, int t1, float ML,
                                           float MR, float T, unsigned long long* __restrict__ bestL,
                                           unsigned* __restrict__ secondL, unsigned long long* __restrict__ bestR,
                                           unsigned* __restrict__ secondR, unsigned const* __restrict__ bits, int ldi,
                                           SieveBest const& out, int* list, int lane)
{
    int const h = lane >> 5;
    int const c32 = lane & 31;
    // blocks past L.n (a multiple of 32) repeat the last one with a bound that nothing exceeds
    v4i B[kSieveBlocks][4];
    float base[kSieveBlocks], arm = ML;
#pragma unroll
    for (int cb = 0; cb < kSieveBlocks; ++cb) {
        int const blk = min(i0 / 32 + cb, L.n / 32 - 1);
        sieve_tile(B[cb], L.q, blk, lane);
        float const r = L.res[(blk * 32 + c32) / kSieveGroup];
        bool const exists = i0 + 32 * cb < L.n;
        // score units * 65536; the 2 covers the roundings here and below
        base[cb] = exists ? (T - r * MR) * 65536.0f - 2.0f : INFINITY;
        arm = fmaxf(arm, ML + r);
    }
    arm *= 65536.0f;
    int cnt = 0;    // uniform
    int stop = t1;  // ... 0 past the limit
    auto tile = [&](v4i(&a)[4], int t) {
        float const* const rt = R.res + t * (kSieveTile / kSieveGroup);
        float const r = fmaxf(fmaxf(rt[0], rt[1]), fmaxf(rt[2], rt[3]));
        // two blocks at a time: four would not fit beside the operands
#pragma unroll
        for (int c0 = 0; c0 < kSieveBlocks; c0 += 2) {
            v16i acc[2] = {};
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    acc[k] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[s], B[c0 + k][s], acc[k], 0, 0, 0);
            if (c0 + 2 == kSieveBlocks) sieve_tile(a, R.q, min(t + 2, t1 - 1), lane);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                int const cb = c0 + k;
                float const thr = fmaf(-arm, r, base[cb]);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64((float)max16(acc[k]) > thr) == 0, 1)) continue;
                int const entry = ((cb * 32 + c32) << 24) | (t * kSieveTile) | (h << 4);
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    bool const hit = (float)acc[k][e] > thr;
                    unsigned long long const m = __builtin_amdgcn_ballot_w64(hit);
                    if (m == 0) continue;
                    int const at = cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                    if (hit && at < out.limit) list[at] = entry | e;
                    cnt += __builtin_popcountll(m);
                }
                if (cnt > out.limit) stop = 0;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    {
        v4i a0[4], a1[4];
        sieve_tile(a0, R.q, t0, lane);
        sieve_tile(a1, R.q, min(t0 + 1, t1 - 1), lane);
        int t = t0;
        for (; t + 1 < stop; t += 2) {
            tile(a0, t);
            tile(a1, t + 1);
        }
        if (t < stop) tile(a0, t);
    }
    if (cnt > 64 && out.gate) {
        if (__hip_atomic_load(out.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;  // the full pass's call
        if (cnt <= out.limit) {
            unsigned sum = 0;
            if (lane == 0) {
                sum = atomicAdd(out.scored, (unsigned)cnt) + (unsigned)cnt;
                if (sum > out.mostScored) __hip_atomic_store(out.gate, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if ((unsigned)__builtin_amdgcn_readfirstlane((int)sum) > out.mostScored) return;
        }
    }
    if (cnt > out.limit) {
        sieve_mark(bestL, i0, min(i0 + 32 * kSieveBlocks, L.n), out.flags, out.cntL, R.n, out, lane);
        sieve_mark(bestR, t0 * kSieveTile, t1 * kSieveTile, out.flags ? out.flags + out.offR : nullptr, out.cntR, L.n,
                   out, lane);
        return;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // LDS operations of one wave are in order
    for (int c = lane; c < cnt; c += 64) {
        // accumulator element r of lane half h: row 8 (r / 4) + 4 h + r % 4 of the tile
        int const e = list[c];
        int const i = i0 + (e >> 24), j = (e & 0xffffe0) + 8 * ((e >> 2) & 3) + 4 * ((e >> 4) & 1) + (e & 3);
        if (bits && ((bits[(size_t)(j >> 5) * ldi + i] >> (j & 31)) & 1u)) continue;  // a removed pair
        float const s = sieve_exact(L.X + (size_t)i * kDim, R.X + (size_t)j * kDim);
        if (!(s > 0.0f)) continue;  // T > 0: cannot matter
        unsigned long long const v = (unsigned long long)__float_as_uint(s) << 32;
        sieve_enter(bestL + i, secondL + i, v | (0xffffffffu - (unsigned)j), cnt > kSieveLook);
        sieve_enter(bestR + j, secondR + j, v | (0xffffffffu - (unsigned)i), cnt > kSieveLook);
    }
}

__global__ __launch_bounds__(256, 3) void k_sieve(SieveSet L, SieveSet R, SievePlan p,
                                                  unsigned const* __restrict__ maxNormBits, float T, SieveBest out,
                                                  unsigned const* __restrict__ bits, int ldi)
{
    __shared__ int lists[4][kSieveList];
    int const wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // neighbouring work-groups of one XCD share a split's right tiles in its L2
    int const b = xcd_block(blockIdx.x, gridDim.x);
    int const split = b / p.groups;
    int const i0 = ((b - split * p.groups) * 4 + wv) * (32 * kSieveBlocks);
    if (i0 >= L.n) return;  // the waves of a group share nothing
    int const t0 = split * p.tiles;
    sieve_wave(L, R, i0, t0, min(t0 + p.tiles, R.n / kSieveTile), __uint_as_float(maxNormBits[0]),
               __uint_as_float(maxNormBits[kMaxNormR]), T, out.best, out.second, out.best + out.offR, out.second + out.offR,
               bits, ldi, out, lists[wv], threadIdx.x & 63);
}

// Splits of the right features: three work-groups of four waves per CU run at a time, and a
// wave's operand load and exact scores cost about four tiles.
SievePlan plan_sieve(int nL, int nR)
{
    SievePlan p;
    p.groups = (nL + 128 * kSieveBlocks - 1) / (128 * kSieveBlocks);
    int const nTiles = nR / kSieveTile;
    long long best = 1LL << 60;
    for (int s = 1; s <= nTiles && s <= 1024; ++s) {
        int const tiles = (nTiles + s - 1) / s;
        int const splits = (nTiles + tiles - 1) / tiles;
        long long const cost = ((long long)p.groups * splits + 767) / 768 * (tiles + 4);
        if (cost < best) {
            best = cost;
            p.splits = splits;
            p.tiles = tiles;
        }
    }
    return p;
}

void launch_sieve(SieveSet const& L, SieveSet const& R, SievePlan const& p, unsigned const* maxNormBits, float T,
                  SieveBest const& b, unsigned const* bits, int ldi, hipStream_t st)
{
    if (L.n <= 0 || R.n <= 0) return;
    hipLaunchKernelGGL(k_sieve, dim3(p.groups * p.splits), dim3(256), 0, st, L, R, p, maxNormBits, T, b, bits, ldi);
}

// Over a batch: item = (pair, group of 512 left features, split, tiles per split), one
// work-group each.
// 256 uneven uint8 pairs: 537 us (2.9 TB/s would read the rows, 3.4 POPS of int8 products) + 13 for
// the decisions, against 2358 + 167 + 23 of the integer-row pass, its merge and its re-check.
__device__ __forceinline__ void sieve_item(BatchDev const& b, BatchSieve const& s, int4 w, int t0, int t1, int n,
                                           int limit, int* list, int wv)
{
    BatchSeg const sl = b.seg[w.x];
    BatchSeg const sr = b.seg[b.nPairs + w.x];
    int const i0 = (w.y * 4 + wv) * (32 * kSieveBlocks);
    t1 = min(t1, sr.n / kSieveTile);
    if (i0 >= sl.n || t0 >= t1) return;
    size_t const l0 = b.imgBase[sl.img], r0 = b.imgBase[sr.img];
    SieveSet const L{b.q8 + l0 * kDim, b.res + l0 / kSieveGroup, b.img + l0 * kDim, sl.n};
    SieveSet const R{b.q8 + r0 * kDim, b.res + r0 / kSieveGroup, b.img + r0 * kDim, sr.n};
    SieveBest out{};  // (marked features are listed by the decisions)
    out.limit = limit;
    if (s.counters) {
        out.gate = s.counters + kBCntGate;
        out.scored = reinterpret_cast<unsigned*>(s.counters + kBCntScored);
        out.mostScored = sieve_most_scored((double)n * s.tiles * (128.0 * kSieveBlocks * kSieveTile));
    }
    sieve_wave(L, R, i0, t0, t1, __uint_as_float(b.maxNorm[sl.img]), __uint_as_float(b.maxNorm[sr.img]), s.T,
               s.best + sl.qOff, s.second + sl.qOff, s.best + sr.qOff, s.second + sr.qOff, nullptr, 0, out, list,
               threadIdx.x & 63);
}

constexpr int kBatchSieveList = 2048;

__global__ __launch_bounds__(256, 3) void k_batch_sieve(BatchDev b, BatchSieve s)
{
    // a wave's run of 64 tiles holds 2^18 scores: longer lists than a pair's, since listing its
    // features for the exact re-check costs far more than scoring some thousand candidates
    __shared__ int lists[4][kBatchSieveList];
    int const wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int4 const w = s.items[blockIdx.x];
    int const limit = min(max(s.tiles * kSieveTile, kSieveList), kBatchSieveList);
    sieve_item(b, s, w, w.z * w.w, (w.z + 1) * w.w, s.nItems, limit, lists[wv], wv);
}

// The items of the pairs that a learned run hands over (counted by an earlier kernel): few, so
// each is cut into runs of kSieveRun tiles, taken by a fixed grid: a run is a wave's shortest
// useful chain.  Whole items, one work-group each, of which the others leave at once: 56 us on the
// 256-pair batch, 31 so.
constexpr int kSieveRun = 8;

__global__ __launch_bounds__(256, 3) void k_batch_sieve_listed(BatchDev b, BatchSieve s)
{
    __shared__ int lists[4][kSieveList];
    int const wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int const n = __builtin_amdgcn_readfirstlane(*s.nItemsDev);
    int const runs = (s.tiles + kSieveRun - 1) / kSieveRun;
    for (int u = blockIdx.x; u < n * runs; u += gridDim.x) {
        int4 const w = s.items[u / runs];
        int const t0 = w.z * w.w + (u % runs) * kSieveRun;
        sieve_item(b, s, w, t0, min(t0 + kSieveRun, (w.z + 1) * w.w), n, kSieveList, lists[wv], wv);
    }
}

void launch_batch_sieve(BatchDev const& b, BatchSieve const& s, hipStream_t st)
{
    if (s.nItems <= 0) return;
    if (s.nItemsDev) hipLaunchKernelGGL(k_batch_sieve_listed, dim3(768), dim3(256), 0, st, b, s);
    else hipLaunchKernelGGL(k_batch_sieve, dim3(s.nItems), dim3(256), 0, st, b, s);
}

// ------------------------------------------------------------------------------ decisions
// The bound of the listed features (v3dm_sieve.h): blocks of 64 candidates each, 128 of the run's
// scores for one; the batch's exact re-check takes 28 pairs per ns.
__global__ __launch_bounds__(256) void k_batch_sieve_decide(BatchDev b, BatchSieve s, float minScore, float minRatio,
                                                            int* __restrict__ sel, int* __restrict__ flagList,
                                                            int* __restrict__ counters,
                                                            int const* __restrict__ segMask)
{
    int const si = b.segOfBlock[blockIdx.x];  // 256 queries of one segment
    if (segMask && !segMask[si]) return;
    int const g = blockIdx.x * kBatchRowAlign + threadIdx.x;
    int const lane = threadIdx.x & 63;
    int const d = sieve_decision(s.best + g, s.second + g, minScore, minRatio);
    sel[g] = d;
    unsigned long long const m = __builtin_amdgcn_ballot_w64(d == kFlag);
    if (m == 0) return;
    int const n = __builtin_popcountll(m);
    int slot = 0;
    if (lane == 0) {
        slot = atomicAdd(&counters[kBCntFlag], n);
        if (s.counters && !__hip_atomic_load(&counters[kBCntGate], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            unsigned const blocks = (unsigned)n * ((b.seg[si].nO + 63) / 64);
            unsigned const sum = atomicAdd(reinterpret_cast<unsigned*>(&counters[kBCntListed]), blocks) + blocks;
            double const items = s.nItemsDev ? *s.nItemsDev : s.nItems;
            if (sum > 16384.0 + items * s.tiles * (128.0 * kSieveBlocks * kSieveTile / 64 / 128))
                __hip_atomic_store(&counters[kBCntGate], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    slot = __builtin_amdgcn_readfirstlane(slot);
    if (d == kFlag)
        flagList[slot + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = g;
}

void launch_batch_sieve_decide(BatchDev const& b, BatchSieve const& s, float minScore, float minRatio, int* sel,
                               int* flagList, int* counters, int const* segMask, hipStream_t st)
{
    static_assert(kBatchRowAlign == 256, "a work-group per query block");
    if (b.qRows <= 0) return;
    hipLaunchKernelGGL(k_batch_sieve_decide, dim3(b.qRows / kBatchRowAlign), dim3(256), 0, st, b, s, minScore, minRatio,
                       sel, flagList, counters, segMask);
}

// ------------------------------------------------------------------------------ rows of a batch
// The int8 tiles and residuals (as the single pair's, v3dm_select.hip): 8 rows per wave, lane =
// 8 * (16 components) + row, so that a store is 8 runs of 128 bytes.  What bounds it: the rows
// (128 bytes in, 128 out) and some 150 vector instructions per 8 rows: 108 us for 2.4 * 10^6 rows of
// uint8 (139 for the FP16 integers of the full pass).
template <bool kU8>
__device__ __forceinline__ void sieve_rows8(BatchDev const& b, size_t row0, signed char* __restrict__ q8,
                                            float* __restrict__ res)
{
    int const lane = threadIdx.x & 63;
    int const c = lane >> 3;
    size_t const row = row0 + (lane & 7);
    float x[16];
    if (kU8) {
        uint4 const w = reinterpret_cast<uint4 const*>(b.u8 + row * kDim)[c];
        float const d = b.denom[row];
        unsigned const u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = dequant_u8_value((unsigned char)(u[k >> 2] >> (8 * (k & 3))), d);
    } else {
        float4 const* const p = reinterpret_cast<float4 const*>(b.img + row * kDim) + 4 * c;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float4 const v = p[k];
            x[4 * k] = v.x, x[4 * k + 1] = v.y, x[4 * k + 2] = v.z, x[4 * k + 3] = v.w;
        }
    }
    unsigned o[4] = {0, 0, 0, 0};
    float r2 = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        float const q = fminf(fmaxf(rintf(x[k] * kSieveScale), -127.0f), 127.0f);
        float const e = x[k] - q * (1.0f / kSieveScale);
        r2 += e * e;
        o[k >> 2] |= ((unsigned)(int)q & 0xffu) << (8 * (k & 3));
    }
    *reinterpret_cast<uint4*>(q8 + (row / kSieveTile) * kSieveTileBytes + c * 512 + (row % kSieveTile) * 16) =
        make_uint4(o[0], o[1], o[2], o[3]);
    r2 += __shfl_xor(r2, 8);
    r2 += __shfl_xor(r2, 16);
    r2 += __shfl_xor(r2, 32);
    r2 = fmaxf(r2, __shfl_xor(r2, 1));
    r2 = fmaxf(r2, __shfl_xor(r2, 2));
    r2 = fmaxf(r2, __shfl_xor(r2, 4));
    if (lane == 0) res[row0 / kSieveGroup] = sqrtf(r2) * 1.001f + 1e-6f;
}

template <bool kU8>
__global__ __launch_bounds__(256) void k_batch_sieve_rows(BatchDev b, signed char* __restrict__ q8,
                                                          float* __restrict__ res)
{
    sieve_rows8<kU8>(b, ((size_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 8, q8, res);
}

// The rows of the flagged segments' images (a learned run's fallback).
template <bool kU8>
__global__ __launch_bounds__(256) void k_batch_sieve_masked(BatchDev b, int const* __restrict__ segMask,
                                                            signed char* __restrict__ q8, float* __restrict__ res)
{
    int const si = b.segOfBlock[blockIdx.x];
    if (!segMask[si]) return;
    BatchSeg const sg = b.seg[si];
    int const q0 = blockIdx.x * kBatchRowAlign - sg.qOff;
    size_t const row0 = (size_t)b.imgBase[sg.img] + q0;
    for (int r = 8 * (threadIdx.x >> 6); r < kBatchRowAlign && q0 + r < sg.n; r += 32)
        sieve_rows8<kU8>(b, row0 + r, q8, res);
}

void launch_batch_sieve_rows(BatchDev const& b, int rows, signed char* q8, float* res, hipStream_t st)
{
    if (rows <= 0) return;
    dim3 const g(rows / 32);  // images are padded to 256 rows
    if (b.u8) hipLaunchKernelGGL(k_batch_sieve_rows<true>, g, dim3(256), 0, st, b, q8, res);
    else hipLaunchKernelGGL(k_batch_sieve_rows<false>, g, dim3(256), 0, st, b, q8, res);
}

void launch_batch_sieve_masked(BatchDev const& b, int const* segMask, signed char* q8, float* res, hipStream_t st)
{
    if (b.qRows <= 0) return;
    dim3 const g(b.qRows / kBatchRowAlign);
    if (b.u8) hipLaunchKernelGGL(k_batch_sieve_masked<true>, g, dim3(256), 0, st, b, segMask, q8, res);
    else hipLaunchKernelGGL(k_batch_sieve_masked<false>, g, dim3(256), 0, st, b, segMask, q8, res);
}

}  // namespace v3dm
