// Selection stage shared by every precision form: per-feature norms, merging of partial
// top-2 states, certified decisions, exact FP64 re-check of open queries, mutual check
// and ordered compaction of the matches.
//
// Reference: the selection kernels and host loop of V3D/CUDA/v3d_cudamatching.cu
// (cu:133-210 column/row top-2 with the ratio test, cu:33-85 without it, cu:546-551 the
// mutual check).
#include "v3dm_device.h"
#include "v3dm_kernels.h"
#include "v3dm_sieve.h"
#include "v3dm_split.h"

namespace v3dm {

// ------------------------------------------------------------------------------ norms
// norm[r] = ||x_r||_2 (FP32) and the maximum over rows.  Norms are >= 0 or NaN, so the
// max can be taken on the uint bits; a NaN wins, which later flags every query.
// One work-group handles 64 rows (16 per wave) and issues one atomic.
__global__ __launch_bounds__(256) void k_norms(float const* __restrict__ X, int n, float* __restrict__ norm,
                                               unsigned int* __restrict__ maxNormBits)
{
    __shared__ unsigned int wmax[4];
    int const lane = threadIdx.x & 63;
    int const wave = threadIdx.x >> 6;
    unsigned int mx = 0;
    for (int k = 0; k < 16; ++k) {
        int const row = blockIdx.x * 64 + wave * 16 + k;
        if (row >= n) break;
        float2 const v = reinterpret_cast<float2 const*>(X + (size_t)row * kDim)[lane];
        float s = v.x * v.x + v.y * v.y;
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        float const nr = sqrtf(s);
        if (lane == 0) norm[row] = nr;
        mx = max(mx, __float_as_uint(nr));
    }
    if (lane == 0) wmax[wave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned int const m = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        atomicMax(maxNormBits, m);
    }
}

void launch_norms(float const* X, int n, float* norm, unsigned int* maxNormBits, hipStream_t st)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_norms, dim3((n + 63) / 64), dim3(256), 0, st, X, n, norm, maxNormBits);
}

// ------------------------------------------------------------------------------ row preparation
// Per row: the FP32 row (from a device array, from uint8 components, or in place), its norm
// (summed as k_norms does) and its split parts, in one launch: the set is read once, where a
// copy or a dequantisation, a fill of the maximum and k_norms took three launches.  A wave
// takes 8 rows at a time, all loads in flight before the first reduction (k_norms waits for
// each row's load in its turn: 14 us for any set up to 16384 rows).  Every work-group leaves
// its largest norm and range flag in a slot and takes a ticket; the last one publishes the
// set's (at most kPrepGroups work-groups, so one thread each reads a slot).  The slots are
// device-coherent stores waited for before the ticket, not fenced: a fence would write back
// the XCD's whole L2 (22 us for 512 work-groups).
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
constexpr int kPrepRows = 8;  // rows per wave and round

__device__ __forceinline__ void split_pair(float2 v, unsigned& hi, unsigned& lo)
{
    float const x = v.x * kSplitScale, y = v.y * kSplitScale;
    v2h const h = {(_Float16)x, (_Float16)y};
    v2h const l = {(_Float16)(x - (float)h.x), (_Float16)(y - (float)h.y)};
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, l);
}

// The sum of each of 8 values over the wave's lanes, the largest of them in every lane: the
// first three steps halve the values a lane carries.
__device__ __forceinline__ float max_of_sums(float (&s)[8], int lane)
{
#pragma unroll
    for (int n = 4, o = 32; n >= 1; n >>= 1, o >>= 1) {
        bool const up = lane & o;
#pragma unroll
        for (int k = 0; k < n; ++k) {
            float const other = __shfl_xor(up ? s[k] : s[n + k], o);
            s[k] = (up ? s[n + k] : s[k]) + other;
        }
    }
    float x = s[0];
    x += __shfl_xor(x, 4);
    x += __shfl_xor(x, 2);
    x += __shfl_xor(x, 1);
    x = fmaxf(x, __shfl_xor(x, 32));
    x = fmaxf(x, __shfl_xor(x, 16));
    return fmaxf(x, __shfl_xor(x, 8));
}

template <int kFrom>
__global__ __launch_bounds__(256) void k_split_rows(void const* __restrict__ src, float* __restrict__ X, int n,
                                                    float* __restrict__ norm, unsigned int* __restrict__ maxNormBits,
                                                    unsigned char* __restrict__ split,
                                                    unsigned char* __restrict__ ints, float* __restrict__ scale,
                                                    signed char* __restrict__ q8, float* __restrict__ res,
                                                    int* __restrict__ info, int* __restrict__ hostFit)
{
    __shared__ unsigned int wmax[4];
    __shared__ int wbad[4];
    __shared__ int last;
    int const lane = threadIdx.x & 63;
    int const wave = threadIdx.x >> 6;
    unsigned int mx = 0;
    bool bad = false;
    for (int row0 = (blockIdx.x * 4 + wave) * kPrepRows; row0 < n; row0 += gridDim.x * 4 * kPrepRows) {
        float2 v[kPrepRows];
        if constexpr (kFrom == kRowsU8) {
            uchar2 q[kPrepRows];
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k)
                q[k] = (row0 + k < n) ? static_cast<uchar2 const*>(src)[(size_t)(row0 + k) * 64 + lane]
                                      : make_uchar2(0, 0);
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) {
                float const d = dequant_u8_denom(q[k]);
                v[k] = (row0 + k < n) ? make_float2(dequant_u8_value(q[k].x, d), dequant_u8_value(q[k].y, d))
                                      : make_float2(0.0f, 0.0f);
                if (row0 + k < n) {
                    v2h const i = {(_Float16)(float)q[k].x, (_Float16)(float)q[k].y};
                    reinterpret_cast<v2h*>(ints + (size_t)(row0 + k) * kIntRowBytes)[lane] = i;
                    if (lane == 0) scale[row0 + k] = d;
                }
            }
        } else {
            float2 const* const rows = kFrom == kRowsF32 ? static_cast<float2 const*>(src)
                                                         : reinterpret_cast<float2 const*>(X);
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k)
                v[k] = (row0 + k < n) ? rows[(size_t)(row0 + k) * 64 + lane] : make_float2(0.0f, 0.0f);
        }
        float s[kPrepRows];
#pragma unroll
        for (int k = 0; k < kPrepRows; ++k) s[k] = v[k].x * v[k].x + v[k].y * v[k].y;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) s[k] += __shfl_xor(s[k], o);
#pragma unroll
        for (int k = 0; k < kPrepRows; ++k) {
            float const nr = sqrtf(s[k]);
            mx = max(mx, __float_as_uint(nr));  // norms are >= 0 or NaN: a NaN wins
            bad = bad || !(nr == 0.0f || (nr >= kSplitNormMin && nr < kSplitNormMax));
            if (row0 + k >= n) break;  // uniform over the wave; rows past n are zero above
            if (lane == 0) norm[row0 + k] = nr;
            if (kFrom != kRowsInPlace) reinterpret_cast<float2*>(X)[(size_t)(row0 + k) * 64 + lane] = v[k];
            unsigned hi, lo;
            split_pair(v[k], hi, lo);
            unsigned* o = reinterpret_cast<unsigned*>(split + (size_t)(row0 + k) * kSplitRowBytes + (lane >> 5) * 256);
            o[lane & 31] = hi;
            o[32 + (lane & 31)] = lo;
        }
        // the sieve's rows (past n: inside the padded buffer, never read)
        float e2[kPrepRows];
#pragma unroll
        for (int k = 0; k < kPrepRows; ++k) {
            float const qx = fminf(fmaxf(rintf(v[k].x * kSieveScale), -127.0f), 127.0f);
            float const qy = fminf(fmaxf(rintf(v[k].y * kSieveScale), -127.0f), 127.0f);
            float const ex = v[k].x - qx * (1.0f / kSieveScale), ey = v[k].y - qy * (1.0f / kSieveScale);
            e2[k] = ex * ex + ey * ey;
            int const row = row0 + k;
            *reinterpret_cast<char2*>(q8 + (size_t)(row / kSieveTile) * kSieveTileBytes + (lane >> 3) * 512 +
                                      (row % kSieveTile) * 16 + (lane & 7) * 2) =
                make_char2((signed char)(int)qx, (signed char)(int)qy);
        }
        float const r2 = max_of_sums(e2, lane);
        if (lane == 0) res[row0 / kSieveGroup] = sqrtf(r2) * 1.001f + 1e-6f;  // rounded up
    }
    if (lane == 0) {
        wmax[wave] = mx;
        wbad[wave] = bad;
    }
    __syncthreads();
    int* const slot = info + kPrepSlot;  // two ints per work-group
    if (threadIdx.x == 0) {
        unsigned int const m = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        int const f = wbad[0] | wbad[1] | wbad[2] | wbad[3];
        __hip_atomic_store(slot + 2 * blockIdx.x, (int)m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(slot + 2 * blockIdx.x + 1, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        int const t = __hip_atomic_fetch_add(info, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = t == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    unsigned int m = 0;
    int f = 0;
    if (threadIdx.x < gridDim.x) {
        m = (unsigned int)__hip_atomic_load(slot + 2 * threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        f = __hip_atomic_load(slot + 2 * threadIdx.x + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    for (int o = 32; o > 0; o >>= 1) {
        m = max(m, __shfl_xor(m, o));
        f |= __shfl_xor(f, o);
    }
    __syncthreads();
    if (lane == 0) {
        wmax[wave] = m;
        wbad[wave] = f;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    *maxNormBits = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    *hostFit = !(wbad[0] | wbad[1] | wbad[2] | wbad[3]);
    __hip_atomic_store(info, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

void launch_split_rows(RowSource from, void const* src, float* X, int n, float* norm, unsigned int* maxNormBits,
                       unsigned char* split, unsigned char* ints, float* scale, signed char* q8, float* res, int* info,
                       int* hostFit, hipStream_t st)
{
    if (n <= 0) return;
    int const per = 4 * kPrepRows;
    dim3 const grid(min((n + per - 1) / per, kPrepGroups));
    if (from == kRowsU8)
        hipLaunchKernelGGL(k_split_rows<kRowsU8>, grid, dim3(256), 0, st, src, X, n, norm, maxNormBits, split, ints,
                           scale, q8, res, info, hostFit);
    else if (from == kRowsF32)
        hipLaunchKernelGGL(k_split_rows<kRowsF32>, grid, dim3(256), 0, st, src, X, n, norm, maxNormBits, split, ints,
                           scale, q8, res, info, hostFit);
    else
        hipLaunchKernelGGL(k_split_rows<kRowsInPlace>, grid, dim3(256), 0, st, src, X, n, norm, maxNormBits, split,
                           ints, scale, q8, res, info, hostFit);
}

// ------------------------------------------------------------------------------ merge + decide
// 8 lanes per query (lane = 8*query + sub); each lane merges every 8th partial, then the
// 8 lanes combine with xor shuffles.  Queries [0, nL) are left features, [nL, nL+nR)
// right features.
__global__ __launch_bounds__(256) void k_merge_decide(Top2 const* __restrict__ colPart, int nColParts, int ldc,
                                                      Top2 const* __restrict__ rowPart, int nRowParts, int ldr,
                                                      int nL, int nR, float const* __restrict__ normL,
                                                      float const* __restrict__ normR,
                                                      unsigned int const* __restrict__ maxNormBits, float epsRel,
                                                      float minScore, float minRatio, int* __restrict__ colMax,
                                                      int* __restrict__ rowMax, int* __restrict__ flagList,
                                                      int flagOffR, int* __restrict__ counters)
{
    int const sub = threadIdx.x & 7;
    int const g = (int)((blockIdx.x * 256u + threadIdx.x) >> 3);
    bool const valid = g < nL + nR;
    int const gq = valid ? g : 0;
    bool const left = gq < nL;
    int const q = left ? gq : gq - nL;
    Top2 const* part = left ? colPart : rowPart;
    int const np = valid ? (left ? nColParts : nRowParts) : 0;
    size_t const ld = left ? (size_t)ldc : (size_t)ldr;
    Top2 s = top2_init();
#pragma unroll 4
    for (int p = sub; p < np; p += 8) s = top2_merge(s, part[(size_t)p * ld + q]);
    s = top2_merge(s, top2_shfl_xor(s, 1));
    s = top2_merge(s, top2_shfl_xor(s, 2));
    s = top2_merge(s, top2_shfl_xor(s, 4));
    if (!valid || sub != 0) return;
    float const nq = left ? normL[q] : normR[q];
    float const mo = __uint_as_float(maxNormBits[left ? 1 : 0]);
    float const eps = epsRel * nq * mo + kEpsAbs;
    int const d = (epsRel > 0.0f) ? decide_certified(s, eps, minScore, minRatio) : kFlag;
    if (d == kFlag) {
        int const slot = atomicAdd(&counters[left ? kCntFlag : kCntFlagR], 1);
        flagList[left ? slot : flagOffR + slot] = q;
    }
    (left ? colMax : rowMax)[q] = d;
}

void launch_merge_decide(Top2 const* colPart, int nColParts, int ldc, Top2 const* rowPart, int nRowParts,
                         int ldr, int nL, int nR, float const* normL, float const* normR,
                         unsigned int const* maxNormBits, float epsRel, float minScore, float minRatio,
                         int* colMax, int* rowMax, int* flagList, int flagOffR, int* counters, hipStream_t st)
{
    int const n = nL + nR;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_merge_decide, dim3((n + 31) / 32), dim3(256), 0, st, colPart, nColParts, ldc, rowPart,
                       nRowParts, ldr, nL, nR, normL, normR, maxNormBits, epsRel, minScore, minRatio, colMax,
                       rowMax, flagList, flagOffR, counters);
}

// ------------------------------------------------------------------------------ exact re-check
// Open queries are listed per direction (left queries at flagList[0..), right queries at
// flagList[flagOffR..)).  A work unit is (one or up to kRecheckGroup queries of one direction, chunk of 64 *
// subs candidates), one wave each, grid-stride over all units; the last wave of a query
// merges its partials and takes the IEEE FP32 decision.  Chunks are as short as the partials'
// buffer allows (kRecheckMaxChunks per listed row of either side, so the fewer queries are
// open, the more chunks each gets): with the usual tens of open queries every unit is one
// step of 64 candidates, 14 us for a few open queries of 16384 x 16384 in one launch (a chain of
// loads, 64 dependent FP64 steps a quarter and the tickets; nothing is near a rate) against
// 38 + 5 us in two.  With every query open (a zero error bound) it is 1.3 times the earlier
// 16 queries a group: 3.7 against 2.8 ms at 8192 x 8192.
constexpr int kRecheckGroup = 4;  // queries per unit: they share the candidates' loads

struct RecheckDir {
    float const* Q;
    float const* C;
    int* sel;
    int nC, cnt, base;  // base: first list entry and row of the partials
    int subs, nCh;
};

__device__ __forceinline__ RecheckDir recheck_dir(bool left, float const* L, float const* R, int nL, int nR, int cnt,
                                                  int rowsL, int rowsR, int* colMax, int* rowMax)
{
    RecheckDir d;
    d.Q = left ? L : R;
    d.C = left ? R : L;
    d.sel = left ? colMax : rowMax;
    d.nC = left ? nR : nL;
    d.cnt = cnt;
    d.base = left ? 0 : rowsL;
    int const nSub = (d.nC + 63) / 64;
    long long const room = (long long)(left ? rowsL : rowsR) * kRecheckMaxChunks / max(cnt, 1);
    int const most = (int)min(room, (long long)nSub);
    d.subs = (nSub + most - 1) / max(most, 1);
    d.nCh = (nSub + d.subs - 1) / d.subs;
    return d;
}

template <int kQ>
__device__ __forceinline__ void recheck_units(RecheckDir const& dl, RecheckDir const& dr, int const* flagList,
                                              Top2* __restrict__ part, int* __restrict__ tickets,
                                              unsigned const* __restrict__ gbits, int ldi, float minScore,
                                              float minRatio, float* __restrict__ stage, double* __restrict__ qd)
{
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * 256 + threadIdx.x) >> 6));
    int const unitsL = (dl.cnt + kQ - 1) / kQ * dl.nCh;
    int const units = unitsL + (dr.cnt + kQ - 1) / kQ * dr.nCh;
    for (int w = wave; w < units; w += gridDim.x * 4) {
        bool const left = w < unitsL;
        RecheckDir const& d = left ? dl : dr;
        int const wl = left ? w : w - unitsL;
        int const g = wl / d.nCh, c = wl - g * d.nCh;
        float const* q[kQ];
        int row[kQ];
        Top2 s[kQ];
#pragma unroll
        for (int j = 0; j < kQ; ++j) {
            int const e = min(g * kQ + j, d.cnt - 1);  // past the end: the last query again, not published
            row[j] = __builtin_amdgcn_readfirstlane(flagList[d.base + e]);
            q[j] = d.Q + (size_t)row[j] * kDim;
            s[j] = top2_init();
        }
        exact_queries<kQ>(q, qd, lane);
        int const c1 = min((c + 1) * d.subs * 64, d.nC);
        for (int c0 = c * d.subs * 64; c0 < c1; c0 += 64) {
            int const ci = c0 + lane;
            float v[kQ];
            exact_scores<kQ>(qd, d.C + (size_t)c0 * kDim, d.nC - c0, stage, lane, v);
#pragma unroll
            for (int j = 0; j < kQ; ++j) {
                if (gbits) {
                    // guided matching: a removed (left, right) pair scores -1e20
                    int const li = left ? row[j] : min(ci, d.nC - 1), rj = left ? min(ci, d.nC - 1) : row[j];
                    v[j] = ((gbits[(size_t)(rj >> 5) * ldi + li] >> (rj & 31)) & 1u) ? -1e20f : v[j];
                }
                if (ci < c1) top2_push(s[j], v[j], ci);
            }
        }
#pragma unroll
        for (int j = 0; j < kQ; ++j) {
            int const e = g * kQ + j;
            if (e >= d.cnt) break;  // uniform
            for (int o = 32; o > 0; o >>= 1) s[j] = top2_merge(s[j], top2_shfl_xor(s[j], o));
            Top2* const p = part + (size_t)d.base * kRecheckMaxChunks + (size_t)e * d.nCh;
            if (publish_partial(s[j], p, c, d.nCh, tickets + d.base + e, lane)) {
                Top2 const t = merge_partials(p, d.nCh, lane);
                if (lane == 0) d.sel[row[j]] = decide_exact(t, minScore, minRatio);
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_recheck(float const* __restrict__ L, float const* __restrict__ R, int nL,
                                                 int nR, int const* __restrict__ flagList, int rowsL, int rowsR,
                                                 int const* __restrict__ counters, Top2* __restrict__ part,
                                                 int* __restrict__ tickets, unsigned const* __restrict__ gbits,
                                                 int ldi, float minScore, float minRatio, int* __restrict__ colMax,
                                                 int* __restrict__ rowMax)
{
    __shared__ __attribute__((aligned(16))) float stage[4][kExactLds];
    __shared__ __attribute__((aligned(16))) double qd[4][kRecheckGroup * kDim];
    int const cntL = __builtin_amdgcn_readfirstlane(counters[kCntFlag]);
    int const cntR = __builtin_amdgcn_readfirstlane(counters[kCntFlagR]);
    RecheckDir const dl = recheck_dir(true, L, R, nL, nR, cntL, rowsL, rowsR, colMax, rowMax);
    RecheckDir const dr = recheck_dir(false, L, R, nL, nR, cntR, rowsL, rowsR, colMax, rowMax);
    int const wv = threadIdx.x >> 6;
    // a query per wave while the grid holds a wave for every unit
    if ((long long)cntL * dl.nCh + (long long)cntR * dr.nCh <= 4LL * gridDim.x)
        recheck_units<1>(dl, dr, flagList, part, tickets, gbits, ldi, minScore, minRatio, stage[wv], qd[wv]);
    else
        recheck_units<kRecheckGroup>(dl, dr, flagList, part, tickets, gbits, ldi, minScore, minRatio, stage[wv],
                                     qd[wv]);
}

void launch_recheck_exact(float const* L, float const* R, int nL, int nR, int const* flagList, int rowsL, int rowsR,
                          int const* counters, float minScore, float minRatio, int* colMax, int* rowMax, Top2* part,
                          int* tickets, int grid, hipStream_t st, unsigned const* gbits, int ldi)
{
    if (nL <= 0 || nR <= 0) return;
    hipLaunchKernelGGL(k_recheck, dim3(grid), dim3(256), 0, st, L, R, nL, nR, flagList, rowsL, rowsR, counters, part,
                       tickets, gbits, ldi, minScore, minRatio, colMax, rowMax);
}

// ------------------------------------------------------------------------------ mutual + compaction
// (k, colMax[k]) is a match iff rowMax[colMax[k]] == k (cu:546-551).  One launch, ordered
// by a decoupled look-back: work-group b takes the 1024 left features [1024 b, 1024 b +
// 1024) (4 per thread), counts its matches, publishes the count (flag 1) in its status
// word, then adds up its predecessors' words from the nearest backwards (64 per step, one
// per lane of wave 0) until it reaches an inclusive prefix (flag 2), publishes its own
// inclusive prefix and writes its matches in ascending k from its exclusive prefix on, so
// the output is sorted by k.  A status word is valid for the call whose epoch it carries,
// so nothing is cleared between calls.  A work-group waits only for lower indices, which
// are dispatched before it; the wait is bounded (mw.spinLimit sleeps), and a work-group
// that runs out of it stores the epoch in counters[kCntMutualError] (its matches then land
// below their place, inside the buffer).  The last work-group also publishes the match,
// re-check and rescoring counts and clears the per-call counters.

// Left feature sampled as sample k of S (evenly spaced over [0, nL)).
__device__ __forceinline__ int sample_row(int k, int nL, int S) { return (int)(((long long)k * nL) / S); }

__device__ __forceinline__ unsigned long long mutual_word(unsigned epoch, unsigned flag, unsigned value)
{
    return ((unsigned long long)epoch << 32) | ((unsigned long long)flag << 30) | value;  // value < 2^30
}

__global__ __launch_bounds__(256) void k_mutual(int const* __restrict__ colMax, int const* __restrict__ rowMax,
                                                int nL, int nR, unsigned long long* __restrict__ status,
                                                unsigned epoch, int* __restrict__ stripes,
                                                int2* __restrict__ pairs, int* __restrict__ counters, SampleOut so,
                                                MutualWait mw)
{
    __shared__ int wsum[4];
    __shared__ int sBase;
    int const tid = threadIdx.x;
    int const lane = tid & 63;
    int const wave = tid >> 6;
    int const b = blockIdx.x;
    int const i0 = b * kMutualSlice + 4 * tid;
    // all four colMax entries in one load, then all four rowMax gathers (indices clamped to
    // [0, max(nR - 1, 0)]: in bounds, rowMax holds at least one row per allocation) before
    // any test: two round trips
    int l[4];
    if (i0 + 3 < nL) {
        int4 const c = *reinterpret_cast<int4 const*>(colMax + i0);
        l[0] = c.x, l[1] = c.y, l[2] = c.z, l[3] = c.w;
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) l[u] = (i0 + u < nL) ? colMax[i0 + u] : -1;
    }
    int r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = rowMax[min(max(l[u], 0), max(nR - 1, 0))];
    bool m[4];
    int cnt = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        m[u] = (l[u] >= 0) && (l[u] < nR) && (r[u] == i0 + u);
        cnt += m[u] ? 1 : 0;
    }
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int const t = __shfl_up(incl, o);
        incl += (lane >= o) ? t : 0;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        off += (w < wave) ? wsum[w] : 0;
        total += wsum[w];
    }
    if (wave == 0) {
        if (lane == 0)
            __hip_atomic_store(&status[b], mutual_word(epoch, b == 0 ? 2u : 1u, (unsigned)total), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        int excl = 0;
        bool failed = false;
        int top = b - 1;  // nearest predecessor not yet added (uniform over the wave)
        unsigned spins = 0;
        while (top >= 0) {
            int const j = top - lane;
            unsigned long long const w =
                (j >= 0) ? __hip_atomic_load(&status[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                         : mutual_word(epoch, 2u, 0u);  // before work-group 0: an inclusive prefix of 0
            unsigned const fl = ((unsigned)(w >> 32) == (epoch ^ mw.readXor)) ? (unsigned)(w >> 30) & 3u : 0u;
            unsigned long long const ready = __ballot(fl != 0u);
            unsigned long long const inclusive = __ballot(fl == 2u);
            int const stop = inclusive ? __ffsll((long long)inclusive) - 1 : 63;  // last lane to add
            unsigned long long const need = (2ull << stop) - 1ull;                 // lanes 0 .. stop
            if ((ready & need) == need) {
                int v = (lane <= stop) ? (int)(w & 0x3fffffffull) : 0;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
                excl += v;
                if (inclusive) break;
                top -= 64;
            } else {
                if (++spins > mw.spinLimit) {
                    failed = true;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
        if (lane == 0) {
            if (b > 0)
                __hip_atomic_store(&status[b], mutual_word(epoch, 2u, (unsigned)(excl + total)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            if (failed) counters[kCntMutualError] = (int)epoch;
            sBase = excl;
        }
    }
    __syncthreads();
    int pos = sBase + off + incl - cnt;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (m[u]) pairs[pos++] = make_int2(i0 + u, l[u]);
    // work-group 0 (off the look-back chain by now): the sampled learned decisions
    if (b == 0 && tid < so.S) so.out[tid] = colMax[sample_row(tid, nL, so.S)];  // vector stores
    if (b != (int)gridDim.x - 1) return;
    // the last work-group: counts of the call
    if (wave == 0) {
        int rescored = 0;
        if (tid < kStripes) {
            rescored = stripes[tid * kStripeStride];
            stripes[tid * kStripeStride] = 0;
        }
        for (int o = 32; o > 0; o >>= 1) rescored += __shfl_xor(rescored, o);
        if (tid == 0) {
            counters[kCntPairs] = sBase + total;
            counters[kCntFlagDone] = counters[kCntFlag] + counters[kCntFlagR];
            counters[kCntFlag] = 0;
            counters[kCntFlagR] = 0;
            counters[kCntRescoredDone] = rescored;
        }
    }
}

void launch_mutual_compact(int const* colMax, int const* rowMax, int nL, int nR, unsigned long long* status,
                           unsigned epoch, int* stripes, int2* pairs, int* counters, hipStream_t st,
                           SampleOut const& so, MutualWait const& mw)
{
    int const nb = (nL + kMutualSlice - 1) / kMutualSlice;
    hipLaunchKernelGGL(k_mutual, dim3(nb > 0 ? nb : 1), dim3(256), 0, st, colMax, rowMax, nL, nR, status, epoch,
                       stripes, pairs, counters, so, mw);
}

// ------------------------------------------------------------------------------ sampled check
// A shortlist result is checked on S evenly spaced left features (S <= 128): their rows and
// norms are gathered into a 128-row block (zero rows past S) and decided by the plain exact
// path; the comparison counts the sampled features the exact rule accepts, those whose
// shortlist decision differs from it (missed), and those the shortlist accepts wrongly.
__global__ __launch_bounds__(256) void k_sample_gather(float const* __restrict__ L, float const* __restrict__ normL,
                                                       int nL, int S, float* __restrict__ Ls,
                                                       float* __restrict__ normS, int* __restrict__ idx,
                                                       int* __restrict__ counters)
{
    if (blockIdx.x == 0 && threadIdx.x < kNumCounters) counters[threadIdx.x] = 0;  // the check's own counters
    int const lane = threadIdx.x & 63;
    int const k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= kSampleRows) return;
    int const i = (k < S) ? sample_row(k, nL, S) : -1;
    float2 const v = (i >= 0) ? reinterpret_cast<float2 const*>(L + (size_t)i * kDim)[lane] : make_float2(0.f, 0.f);
    reinterpret_cast<float2*>(Ls + (size_t)k * kDim)[lane] = v;
    if (lane == 0) {
        normS[k] = (i >= 0) ? normL[i] : 0.0f;
        idx[k] = i;
    }
}

void launch_sample_gather(float const* L, float const* normL, int nL, int S, float* Ls, float* normS, int* idx,
                          int* counters, hipStream_t st)
{
    hipLaunchKernelGGL(k_sample_gather, dim3(kSampleRows / 4), dim3(256), 0, st, L, normL, nL, S, Ls, normS, idx,
                       counters);
}

// The sampled rows' decisions: one wave per sampled left feature merges its split
// partials (lane l takes every 64th), then the certified decision as in k_merge_decide.
__global__ __launch_bounds__(256) void k_sample_decide(Top2 const* __restrict__ colPart, int nParts, int ldc, int S,
                                                       float const* __restrict__ normS,
                                                       unsigned int const* __restrict__ maxNormBits, float epsRel,
                                                       float minScore, float minRatio, int* __restrict__ dec,
                                                       int* __restrict__ flagList, int* __restrict__ counters)
{
    int const lane = threadIdx.x & 63;
    int const q = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (q >= S) return;  // uniform per wave
    Top2 s = top2_init();
    for (int p = lane; p < nParts; p += 64) s = top2_merge(s, colPart[(size_t)p * ldc + q]);
    for (int o = 32; o > 0; o >>= 1) s = top2_merge(s, top2_shfl_xor(s, o));
    if (lane != 0) return;
    float const eps = epsRel * normS[q] * __uint_as_float(maxNormBits[1]) + kEpsAbs;
    int const d = (epsRel > 0.0f) ? decide_certified(s, eps, minScore, minRatio) : kFlag;
    if (d == kFlag) flagList[atomicAdd(&counters[kCntFlag], 1)] = q;
    dec[q] = d;
}

void launch_sample_decide(Top2 const* colPart, int nParts, int ldc, int S, float const* normS,
                          unsigned int const* maxNormBits, float epsRel, float minScore, float minRatio, int* dec,
                          int* flagList, int* counters, hipStream_t st)
{
    if (S <= 0) return;
    hipLaunchKernelGGL(k_sample_decide, dim3((S + 3) / 4), dim3(256), 0, st, colPart, nParts, ldc, S, normS,
                       maxNormBits, epsRel, minScore, minRatio, dec, flagList, counters);
}


}  // namespace v3dm
