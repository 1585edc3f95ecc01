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
// Per row: the FP32 row (from a device array, from uint8 components, or in place), its norm and
// its int8 row for the sieve, in one launch: the set is read once, where a copy or a
// dequantisation, a fill of the maximum and k_norms took three launches.  A wave takes 8 rows at
// a time, all loads in flight before the first reduction (k_norms waits for each row's load in
// its turn: 14 us for any set up to 16384 rows), and reduces the 8 rows' sums together.  The
// split rows of the full pass are made where that pass runs (k_split_sets).  The set's largest
// norm is an atomic maximum under the call's epoch, so nothing is cleared and no work-group waits
// for another; a row out of range clears the host's flag, which the host has set.
//
// What bounds it: latency (the loads, two reductions, the stores: 7 us for any small set); a set
// of 32768 rows moves 38 MB in 12 us.  With the split rows made here and a ticket for the last
// work-group, which published the maximum: 8 us for small sets, 18 for 32768 rows.
constexpr int kPrepRows = 8;  // rows per wave and round

// The sums of 8 values over the wave's lanes: lane l gets the sum of value l / 8.  The first
// three steps halve the values a lane carries (10 shuffles instead of 48).
__device__ __forceinline__ float sums_of8(float (&s)[8], int lane)
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
    return x + __shfl_xor(x, 1);
}

template <int kFrom, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void k_prep_rows(void const* __restrict__ src, float* __restrict__ X, int n,
                                                   float* __restrict__ norm, unsigned long long* __restrict__ maxNorm,
                                                   unsigned epoch, float* __restrict__ scale,
                                                   signed char* __restrict__ q8, float* __restrict__ res,
                                                   int* __restrict__ hostFit)
{
    __shared__ unsigned int wmax[kWaves];
    int const lane = threadIdx.x & 63;
    int const wave = threadIdx.x >> 6;
    unsigned int mx = 0;
    int bad = 0;
    for (int row0 = (blockIdx.x * kWaves + wave) * kPrepRows; row0 < n;
         row0 += gridDim.x * kWaves * kPrepRows) {
        // n is a multiple of 32: no round is partial
        float2 v[kPrepRows];
        if constexpr (kFrom == kRowsU8) {
            uchar2 q[kPrepRows];
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) q[k] = static_cast<uchar2 const*>(src)[(size_t)(row0 + k) * 64 + lane];
            // the sums of squares are exact in any order (dequant_u8_denom)
            float s[kPrepRows];
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) s[k] = (float)q[k].x * (float)q[k].x + (float)q[k].y * (float)q[k].y;
            float const mine = dequant_u8_scale(sums_of8(s, lane));
            if ((lane & 7) == 0) scale[row0 + (lane >> 3)] = mine;
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) {
                float const d = __shfl(mine, 8 * k);
                v[k] = make_float2(dequant_u8_value(q[k].x, d), dequant_u8_value(q[k].y, d));
            }
        } else {
            float2 const* const rows = kFrom == kRowsF32 ? static_cast<float2 const*>(src)
                                                         : reinterpret_cast<float2 const*>(X);
#pragma unroll
            for (int k = 0; k < kPrepRows; ++k) v[k] = rows[(size_t)(row0 + k) * 64 + lane];
        }
        float s[kPrepRows], e2[kPrepRows];
#pragma unroll
        for (int k = 0; k < kPrepRows; ++k) {
            s[k] = v[k].x * v[k].x + v[k].y * v[k].y;
            if (kFrom != kRowsInPlace) reinterpret_cast<float2*>(X)[(size_t)(row0 + k) * 64 + lane] = v[k];
            float const qx = fminf(fmaxf(rintf(v[k].x * kSieveScale), -127.0f), 127.0f);
            float const qy = fminf(fmaxf(rintf(v[k].y * kSieveScale), -127.0f), 127.0f);
            float const ex = v[k].x - qx * (1.0f / kSieveScale), ey = v[k].y - qy * (1.0f / kSieveScale);
            e2[k] = ex * ex + ey * ey;
            int const row = row0 + k;
            *reinterpret_cast<char2*>(q8 + (size_t)(row / kSieveTile) * kSieveTileBytes + (lane >> 3) * 512 +
                                      (row % kSieveTile) * 16 + (lane & 7) * 2) =
                make_char2((signed char)(int)qx, (signed char)(int)qy);
        }
        float const nr = sqrtf(sums_of8(s, lane));
        if ((lane & 7) == 0) norm[row0 + (lane >> 3)] = nr;
        mx = max(mx, __float_as_uint(nr));  // norms are >= 0 or NaN: a NaN wins
        bad |= !(nr == 0.0f || (nr >= kSplitNormMin && nr < kSplitNormMax));
        float r2 = sums_of8(e2, lane);
#pragma unroll
        for (int o = 32; o >= 8; o >>= 1) r2 = fmaxf(r2, __shfl_xor(r2, o));
        if (lane == 0) res[row0 / kSieveGroup] = sqrtf(r2) * 1.001f + 1e-6f;  // rounded up
    }
#pragma unroll
    for (int o = 32; o >= 8; o >>= 1) {
        mx = max(mx, __shfl_xor(mx, o));
        bad |= __shfl_xor(bad, o);
    }
    if (lane == 0) {
        wmax[wave] = mx;
        if (bad) *hostFit = 0;
    }
    __syncthreads();
    if (threadIdx.x >= kWaves) return;
    mx = wmax[threadIdx.x];
#pragma unroll
    for (int o = kWaves / 2; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
    // atomics of one address take about 10 ns each: one a work-group, and only with a new maximum
    unsigned long long const word = ((unsigned long long)epoch << 32) | mx;
    if (threadIdx.x == 0 && __hip_atomic_load(maxNorm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < word)
        atomicMax(maxNorm, word);
}

template <int kFrom>
void launch_prep_from(void const* src, float* X, int n, float* norm, unsigned long long* maxNorm, unsigned epoch,
                      float* scale, signed char* q8, float* res, int* hostFit, hipStream_t st)
{
    int const small = (n + 4 * kPrepRows - 1) / (4 * kPrepRows), large = (n + 16 * kPrepRows - 1) / (16 * kPrepRows);
    if (small <= kPrepGroups)
        hipLaunchKernelGGL((k_prep_rows<kFrom, 4>), dim3(small), dim3(256), 0, st, src, X, n, norm, maxNorm, epoch,
                           scale, q8, res, hostFit);
    else
        hipLaunchKernelGGL((k_prep_rows<kFrom, 16>), dim3(min(large, kPrepGroups)), dim3(1024), 0, st, src, X, n, norm,
                           maxNorm, epoch, scale, q8, res, hostFit);
}

// Work-groups of 4 waves while one round of kPrepGroups of them holds the set (8192 rows), of 16
// above: a maximum's atomic a work-group is what the larger ones save (16384 rows 14 -> 11 us,
// 32768 rows 17 -> 12 us), and below they would leave compute units idle (1920 rows of uint8 8.5
// against 10.5 us).
void launch_prep_rows(RowSource from, void const* src, float* X, int n, float* norm, unsigned int* maxNorm,
                      unsigned epoch, float* scale, signed char* q8, float* res, int* hostFit, hipStream_t st)
{
    if (n <= 0) return;
    auto* const mx = reinterpret_cast<unsigned long long*>(maxNorm);
    if (from == kRowsU8) launch_prep_from<kRowsU8>(src, X, n, norm, mx, epoch, scale, q8, res, hostFit, st);
    else if (from == kRowsF32) launch_prep_from<kRowsF32>(src, X, n, norm, mx, epoch, scale, q8, res, hostFit, st);
    else launch_prep_from<kRowsInPlace>(src, X, n, norm, mx, epoch, scale, q8, res, hostFit, st);
}

// The rows of the full pass for both sets in one launch, a chunk of 8 components per thread:
// the split parts, and where a set has scales (uint8 uploads) its components as FP16 integers
// (x = fl(q d) with d > 0, so q is the integer next to x / d).  Made when the full pass first
// needs them: with the sieve few calls do.
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

__global__ __launch_bounds__(256) void k_split_sets(SplitRowsOf a, SplitRowsOf b, int* __restrict__ gated)
{
    if (gated) {
        if (!gated[kCntGate]) return;
        // the sieve's list is void, the full pass makes its own
        if (blockIdx.x == 0 && threadIdx.x == 0) gated[kCntFlag] = gated[kCntFlagR] = 0;
    }
    int const t = blockIdx.x * 256 + threadIdx.x;
    bool const first = (t >> 4) < a.n;
    SplitRowsOf const& s = first ? a : b;
    int const row = first ? t >> 4 : (t >> 4) - a.n;
    int const c = t & 15;
    if (row >= s.n) return;
    float4 const* const p = reinterpret_cast<float4 const*>(s.X + (size_t)row * kDim) + 2 * c;
    float4 const u = p[0], w = p[1];
    float const x[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
    v8h hi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float const y = x[k] * kSplitScale;
        hi[k] = (_Float16)y;
        lo[k] = (_Float16)(y - (float)hi[k]);
    }
    unsigned char* const o = s.split + (size_t)row * kSplitRowBytes + (c >> 3) * 256 + (c & 7) * 16;
    *reinterpret_cast<v8h*>(o) = hi;
    *reinterpret_cast<v8h*>(o + 128) = lo;
    if (!s.ints) return;
    float const d = s.scale[row];
    v8h q;
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = x[k] == 0.0f ? (_Float16)0.0f : (_Float16)rintf(__fdiv_rn(x[k], d));
    *reinterpret_cast<v8h*>(s.ints + (size_t)row * kIntRowBytes + c * 16) = q;
}

void launch_split_sets(SplitRowsOf const& a, SplitRowsOf const& b, int* gated, hipStream_t st)
{
    int const rows = a.n + b.n;
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_split_sets, dim3((rows + 15) / 16), dim3(256), 0, st, a, b, gated);
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
                                                      int flagOffR, int* __restrict__ counters,
                                                      int const* __restrict__ gate)
{
    if (gate && !*gate) return;
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
    float const mo = __uint_as_float(maxNormBits[left ? kMaxNormR : 0]);
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
                         int* colMax, int* rowMax, int* flagList, int flagOffR, int* counters, hipStream_t st,
                         int const* gate)
{
    int const n = nL + nR;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_merge_decide, dim3((n + 31) / 32), dim3(256), 0, st, colPart, nColParts, ldc, rowPart,
                       nRowParts, ldr, nL, nR, normL, normR, maxNormBits, epsRel, minScore, minRatio, colMax,
                       rowMax, flagList, flagOffR, counters, gate);
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
// 38 + 5 us in two.  With every query open (a zero error bound, or equal rows) LDS reads bound
// it, with conversions close behind: eight queries a unit, kept as floats, and no more units than
// four a wave (each loads its queries and publishes its partials): 8192 x 8192 2.1 ms, 4096 x 4096
// 0.6; four queries as doubles in units of 64 or 128 candidates 3.7 and 1.3, 16 queries a
// work-group 2.8 and 0.8.
constexpr int kRecheckGroup = 4;  // queries per unit: they share the candidates' loads
constexpr int kRecheckWide = 8;   // ... where every wave has two such units

struct RecheckDir {
    float const* Q;
    float const* C;
    int* sel;
    int nC, cnt, base;  // base: first list entry and row of the partials
    int subs, nCh;
};

__device__ __forceinline__ RecheckDir recheck_dir(bool left, float const* L, float const* R, int nL, int nR, int cnt,
                                                  int rowsL, int rowsR, int* colMax, int* rowMax, int target)
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
    int const most = (int)min(room, (long long)min(nSub, target));
    d.subs = (nSub + most - 1) / max(most, 1);
    d.nCh = (nSub + d.subs - 1) / d.subs;
    return d;
}

template <int kQ, class T>
__device__ __forceinline__ void recheck_units(RecheckDir const& dl, RecheckDir const& dr, int const* flagList,
                                              Top2* __restrict__ part, int* __restrict__ tickets,
                                              unsigned const* __restrict__ gbits, int ldi, float minScore,
                                              float minRatio, float* __restrict__ stage, T* __restrict__ qd)
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

template <bool kSieve>
__global__ __launch_bounds__(256, 3) void k_recheck(float const* __restrict__ L, float const* __restrict__ R, int nL,
                                                 int nR, int const* __restrict__ flagList, int rowsL, int rowsR,
                                                 int const* __restrict__ counters, Top2* __restrict__ part,
                                                 int* __restrict__ tickets, unsigned const* __restrict__ gbits,
                                                 int ldi, float minScore, float minRatio, int* __restrict__ colMax,
                                                 int* __restrict__ rowMax, SieveBest sieve)
{
    __shared__ __attribute__((aligned(16))) float stage[4][kExactLds];
    __shared__ __attribute__((aligned(16))) double qd[4][kRecheckGroup * kDim];
    bool given = false;  // the call is the full pass's
    if constexpr (kSieve) {
        given = sieve.gate && *sieve.gate;
        // the other queries' decisions; the listed ones' follow below
        for (int g = blockIdx.x * 256 + threadIdx.x; g < nL + nR; g += gridDim.x * 256) {
            int const q = g < nL ? g : g - nL;
            int const at = g < nL ? q : sieve.offR + q;
            int const d = sieve_decision(sieve.best + at, sieve.second + at, minScore, minRatio);
            if (d != kFlag) (g < nL ? colMax : rowMax)[q] = d;
        }
    }
    if (given || (!kSieve && sieve.gate && !*sieve.gate)) return;
    int const cntL = __builtin_amdgcn_readfirstlane(counters[kCntFlag]);
    int const cntR = __builtin_amdgcn_readfirstlane(counters[kCntFlagR]);
    // with many queries open no more chunks than give every wave four wide units
    int const target = max(16 * kRecheckWide * (int)gridDim.x / max(cntL + cntR, 1), 1);
    RecheckDir const dl = recheck_dir(true, L, R, nL, nR, cntL, rowsL, rowsR, colMax, rowMax, target);
    RecheckDir const dr = recheck_dir(false, L, R, nL, nR, cntR, rowsL, rowsR, colMax, rowMax, target);
    int const wv = threadIdx.x >> 6;
    // a query per wave while the grid holds a wave for every unit
    long long const single = (long long)cntL * dl.nCh + (long long)cntR * dr.nCh;
    static_assert(kRecheckWide * sizeof(float) <= kRecheckGroup * sizeof(double), "the queries' room");
    if (single <= 4LL * gridDim.x)
        recheck_units<1>(dl, dr, flagList, part, tickets, gbits, ldi, minScore, minRatio, stage[wv], qd[wv]);
    else if (single >= 8LL * kRecheckWide * gridDim.x)
        recheck_units<kRecheckWide>(dl, dr, flagList, part, tickets, gbits, ldi, minScore, minRatio, stage[wv],
                                    reinterpret_cast<float*>(qd[wv]));
    else
        recheck_units<kRecheckGroup>(dl, dr, flagList, part, tickets, gbits, ldi, minScore, minRatio, stage[wv],
                                     reinterpret_cast<float*>(qd[wv]));
}

void launch_recheck_exact(float const* L, float const* R, int nL, int nR, int const* flagList, int rowsL, int rowsR,
                          int const* counters, float minScore, float minRatio, int* colMax, int* rowMax, Top2* part,
                          int* tickets, int grid, hipStream_t st, unsigned const* gbits, int ldi, int* gate)
{
    if (nL <= 0 || nR <= 0) return;
    SieveBest none{};
    none.gate = gate;
    hipLaunchKernelGGL(k_recheck<false>, dim3(grid), dim3(256), 0, st, L, R, nL, nR, flagList, rowsL, rowsR, counters,
                       part, tickets, gbits, ldi, minScore, minRatio, colMax, rowMax, none);
}

// A thread per query; hardly ever is a query listed, and then a bounded number (SieveBest).
void launch_sieve_finish(float const* L, float const* R, int nL, int nR, SieveBest const& b, int const* flagList,
                         int rowsL, int rowsR, int const* counters, float minScore, float minRatio, int* colMax,
                         int* rowMax, Top2* part, int* tickets, unsigned const* gbits, int ldi, hipStream_t st)
{
    if (nL <= 0 || nR <= 0) return;
    hipLaunchKernelGGL(k_recheck<true>, dim3(kRecheckGrid), dim3(256), 0, st, L, R, nL, nR, flagList, rowsL, rowsR, counters,
                       part, tickets, gbits, ldi, minScore, minRatio, colMax, rowMax, b);
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
// re-check and rescoring counts and clears the per-call counters.  Matches and counts also go
// straight to the handle's pinned host block: a copy after the kernel cost about 10 us a call.

// Left feature sampled as sample k of S (evenly spaced over [0, nL)).
__device__ __forceinline__ int sample_row(int k, int nL, int S) { return (int)(((long long)k * nL) / S); }

__device__ __forceinline__ unsigned long long mutual_word(unsigned epoch, unsigned flag, unsigned value)
{
    return ((unsigned long long)epoch << 32) | ((unsigned long long)flag << 30) | value;  // value < 2^30
}

__global__ __launch_bounds__(256) void k_mutual(int const* __restrict__ colMax, int const* __restrict__ rowMax,
                                                int nL, int nR, unsigned long long* __restrict__ status,
                                                unsigned epoch, int* __restrict__ stripes,
                                                int2* __restrict__ pairs, int* __restrict__ counters,
                                                int* __restrict__ host, SampleOut so, MutualWait mw)
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
            if (failed) {
                counters[kCntMutualError] = (int)epoch;
                if (host) host[kCntMutualError] = (int)epoch;
            }
            sBase = excl;
        }
    }
    __syncthreads();
    int pos = sBase + off + incl - cnt;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (m[u]) {
            int2 const pr = make_int2(i0 + u, l[u]);
            if (host) reinterpret_cast<int2*>(host + kNumCounters)[pos] = pr;
            pairs[pos++] = pr;
        }
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
            int const open = counters[kCntFlag] + counters[kCntFlagR];
            counters[kCntPairs] = sBase + total;
            counters[kCntFlagDone] = open;
            counters[kCntFlag] = 0;
            counters[kCntFlagR] = 0;
            counters[kCntRescoredDone] = rescored;
            if (host) {
                host[kCntPairs] = sBase + total;
                host[kCntFlagDone] = open;
                host[kCntGate] = counters[kCntGate];
                host[kCntRescoredDone] = rescored;
            }
            counters[kCntGate] = 0;
            counters[kCntScored] = 0;
        }
    }
}

void launch_mutual_compact(int const* colMax, int const* rowMax, int nL, int nR, unsigned long long* status,
                           unsigned epoch, int* stripes, int2* pairs, int* counters, int* host, hipStream_t st,
                           SampleOut const& so, MutualWait const& mw)
{
    int const nb = (nL + kMutualSlice - 1) / kMutualSlice;
    hipLaunchKernelGGL(k_mutual, dim3(nb > 0 ? nb : 1), dim3(256), 0, st, colMax, rowMax, nL, nR, status, epoch,
                       stripes, pairs, counters, host, so, mw);
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
    float const eps = epsRel * normS[q] * __uint_as_float(maxNormBits[kMaxNormR]) + kEpsAbs;
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
