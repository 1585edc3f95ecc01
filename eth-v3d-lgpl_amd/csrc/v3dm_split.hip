// Plain FP32 putative matching on FP16 matrix instructions (gfx950): the fused score pass of
// v3dm_fp32.hip with every descriptor split in two FP16 parts (v3dm_split.h).
//
// v_mfma_f32_32x32x2_f32 runs at 1/16 of v_mfma_f32_32x32x16_f16's rate; three FP16
// products per score give the FP32 product's accuracy at 3/16 of its matrix time.
//
// Reference path: V3D_CUDA::SIFT_Matching::findPutativeMatches
// (V3D/CUDA/v3d_cudamatching.cu:522-552); as there, scores, best and second best are FP32.
#include <type_traits>

#include "v3dm_device.h"
#include "v3dm_kernels.h"
#include "v3dm_split.h"

namespace v3dm {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

// ------------------------------------------------------------------------------ score pass
// Work-group: kW waves of 64 left features each (two 32-column blocks whose hi and lo parts
// are the resident B operands, 128 VGPRs), streaming 32-row tiles of right features through
// two LDS stages filled by direct global->LDS loads.  Why this shape: a tile's parts (16 KiB)
// are read from LDS once per wave for two column blocks, so 48 matrix instructions (1536
// cycles) stand against 16 KiB of operand reads, 16 KiB of the score transpose below (256
// LDS cycles a wave together, 1024 of the CU's per tile) and about 300 vector instructions
// (1200 cycles) that the SIMD's other wave overlaps; 256 VGPRs leave two waves per SIMD, and
// the 70 KiB of LDS two work-groups per CU, which drift apart and fill each other's gaps.
// Counts are multiples of 32, so no tile and no column block is partial; a wave's second (or
// every) block past nL is skipped.
//
// Lane l holds column c = l % 32 and rows j = 8 (r / 4) + 4 (l / 32) + r % 4 of each 32x32
// block.  Per left feature the running top-2 stays in registers (the position inside the tile
// as r, the tile noted once per tile when the best changed); per right feature each wave
// writes its scores to its own LDS rows, reads them back a row per lane pair, and the waves'
// partial top-2 of a tile are merged by one of them after the next tile's barrier, so a tile
// costs one barrier.
//
// k index of matrix step s: h*64 + 8*s + v (h = l / 32); the parts of one score are added
// small products first (lo hi, hi lo, then hi hi) step by step.
//
// What bounds it: matrix instructions on real descriptors, which draw the card's power limit
// (three products of 16384 x 16384 run at 1.05 PFLOP/s here; a loop of nothing but the
// instruction reaches 1.48, the library's 8192^3 product 1.2), then the selection beside them
// (the products and operand reads alone take 164 us of the 196).
// 16384 x 16384: 196 us against 605-635 us of k_fused_fp32; 8192 x 7936: 59 against 185 us.
// One tile's selection after its products instead of beside the next tile's: 210 us; every
// position tracked instead of looked for: 215 against 195 us (same box).
constexpr int kSplitTileBytes = kSplitTile * kSplitRowBytes;  // 16 KiB
constexpr int kSplitPair = 1024 + 16;                         // two rows and a pad
constexpr int kSplitStage = (kSplitTile / 2) * kSplitPair;
constexpr int kTRow = 36;                            // floats per row of the transposed block

template <int kW>
struct SplitLds {
    __attribute__((aligned(16))) unsigned char stage[2][kSplitStage];
    __attribute__((aligned(16))) float trans[kW][2][kSplitTile * kTRow];
    float absent[kSplitTile * kTRow];  // where column blocks past nL write their scores
    float rowB1[2][kW][kSplitTile], rowB2[2][kW][kSplitTile];
    int rowA1[2][kW][kSplitTile];
};

// Stage layout: a direct load fills 1 KiB (two rows as they lie in memory, lane L at +16 L)
// and the next pair of rows starts 16 bytes further on; in odd rows hi and lo are swapped (each lane
// fetches the chunk that belongs at its slot).  The 16 rows that a group of lanes reads one
// chunk of then lie on distinct 16-byte columns of the 256 bytes of banks (with the two
// 64-byte halves swapped instead, a quarter of the LDS cycles were conflicts), and a lane's
// chunks need two addresses (hi and lo) with constant offsets.
__device__ __forceinline__ int split_src(int tid) { return (tid * 16) ^ ((tid & 32) << 2); }

// R as a raw buffer resource: a tile's loads take one scalar offset and the 32-bit lane offset
// (64-bit lane addresses would not leave room for the operands).
template <int kW>
__device__ __forceinline__ void split_stage(__amdgpu_buffer_rsrc_t R, int t, unsigned char* stage, int src, int wv)
{
#pragma unroll
    for (int p = 0; p < kSplitTile / (2 * kW); ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(R, (lds_void*)(stage + (kW * p + wv) * kSplitPair), 16, src,
                                                 t * kSplitTileBytes + p * (1024 * kW), 0, 0);
}

// Best and second best of a stream of scores, without the position: 13 instructions per 8
// scores (two triples by max3 / med3, a pair, three states merged by max3 / med3) where
// pushing them one by one with the position took 32.
struct Best2 {
    float b1, b2;
};

__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

__device__ __forceinline__ Best2 best2_of8(float const (&x)[8])
{
    float const h0 = max3(x[0], x[1], x[2]), m0 = __builtin_amdgcn_fmed3f(x[0], x[1], x[2]);
    float const h1 = max3(x[3], x[4], x[5]), m1 = __builtin_amdgcn_fmed3f(x[3], x[4], x[5]);
    float const h2 = fmaxf(x[6], x[7]), m2 = fminf(x[6], x[7]);
    return Best2{max3(h0, h1, h2), fmaxf(__builtin_amdgcn_fmed3f(h0, h1, h2), max3(m0, m1, m2))};
}

__device__ __forceinline__ Best2 best2_merge(Best2 a, Best2 b)
{
    return Best2{fmaxf(a.b1, b.b1), max3(a.b2, b.b2, fminf(a.b1, b.b1))};
}

// 2^-28 of a best or second best; the initial state stays kInit.
__device__ __forceinline__ float split_back(float b) { return b > -1e29f ? b * kSplitBack : kInit; }

// The partial top-2 of tile t's right features from the waves' LDS entries.
template <int kW>
__device__ __forceinline__ void split_merge_rows(SplitLds<kW> const& lds, int t, int lane, Top2* __restrict__ rowPart)
{
    if (lane >= kSplitTile) return;
    Top2 s = top2_init();
#pragma unroll
    for (int w = 0; w < kW; ++w)
        s = top2_merge(s, Top2{lds.rowB1[t & 1][w][lane], lds.rowB2[t & 1][w][lane], lds.rowA1[t & 1][w][lane]});
    s.b1 = split_back(s.b1);
    s.b2 = split_back(s.b2);
    // transposed row 16 h + r holds row 8 (r / 4) + 4 h + r % 4 of the tile
    rowPart[t * kSplitTile + 8 * ((lane & 15) >> 2) + 4 * (lane >> 4) + (lane & 3)] = s;
}

// Running state of one left feature: at = 16 * tile + r of the best, kept only while the
// best exceeds the caller's minimum score.
struct ColState {
    Best2 s;
    int at;
};

// Where a lane's stream position p (a multiple of 4) lies in its wave's transposed blocks.
constexpr int split_tr(int p) { return (p >> 4) * (kSplitTile * kTRow) + (p & 15); }

// The selection of one tile (both directions) in eight parts, one per matrix step of the
// next tile: parts 0-3 the left features (and the scores to LDS), parts 4-7 the right
// features, read back a part ahead.
//
// A position is looked for only where a new best exceeds thr (the caller's minimum score):
// a query whose best does not is rejected or re-checked exactly whatever the position, and a
// query that is accepted has its best above it.  At the usual 0.9 one tile in twenty of a
// wave holds such a score; with a minimum below most scores the search costs what tracking
// the position of every score would.
struct Selection {
    Best2 row;
    float old;
    float4 next[2];  // the coming columns
};

template <bool kGuided, int kW>
__device__ __forceinline__ void select_part(int part, Selection& x, v16f (&acc)[2], unsigned const (&gw)[2],
                                            ColState (&col)[2], int t, float* const (&tw)[2], float const* tr,
                                            SplitLds<kW>& lds, int wv, int lane, int i0, float thr)
{
    if (part < 4) {
        int const cb = part >> 1, r0 = 8 * (part & 1);
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            int const e = r0 + r;
            if (kGuided)
                acc[cb][e] = ((gw[cb] >> (8 * (e >> 2) + (e & 3))) & 1u) ? -1e20f / kSplitBack : acc[cb][e];
            v[r] = acc[cb][e];
            tw[cb][e * kTRow] = v[r];
        }
        if (r0 == 0) x.old = col[cb].s.b1;
        col[cb].s = best2_merge(col[cb].s, best2_of8(v));
        if (r0 != 0) {
            float const b = col[cb].s.b1;
            bool const better = b > fmaxf(x.old, thr);
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(better) != 0, 0)) {
                int at = 0;
#pragma unroll
                for (int r = 15; r >= 0; --r) at = acc[cb][r] == b ? r : at;  // the first of equal bests
                col[cb].at = better ? 16 * t + at : col[cb].at;
            }
        }
        // the wave's own LDS rows: its writes come before its reads (LDS operations of one
        // wave are in order)
        if (part == 3) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
        float const v[8] = {x.next[0].x, x.next[0].y, x.next[0].z, x.next[0].w,
                            x.next[1].x, x.next[1].y, x.next[1].z, x.next[1].w};
        Best2 const b = best2_of8(v);
        x.row = part == 4 ? b : best2_merge(x.row, b);
    }
    if (part >= 3 && part < 7) {
        x.next[0] = *reinterpret_cast<float4 const*>(tr + split_tr(8 * (part - 3)));
        x.next[1] = *reinterpret_cast<float4 const*>(tr + split_tr(8 * (part - 3) + 4));
    }
    if (part == 7) {
        // the two halves of the wave hold 32 columns of a row each; both end with the merged
        // state and write it
        float const o1 = __shfl_xor(x.row.b1, 32), o2 = __shfl_xor(x.row.b2, 32);
        Best2 const both = best2_merge(x.row, Best2{o1, o2});
        int a1 = -1;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(both.b1 > thr) != 0, 0)) {
            // position p of the lane's stream: column block p / 16, column 16 h + p % 16
            int q = 64;
#pragma unroll
            for (int p = 28; p >= 0; p -= 4) {
                float4 const v = *reinterpret_cast<float4 const*>(tr + split_tr(p));
                q = v.w == both.b1 ? p + 3 : q;
                q = v.z == both.b1 ? p + 2 : q;
                q = v.y == both.b1 ? p + 1 : q;
                q = v.x == both.b1 ? p : q;
            }
            int at = q == 64 ? 0x7fffffff : i0 + (q >> 4) * 32 + 16 * (lane >> 5) + (q & 15);
            at = min(at, __shfl_xor(at, 32));  // the first of equal bests
            a1 = both.b1 > thr ? at : -1;
        }
        lds.rowB1[t & 1][wv][lane & 31] = both.b1;
        lds.rowB2[t & 1][wv][lane & 31] = both.b2;
        lds.rowA1[t & 1][wv][lane & 31] = a1;
    }
}

// One work unit: left block lb (64 * kW features) against right tiles [t0, t1) -> colPart[i],
// rowPart[j] (the caller's split and left block offsets applied).
template <bool kGuided, int kW>
__device__ __forceinline__ void split_block(unsigned char const* __restrict__ L, unsigned char const* __restrict__ R,
                                            int nL, int lb, int t0, int t1, Top2* __restrict__ colPart,
                                            Top2* __restrict__ rowPart, unsigned const* __restrict__ bits, int ldi,
                                            SplitLds<kW>& lds, float thr)
{
    int tid = threadIdx.x;
    __asm__ volatile("" : "+v"(tid));
    int const lane = tid & 63;
    int const wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const h = lane >> 5;
    int const c32 = lane & 31;
    int const i0 = lb * (64 * kW) + wv * 64;
    int const nBlk = min(max((nL - i0) / 32, 0), 2);  // column blocks of this wave that exist

    int const src = split_src(tid);
    __amdgpu_buffer_rsrc_t const rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(R), 0, t1 * kSplitTileBytes, 0x00027000);
    split_stage<kW>(rs, t0, lds.stage[0], src, wv);

    // rows past nL are inside the buffer (a multiple of kSplitRowPad rows) and never used
    v8h bh[2][8], bl[2][8];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        uint4 const* p = reinterpret_cast<uint4 const*>(L + (size_t)(i0 + cb * 32 + c32) * kSplitRowBytes + h * 256);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            bh[cb][s] = __builtin_bit_cast(v8h, p[s]);
            bl[cb][s] = __builtin_bit_cast(v8h, p[8 + s]);
        }
    }

    // scores of a column block past nL go to `absent`; the rows read for it hold -3e30, below
    // the initial state, and never count
    float* tw[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        float* const own = lds.trans[wv][cb];
        tw[cb] = (cb < nBlk ? own : lds.absent) + 16 * h * kTRow + c32;
        if (cb >= nBlk)
            for (int k = lane; k < kSplitTile * kTRow; k += 64) own[k] = -3e30f;
    }
    float const* const tr = lds.trans[wv][0] + c32 * kTRow + 16 * h;

    ColState col[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) col[cb] = ColState{Best2{kInit, kInit}, -1};
    unsigned gw[2] = {0, 0}, gp[2] = {0, 0};
    v16f acc[2], prev[2];

    int const at = (c32 >> 1) * kSplitPair + (c32 & 1) * 512 + h * 256;  // the lane's half row of a stage

    // Tile t's products beside the selection of tile t - 1 from `prev`
    auto step = [&](int t, auto select) {
        wait_lds_loads();
        __syncthreads();  // tile t is staged; every wave is done with the other stage
        int const cur = (t - t0) & 1;
        if (t + 1 < t1) split_stage<kW>(rs, t + 1, lds.stage[cur ^ 1], src, wv);
        // the partials of tile t - 2 were written before this barrier
        if (t >= t0 + 2 && wv == t % kW) split_merge_rows<kW>(lds, t - 2, lane, rowPart);
        if (kGuided) {
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
                if (cb < nBlk) gw[cb] = bits[(size_t)t * ldi + i0 + cb * 32 + c32] >> (4 * h);
        }
        unsigned char const* const Ah = lds.stage[cur] + at + 128 * (c32 & 1);
        unsigned char const* const Al = lds.stage[cur] + at + 128 * (~c32 & 1);
        v8h al = *reinterpret_cast<v8h const*>(Al), ah = *reinterpret_cast<v8h const*>(Ah);
        acc[0] = v16f{};
        acc[1] = v16f{};
        Selection x;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[0][s], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[1][s], acc[1], 0, 0, 0);
            if (s < 7) al = *reinterpret_cast<v8h const*>(Al + 16 * (s + 1));
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[0][s], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[1][s], acc[1], 0, 0, 0);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[0][s], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[1][s], acc[1], 0, 0, 0);
            if (s < 7) ah = *reinterpret_cast<v8h const*>(Ah + 16 * (s + 1));
            if (decltype(select)::value) {
                select_part<kGuided, kW>(s, x, prev, gp, col, t - 1, tw, tr, lds, wv, lane, i0, thr);
                // one matrix instruction per six of the selection's; nothing moves between steps
#pragma unroll
                for (int k = 0; k < 6; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x080, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            prev[cb] = acc[cb];
            gp[cb] = gw[cb];
        }
    };
    step(t0, std::false_type{});
    for (int t = t0 + 1; t < t1; ++t) step(t, std::true_type{});
    {
        Selection x;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            select_part<kGuided, kW>(s, x, prev, gp, col, t1 - 1, tw, tr, lds, wv, lane, i0, thr);
    }
    __syncthreads();  // the last tiles' partials (and, in a persistent kernel, the stages)
    if (wv == t1 % kW) split_merge_rows<kW>(lds, t1 - 1, lane, rowPart);
    if (t1 - t0 >= 2 && wv == (t1 + 1) % kW) split_merge_rows<kW>(lds, t1 - 2, lane, rowPart);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        int const p = col[cb].at;
        int const j = p < 0 ? -1 : (p >> 4) * kSplitTile + 8 * ((p & 15) >> 2) + 4 * h + (p & 3);
        Top2 cs{col[cb].s.b1, col[cb].s.b2, j};
        cs = top2_merge(cs, top2_shfl_xor(cs, 32));
        cs.b1 = split_back(cs.b1);
        cs.b2 = split_back(cs.b2);
        if (h == 0 && cb < nBlk) colPart[i0 + cb * 32 + c32] = cs;
    }
}

template <bool kGuided>
__global__ __launch_bounds__(256, 2) void k_split_pass(unsigned char const* __restrict__ L,
                                                       unsigned char const* __restrict__ R, int nL, int nR,
                                                       int leftBlocks, int tilesPerSplit, Top2* __restrict__ colPart,
                                                       int ldc, Top2* __restrict__ rowPart, int ldr,
                                                       unsigned const* __restrict__ bits, int ldi, float thr)
{
    __shared__ SplitLds<4> lds;
    // neighbouring work-groups of one XCD share a split's right tiles in its L2
    int const b = xcd_block(blockIdx.x, gridDim.x);
    int const split = b / leftBlocks, lb = b - split * leftBlocks;
    int const t0 = split * tilesPerSplit;
    int const t1 = min(t0 + tilesPerSplit, nR / kSplitTile);
    split_block<kGuided, 4>(L, R, nL, lb, t0, t1, colPart + (size_t)split * ldc, rowPart + (size_t)lb * ldr, bits, ldi,
                            lds, thr);
}

// The pass's scores of one 32x32 block per wave, written out (v3dm_score_block): the same
// operands, instructions and order as split_block.
__global__ __launch_bounds__(64) void k_split_scores(unsigned char const* __restrict__ L,
                                                     unsigned char const* __restrict__ R, int nRows, int nCols,
                                                     float* __restrict__ out)
{
    int const lane = threadIdx.x;
    int const h = lane >> 5;
    int const c32 = lane & 31;
    int const i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
    uint4 const* q = reinterpret_cast<uint4 const*>(L + (size_t)(i0 + c32) * kSplitRowBytes + h * 256);
    uint4 const* c = reinterpret_cast<uint4 const*>(R + (size_t)(j0 + c32) * kSplitRowBytes + h * 256);
    v16f acc = v16f{};
    for (int s = 0; s < 8; ++s) {
        v8h const ah = __builtin_bit_cast(v8h, c[s]), al = __builtin_bit_cast(v8h, c[8 + s]);
        v8h const bh = __builtin_bit_cast(v8h, q[s]), bl = __builtin_bit_cast(v8h, q[8 + s]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc, 0, 0, 0);
    }
    int const i = i0 + c32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        int const j = j0 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (i < nRows && j < nCols) out[(size_t)i * nCols + j] = acc[r] * kSplitBack;
    }
}

void launch_score_block_split(unsigned char const* L, unsigned char const* R, int nRows, int nCols, float* out,
                              hipStream_t st)
{
    dim3 const grid((nCols + 31) / 32, (nRows + 31) / 32);
    hipLaunchKernelGGL(k_split_scores, grid, dim3(64), 0, st, L, R, nRows, nCols, out);
}

// Splits of the right features: the work-groups run in rounds of 512 (two per CU), so the
// pass takes about ceil(groups / 512) * (tiles per split + the operand load and the column
// merge, about two tiles); the smallest of that, fewer splits on a tie.
FusedPlan plan_split(int nL, int nR)
{
    FusedPlan p;
    p.leftBlocks = (nL + 255) / 256;
    int const nTiles = nR / kSplitTile;
    int best = 0x7fffffff;
    for (int s = 1; s <= kMaxSplits && s <= nTiles; ++s) {
        int const tiles = (nTiles + s - 1) / s;
        int const splits = (nTiles + tiles - 1) / tiles;
        int const rounds = (int)(((long long)p.leftBlocks * splits + 511) / 512);
        int const cost = rounds * (tiles + 2);
        if (cost < best) {
            best = cost;
            p.splits = splits;
            p.tilesPerSplit = tiles;
        }
    }
    return p;
}

void launch_split_pass(unsigned char const* L, unsigned char const* R, int nL, int nR, FusedPlan const& p,
                       Top2* colPart, int ldc, Top2* rowPart, int ldr, unsigned const* bits, int ldi, float minScore,
                       hipStream_t st)
{
    if (nL <= 0 || nR <= 0) return;
    dim3 const grid(p.leftBlocks * p.splits);
    float const thr = minScore / kSplitBack;  // exact: a power of two
    if (bits)
        hipLaunchKernelGGL(k_split_pass<true>, grid, dim3(256), 0, st, L, R, nL, nR, p.leftBlocks, p.tilesPerSplit,
                           colPart, ldc, rowPart, ldr, bits, ldi, thr);
    else
        hipLaunchKernelGGL(k_split_pass<false>, grid, dim3(256), 0, st, L, R, nL, nR, p.leftBlocks, p.tilesPerSplit,
                           colPart, ldc, rowPart, ldr, bits, ldi, thr);
}

}  // namespace v3dm
