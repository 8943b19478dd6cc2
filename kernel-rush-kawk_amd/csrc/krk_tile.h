// Tall-tile MFMA skinny GEMM (gfx950): y = epilogue(x[M,K] · W[N,K]ᵀ) for 65
// to 128 rows in one launch, so that a batch of more than 64 rows reads W
// once instead of once per 64 rows; and for 49 to 64 rows of the shapes that
// it is faster on (tile_rows_ok, with the figures).
//
// Reference counterparts: _skinny_kernel / _gateup_kernel with split-K and
// their sum kernels (engine/kernels/gemm.py:54-104, 116-170); the reference
// leaves these row counts to cuBLAS (a tree of 4 rows for each of 32
// sequences, engine/engine.py:501, 571-576).
//
// What bounds it (measured on an MI355X, N x K the Qwen3-4B projections, 128
// rows): the stage loop without loads (LDS fragment reads, MFMAs, a barrier per
// 128 k) takes 17.1 us of gate_up's 32.3 and 8.0 of qkv's 17.2, x loads alone
// add 4 us to it, W loads alone 3-6, both 9-15: a CU takes in 32-49 B/ns of the
// mix, W from HBM and x from L2.  At 128 rows a workgroup that keeps K whole
// reads more x than W, so the time follows the bytes each CU takes in, (rows +
// channels) x K of its split, and splitting K, which shrinks x's share, pays
// for a second launch (4.5 us) only where channels per CU are few (o, down).  A
// wave reads its next fragments, across the stage's barrier, before it
// multiplies the present ones (gate_up 3-4 us faster).
// Against two launches of 64 rows, M = 128: qkv 25.1 -> 17.6 us, gate_up 49.2 ->
// 33.2, down 36.6 -> 24.7, o 23.8 -> 14.6, lm_head 268 -> 230.
//
// Work split: a workgroup owns `cb` output channels (NT tiles of 16 W rows;
// SILU: 8 gate and the matching 8 up rows per tile, as in the stream kernel)
// and one of `splits` ranges of 128-k stages, for all 16·MT rows.  W and x
// pieces of a stage (256 bytes of each row, 4 rows per DMA) go straight to an
// LDS ring of D stages by LDS DMA, D - 1 of them in flight; tile rows are
// XOR-swizzled by 16-byte piece so that fragment reads hit distinct banks.
// The waves form a grid of WM row groups x 2 halves of each stage's k: x is
// read from LDS once, W WM times.  The two halves are added through LDS at
// the end.  W is the MFMA's A operand, so a lane ends with 4 consecutive
// channels of one row and stores them as 8 bytes (SILU: lanes 32-63 hold the
// up sums of lanes 0-31's gates).
//
// Split K: the fp32 sums go to `part` in fragment order (whole 1 KB runs) and
// tile_reduce_kernel adds the splits in order s = 0, 1, ... in a second
// launch.  (The in-kernel fix-up of krk_epilogue.h makes one workgroup per
// block read every split's sums: at 8 splits it cost 7-8 us, this launch 4.5.)
//
// Rows past M and channels past the block load clamped in-range rows, whose
// outputs are not stored; k past K is zeroed in both operands.
#pragma once

#include "krk_epilogue.h"
#include "krk_sync.h"

namespace krk {

constexpr int kTileKC = 128;       // k per stage
constexpr int kTileMaxRows = 128;  // rows per launch
constexpr int kTileMaxNT = 5;
constexpr int kTileMaxSplits = 4;

// Row groups: two m tiles per wave, and two waves per group (halves of k).
__host__ __device__ constexpr int tile_wm(int MT) { return MT / 2; }
__host__ __device__ constexpr int tile_waves(int MT) { return 2 * tile_wm(MT); }
__host__ __device__ constexpr size_t tile_slot_bytes(int MT, int NT) { return (size_t)16 * (MT + NT) * 2 * kTileKC; }
// Ring stages that fit `lds` bytes, 3 to 6.
__host__ __device__ constexpr int tile_depth(int MT, int NT, size_t lds) {
    const int d = (int)(lds / tile_slot_bytes(MT, NT));
    return d > 6 ? 6 : d;
}
__host__ __device__ constexpr size_t tile_lds_bytes(int MT, int NT, int D) {
    const size_t ring = D * tile_slot_bytes(MT, NT), red = (size_t)MT * NT * 1024;
    return ring > red ? ring : red;
}
// fp32 partial sums of one split: whole tiles.
__host__ __device__ constexpr size_t tile_part_bytes(int MT, int NT, int nblk) { return (size_t)nblk * MT * NT * 1024; }

struct TileArgs {
    const uint16_t* x;
    int64_t ldx;
    const uint16_t* w;
    int64_t ldw;
    uint16_t* y;
    int64_t ldy;
    int M, N, K, splits, cb, nblk;
    float* part;
};

// Four consecutive output channels of row m, from channel cl of block blk:
// v = the lane's sums.  Called by all lanes of a wave.
template <bool SILU>
__device__ __forceinline__ void tile_store(const TileArgs& a, int blk, int t, int q, int m, const f32x4& v, bool vec) {
    uint32_t o[4];
    if constexpr (SILU) {
        // Tile rows 0-7 are gates (lanes 0-31), rows 8-15 ups (lanes 32-63).
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const auto gu = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[e]), __float_as_uint(v[e]), false, false);
            o[e] = silu_mul_bf16(__uint_as_float(gu[0]), __uint_as_float(gu[1]));
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f32_to_bf16(v[e]);
    }
    const int Nout = SILU ? a.N >> 1 : a.N;
    const int cl = SILU ? 8 * t + 4 * (q & 1) : 16 * t + 4 * q;
    const int c = blk * a.cb + cl;
    if (m >= a.M || (SILU && q >= 2)) return;
    uint16_t* d = a.y + (int64_t)m * a.ldy + c;
    if (vec && cl + 4 <= a.cb && c + 4 <= Nout) {
        *reinterpret_cast<uint2*>(d) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (cl + e < a.cb && c + e < Nout) d[e] = (uint16_t)o[e];
    }
}
// 8-byte stores: y and its rows 8-byte aligned (cb is a multiple of 4).
__device__ __forceinline__ bool tile_vec_ok(const TileArgs& a) {
    return (reinterpret_cast<uintptr_t>(a.y) & 7) == 0 && (a.ldy & 3) == 0;
}

// MT 16-row x tiles, NT 16-row W tiles, D ring stages.  Grid: nblk x splits
// workgroups, split = blockIdx % splits.
template <int MT, int NT, int D, bool SILU>
__global__ void __launch_bounds__(64 * tile_waves(MT))
tile_gemm_kernel(TileArgs a) {
    constexpr int KC = kTileKC, WM = tile_wm(MT), WV = tile_waves(MT), MTW = 2, KPW = 2;
    constexpr int RB = 2 * KC, RG = 1024 / RB, LR = 64 / RG;  // bytes per tile row, rows and lanes per row of a DMA
    constexpr int NR = 16 * NT, MX = 16 * MT, G = (NR + MX) / RG;
    constexpr int LO = G / WV, REM = G % WV, HI = LO + (REM ? 1 : 0);  // DMAs per wave and stage: HI on waves < REM
    constexpr int SLOT = (NR + MX) * RB;
    static_assert(MT % 2 == 0 && MT <= 8, "two m tiles per wave");
    static_assert(KC / 32 == 2 * KPW && LR == 16, "two k-steps per wave and stage");
    static_assert(D >= 3 && D <= 8 && (D - 2) * HI < 64, "waits count up to 63 DMAs");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int wm = wave % WM, wk = wave / WM;
    const int s = a.splits == 1 ? 0 : blockIdx.x % a.splits;
    // Unsplit: each XCD's blocks adjacent, so the partial lines of y that
    // neighbouring blocks write meet in one L2.
    const int blk = a.splits == 1 ? xcd_block(blockIdx.x, a.nblk) : blockIdx.x / a.splits;
    const int Nout = SILU ? a.N >> 1 : a.N;

    // Source row and swizzled piece of each DMA: tile rows W first, then x.
    const uint16_t* src[HI];
    int kof[HI];
#pragma unroll
    for (int j = 0; j < HI; ++j) {
        int g = wave + WV * j;
        g = g < G ? g : 0;  // a wave without a last DMA
        const int row = RG * g + lane / LR;
        kof[j] = 8 * ((lane % LR) ^ (row & 15));
        if (row < NR) {
            int cl = SILU ? 8 * (row >> 4) + (row & 7) : row;
            cl = cl < a.cb ? cl : a.cb - 1;
            int ch = blk * a.cb + cl;
            ch = ch < Nout ? ch : Nout - 1;
            src[j] = a.w + (int64_t)((SILU && (row & 8)) ? ch + Nout : ch) * a.ldw;
        } else {
            const int m = row - NR;
            src[j] = a.x + (int64_t)(m < a.M ? m : a.M - 1) * a.ldx;
        }
    }
    const int KST = (a.K + KC - 1) / KC;
    const int sb = (int)(((int64_t)s * KST) / a.splits);
    const int se = (int)(((int64_t)(s + 1) * KST) / a.splits);
    const int nst = se - sb;
    const bool ragged = a.K % KC != 0 && se == KST;  // the last stage ends past K

    auto issue = [&](int t) {
        const int k0 = (sb + t) * KC;
        unsigned char* const slot = smem + (t % D) * SLOT;
        const bool tail = ragged && t == nst - 1;
#pragma unroll
        for (int j = 0; j < HI; ++j) {
            const int g = wave + WV * j;
            if (j < LO || wave < REM) {
                int k = k0 + kof[j];
                if (tail) k = k < a.K ? k : 0;  // any in-range piece: zeroed at use
                if (RG * g < NR) dma_row_stream(src[j] + k, slot + g * 1024);
                else dma_row(src[j] + k, slot + g * 1024);
            }
        }
    };
    // Stage t readable by every wave and the slot of stage t - 1 free: this
    // wave's DMAs of it have landed, all waves' after the barrier.
    auto landed = [&](int t) {
        const int ahead = nst - 1 - t < D - 2 ? nst - 1 - t : D - 2;
        if (REM && wave < REM) vm_wait_stages<HI>(ahead);
        else vm_wait_stages<LO>(ahead);
        bare_barrier();
        if (t + D - 1 < nst) issue(t + D - 1);
    };
    u32x4 F[2][NT + MTW];
    auto read = [&](u32x4 (&f)[NT + MTW], const unsigned char* slot, int kk) {
        const int lo = 16 * ((4 * (wk * KPW + kk) + q) ^ r);
#pragma unroll
        for (int t = 0; t < NT; ++t) f[t] = *reinterpret_cast<const u32x4*>(slot + (16 * t + r) * RB + lo);
#pragma unroll
        for (int i = 0; i < MTW; ++i)
            f[NT + i] = *reinterpret_cast<const u32x4*>(slot + (NR + 16 * (wm * MTW + i) + r) * RB + lo);
    };
    f32x4 acc[MTW][NT];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mma = [&](u32x4 (&f)[NT + MTW], int t, int kk) {
        if (ragged && t == nst - 1) {
            const uint32_t mk = (sb + t) * KC + 8 * (4 * (wk * KPW + kk) + q) < a.K ? 0xffffffffu : 0u;
#pragma unroll
            for (int z = 0; z < NT + MTW; ++z) f[z] &= mk;
        }
#pragma unroll
        for (int i = 0; i < MTW; ++i)
#pragma unroll
            for (int t2 = 0; t2 < NT; ++t2)
                acc[i][t2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, f[t2]), __builtin_bit_cast(bf16x8, f[NT + i]), acc[i][t2], 0, 0, 0);
    };

    for (int d = 0; d < D - 1 && d < nst; ++d) issue(d);
    if (nst > 0) {
        landed(0);
        read(F[0], smem, 0);
        int sl = 0;
        for (int t = 0; t < nst; ++t) {
            const unsigned char* const slot = smem + sl * SLOT;
            sl = sl + 1 == D ? 0 : sl + 1;
            read(F[1], slot, 1);
            __builtin_amdgcn_sched_barrier(0);
            mma(F[0], t, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1 < nst) {
                lds_wait();  // this wave has read all of stage t
                landed(t + 1);
                read(F[0], smem + sl * SLOT, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            mma(F[1], t, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The second halves' sums through LDS (every wave is done with the ring).
    f32x4* const red = reinterpret_cast<f32x4*>(smem);
    lds_wait();
    bare_barrier();
    if (wk) {
#pragma unroll
        for (int i = 0; i < MTW; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) red[((wm * MTW + i) * NT + t) * 64 + lane] = acc[i][t];
    }
    lds_wait();
    bare_barrier();
    if (wk) return;
    const bool vec = tile_vec_ok(a);
#pragma unroll
    for (int i = 0; i < MTW; ++i) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int tile = (wm * MTW + i) * NT + t;
            const f32x4 v = acc[i][t] + red[tile * 64 + lane];
            if (a.splits == 1) {
                tile_store<SILU>(a, blk, t, q, 16 * (wm * MTW + i) + r, v, vec);
            } else {
                float* const p = a.part + ((size_t)s * a.nblk + blk) * (MT * NT * 256) + tile * 256 + lane * 4;
                *reinterpret_cast<f32x4*>(p) = v;
            }
        }
    }
}

constexpr int kTileReduceThreads = 256;

// Adds the S splits' partial sums in order and applies the epilogue: one
// thread per (block, tile, lane) of tile_gemm_kernel<MT, NT, ...>.
template <int S, bool SILU>
__global__ void __launch_bounds__(kTileReduceThreads)
tile_reduce_kernel(TileArgs a, int MT, int NT) {
    const int per = MT * NT * 64;
    const int id = blockIdx.x * kTileReduceThreads + threadIdx.x;
    const int blk = id / per;
    if (blk >= a.nblk) return;  // whole waves: per is a multiple of 64
    const int rem = id - blk * per;
    const int tile = rem >> 6, lane = rem & 63;
    const int i = tile / NT, t = tile - i * NT;
    const size_t stride = (size_t)a.nblk * per * 4;
    const float* const p = a.part + (size_t)id * 4;
    f32x4 v[S];
#pragma unroll
    for (int z = 0; z < S; ++z) v[z] = *reinterpret_cast<const f32x4*>(p + z * stride);
    f32x4 sum = v[0];
#pragma unroll
    for (int z = 1; z < S; ++z) sum += v[z];
    tile_store<SILU>(a, blk, t, lane >> 4, 16 * i + (lane & 15), sum, tile_vec_ok(a));
}

}  // namespace krk
