// float16/bfloat16 GEMM for large problems on gfx950: 256x256 workgroup tiles,
// 8 waves (two per SIMD), v_mfma_f32_16x16x32, operands fetched from global
// memory straight into LDS by buffer loads (no register staging) through a
// ring of four 32-k stages.
//
// Reference semantics: the same operand model and epilogue as the other
// tvk_gemm kernels (src/shaders/helpers/gemm.slang:3-9,
// src/shaders/helpers/gemm_simd.slang:67-99); only the summation order inside
// a 32-k step differs (the MFMA's), as with the reference's coop-matrix path
// (src/shaders/ops/matmul_coop.slang:172-222).
//
// LDS layouts (per stage, per operand, 16 KB). gfx950's LDS has 64 banks of
// 4 bytes; a ds_read_b128 is served 16 lanes a cycle, in the lane groups
// {0-3, 12-15, 20-27}, {16-19, 28-31, 4-11} and the same two shifted by 32
// (measured: bank-conflict counters over address patterns that tell the
// groupings apart); a ds_read_b64 (also the transposing one) 32 lanes a
// cycle. A read is conflict-free when each group's 16-byte (8-byte) units
// fall on distinct banks.
//   k-contiguous operand ("KM"): BM or BN rows x 32 k, 64 B per row. Row r's
//     16-byte chunk c sits at slot c ^ swz_km(r). With the wide swizzle,
//     (r >> 1) & 3, each lane group of a fragment read (16 rows x one chunk)
//     lands on 16 distinct 16-byte bank slots; the narrow one,
//     ((r >> 1) ^ (r >> 3)) & 3, puts two units of a group on one slot.
//   m/n-contiguous operand ("MN"): 32 k-rows x W columns (W >= 128), 2W bytes
//     per row, chunk slot c ^ swz_mn(k). Fragments are read with
//     ds_read_b64_tr_b16, which transposes 4 k-rows x 16 columns across each
//     16-lane group; the 32 lanes served together read k-rows 8g + 0..3 and
//     8(g+1) + 0..3. The wide swizzle spreads them over all 64 banks (bit 3
//     of the k-row selects the other half of the bank window); the narrow one
//     leaves the two row groups on the same banks (two cycles a read).
// The 128x128 tiles use the wide swizzles; the 256x256 tile the narrow ones,
// measured 1 % faster there (its LDS reads are not what limits it, and the
// wide MN swizzle spills registers when A is the MN operand).
// Each buffer load writes one contiguous 1 KB block of LDS (lane l's 16 bytes
// at offset 16*l), so every block is 16 KM rows or 2 MN rows.
//
// Pipeline, per 32-k stage kt (each wave: 32 MFMAs of 16x16x32 on a 128x64
// wave tile): the MFMAs use fragments already in registers; between them the
// wave reads the next stage's fragments and issues its share of the loads of
// stage kt+4 into the slot stage kt occupied (free: every wave read it before
// the previous barrier). One barrier per stage, after waiting until stage kt+2
// has landed. The loads are issued from inline assembly: a compiler-visible
// LDS-DMA would make every later LDS read wait for all of them.
#pragma once

#include "gemm_common.h"

#include <type_traits>

namespace tvk {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define TVK_LDS __attribute__((address_space(3)))

constexpr int D_BK = 32;

// Tile configurations: 256x256 runs 8 waves of 128x64; the others 64x64 wave
// tiles (128x128: 4 waves, 256x128 and 128x256: 8 waves).
template <int BM_, int BN_>
struct DCfg {
    static constexpr int BM = BM_, BN = BN_;
    static constexpr bool BIG = BM == 256 && BN == 256;
    static constexpr int NW = BIG ? 8 : (BM / 64) * (BN / 64);
    static constexpr int NT = 64 * NW;
    static constexpr int WN = BIG ? 4 : BN / 64;           // waves along N
    static constexpr int WMW = NW / WN;                     // waves along M
    static constexpr int WTM = BM / WMW, WTN = BN / WN;     // wave tile
    static constexpr int FM = WTM / 16, FN = WTN / 16;
    static constexpr int OPA = BM * D_BK * 2, OPB = BN * D_BK * 2;   // bytes per operand per stage
    static constexpr int STB = OPA + OPB;
    static constexpr int DA = OPA / 1024 / NW, DB = OPB / 1024 / NW; // loads per wave per stage
    static constexpr int DS = DA + DB;
    static_assert(DA >= 1 && DB >= 1 && WTN == 64, "tile configuration");
};

// Buffer resource over [p, p + bytes): loads past the end return zeros.
__device__ inline i32x4 dma_rsrc(const void* p, int64_t bytes) {
    const uint64_t a = (uint64_t)p;
    return i32x4{(int)(uint32_t)a, (int)((a >> 32) & 0xffff), (int)min(bytes, (int64_t)0x7fffffff), 0x00020000};
}

// 16 bytes per lane from r + voff into LDS at lds_addr + 16 * lane (lds_addr
// is wave-uniform; it travels in M0).
__device__ inline void dma16(i32x4 r, uint32_t lds_addr, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(r) : "memory");
}

template <int N>
__device__ inline void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

template <bool WIDE>
__device__ inline int swz_km(int row) { return WIDE ? (row >> 1) & 3 : ((row >> 1) ^ (row >> 3)) & 3; }
template <bool WIDE>
__device__ inline int swz_mn(int kr) { return WIDE ? ((kr & 3) | (((kr >> 3) & 1) << 2)) * 2 : (kr & 3) * 2; }

// Per-lane source offsets (bytes, at k = 0) of one operand's loads. Rows or
// columns outside the matrix start at kOOB, so with the k advance added they
// stay past the buffer's end and load zeros.
// D loads per wave; W = the tile's extent along this operand's rows (m or n):
// an MN tile has k-rows of 2W bytes, 1024 / (2W) of them per 1 KB load; XS:
// the wide swizzles.
template <bool KM, int D, int W, bool XS>
struct DmaSrc {
    static_assert(KM || W >= 128, "the MN swizzle moves chunks within 16-chunk blocks");
    uint32_t off[D];
    uint32_t tail[D];   // added in the last stage: past the buffer for a KM chunk at or past k_left, else 0
    uint32_t kstep;     // bytes per stage along k
    __device__ inline void init(int64_t s_row, int64_t s_k, int row0, int rows, int wave, int lane, int k_left) {
        constexpr int CPR = 2 * W / 16;   // 16-byte chunks per MN k-row
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int blk = wave * D + i;
            if constexpr (KM) {
                const int row = blk * 16 + lane / 4;
                const int c = (lane % 4) ^ swz_km<XS>(row);
                const int gr = row0 + row;
                off[i] = gr < rows ? (uint32_t)(((int64_t)gr * s_row + c * 8) * 2) : kOOB;
                tail[i] = c * 8 >= k_left && gr < rows ? kOOB : 0;
            } else {
                const int kr = blk * (64 / CPR) + lane / CPR;
                const int c = (lane % CPR) ^ swz_mn<XS>(kr);
                const int gc = row0 + c * 8;
                off[i] = gc < rows ? (uint32_t)(((int64_t)kr * s_k + gc) * 2) : kOOB;
                tail[i] = 0;
            }
        }
        kstep = KM ? (uint32_t)(D_BK * 2) : (uint32_t)(D_BK * s_k * 2);
    }
};

// One 16x16x32 operand fragment: lane l holds row (or column) l % 16 and
// k = (l / 16) * 8 .. + 7 of the stage.
template <bool KM, int W, bool XS>
__device__ inline u32x4 read_frag(uint32_t base, int row_base, int lane) {
    if constexpr (KM) {
        const int row = row_base + lane % 16;
        const int chunk = lane / 16;
        return *(const TVK_LDS u32x4*)(uintptr_t)(base + row * (2 * D_BK) + ((chunk ^ swz_km<XS>(row)) * 16));
    } else {
        // source lane s of group g points at k-row 8g + 4rr + s/4, columns 4(s%4)..+3;
        // the transpose hands lane s the four k values of column s
        const int g = lane / 16, s = lane % 16;
        const int col = row_base + (s % 4) * 4;
        const int chunk = col / 8, within = (col % 8) * 2;
        u32x4 out;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int kr = g * 8 + rr * 4 + s / 4;
            TVK_LDS s16x4* ptr = (TVK_LDS s16x4*)(uintptr_t)(base + kr * (2 * W) + ((chunk ^ swz_mn<XS>(kr)) * 16) + within);
            const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(ptr));
            out[rr * 2] = w.x;
            out[rr * 2 + 1] = w.y;
        }
        return out;
    }
}

template <int DT>
__device__ inline f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == TVK_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

constexpr int dma_threads(int bm, int bn) { return 64 * ((bm == 256 && bn == 256) ? 8 : (bm / 64) * (bn / 64)); }

// NS: stages in the ring (4, or 8 for 128x128 tiles whose loads need more
// lookahead to cover memory latency: short K, one workgroup per CU).
// BL: C-in staged through the ring (256x256 tiles with a bias; a variant of
// its own because the bias loads' offsets cost the k loop registers).
// KT: the last k step masks a k-contiguous operand's chunks past K (kmask).
template <int DT, bool AK, bool BK, int BM, int BN, int NS, bool BL = false, bool KT = false>
__global__ __launch_bounds__(dma_threads(BM, BN)) void gemm16_dma_kernel(GemmArgs p) {
    constexpr int D_NS = NS;
    typedef DCfg<BM, BN> G;
    constexpr int D_BM = BM, D_BN = BN, D_NT = G::NT, D_FM = G::FM, D_FN = G::FN, D_WTM = G::WTM, D_WTN = G::WTN;
    constexpr int D_OPB = G::OPA, D_STB = G::STB, D_DPS = G::DS;
    static_assert(dma_threads(BM, BN) == G::NT, "thread count");
    // BL: 32 KB past the ring for the epilogue's float32 staging
    __shared__ __attribute__((aligned(1024))) char lds_raw[D_NS * D_STB + (G::BIG && BL ? 32768 : 0)];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(TVK_LDS char*)lds_raw);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wm = wave / G::WN, wn = wave % G::WN;
    const int b = blockIdx.y;
    int tm, tn;
    tile_of(blockIdx.x, p.tiles_m * p.tiles_n, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * D_BM, n0 = tn * D_BN;

    // A: (m, k) at m*sa[1] + k*sa[2]; B: (k, n) at k*sb[1] + n*sb[2]
    const char* A = reinterpret_cast<const char*>(p.a) + a_boff(p, b) * 2;
    const char* B = reinterpret_cast<const char*>(p.b) + b_boff(p, b) * 2;
    const i32x4 ra = dma_rsrc(A, p.a_ext ? p.a_ext : 2 * ((int64_t)(p.M - 1) * p.sa[1] + (int64_t)(p.K - 1) * p.sa[2] + 1));
    const i32x4 rb = dma_rsrc(B, p.b_ext ? p.b_ext : 2 * ((int64_t)(p.N - 1) * p.sb[2] + (int64_t)(p.K - 1) * p.sb[1] + 1));
    constexpr bool XS = !G::BIG;   // the wide (conflict-free) swizzles
    DmaSrc<AK, G::DA, BM, XS> da;
    DmaSrc<BK, G::DB, BN, XS> db;
    const int k_left = p.K % D_BK;   // (KT only)
    da.init(p.sa[1], p.sa[2], m0, p.M, wave, lane, k_left);
    db.init(p.sb[2], p.sb[1], n0, p.N, wave, lane, k_left);
    const uint32_t k_last = (uint32_t)(p.K / D_BK);   // the stage that holds K's end
    // split-K (grid z): this workgroup's k range starts at stage kt0
    const int kt0 = p.split > 1 ? (int)blockIdx.z * (p.k_chunk / D_BK) : 0;
    // (a K off the 32 grid runs its last step whole: split chunks are whole
    // multiples of 64, and the loads past K return zeros, kzero)
    const int nk = ((p.split > 1 ? min(p.k_chunk, p.K - (int)blockIdx.z * p.k_chunk) : p.K) + D_BK - 1) / D_BK;
    // The ring issues the same loads every stage, also for the NS stages past
    // this workgroup's k range (the waits count on them). Those go through
    // resources of no records: out of range, so they return zeros without
    // reading memory (past the end of K, a k-contiguous operand's addresses
    // run into its next row, and a split's into the next split's range).
    const i32x4 ra_none = dma_rsrc(A, 0), rb_none = dma_rsrc(B, 0);
    // C-in through the ring (BL: 256x256 tiles; 16-byte bias and output rows,
    // N a multiple of 8): the loads of stages nk .. nk + 3 bring the bias
    // tile, 64 rows of 512 bytes a slot, instead of nothing, so it arrives
    // with the operands rather than after the k loop
    bool bias_lds = false;
    i32x4 rbias{0, 0, 0, 0};
    uint32_t bias_lane = 0;
    if constexpr (G::BIG && BL) {
        const char* Bias = reinterpret_cast<const char*>(p.bias) + bias_boff(p, b) * 2;
        auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
        bias_lds = p.split <= 1 && p.has_bias && p.sbias[2] == 1 && p.sbias[1] % 8 == 0 && al16(Bias) && p.sc[2] == 1 &&
                   p.sc[1] % 8 == 0 && al16(reinterpret_cast<const char*>(p.c) + c_boff(p, b) * 2) && p.N % 8 == 0 &&
                   2 * ((int64_t)(p.M + 256) * p.sbias[1] + p.N) < (int64_t(1) << 31);
        // an instruction's two rows start 2 u rows past its quarter's first: lane -> row lane / 32, chunk lane % 32
        rbias = dma_rsrc(Bias + ((int64_t)m0 * p.sbias[1] + n0) * 2, bias_lds ? 2 * ((int64_t)(p.M - 1 - m0) * p.sbias[1] + p.N - n0) : 0);
        bias_lane = (uint32_t)((lane / 32) * p.sbias[1] * 2 + (lane % 32) * 16);
    }
    auto dma_one = [&](int kt, int q) {   // q-th load (of D_DPS) of this wave for stage kt
        const uint32_t slot = lds0 + (uint32_t)((kt % D_NS) * D_STB);
        const uint32_t kg = (uint32_t)(kt0 + kt);
        const bool live = kt < nk;
        if constexpr (G::BIG && BL) {
            if (!live && bias_lds) {
                const int u = wave * D_DPS + q;
                dma16(rbias, slot + (uint32_t)(u * 1024), bias_lane + (uint32_t)(((kt - nk) * 64 + 2 * u) * p.sbias[1] * 2));
                return;
            }
        }
        const uint32_t end = KT && kg == k_last ? ~0u : 0u;
        if (q < G::DA) dma16(live ? ra : ra_none, slot + (uint32_t)((wave * G::DA + q) * 1024),
                             da.off[q] + kg * da.kstep + (KT && AK ? da.tail[q] & end : 0u));
        else dma16(live ? rb : rb_none, slot + D_OPB + (uint32_t)((wave * G::DB + q - G::DA) * 1024),
                   db.off[q - G::DA] + kg * db.kstep + (KT && BK ? db.tail[q - G::DA] & end : 0u));
    };

    f32x4 acc[D_FM][D_FN];
#pragma unroll
    for (int i = 0; i < D_FM; ++i)
#pragma unroll
        for (int j = 0; j < D_FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    u32x4 fa[2][D_FM], fb[2][D_FN];
    // prologue: stages 0..3 in flight; stage 0's fragments in registers once it
    // has landed, stage 1 landed before the loop reads it
#pragma unroll
    for (int s = 0; s < D_NS; ++s)
#pragma unroll
        for (int q = 0; q < D_DPS; ++q) dma_one(s, q);
    wait_vmcnt<D_DPS * (D_NS - 1)>();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < D_FM; ++i) fa[0][i] = read_frag<AK, BM, XS>(lds0, wm * D_WTM + i * 16, lane);
#pragma unroll
    for (int j = 0; j < D_FN; ++j) fb[0][j] = read_frag<BK, BN, XS>(lds0 + D_OPB, wn * D_WTN + j * 16, lane);
    wait_vmcnt<D_DPS * (D_NS - 2)>();
    __syncthreads();

    // Stage kt: MFMAs from register set `cur`; in between, one fragment read
    // of stage kt+1 (into set cur^1) after each even MFMA and one load of
    // stage kt+4 after each odd one, in this exact order (sched_barrier).
    auto body = [&](int kt, auto cur_c) {
        constexpr int cur = decltype(cur_c)::value;
        const uint32_t st_next = lds0 + (uint32_t)(((kt + 1) % D_NS) * D_STB);
#pragma unroll
        for (int q = 0; q < D_FM * D_FN; ++q) {
            const int i = q / D_FN, j = q % D_FN;
            acc[i][j] = mfma16<DT>(fa[cur][i], fb[cur][j], acc[i][j]);
            if (q % 2 == 0) {
                const int r = q / 2;
                if (r < D_FM) fa[cur ^ 1][r] = read_frag<AK, BM, XS>(st_next, wm * D_WTM + r * 16, lane);
                else if (r < D_FM + D_FN) fb[cur ^ 1][r - D_FM] = read_frag<BK, BN, XS>(st_next + D_OPB, wn * D_WTN + (r - D_FM) * 16, lane);
            } else if (q / 2 < D_DPS) {
                dma_one(kt + D_NS, q / 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // stage kt+2 landed for this wave; after the barrier, for all waves
        wait_vmcnt<D_DPS * (D_NS - 2)>();
        __syncthreads();
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        body(kt, std::integral_constant<int, 0>{});
        body(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) body(kt, std::integral_constant<int, 0>{});
    // the (empty) loads of stages past the end are still in flight: drain
    // them before the workgroup's LDS can be handed to another
    wait_vmcnt<0>();

    // The output tile goes through LDS 64 rows a pass (once the ring is free):
    // the waves holding a pass's rows write their float32 accumulators there
    // (layout of v_mfma_f32_16x16x32: lane l holds column l % 16, register r
    // row (l / 16) * 4 + r), E_LD floats a row, and the threads read it back
    // along the rows.
    constexpr int E_LD = D_BN + 4;
    float* const et = reinterpret_cast<float*>(lds_raw);
    auto stage_pass = [&](int pass) {
        if (wm == pass * 64 / D_WTM) {
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
                const int i = (pass * 64 % D_WTM) / 16 + ii;
#pragma unroll
                for (int j = 0; j < D_FN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        et[(ii * 16 + (lane / 16) * 4 + r) * E_LD + wn * D_WTN + j * 16 + lane % 16] = acc[i][j][r];
            }
        }
    };

    if (p.split > 1) {
        // float32 partials part[z][batch][M][np]
        float* part = p.part + ((int64_t)blockIdx.z * p.batch + b) * p.M * p.np;
        if (p.np % 4 == 0 && (reinterpret_cast<uintptr_t>(p.part) & 15) == 0) {
            // through the LDS tile: 16-byte row chunks a thread (a lane's
            // accumulators hold four rows of one column; stored directly they
            // are 4-byte stores, which took 2.1 us a workgroup at 128x128)
            constexpr int SPASS = D_BM / 64, SCH = 64 * (D_BN / 4) / D_NT;
            static_assert(SCH * D_NT == 64 * (D_BN / 4), "whole chunks per thread");
            __syncthreads();   // every wave is done with the ring
#pragma unroll
            for (int pass = 0; pass < SPASS; ++pass) {
                stage_pass(pass);
                __syncthreads();
#pragma unroll
                for (int j = 0; j < SCH; ++j) {
                    const int q = tid + j * D_NT;
                    const int rl = q / (D_BN / 4), cc = (q % (D_BN / 4)) * 4;
                    const int row = m0 + pass * 64 + rl, col = n0 + cc;
                    if (row < p.M && col < p.N)
                        *reinterpret_cast<f32x4*>(part + (int64_t)row * p.np + col) = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc);
                }
                __syncthreads();
            }
            return;
        }
        // straight from the accumulators
#pragma unroll
        for (int i = 0; i < D_FM; ++i)
#pragma unroll
            for (int j = 0; j < D_FN; ++j) {
                const int col = n0 + wn * D_WTN + j * 16 + lane % 16;
                if (col >= p.N) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = m0 + wm * D_WTM + i * 16 + (lane / 16) * 4 + r;
                    if (row < p.M) part[(int64_t)row * p.np + col] = acc[i][j][r];
                }
            }
        return;
    }

    __syncthreads();   // every wave is done with the ring: it now holds the output tile
    if constexpr (G::BIG && BL) {
        typedef typename elem<DT>::T T;
        if (bias_lds) {
            // 32 rows a pass: the waves holding them write their accumulators
            // into a float32 tile past the ring ([32][256], 16-byte chunk c of
            // row r at c ^ ((r >> 2) & 3) * 4: the four row groups of a write
            // meet on distinct banks); then each thread finishes 8 columns of a
            // row against its bias chunk from the ring and stores 16 bytes
            float* et = reinterpret_cast<float*>(lds_raw + D_NS * D_STB);
            T* Cb = reinterpret_cast<T*>(p.c) + c_boff(p, b);
            auto et_at = [](int r, int col) { return r * 256 + (((col / 4) ^ (((r >> 2) & 3) * 4)) * 4) + col % 4; };
#pragma unroll
            for (int pass = 0; pass < 8; ++pass) {
                if (wm == pass / 4) {
#pragma unroll
                    for (int ii = 0; ii < 2; ++ii) {
                        const int i = (pass % 4) * 2 + ii;
#pragma unroll
                        for (int j = 0; j < D_FN; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                et[et_at(ii * 16 + (lane / 16) * 4 + r, wn * D_WTN + j * 16 + lane % 16)] = acc[i][j][r];
                    }
                }
                __syncthreads();
#pragma unroll
                for (int jj = 0; jj < 32 * 32 / D_NT; ++jj) {
                    const int q = tid + jj * D_NT, rl = q / 32, cc = (q % 32) * 8;
                    const int rt = pass * 32 + rl, row = m0 + rt, col = n0 + cc;
                    if (row >= p.M || col >= p.N) continue;
                    const f32x4 lo = *reinterpret_cast<const f32x4*>(et + et_at(rl, cc));
                    const f32x4 hi = *reinterpret_cast<const f32x4*>(et + et_at(rl, cc + 4));
                    const u32x4 w = *reinterpret_cast<const u32x4*>(lds_raw + ((nk + rt / 64) % D_NS) * D_STB + (rt % 64) * 512 + cc * 2);
                    const float a8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                    const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
                    uint32_t o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float b0 = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] & 0xffffu)));
                        const float b1 = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] >> 16)));
                        const uint16_t h0 = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(epilogue(a8[2 * e], p.alpha, 1, b0, p.beta, p.act)));
                        const uint16_t h1 = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(epilogue(a8[2 * e + 1], p.alpha, 1, b1, p.beta, p.act)));
                        o[e] = (uint32_t)h0 | ((uint32_t)h1 << 16);
                    }
                    st_nt(reinterpret_cast<u32x4*>(Cb + (int64_t)row * p.sc[1] + col), u32x4{o[0], o[1], o[2], o[3]});
                }
                __syncthreads();
            }
            return;
        }
    }

    // Output through LDS, 64 rows at a time. The waves write their float32
    // accumulators (layout of v_mfma_f32_16x16x32: lane l holds column l % 16,
    // register r row (l / 16) * 4 + r); then each thread finishes 8 consecutive
    // columns of one row (alpha, bias, activation, one rounding) and stores
    // them with a single 16-byte store where the output rows allow it.
    typedef typename elem<DT>::T T;
    T* Cb = reinterpret_cast<T*>(p.c) + c_boff(p, b);
    const T* Bb = p.has_bias ? reinterpret_cast<const T*>(p.bias) + bias_boff(p, b) : nullptr;
    auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    // contiguous output rows: 16-byte stores, of any alignment
    const bool vec_c = p.sc[2] == 1;
    const bool vec_b = p.has_bias && p.sbias[2] == 1 && p.sbias[1] % 8 == 0 && al16(Bb);
    const bool plain = !p.has_bias && p.act == TVK_ACT_NONE;
    // thread tid finishes chunk q = tid + j * D_NT (j < 4) of each 64-row pass:
    // row q / 32, columns 8 * (q % 32); the bias chunks of all four passes are
    // requested up front so their latency overlaps
    constexpr int NPASS = D_BM / 64, CPT = 64 * (D_BN / 8) / D_NT;   // passes; chunks per thread per pass
    static_assert(CPT * D_NT == 64 * (D_BN / 8), "whole chunks per thread");
    static_assert(64 * (D_BN + 4) * 4 <= D_NS * D_STB, "epilogue tile fits the ring");
    if (plain && vec_c) {
        // No bias, no activation, contiguous output rows (most products): each
        // element is its sum times alpha, rounded once, as in the general loop
        // below, with no per-element branches and no bias registers live.
        // (The general loop spends about 500 instructions a chunk on its
        // variants, and its code is fetched cold by every workgroup.)
#pragma unroll
        for (int pass = 0; pass < NPASS; ++pass) {
            stage_pass(pass);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const int q = tid + j * D_NT;
                const int rl = q / (D_BN / 8), cc = (q % (D_BN / 8)) * 8;
                const int row = m0 + pass * 64 + rl, col = n0 + cc;
                if (row >= p.M || col >= p.N) continue;
                const f32x4 lo = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc);
                const f32x4 hi = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc + 4);
                const float a8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                uint16_t h[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
                    const float v = a8[e] * p.alpha;
                    h[e] = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(v));
                }
                T* cp = Cb + (int64_t)row * p.sc[1] + col;
                store_row8(reinterpret_cast<uint16_t*>(cp), u32x4{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16),
                                                                  (uint32_t)h[4] | ((uint32_t)h[5] << 16), (uint32_t)h[6] | ((uint32_t)h[7] << 16)},
                           p.N - col);
            }
            __syncthreads();
        }
        return;
    }
    u32x4 bpre[NPASS][CPT];
    if (vec_b) {
#pragma unroll
        for (int pass = 0; pass < NPASS; ++pass)
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const int q = tid + j * D_NT;
                const int row = m0 + pass * 64 + q / (D_BN / 8), col = n0 + (q % (D_BN / 8)) * 8;
                bpre[pass][j] = u32x4{0, 0, 0, 0};
                if (row < p.M && col + 8 <= p.N)
                    bpre[pass][j] = *reinterpret_cast<const u32x4*>(Bb + (int64_t)row * p.sbias[1] + col);
            }
    }
    if (vec_c && p.act != TVK_ACT_GELU && (!p.has_bias || vec_b)) {
        // contiguous output rows, no GELU, and a bias with 16-byte rows or ReLU:
        // the epilogue of the general loop below (sum times alpha, plus bias
        // times beta, ReLU, one rounding) with selects in place of its
        // per-element branches
        const bool hb = p.has_bias, relu = p.act == TVK_ACT_RELU;
#pragma unroll
        for (int pass = 0; pass < NPASS; ++pass) {
            stage_pass(pass);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const int q = tid + j * D_NT;
                const int rl = q / (D_BN / 8), cc = (q % (D_BN / 8)) * 8;
                const int row = m0 + pass * 64 + rl, col = n0 + cc;
                if (row >= p.M || col >= p.N) continue;
                const bool full = col + 8 <= p.N;
                const f32x4 lo = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc);
                const f32x4 hi = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc + 4);
                const float a8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                float bv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                if (hb) {
                    if (full) {
                        const u32x4 w = bpre[pass][j];
                        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            bv[2 * e] = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] & 0xffffu)));
                            bv[2 * e + 1] = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] >> 16)));
                        }
                    } else {
                        const T* bp = Bb + (int64_t)row * p.sbias[1] + col;
                        for (int e = 0; e < 8 && col + e < p.N; ++e) bv[e] = elem<DT>::to_f32(bp[e]);
                    }
                }
                uint16_t h[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
                    float v = a8[e] * p.alpha;
                    const float t = bv[e] * p.beta;
                    v = hb ? v + t : v;
                    const float r = v > 0.0f ? v : (v != v ? v : 0.0f);
                    v = relu ? r : v;
                    h[e] = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(v));
                }
                T* cp = Cb + (int64_t)row * p.sc[1] + col;
                store_row8(reinterpret_cast<uint16_t*>(cp), u32x4{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16),
                                                                  (uint32_t)h[4] | ((uint32_t)h[5] << 16), (uint32_t)h[6] | ((uint32_t)h[7] << 16)},
                           p.N - col);
            }
            __syncthreads();
        }
        return;
    }
#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) {
        stage_pass(pass);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int q = tid + j * D_NT;
            const int rl = q / (D_BN / 8), cc = (q % (D_BN / 8)) * 8;
            const int row = m0 + pass * 64 + rl, col = n0 + cc;
            if (row >= p.M || col >= p.N) continue;
            const f32x4 lo = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(et + rl * E_LD + cc + 4);
            const float a8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const bool full = col + 8 <= p.N;
            float bv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            if (p.has_bias) {
                if (vec_b && full) {
                    const u32x4 w = bpre[pass][j];
                    const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        bv[2 * e] = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] & 0xffffu)));
                        bv[2 * e + 1] = elem<DT>::to_f32(__builtin_bit_cast(T, (uint16_t)(ww[e] >> 16)));
                    }
                } else {
                    const T* bp = Bb + (int64_t)row * p.sbias[1] + (int64_t)col * p.sbias[2];
                    for (int e = 0; e < 8 && col + e < p.N; ++e) bv[e] = elem<DT>::to_f32(bp[(int64_t)e * p.sbias[2]]);
                }
            }
            uint16_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v;
                if (plain) {
#pragma clang fp contract(off)
                    v = a8[e] * p.alpha;
                } else {
                    v = epilogue(a8[e], p.alpha, p.has_bias, bv[e], p.beta, p.act);
                }
                h[e] = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(v));
            }
            T* cp = Cb + (int64_t)row * p.sc[1] + (int64_t)col * p.sc[2];
            if (vec_c) {
                store_row8(reinterpret_cast<uint16_t*>(cp), u32x4{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16),
                                                                  (uint32_t)h[4] | ((uint32_t)h[5] << 16), (uint32_t)h[6] | ((uint32_t)h[7] << 16)},
                           p.N - col);
            } else {
                for (int e = 0; e < 8 && col + e < p.N; ++e) cp[(int64_t)e * p.sc[2]] = __builtin_bit_cast(T, h[e]);
            }
        }
        __syncthreads();
    }
}

}  // namespace

// Launches the kernel on BM x BN tiles for the operand layout (any split).
template <int DT, int BM, int BN, int NS>
void launch_dma_tile(GemmArgs& p, bool a_kmajor, bool b_kmajor, hipStream_t s) {
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    const dim3 grid(p.tiles_m * p.tiles_n, p.batch, p.split > 1 ? p.split : 1), block(DCfg<BM, BN>::NT);
    if constexpr (DCfg<BM, BN>::BIG) {
        if (p.has_bias && p.split <= 1 && !p.kmask) {
            if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, true, BM, BN, NS, true>), grid, block, 0, s, p);
            else if (a_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, false, BM, BN, NS, true>), grid, block, 0, s, p);
            else if (b_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, false, true, BM, BN, NS, true>), grid, block, 0, s, p);
            else hipLaunchKernelGGL((gemm16_dma_kernel<DT, false, false, BM, BN, NS, true>), grid, block, 0, s, p);
            return;
        }
    }
    if constexpr (NS == 4 && !(BM == 256 && BN == 128)) if (p.kmask) {
        if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, true, BM, BN, NS, false, true>), grid, block, 0, s, p);
        else if (a_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, false, BM, BN, NS, false, true>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((gemm16_dma_kernel<DT, false, true, BM, BN, NS, false, true>), grid, block, 0, s, p);
        return;
    }
    if (a_kmajor && b_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, true, BM, BN, NS>), grid, block, 0, s, p);
    else if (a_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, true, false, BM, BN, NS>), grid, block, 0, s, p);
    else if (b_kmajor) hipLaunchKernelGGL((gemm16_dma_kernel<DT, false, true, BM, BN, NS>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((gemm16_dma_kernel<DT, false, false, BM, BN, NS>), grid, block, 0, s, p);
}

// The 128x128 instantiations live in gemm_dma128.hip, compiled with the MFMA
// results in VGPRs (in the AGPR form hipcc rotates their accumulators through
// AGPR copies inside the k loop); the 256x256 ones keep the default form,
// in which they allocate cleanly while the VGPR form spills.
void launch_dma128(int dtype, GemmArgs& p, bool a_kmajor, bool b_kmajor, hipStream_t s, int stages);
// 128x256 (wide) and 256x128 tiles, 8 waves of 64x64 (gemm_dma128.hip, the same form)
void launch_dma_rect(int dtype, GemmArgs& p, bool a_kmajor, bool b_kmajor, hipStream_t s, bool wide);

}  // namespace tvk
