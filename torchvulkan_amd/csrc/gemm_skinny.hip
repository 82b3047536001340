// M <= 16 GEMM as an HBM stream over B (the decode-like shapes of the path:
// C5 "skinny" [16,4096]x[4096,14336] and small-batch linears).
//
// With M <= 16 the product is bound by reading B once: 2*K*N bytes against
// 2*M*K*N flops. A workgroup owns CW (64) columns, one 128-byte line of each
// row of B, and all of K; its eight waves take 64-row blocks of K in turn and
// reduce their partial sums in LDS at the end, so no
// workgroup ever waits for another (a cross-XCD handoff would need an L2
// write-back per workgroup). Per 32 k a wave issues v_mfma_f32_16x16x32 per 16
// columns against the 16 rows of A. B stored k-contiguous ([N][K], a transposed
// weight view) is loaded straight into MFMA operands; B stored n-contiguous
// ([K][N]) is written to a wave-private LDS tile as it arrives and read back
// along k. It runs the layouts without 16-byte rows, n-contiguous B where the
// ring below does not apply, and k-contiguous B where its ring does not pay
// (kring_pays).
//
// B n-contiguous with 16-byte aligned rows ([K][N], the C5 layout) takes a
// second kernel, gemm16_skinny_ring: workgroups of 8 waves own 128 columns
// (256 bytes of each row of B) and a K range; B and A arrive by buffer loads
// straight into a 4-stage LDS ring (no register staging), each wave reads its
// 16 columns back along k with ds_read_b64_tr_b16 and issues one
// v_mfma_f32_16x16x32 per 32 k. The K range is split between workgroups
// until about one workgroup per CU runs; float32 partials are then summed in
// split order by a second kernel that applies the epilogue.
//
// Epilogue semantics are the reference's (src/shaders/helpers/gemm_simd.slang:67-99).
#include "gemm_common.h"

#include <algorithm>

namespace tvk {
namespace {

constexpr int SK_NW = 8;      // waves per workgroup (K split over them)
constexpr int SK_CW = 64;     // columns per workgroup: 128-byte rows of B
constexpr int SK_NG = SK_CW / 16;
constexpr int SK_KSTEP = 32;  // k per MFMA
constexpr int SK_U = 2;       // k steps per wave iteration
constexpr int SK_KI = SK_U * SK_KSTEP;
constexpr int SK_LDW = SK_CW + 8;  // LDS row (halfs) of the [k][col] transpose tile

template <int DT>
__device__ inline f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == TVK_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int DT, bool BKM, bool VEC>
__global__ __launch_bounds__(64 * SK_NW) void gemm_skinny_kernel(GemmArgs p) {
    constexpr int TILE_H = SK_KI * SK_LDW;              // halfs per wave
    constexpr int RED_F = SK_NW * 16 * (SK_CW + 4);     // floats
    constexpr int TILE_BYTES = BKM ? 0 : SK_NW * TILE_H * 2;
    constexpr int BYTES = TILE_BYTES > RED_F * 4 ? TILE_BYTES : RED_F * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[BYTES];

    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    // strips are dealt to the 8 XCDs round robin by block id: give each XCD a
    // contiguous run of strips (neighbouring strips share DRAM rows of B)
    int strip = blockIdx.x;
    if (gridDim.x % 8 == 0) strip = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    const int n0 = strip * SK_CW, b = blockIdx.z;

    const uint16_t* A = reinterpret_cast<const uint16_t*>(p.a) + a_boff(p, b);
    const uint16_t* B = reinterpret_cast<const uint16_t*>(p.b) + b_boff(p, b);
    const int64_t a_bytes = 2 * ((int64_t)(p.M - 1) * p.sa[1] + (int64_t)(p.K - 1) * p.sa[2] + 1);
    const int64_t b_bytes = 2 * ((int64_t)(p.N - 1) * p.sb[2] + (int64_t)(p.K - 1) * p.sb[1] + 1);
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)min(a_bytes, (int64_t)0x7fffffff), 0x00020000);
    __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)min(b_bytes, (int64_t)0x7fffffff), 0x00020000);

    const int j = lane % 16, g = lane / 16;
    // n-contiguous B: lane loads 8 columns (chunk lane%8) of rows lane/8 + 8q
    const int tc = (lane % 8) * 8, tr = lane / 8;
    uint16_t* tile = reinterpret_cast<uint16_t*>(smem) + wave * TILE_H;

    f32x4 acc[SK_NG];
#pragma unroll
    for (int e = 0; e < SK_NG; ++e) acc[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // The waves of the workgroup take 64-row blocks of B in turn (block
    // wave, wave+8, ...), so at any time they sweep neighbouring rows
    // together. The loads of a wave's next block are in flight while the
    // current one is transposed and multiplied (two register sets).
    u32x4 av[2][SK_U], bv[2][SK_U][SK_NG];
    auto issue = [&](int set, int k0) {
#pragma unroll
        for (int u = 0; u < SK_U; ++u) {
            const int kk = k0 + u * SK_KSTEP + g * 8;
            av[set][u] = load_chunk<VEC>(ra, j < p.M, (int64_t)j * p.sa[1] + (int64_t)kk * p.sa[2], p.sa[2], p.K - kk);
            if constexpr (BKM) {
#pragma unroll
                for (int e = 0; e < SK_NG; ++e) {
                    const int n = n0 + 16 * e + j;
                    bv[set][u][e] = load_chunk<VEC>(rb, n < p.N, (int64_t)n * p.sb[2] + (int64_t)kk * p.sb[1], p.sb[1], p.K - kk);
                }
            } else {
                const int n = n0 + tc;
#pragma unroll
                for (int q = 0; q < SK_NG; ++q) {
                    const int kr = k0 + u * SK_KSTEP + tr + 8 * q;
                    bv[set][u][q] = load_chunk<VEC>(rb, kr < p.K, (int64_t)kr * p.sb[1] + (int64_t)n * p.sb[2], p.sb[2], p.N - n);
                }
            }
        }
    };
    auto consume = [&](int set) {
        if constexpr (!BKM) {
            // rows arrive n-contiguous: park them in the wave's [k][col] tile,
            // then gather 8 k of one column per lane
#pragma unroll
            for (int u = 0; u < SK_U; ++u)
#pragma unroll
                for (int q = 0; q < SK_NG; ++q)
                    *reinterpret_cast<u32x4*>(tile + (u * SK_KSTEP + tr + 8 * q) * SK_LDW + tc) = bv[set][u][q];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < SK_U; ++u)
#pragma unroll
                for (int e = 0; e < SK_NG; ++e) {
                    const uint16_t* src = tile + (u * SK_KSTEP + g * 8) * SK_LDW + 16 * e + j;
                    uint32_t h[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) h[i] = src[i * SK_LDW];
                    bv[set][u][e] = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
                }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int u = 0; u < SK_U; ++u)
#pragma unroll
            for (int e = 0; e < SK_NG; ++e) acc[e] = mfma16<DT>(av[set][u], bv[set][u][e], acc[e]);
    };
    const int kstride = SK_NW * SK_KI;
    int k0 = wave * SK_KI;
    if (k0 < p.K) issue(0, k0);
    while (k0 < p.K) {
        if (k0 + kstride < p.K) issue(1, k0 + kstride);
        consume(0);
        k0 += kstride;
        if (k0 >= p.K) break;
        if (k0 + kstride < p.K) issue(0, k0 + kstride);
        consume(1);
        k0 += kstride;
    }

    // reduce the waves' partial sums (16x16 accumulator layout: lane holds
    // column lane%16, rows (lane/16)*4 + r)
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int e = 0; e < SK_NG; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * 16 + g * 4 + r) * (SK_CW + 4) + 16 * e + j] = acc[e][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < (16 * SK_CW) / (64 * SK_NW); ++q) {
        const int idx = tid + 64 * SK_NW * q;
        const int m = idx / SK_CW, cl = idx % SK_CW;
        float v = red[m * (SK_CW + 4) + cl];
#pragma unroll
        for (int w = 1; w < SK_NW; ++w) v += red[(w * 16 + m) * (SK_CW + 4) + cl];
        const int n = n0 + cl;
        if (m < p.M && n < p.N) store_out<DT, true>(p, b, m, n, v);
    }
}


// ---------------------------------------------------------------------------
// gemm16_skinny_ring
// ---------------------------------------------------------------------------

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define TVK_LDS __attribute__((address_space(3)))

constexpr int SR_NB = 128;                 // columns per workgroup
constexpr int SR_NW = 8;                   // waves, 16 columns each
constexpr int SR_NS = 4;                   // ring stages of 32 k
constexpr int SR_ROW = SR_NB * 2;          // bytes of one k-row of the B tile
constexpr int SR_BST = 32 * SR_ROW;        // B bytes per stage: 8 loads of 1 KB, one per wave
constexpr int SR_STB = SR_BST + 1024;      // + A: 16 rows x 32 k, one load (wave 0)

__device__ inline i32x4 sr_rsrc(const void* ptr, int64_t bytes) {
    const uint64_t a = (uint64_t)ptr;
    return i32x4{(int)(uint32_t)a, (int)((a >> 32) & 0xffff), (int)min(bytes, (int64_t)0x7fffffff), 0x00020000};
}

// 16 bytes per lane into LDS at lds_addr + 16 * lane (lds_addr wave-uniform,
// carried in M0). Issued from asm so the compiler does not order every later
// LDS read behind it; the waits are explicit.
__device__ inline void sr_dma16(i32x4 r, uint32_t lds_addr, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(lds_addr), "v"(voff), "s"(r) : "memory");
}
template <int N>
__device__ inline void sr_wait() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

__device__ inline int sr_swz(int kr) { return (kr & 3) * 2; }

// grid (strips, splits, batch); requires A k-contiguous, B n-contiguous, rows
// of both 16-byte aligned, N % 8 == 0 and k_chunk % 32 == 0.
template <int DT>
__global__ __launch_bounds__(64 * SR_NW) void gemm_skinny_ring_kernel(GemmArgs p) {
    __shared__ __attribute__((aligned(1024))) char lds_raw[SR_NS * SR_STB];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(TVK_LDS char*)lds_raw);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int n0 = blockIdx.x * SR_NB, z = blockIdx.y, b = blockIdx.z;
    const int kb = p.split > 1 ? z * p.k_chunk : 0;
    const int klen = p.split > 1 ? p.k_chunk : p.K;
    const int nk = klen / 32;

    const char* A = reinterpret_cast<const char*>(p.a) + a_boff(p, b) * 2;
    const char* B = reinterpret_cast<const char*>(p.b) + b_boff(p, b) * 2;
    const i32x4 ra = sr_rsrc(A, 2 * ((int64_t)(p.M - 1) * p.sa[1] + p.K));
    const i32x4 rb = sr_rsrc(B, 2 * ((int64_t)(p.K - 1) * p.sb[1] + p.N));
    // wave w loads B block w (k-rows 4w..4w+3 of the stage); wave 0 also loads A
    const int kr = wave * 4 + lane / 16;
    const int bc = (lane % 16) ^ sr_swz(kr);
    const int gc = n0 + bc * 8;
    const uint32_t b_off = gc < p.N ? (uint32_t)(((int64_t)(kb + kr) * p.sb[1] + gc) * 2) : kOOB;
    const uint32_t b_step = (uint32_t)(32 * p.sb[1] * 2);
    const int ar = lane / 4;
    const uint32_t a_off = ar < p.M ? (uint32_t)(((int64_t)ar * p.sa[1] + kb + (lane % 4) * 8) * 2) : kOOB;
    auto issue = [&](int s) {
        if (s >= nk) return;
        const uint32_t slot = lds0 + (uint32_t)((s % SR_NS) * SR_STB);
        sr_dma16(rb, slot + (uint32_t)(wave * 1024), b_off + (uint32_t)s * b_step);
        if (wave == 0) sr_dma16(ra, slot + SR_BST, a_off + (uint32_t)s * 64);
    };

    f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < SR_NS - 1; ++s) issue(s);
    // this wave's B fragment: 16 columns, lane s of group g gets k 8g..8g+7 of column s
    const int g = lane / 16, sl = lane % 16;
    const int col = wave * 16 + (sl % 4) * 4;
    const int chunk = col / 8, within = (col % 8) * 2;
    for (int kt = 0; kt < nk; ++kt) {
        // stage kt landed; the two stages issued after it may be in flight
        if (nk - 1 - kt >= SR_NS - 2) {
            if (wave == 0) sr_wait<2 * (SR_NS - 2)>();
            else sr_wait<SR_NS - 2>();
        } else {
            sr_wait<0>();
        }
        __syncthreads();
        issue(kt + SR_NS - 1);
        const uint32_t st = lds0 + (uint32_t)((kt % SR_NS) * SR_STB);
        const u32x4 af = *(const TVK_LDS u32x4*)(uintptr_t)(st + SR_BST + (lane % 16) * 64 + (lane / 16) * 16);
        u32x4 bf;
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int r = g * 8 + rr * 4 + sl / 4;
            TVK_LDS s16x4* ptr = (TVK_LDS s16x4*)(uintptr_t)(st + r * SR_ROW + ((chunk ^ sr_swz(r)) * 16) + within);
            const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(ptr));
            bf[rr * 2] = w.x;
            bf[rr * 2 + 1] = w.y;
        }
        acc = mfma16<DT>(af, bf, acc);
    }
    sr_wait<0>();

    // lane l holds column l % 16 of the wave's 16, rows (l / 16) * 4 + r
    const int n = n0 + wave * 16 + lane % 16;
    if (n < p.N) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = (lane / 16) * 4 + r;
            if (m >= p.M) continue;
            const int64_t pi = (((int64_t)z * p.batch + b) * p.M + m) * p.N + n;
            if (p.split > 1 && p.tile_count) part_store(part_rsrc(p), pi, acc[r]);   // written through (split_fixup)
            else if (p.split > 1) p.part[pi] = acc[r];
            else store_out<DT, true>(p, b, m, n, acc[r]);
        }
    }
    // every wave has drained its loads into the ring: its first word serves
    // as the fixup's flag (the fixup's first barrier orders that)
    if (p.split > 1 && p.tile_count)
        split_fixup<DT, 64 * SR_NW, 16, SR_NB>(p, b, 0, n0, p.tile_count + (int64_t)b * gridDim.x + blockIdx.x,
                                               reinterpret_cast<int*>(lds_raw));
}

// Splits of K for the ring kernel: powers of two while the grid stays within
// about one workgroup per CU and every split keeps at least 4 stages.
int ring_splits(const GemmArgs& p) {
    const int64_t wgs = (int64_t)((p.N + SR_NB - 1) / SR_NB) * p.batch;
    int split = 1;
    while (wgs * split * 2 <= 256 && p.K % (64 * split) == 0 && p.K / (2 * split) >= 128) split *= 2;
    return split;
}

// ---------------------------------------------------------------------------
// The ring for B k-contiguous (nn.Linear's weight [N][K]) with 16-byte rows, M <= 64
// ---------------------------------------------------------------------------
// Bound by reading B once, as the ring above; what the split has to get right
// is how B's rows meet the memory channels.
//   - A workgroup of 8 waves owns 64 columns: four 16-column groups x two k
//     halves of a 256-k stage, so a stage reads 512 bytes of each of 64 rows
//     (the direct-to-register kernel read 64-byte pieces: 3.9 TB/s on bfloat16
//     16 x 4096 x 14336, 30.6 us). B and A arrive by buffer loads straight into
//     a ring of 2-4 stages; each wave reads only its own 4 KB of a B stage, A
//     is shared. The halves' sums meet in LDS at the end. 128 columns and one
//     k half (256 bytes a row, and twice as many K chunks for the same
//     workgroups) took 27.4 us where this takes 22.8 (5.2 TB/s).
//   - With rows a multiple of 4 KB apart the same stage of every row lies on
//     the same channels, of memory and of an XCD's L2: workgroups start their
//     k loop at different stages, counted so that the workgroups of one XCD
//     (every eighth) take all of them (26.8 -> 22.8 us there; 8192 x 8192
//     44 us with the workgroups of an XCD on two stages, 35.6 unrotated, 26.7
//     so). A fixed order for a shape: the same bits every run.
//   - K is split between workgroups up to about one per CU in chunks of at
//     least four stages (the exchange costs about 1.5 us: 7 x 1000 -> 500 takes
//     5.2 us whole, 6.2 in two), summed by the last workgroup of a strip
//     (split_fixup) or a second launch; without memory for partials a
//     workgroup takes a strip's chunks in turn (SERIAL).
//   - MF 16-row blocks of A: up to 64 rows (4096 -> 14336: 24.3 us for 32 rows,
//     31.7 for 64; the split 128 x 128 ring took 33.1 and 36.8). Above 32 rows A
//     weighs as much as B in the ring, and from K = 8192 the 128 x 128 tiles
//     are as fast (64 x 14336 x 4096: 32.7 us there, 34.2 here).
constexpr int SKR_K = 128;                   // k per wave and stage: 256 bytes of each row
constexpr int SKR_KG = 2;                    // k groups of a workgroup
constexpr int SKR_NB = 16 * SR_NW / SKR_KG;  // columns of a workgroup
constexpr int SKR_KST = SKR_K * SKR_KG;      // k per stage
constexpr int SKR_B = SR_NW * 16 * SKR_K * 2;   // B bytes per stage: 32 KB, 4 KB per wave

// LDS bytes of a stage (MF 16-row blocks of A) and ring depth in 160 KB
constexpr int kring_stage(int mf) { return SKR_B + mf * SKR_KG * 4096; }
constexpr int kring_depth(int mf) { return std::min(4, 160 * 1024 / kring_stage(mf)); }

// SERIAL: one workgroup takes a strip's K chunks one after another, for calls
// without memory for partials. It adds the chunks' sums in chunk order, the
// additions of split_fixup, so a call gives the same bits either way. The k
// halves meet in a ring slot: an array of their own cost the ring a stage (four
// captured 1 x 512 x 8192 22.5 us so, 21.2 now; 16.0 split over workgroups,
// 32.5 on the register kernel).
template <int DT, int MF, bool SERIAL>
__global__ __launch_bounds__(64 * SR_NW) void gemm_skinny_kring_kernel(GemmArgs p) {
    constexpr int CG = SR_NW / SKR_KG;   // 16-column groups
    constexpr int NS = kring_depth(MF), STB = kring_stage(MF);
    constexpr int AL = 4 * MF * SKR_KG / SR_NW;   // A loads per wave
    static_assert(AL * SR_NW == 4 * MF * SKR_KG, "whole loads");
    __shared__ __attribute__((aligned(1024))) char lds_raw[NS * STB];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(TVK_LDS char*)lds_raw);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int cg = wave % CG, kg = wave / CG;
    const int n0 = blockIdx.x * SKR_NB, z = blockIdx.y, b = blockIdx.z;
    const bool split = !SERIAL && p.split > 1;
    const int kb = split ? z * p.k_chunk : 0;
    const int kend = split ? min(p.K, kb + p.k_chunk) : p.K;
    const int nk = (kend - kb + SKR_KST - 1) / SKR_KST;
    __builtin_assume(nk > 0);   // (without it the loop is laid out behind the epilogue, and fetched cold)
    const int per = SERIAL ? p.k_chunk / SKR_KST : nk;   // stages of a chunk
    // the stage that the s-th load brings: a chunk's stages from its workgroup's first one round (found once where
    // there is one chunk: per load its remainder added 0.4 us to 7 x 512 x 512)
    auto first_of = [&](int n) { return p.sb[2] % 2048 == 0 ? (int)((blockIdx.x + blockIdx.x / 8) % (unsigned)n) : 0; };
    const int rot = SERIAL ? 0 : first_of(nk);
    auto stage_at = [&](int s) {
        const int c0 = SERIAL ? s / per * per : 0, n = SERIAL ? min(per, nk - c0) : nk;
        const int i = s - c0 + (SERIAL ? first_of(n) : rot);
        return c0 + (i >= n ? i - n : i);
    };

    const char* A = reinterpret_cast<const char*>(p.a) + a_boff(p, b) * 2;
    const char* B = reinterpret_cast<const char*>(p.b) + b_boff(p, b) * 2;
    const i32x4 ra = sr_rsrc(A, 2 * ((int64_t)(p.M - 1) * p.sa[1] + p.K));
    const i32x4 rb = sr_rsrc(B, 2 * ((int64_t)(p.N - 1) * p.sb[2] + p.K));
    // a load brings 4 rows of 256 bytes; LDS slot c of row r holds 16-byte chunk c ^ (r % 16)
    uint32_t b_off[4], a_off[AL];
    int b_k[4], a_k[AL];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = 4 * q + lane / 16, n = n0 + cg * 16 + row;
        b_k[q] = kg * SKR_K + ((lane % 16) ^ row) * 8;
        b_off[q] = n < p.N ? (uint32_t)(((int64_t)n * p.sb[2] + kb + b_k[q]) * 2) : kOOB;
    }
#pragma unroll
    for (int q = 0; q < AL; ++q) {
        const int blk = wave * AL + q, row = (blk % (4 * MF)) * 4 + lane / 16;
        a_k[q] = blk / (4 * MF) * SKR_K + ((lane % 16) ^ (row % 16)) * 8;
        a_off[q] = row < p.M ? (uint32_t)(((int64_t)row * p.sa[1] + kb + a_k[q]) * 2) : kOOB;
    }
    auto issue = [&](int s) {
        if (s >= nk) return;
        const uint32_t slot = lds0 + (uint32_t)((s % NS) * STB);
        const int ks = stage_at(s);
        const int left = p.K - kb - ks * SKR_KST;   // chunks at or past it would read the next row: zeros instead
        const uint32_t step = (uint32_t)(ks * SKR_KST * 2);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            sr_dma16(rb, slot + (uint32_t)(wave * 4096 + q * 1024), b_k[q] < left ? b_off[q] + step : kOOB);
#pragma unroll
        for (int q = 0; q < AL; ++q)
            sr_dma16(ra, slot + SKR_B + (uint32_t)((wave * AL + q) * 1024), a_k[q] < left ? a_off[q] + step : kOOB);
    };

    f32x4 acc[MF], total[MF];   // (total: SERIAL only)
#pragma unroll
    for (int m = 0; m < MF; ++m) acc[m] = total[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // the second k half's sums onto the first's, through a ring slot that every wave has left
    auto add_halves = [&](int slot) {
        f32x4* red = reinterpret_cast<f32x4*>(lds_raw + slot * STB);
        if (kg > 0) {
#pragma unroll
            for (int m = 0; m < MF; ++m) red[(cg * MF + m) * 64 + lane] = acc[m];
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int m = 0; m < MF; ++m) acc[m] += red[(cg * MF + m) * 64 + lane];
        }
    };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(s);
    const int g = lane / 16, c16 = lane % 16;
    for (int kt = 0; kt < nk; ++kt) {
        // stage kt landed; the stages issued after it may be in flight
        if (nk - 1 - kt >= NS - 2) sr_wait<(4 + AL) * (NS - 2)>();
        else sr_wait<0>();
        __syncthreads();
        issue(kt + NS - 1);
        const uint32_t st = lds0 + (uint32_t)((kt % NS) * STB);
#pragma unroll
        for (int ks = 0; ks < SKR_K / 32; ++ks) {
            const uint32_t at = (uint32_t)(c16 * 256 + (((ks * 4 + g) ^ c16) * 16));
            const u32x4 bf = *(const TVK_LDS u32x4*)(uintptr_t)(st + wave * 4096 + at);
#pragma unroll
            for (int m = 0; m < MF; ++m) {
                const u32x4 af = *(const TVK_LDS u32x4*)(uintptr_t)(st + SKR_B + (kg * MF + m) * 4096 + at);
                acc[m] = mfma16<DT>(af, bf, acc[m]);
            }
        }
        if (SERIAL && ((kt + 1) % per == 0 || kt == nk - 1)) {
            __syncthreads();
            add_halves(kt % NS);   // stage kt's slot, loaded again after the next stage's barrier
#pragma unroll
            for (int m = 0; m < MF; ++m) {
                total[m] = kt < per ? acc[m] : total[m] + acc[m];
                acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    }
    sr_wait<0>();
    __syncthreads();
    if constexpr (SERIAL) {
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[m] = total[m];
    } else {
        add_halves(0);
    }

    // lane l holds column l % 16 of the wave's 16, rows 16 m + (l / 16) * 4 + r
    const int n = n0 + cg * 16 + c16;
    if (kg == 0 && n < p.N) {
#pragma unroll
        for (int m = 0; m < MF; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m * 16 + g * 4 + r;
                if (row >= p.M) continue;
                const int64_t pi = (((int64_t)z * p.batch + b) * p.M + row) * p.np + n;
                if (split && p.tile_count) part_store(part_rsrc(p), pi, acc[m][r]);
                else if (split) p.part[pi] = acc[m][r];
                else store_out<DT, true>(p, b, row, n, acc[m][r]);
            }
    }
    if (split && p.tile_count)
        split_fixup<DT, 64 * SR_NW, 16 * MF, SKR_NB>(p, b, 0, n0, p.tile_count + (int64_t)b * gridDim.x + blockIdx.x,
                                                   reinterpret_cast<int*>(lds_raw));
}

// The range where the ring leads the kernels that take these products without
// it (up to 16 rows gemm_skinny_kernel, above it the 64x64 tiles and from
// K = 2048 the split 128x128 tiles). It runs one workgroup a CU, whose stages
// are 256 k, so it wants about one round of workgroups and a whole stage:
//   - M <= 16, K >= 256 (8 rows, 32 x 2048 x 64: 1.15x the other kernel's
//     time, K = 128 1.07x, 256 0.92x), and up to 384 workgroups (1024 for one
//     row: batch 64 of 1 x 512 x 512 0.79x, of 4 1.06x) or K >= 1536 (4 x 128256
//     x 256 1.22x, x 1024 1.03x, x 1536 0.87x).
//   - above, K >= 4 M, from 33 rows 8 M: a stage does the products of whole
//     16-row blocks, 4 of them from there (64 x 4096 x 256 1.12x, x 512 0.99x; 32
//     x 4096 x 64 1.02x, x 128 0.94x).
//   - at most one round of workgroups (64 x 20000 x 1024, 313 of them, 1.43x;
//     batch 64 of 64 x 512 x 1000 1.29x; 33 x 16384 x 1024, 256 of them, 0.70x),
//     two over one weight with K off the 32 grid, which the tiles stage through
//     registers (33 x 32000 x 1000 0.90x; from K = 2048 they split, x 5000 1.2x),
//     and any number over one long wide weight up to 32 rows, where the tiles
//     starve too (32 x 32000 x 5000 0.66x).
//   - batches split K less well than the tiles, which do from K = 2048: above 32
//     rows half a round there (batch 16 of 64 x 512 x 2048 1.03x, 256 of 64 x 64 x
//     2048 1.15x; of 17 x 1000 0.76x) and a quarter from K = 4096, up to 32 rows a
//     quarter from 8192 (batch 16 of 32 x 512 x 8192, 128 workgroups, 1.17x; 4 of
//     17 x 4096 x 4096, 256, 0.85x).
bool kring_pays(const GemmArgs& p) {
    const int64_t wgs = (int64_t)((p.N + SKR_NB - 1) / SKR_NB) * p.batch;
    if (p.M <= 16) return p.K >= 256 && (wgs <= (p.M == 1 ? 1024 : 384) || p.K >= 1536);
    if (p.M > (p.K < 8192 ? 64 : 32) || p.K < (p.M <= 32 ? 4 : 8) * p.M) return false;
    if (p.batch > 1 && p.M <= 32) return wgs <= (p.K >= 8192 ? 64 : 256);
    if (p.batch > 1) return wgs <= (p.K >= 4096 ? 64 : p.K >= 2048 ? 128 : 256);
    if (p.M <= 32 && p.K >= 4096) return true;
    return wgs <= (p.K % 32 != 0 && p.K >= 768 && p.K < 2048 ? 512 : 256);
}

bool kring_applies(const GemmArgs& p, bool b_kmajor, bool vec) {
    if (!kring_pays(p)) return false;
    auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    if (!b_kmajor || !vec || !al16(p.a) || !al16(p.b) || p.sa[2] != 1 || p.sb[1] != 1) return false;
    if (p.K % 8 != 0 || (p.M > 1 && p.sa[1] % 8 != 0) || (p.N > 1 && p.sb[2] % 8 != 0)) return false;
    if (p.batch > 1 && (p.sa[0] % 8 != 0 || p.sb[0] % 8 != 0)) return false;
    if (p.bh > 1 && (p.sa_h % 8 != 0 || p.sb_h % 8 != 0)) return false;
    return true;
}

// Strips of columns, K chunks (whole stages) and their length.
struct KringShape {
    int strips, split, chunk;
};

KringShape kring_shape(const GemmArgs& p) {
    KringShape r;
    r.strips = (p.N + SKR_NB - 1) / SKR_NB;
    const int stages = (p.K + SKR_KST - 1) / SKR_KST;
    const int64_t want = std::min<int64_t>(256 / ((int64_t)r.strips * p.batch), stages / 4);
    const int per = want > 1 ? (int)((stages + want - 1) / want) : stages;
    r.chunk = per * SKR_KST;
    r.split = (stages + per - 1) / per;
    return r;
}

// Bytes of the partials of `split` chunks: rows of N rounded up to 4, which the
// fixup and the second launch read 16 bytes at a time.
int kring_pitch(const GemmArgs& p) { return (p.N + 3) / 4 * 4; }
size_t kring_part_bytes(const GemmArgs& p, int split) {
    return split > 1 ? (size_t)split * p.batch * p.M * kring_pitch(p) * 4 : 0;
}

template <int DT, bool SERIAL>
void launch_kring(const GemmArgs& q, const KringShape& ks, hipStream_t s) {
    const dim3 grid(ks.strips, SERIAL ? 1 : q.split, q.batch), block(64 * SR_NW);
    if (q.M <= 16) hipLaunchKernelGGL((gemm_skinny_kring_kernel<DT, 1, SERIAL>), grid, block, 0, s, q);
    else if (q.M <= 32) hipLaunchKernelGGL((gemm_skinny_kring_kernel<DT, 2, SERIAL>), grid, block, 0, s, q);
    else hipLaunchKernelGGL((gemm_skinny_kring_kernel<DT, 4, SERIAL>), grid, block, 0, s, q);
}

// The kernel, and where K is split into a pool's or the caller's partials
// without counters their reduction.
template <int DT>
void launch_kring_all(const GemmArgs& q, const KringShape& ks, hipStream_t s) {
    if (q.split > 1 && !q.part) return launch_kring<DT, true>(q, ks, s);
    launch_kring<DT, false>(q, ks, s);
    if (q.split > 1 && !q.tile_count) launch_split_reduce<DT>(q, s);
}

// Whether a call that may not share memory with others, or must not allocate,
// splits K over workgroups all the same: up to 16 rows, and below K = 2048,
// such products have always been summed without partials.
bool kring_shared_split(const GemmArgs& p) { return p.M > 16 && p.K >= 2048; }

bool ring_applies(const GemmArgs& p, bool b_kmajor, bool vec) {
    if (b_kmajor || !vec) return false;
    auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    if (!al16(p.a) || !al16(p.b) || p.sa[2] != 1 || p.sb[2] != 1) return false;
    if (p.K % 32 != 0 || p.N % 8 != 0 || (p.M > 1 && p.sa[1] % 8 != 0) || (p.K > 1 && p.sb[1] % 8 != 0)) return false;
    if (p.batch > 1 && (p.sa[0] % 8 != 0 || p.sb[0] % 8 != 0)) return false;
    if (p.bh > 1 && (p.sa_h % 8 != 0 || p.sb_h % 8 != 0)) return false;
    return true;
}
}  // namespace

bool skinny_applies(int64_t M, int64_t N, int64_t K, int64_t batch) {
    return M >= 1 && M <= 16 && N >= 64 && K >= 64 && batch <= 65535;
}

bool skinny_wide_applies(const GemmArgs& p, bool b_kmajor, bool vec) {
    return p.M > 16 && skinny_applies(16, p.N, p.K, p.batch) && kring_applies(p, b_kmajor, vec);
}

const char* skinny_name(const GemmArgs& p, bool b_kmajor, bool vec) {
    if (ring_applies(p, b_kmajor, vec)) return ring_splits(p) > 1 ? "gemm16_skinny_ring_splitk" : "gemm16_skinny_ring";
    return b_kmajor ? "gemm16_skinny_bk" : "gemm16_skinny_bn";
}

size_t skinny_scratch_bytes(const GemmArgs& p, bool b_kmajor, bool vec) {
    if (kring_applies(p, b_kmajor, vec)) return kring_shared_split(p) ? kring_part_bytes(p, kring_shape(p).split) : 0;
    if (!ring_applies(p, b_kmajor, vec)) return 0;
    const int split = ring_splits(p);
    return split > 1 ? (size_t)split * p.batch * p.M * p.N * 4 : 0;
}

hipError_t launch_skinny(int dtype, const GemmArgs& p, bool b_kmajor, bool vec, hipStream_t s, float* part) {
    if (kring_applies(p, b_kmajor, vec)) {
        GemmArgs q = p;
        const KringShape ks = kring_shape(p);
        q.np = kring_pitch(p);
        q.split = ks.split;
        q.k_chunk = ks.chunk;
        Scratch scratch;
        q.part = nullptr;   // (without partials a workgroup takes a strip's chunks one after another)
        if (q.split > 1 && part) {   // the caller's memory, which its calls on other streams share
            if (kring_shared_split(p)) q.part = part;
        } else if (q.split > 1) {
            // A captured call takes memory of the graph's own where the tiled plans, which split from K = 2048 above 16
            // rows, take it too, and sums the partials in a second launch (in one workgroup a strip few strips leave
            // most CUs idle: bfloat16 33 x 8000 x 256 29.1 us, 10.9 on split tiles, 9.7 so).
            const size_t bytes = kring_part_bytes(p, q.split);
            if (bytes < (size_t)1 << 31 && (scratch_usable(s) || (kring_shared_split(p) && s != hipStreamPerThread)))
                q.part = static_cast<float*>(scratch.get(bytes, s));
            if (q.part) q.tile_count = split_counters(s, (int64_t)ks.strips * p.batch);   // (NULL under capture)
        }
        if (dtype == TVK_F16) launch_kring_all<TVK_F16>(q, ks, s);
        else launch_kring_all<TVK_BF16>(q, ks, s);
        return hipGetLastError();
    }
    if (ring_applies(p, b_kmajor, vec)) {
        GemmArgs q = p;
        q.np = q.N;
        q.split = ring_splits(p);
        q.k_chunk = p.K / q.split;
        Scratch scratch;
        if (q.split > 1) {
            q.part = part ? part : static_cast<float*>(scratch.get((size_t)q.split * p.batch * p.M * p.N * 4, s));
            if (!q.part) return hipErrorOutOfMemory;
        }
        const dim3 grid((p.N + SR_NB - 1) / SR_NB, q.split, p.batch);
        // the reduction in the same launch, except on caller-provided scratch
        // (the allocation-free entry point keeps its second launch)
        if (q.split > 1 && !part && (int64_t)q.split * p.batch * p.M * p.N * 4 < (int64_t(1) << 31))
            q.tile_count = split_counters(s, (int64_t)grid.x * p.batch);
        if (dtype == TVK_F16) hipLaunchKernelGGL(gemm_skinny_ring_kernel<TVK_F16>, grid, dim3(64 * SR_NW), 0, s, q);
        else hipLaunchKernelGGL(gemm_skinny_ring_kernel<TVK_BF16>, grid, dim3(64 * SR_NW), 0, s, q);
        if (q.split > 1 && !q.tile_count) {
            if (dtype == TVK_F16) launch_split_reduce<TVK_F16>(q, s);
            else launch_split_reduce<TVK_BF16>(q, s);
        }
        return hipGetLastError();
    }
    const int strips = (p.N + SK_CW - 1) / SK_CW;
    dim3 grid(strips, 1, p.batch);
#define TVK_SK(D, BKM, V) hipLaunchKernelGGL((gemm_skinny_kernel<D, BKM, V>), grid, dim3(64 * SK_NW), 0, s, p)
    if (dtype == TVK_F16) {
        if (b_kmajor) { if (vec) TVK_SK(TVK_F16, true, true); else TVK_SK(TVK_F16, true, false); }
        else { if (vec) TVK_SK(TVK_F16, false, true); else TVK_SK(TVK_F16, false, false); }
    } else {
        if (b_kmajor) { if (vec) TVK_SK(TVK_BF16, true, true); else TVK_SK(TVK_BF16, true, false); }
        else { if (vec) TVK_SK(TVK_BF16, false, true); else TVK_SK(TVK_BF16, false, false); }
    }
#undef TVK_SK
    return hipGetLastError();
}

}  // namespace tvk
