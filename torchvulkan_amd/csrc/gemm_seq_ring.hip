// float32 GEMM in the reference SIMD tile's order on 64x64 tiles, operands
// loaded straight into an LDS ring (the products with few tiles; larger ones
// keep the 128x128 tiles of gemm.hip).
//
// Every output accumulates fmaf(a_k, b_k, acc) for k = 0, 1, 2, ... on
// v_mfma_f32_16x16x1_4b_f32 (src/shaders/helpers/gemm_simd.slang:219-239; each
// wave owns 16 rows x 64 columns, its row's A value in all four blocks, one
// 16x64 rank-1 update an instruction), the bits of gemm_seq16_kernel.
//
// A wave is one chain of K dependent instructions, so the call is bound by
// keeping that chain fed: 1024^3 runs one wave a SIMD. Staged through registers
// one 16-k step ahead, a step waited for its loads (about 500 cycles of
// products against 1200-1900 of latency) and for most of its LDS reads: 35.4
// us. Here four 16-k stages (32 KB, so that several workgroups share a CU) are
// loaded straight into LDS, three of them in flight, and a stage's fragments are
// read into a second register set during the products of the stage before: 29.5
// us, about 61 cycles an instruction, which is its dependent latency (eight
// stages: the same; 13.7 us at its issue rate). 2048^3: 165 -> 155 us (eight
// stages, two workgroups a CU: 167). Two or four shorter chains a wave on
// v_mfma_f32_4x4x1_16b_f32 (8 waves of 8 rows) took 34.9 and 195 us. Rows that
// are no 16-byte multiples load four bytes a lane into the same layout: 1000 x
// 333 x 1777 97.5 -> 61.5 us.
#include "gemm_common.h"

#include <type_traits>

namespace tvk {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
#define TVK_LDS __attribute__((address_space(3)))

constexpr int SQ_BK = 16;                  // k per stage
constexpr int SQ_NS = 4;                   // stages in the ring
constexpr int SQ_OP = 64 * SQ_BK * 4;      // bytes of an operand's stage: 4 KB, 1 KB per wave
constexpr int SQ_ST = 2 * SQ_OP;

__device__ inline i32x4 sq_rsrc(const void* ptr, int64_t bytes) {
    const uint64_t a = (uint64_t)ptr;
    return i32x4{(int)(uint32_t)a, (int)((a >> 32) & 0xffff), (int)min(bytes, (int64_t)0x7fffffff), 0x00020000};
}
// 16 or 4 bytes per lane into LDS at lds_addr + 16 (or 4) * lane; the waits are explicit.
template <bool VEC>
__device__ inline void sq_dma(i32x4 r, uint32_t lds_addr, uint32_t voff) {
    if constexpr (VEC)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     :: "s"(lds_addr), "v"(voff), "s"(r) : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                     :: "s"(lds_addr), "v"(voff), "s"(r) : "memory");
}
template <int N>
__device__ inline void sq_wait() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

// Chunk swizzle of a k-contiguous operand's 64-byte LDS rows: the 16 rows of
// a served lane group meet 16 distinct 16-byte slots.
__device__ inline int sq_swz(int row) { return (row >> 2) & 3; }

// One operand's loads: its 64 rows (m or n) x 16 k of a stage. KM
// (k-contiguous): LDS rows of 16 k; else 16 k-rows of 64 values. Wave w fills
// the operand's w-th 1 KB with L loads.
template <bool KM, bool VEC>
struct SqSrc {
    static constexpr int L = VEC ? 1 : 4, E = VEC ? 4 : 1;   // loads a stage, elements a lane
    uint32_t off[L];
    int k[L];          // the lane's k within a stage
    uint32_t kstep;
    __device__ inline void init(int64_t s_row, int64_t s_k, int row0, int rows, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int e = (wave * 256 + i * 64 * E) + lane * E;   // the lane's first value in the operand's stage
            int r;
            if constexpr (KM) {
                r = e / SQ_BK;
                const int f = e % SQ_BK;
                k[i] = ((f / 4) ^ sq_swz(r)) * 4 + f % 4;
            } else {
                r = e % 64;
                k[i] = e / 64;
            }
            off[i] = row0 + r < rows ? (uint32_t)(((int64_t)(row0 + r) * s_row + (int64_t)k[i] * s_k) * 4) : kOOB;
        }
        kstep = (uint32_t)(SQ_BK * s_k * 4);
    }
    // k at or past K (left: K minus the stage's first k) loads zeros
    __device__ inline void issue(i32x4 rs, uint32_t at, int stage, int left) const {
#pragma unroll
        for (int i = 0; i < L; ++i)
            sq_dma<VEC>(rs, at + (uint32_t)(i * 64 * E * 4), k[i] < left ? off[i] + (uint32_t)stage * kstep : kOOB);
    }
};

// The k values 4 q4 .. + 3 of a stage for the lane's row (or column).
template <bool KM>
__device__ inline f32x4 sq_read(uint32_t base, int row, int q4) {
    if constexpr (KM) {
        return *(const TVK_LDS f32x4*)(uintptr_t)(base + row * 64 + ((q4 ^ sq_swz(row)) * 16));
    } else {
        const TVK_LDS float* s = (const TVK_LDS float*)(uintptr_t)(base + q4 * 4 * 256 + row * 4);
        return f32x4{s[0], s[64], s[128], s[192]};
    }
}

template <bool AK, bool BK, bool VEC>
__global__ __launch_bounds__(256) void gemm_seq_ring_kernel(GemmArgs p) {
    constexpr int PER = SqSrc<AK, VEC>::L + SqSrc<BK, VEC>::L;   // loads a wave and stage
    __shared__ __attribute__((aligned(1024))) char lds[SQ_NS * SQ_ST];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(TVK_LDS char*)lds);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int b = blockIdx.y;
    int tm, tn;
    tile_of(blockIdx.x, p.tiles_m * p.tiles_n, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * 64, n0 = tn * 64;
    const char* A = reinterpret_cast<const char*>(p.a) + a_boff(p, b) * 4;
    const char* B = reinterpret_cast<const char*>(p.b) + b_boff(p, b) * 4;
    const i32x4 ra = sq_rsrc(A, 4 * ((int64_t)(p.M - 1) * p.sa[1] + (int64_t)(p.K - 1) * p.sa[2] + 1));
    const i32x4 rb = sq_rsrc(B, 4 * ((int64_t)(p.N - 1) * p.sb[2] + (int64_t)(p.K - 1) * p.sb[1] + 1));
    SqSrc<AK, VEC> sa;
    SqSrc<BK, VEC> sb;
    sa.init(p.sa[1], p.sa[2], m0, p.M, wave, lane);
    sb.init(p.sb[2], p.sb[1], n0, p.N, wave, lane);
    const int nk = (p.K + SQ_BK - 1) / SQ_BK;
    auto issue = [&](int s) {
        if (s >= nk) return;
        const uint32_t at = lds0 + (uint32_t)((s % SQ_NS) * SQ_ST + wave * 1024);
        const int left = p.K - s * SQ_BK;
        sa.issue(ra, at, s, left);
        sb.issue(rb, at + SQ_OP, s, left);
    };

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int arow = wave * 16 + lane % 16;   // the same row in all four blocks
    const int bcol = lane;                    // block lane / 16, column lane % 16
    f32x4 av[2][4], bv[2][4];

#pragma unroll
    for (int s = 0; s < SQ_NS - 1; ++s) issue(s);
    if (nk >= SQ_NS - 1) sq_wait<PER * (SQ_NS - 2)>(); else sq_wait<0>();
    __syncthreads();   // stage 0 is in LDS
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        av[0][q] = sq_read<AK>(lds0, arow, q);
        bv[0][q] = sq_read<BK>(lds0 + SQ_OP, bcol, q);
    }
    auto body = [&](int kt, auto cur_c) {
        constexpr int cur = decltype(cur_c)::value;
        // stage kt + 1 landed, in every wave; stage kt - 1's slot was read for the last time two barriers ago
        if (kt + SQ_NS - 2 < nk) sq_wait<PER * (SQ_NS - 3)>(); else sq_wait<0>();
        __syncthreads();
        issue(kt + SQ_NS - 1);
        const uint32_t st = lds0 + (uint32_t)(((kt + 1) % SQ_NS) * SQ_ST);
        // (past the last stage the reads fetch a slot whose values are not used)
#pragma unroll
        for (int k = 0; k < SQ_BK; ++k) {
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(av[cur][k / 4][k % 4], bv[cur][k / 4][k % 4], acc, 0, 0, 0);
            if (k % 2 == 0 && k < 8) av[cur ^ 1][k / 2] = sq_read<AK>(st, arow, k / 2);
            if (k % 2 == 1 && k < 8) bv[cur ^ 1][k / 2] = sq_read<BK>(st + SQ_OP, bcol, k / 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        body(kt, std::integral_constant<int, 0>{});
        body(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) body(kt, std::integral_constant<int, 0>{});

    // register r: block r / 4 (columns 16 (r / 4) ..), row (lane / 16) * 4 + r % 4, column lane % 16
    if (!p.has_bias && p.act == TVK_ACT_NONE) {
        // no bias, no activation: alpha times the sum, as store_out computes it,
        // with the batch offset once for the lane's 16 outputs
        float* c = reinterpret_cast<float*>(p.c) + c_boff(p, b);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = m0 + wave * 16 + (lane / 16) * 4 + r % 4;
            const int col = n0 + (r / 4) * 16 + lane % 16;
            if (row < p.M && col < p.N) {
#pragma clang fp contract(off)
                const float o = acc[r] * p.alpha;
                c[(int64_t)row * p.sc[1] + (int64_t)col * p.sc[2]] = o;
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + wave * 16 + (lane / 16) * 4 + r % 4;
        const int col = n0 + (r / 4) * 16 + lane % 16;
        if (row < p.M && col < p.N) store_out<TVK_F32, true>(p, b, row, col, acc[r]);
    }
}

template <bool AK, bool BK, bool VEC>
void launch(const GemmArgs& p, hipStream_t s) {
    hipLaunchKernelGGL((gemm_seq_ring_kernel<AK, BK, VEC>), dim3(p.tiles_m * p.tiles_n, p.batch), dim3(256), 0, s, p);
}

}  // namespace

void launch_seq_ring(const GemmArgs& p, bool a_kmajor, bool b_kmajor, bool vec, hipStream_t s) {
    if (a_kmajor && b_kmajor) vec ? launch<true, true, true>(p, s) : launch<true, true, false>(p, s);
    else if (a_kmajor) vec ? launch<true, false, true>(p, s) : launch<true, false, false>(p, s);
    else if (b_kmajor) vec ? launch<false, true, true>(p, s) : launch<false, true, false>(p, s);
    else vec ? launch<false, false, true>(p, s) : launch<false, false, false>(p, s);
}

}  // namespace tvk
