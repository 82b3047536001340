// Attention over a key/value cache for a few new queries (L <= 16, no causal
// mask): the call reads K and V once and is bound by that stream.
//
// The tiled forward gives every (batch, query head) a workgroup of 64 query
// slots: one new token fills one of them, each query head of a group reads
// its key/value head again, and few long sequences leave the chip idle (8
// sequences of 32/8 heads over 4001 keys of 128: 256 workgroups, 78 us, 1.7
// TB/s). Here the L * group query rows that share a key/value head are packed
// as the 16 (or 32) columns of the products, and the keys are split between
// workgroups (28 us, 4.7 TB/s there).
//
// A workgroup is 4 waves; each wave streams 32-key tiles of its own (wave w
// takes tiles w, w + 4, ... of the workgroup's range), so no barrier stands
// between a wave and its loads: K rows go straight from memory into the A
// operand of S^T = K Q^T, V rows through a wave-private LDS tile that is read
// back transposed for O^T += V^T P^T; both tiles of the next step are in
// flight while one is computed. The softmax is the tiled forward's (log2
// units, or natural ones with a bias; running max, per-lane sums). At the end
// the waves' (max, sum, O) are merged through LDS in wave order. With one
// split the workgroup writes the output; with more, float32 partials are
// written through to memory (system scope, no fence, as the skinny GEMM's
// split_fixup) and the last workgroup of a row block merges them in split
// order; where the stream has no counters, attn_decode_merge_kernel does the
// same in a second launch. Both give the same bits every run.
#include "attention_kernels.h"

namespace tvk {

namespace {

constexpr int DC_WAVES = 4;
constexpr int DC_BN = 32;   // keys per tile

struct DecodeArgs {
    AttnArgs a;
    int rows;      // L * group: query rows of one key/value head
    int nrb;       // row blocks per key/value head
    int kvh;       // key/value heads
    int per;       // key tiles per split
    int splits;
    float* part_o;   // [split][batch * kvh][rows][hd], or NULL with one split
    float* part_ml;  // [split][batch * kvh][rows][2]: max, sum
    unsigned part_bytes;   // of both
    unsigned* count; // one per row block, zero before and after the launch; NULL: a second launch merges
};

// Output row of packed row r: head r / L of the group, query r % L.
__device__ inline void decode_row(const DecodeArgs& p, int r, int hk, int& h, int& qi) {
    const int hg = r / p.a.L;
    h = hk * p.a.group + hg;
    qi = r - hg * p.a.L;
}

template <int DT>
__device__ inline void decode_store(const AttnArgs& a, int b, int h, int qi, int dv, f32x4 o) {
    uint16_t* op = a.out + (int64_t)b * a.so[0] + (int64_t)h * a.so[1] + (int64_t)qi * a.so[2] + (int64_t)dv * a.so[3];
    if (a.out_vec) {
        *reinterpret_cast<u32x2*>(op) = u32x2{pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3])};
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) op[(int64_t)r * a.so[3]] = __builtin_bit_cast(uint16_t, elem<DT>::from_f32(o[r]));
    }
}

__device__ inline __amdgpu_buffer_rsrc_t decode_rsrc(const DecodeArgs& p) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p.part_o, 0, (int)p.part_bytes, 0x00020000);
}
// Byte offsets of the partials: below 2 GiB (attn_decode_fwd).
__device__ inline int decode_o_at(const DecodeArgs& p, int64_t row, int dv) { return (int)((row * p.a.hd + dv) * 4); }
__device__ inline int decode_ml_at(const DecodeArgs& p, int64_t row) {
    return (int)((const char*)(p.part_ml + row * 2) - (const char*)p.part_o);
}

// Merges columns dv .. dv + 3 of a query row's partials in split order (reads
// that miss the L2, whose lines may be older than other XCDs' stores) and
// writes the output; row counts all rows of the call, all_rows of them.
template <int DT, bool BIAS>
__device__ inline void decode_merge(const DecodeArgs& p, int64_t row, int64_t all_rows, int dv) {
    constexpr float UNIT = BIAS ? AT_LOG2E : 1.0f;
    const AttnArgs& a = p.a;
    const __amdgpu_buffer_rsrc_t rs = decode_rsrc(p);
    float m = -INFINITY, l = 0.0f;
    f32x4 o = f32x4{0, 0, 0, 0};
    // groups of splits, their loads in flight together, on a running max
    constexpr int U = 8;
    auto merge_group = [&](int s0, auto part_c) {
        constexpr bool SOME = decltype(part_c)::value;   // the last group, of fewer than U splits
        u32x2 w[U];
        u32x4 os[U];
        // past the last split it is read again, and its maxima and sums masked to -inf and 0: a weight of 0 would make
        // NaN of an infinite sum, and a branch lets the loads sink to their uses (1 x 32/1 heads x 8000 x 128: 45 us, 22 so)
        auto at = [&](int u) { return (SOME ? min(s0 + u, p.splits - 1) : s0 + u) * all_rows + row; };
#pragma unroll
        for (int u = 0; u < U; ++u)
            w[u] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, decode_ml_at(p, at(u)), 0, kCoherent));
#pragma unroll
        for (int u = 0; u < U; ++u)
            os[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, decode_o_at(p, at(u), dv), 0, kCoherent));
        if (SOME) __builtin_amdgcn_sched_barrier(0);
        float mn = m;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (SOME && s0 + u >= p.splits) w[u][0] = 0xff800000u;
            mn = fmaxf(mn, __builtin_bit_cast(float, (uint32_t)w[u][0]));
        }
        const float f0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * UNIT);
        l *= f0;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= f0;
        m = mn;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float ms = __builtin_bit_cast(float, (uint32_t)w[u][0]), ls = __builtin_bit_cast(float, (uint32_t)w[u][1]);
            const float f = ms == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((ms - m) * UNIT);
            l += ls * f;
            if (SOME) os[u] = os[u] & (s0 + u < p.splits ? ~0u : 0u);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += __builtin_bit_cast(f32x4, os[u])[e] * f;
        }
    };
    int s0 = 0;
    for (; s0 + U <= p.splits; s0 += U) merge_group(s0, std::integral_constant<bool, false>{});
    if (s0 < p.splits) merge_group(s0, std::integral_constant<bool, true>{});
    const int bhk = (int)(row / p.rows), r = (int)(row - (int64_t)bhk * p.rows);
    const int b = bhk / p.kvh, hk = bhk % p.kvh;
    int h, qi;
    decode_row(p, r, hk, h, qi);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    decode_store<DT>(a, b, h, qi, dv, f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
    if (dv == 0)
        a.lse[(int64_t)b * a.sl[0] + (int64_t)h * a.sl[1] + (int64_t)qi * a.sl[2]] =
            l > 0.0f ? m * (BIAS ? 1.0f : AT_LN2) + logf(l) : INFINITY;
}

template <int DT, int D, bool BIAS, int CT, bool PART>
__global__ __launch_bounds__(64 * DC_WAVES, 2) void attn_decode_kernel(DecodeArgs p) {
    constexpr int DS = D / 32, DT16 = D / 16;
    constexpr int LDV = D + 16;                       // as the tiled forward's V rows
    constexpr int VCH = DC_BN * D / 8 / 64;           // 16-byte V chunks per lane and tile
    constexpr int LDO = D + 4;                        // floats per merged row
    constexpr float UNIT = BIAS ? AT_LOG2E : 1.0f;    // softmax_tile's units
    __shared__ __attribute__((aligned(16))) uint16_t vs[DC_WAVES][DC_BN * LDV];
    __shared__ float ml[2][DC_WAVES][16 * CT];
    static_assert(sizeof(vs) >= DC_WAVES * 16 * LDO * sizeof(float), "the merge reuses the V tiles");

    const AttnArgs& a = p.a;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int g = lane / 16, c16 = lane % 16;
    const int rb = blockIdx.x % p.nrb, bhk = blockIdx.x / p.nrb;
    const int b = bhk / p.kvh, hk = bhk % p.kvh;
    const int r0 = rb * 16 * CT;

    u32x4 qf[CT][DS];
    const uint16_t* bias[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int r = r0 + 16 * ct + c16;
        int h = hk * a.group, qi = 0;
        if (r < p.rows) decode_row(p, r, hk, h, qi);
        const uint16_t* Q = a.q + (int64_t)b * a.sq[0] + (int64_t)h * a.sq[1] + (int64_t)qi * a.sq[2];
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const bool in = r < p.rows && (!PART || 32 * ds + 8 * g < a.hd);
            u32x4 x = in ? *reinterpret_cast<const u32x4*>(Q + 32 * ds + 8 * g) : u32x4{0, 0, 0, 0};
            if (!BIAS) x ^= a.qflip;
            qf[ct][ds] = x;
        }
        bias[ct] = BIAS ? a.bias + (int64_t)b * a.sb[0] + (int64_t)h * a.sb[1] + (int64_t)qi * a.sb[2] : nullptr;
    }

    f32x4 oacc[DT16][CT];
    float m_run[CT], l_run[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
        for (int i = 0; i < DT16; ++i) oacc[i][ct] = f32x4{0, 0, 0, 0};
        m_run[ct] = -INFINITY;
        l_run[ct] = 0.0f;
    }

    const char* Kh = reinterpret_cast<const char*>(a.k + (int64_t)b * a.sk[0] + (int64_t)hk * a.sk[1]);
    const char* Vh = reinterpret_cast<const char*>(a.v + (int64_t)b * a.sv[0] + (int64_t)hk * a.sv[1]);
    const int64_t kstep = (int64_t)DC_BN * a.sk[2] * 2, vstep = (int64_t)DC_BN * a.sv[2] * 2;
    const int tiles = (a.S + DC_BN - 1) / DC_BN;
    const int t0 = blockIdx.y * p.per, t1 = min(tiles, t0 + p.per);

    u32x4 kr[2][DS], vr[VCH];
    auto load_k = [&](int t) {
        const char* kt = Kh + (int64_t)t * kstep;
        const bool whole = !PART && t * DC_BN + DC_BN <= a.S;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                const int row = 16 * kb + c16, d = 32 * ds + 8 * g;
                const bool in = whole || (t * DC_BN + row < a.S && (!PART || d < a.hd));
                kr[kb][ds] = in ? *reinterpret_cast<const u32x4*>(kt + (uint32_t)((row * (int)a.sk[2] + d) * 2)) : u32x4{0, 0, 0, 0};
            }
    };
    auto load_v = [&](int t) {
        const char* vt = Vh + (int64_t)t * vstep;
        const bool whole = !PART && t * DC_BN + DC_BN <= a.S;
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int c = lane + 64 * i, row = c / (D / 8), d = (c % (D / 8)) * 8;
            const bool in = whole || (t * DC_BN + row < a.S && (!PART || d < a.hd));
            vr[i] = in ? *reinterpret_cast<const u32x4*>(vt + (uint32_t)((row * (int)a.sv[2] + d) * 2)) : u32x4{0, 0, 0, 0};
        }
    };

    int t = t0 + wave;
    if (t < t1) {
        load_k(t);
        load_v(t);
    }
    for (; t < t1; t += DC_WAVES) {
        // ---- S^T = K Q^T
        f32x4 sacc[2][CT];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                sacc[kb][ct] = f32x4{0, 0, 0, 0};
#pragma unroll
                for (int ds = 0; ds < DS; ++ds) sacc[kb][ct] = mfma16<DT>(kr[kb][ds], qf[ct][ds], sacc[kb][ct]);
            }
        // V rows to the wave's own tile (its reads of the tile before are done: one wave's LDS accesses stay in order)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int c = lane + 64 * i, row = c / (D / 8), d = (c % (D / 8)) * 8;
            *reinterpret_cast<u32x4*>(&vs[wave][row * LDV + d]) = vr[i];
        }
        __builtin_amdgcn_wave_barrier();
        if (t + DC_WAVES < t1) {
            load_k(t + DC_WAVES);
            load_v(t + DC_WAVES);
        }
        // ---- online softmax per column
        const int k0 = t * DC_BN;
        const bool plain = !BIAS && k0 + DC_BN <= a.S;
        float alpha[CT];
        bool rescale = false;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float tmax = -INFINITY;
            if (!plain) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int kj = k0 + 16 * kb + 4 * g + r;
                        float s = sacc[kb][ct][r] * (BIAS ? a.scale : a.c2);
                        if (BIAS && kj < a.S)
                            s = s + elem<DT>::to_f32(__builtin_bit_cast(typename elem<DT>::T, bias[ct][(int64_t)kj * a.sb[3]]));
                        sacc[kb][ct][r] = kj < a.S ? s : -INFINITY;
                    }
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sacc[kb][ct][r]);
            tmax = lanes4_max(tmax);
            if (plain) tmax *= a.c2;
            const float m_old = m_run[ct], m_new = fmaxf(m_old, tmax);
            const float m_use = m_new == -INFINITY ? 0.0f : m_new;
            alpha[ct] = (m_old == m_new || m_old == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f((m_old - m_use) * UNIT);
            rescale = rescale || alpha[ct] != 1.0f;
            float rsum = 0.0f;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = plain ? __builtin_fmaf(sacc[kb][ct][r], a.c2, -m_use) : (sacc[kb][ct][r] - m_use) * UNIT;
                    const float e = __builtin_amdgcn_exp2f(x);
                    sacc[kb][ct][r] = e;
                    rsum += e;
                }
            l_run[ct] = l_run[ct] * alpha[ct] + rsum;
            m_run[ct] = m_new;
        }
        if (__any(rescale)) {
#pragma unroll
            for (int i = 0; i < DT16; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int r = 0; r < 4; ++r) oacc[i][ct][r] *= alpha[ct];
        }
        // ---- O^T += V^T P^T
        u32x4 pf[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const f32x4 x = sacc[0][ct], y = sacc[1][ct];
            pf[ct] = u32x4{pack2<DT>(x[0], x[1]), pack2<DT>(x[2], x[3]), pack2<DT>(y[0], y[1]), pack2<DT>(y[2], y[3])};
        }
#pragma unroll
        for (int i = 0; i < DT16; ++i) {
            const u32x4 vf = read_tr<LDV>(vs[wave], 0, i, g, c16);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) oacc[i][ct] = mfma16<DT>(vf, pf[ct], oacc[i][ct]);
        }
    }

    // ---- merge the waves, one 16-column block at a time through the V tiles
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const float l_tot = lanes4_sum(l_run[ct]);
        if (g == 0) {
            ml[0][wave][16 * ct + c16] = m_run[ct];
            ml[1][wave][16 * ct + c16] = l_tot;
        }
    }
    float* red = reinterpret_cast<float*>(&vs[0][0]);
    const int64_t all_rows = (int64_t)(gridDim.x / p.nrb) * p.rows;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        __syncthreads();   // every wave has left its V tile, and the block before has been read
#pragma unroll
        for (int i = 0; i < DT16; ++i)
            *reinterpret_cast<f32x4*>(&red[(wave * 16 + c16) * LDO + 16 * i + 4 * g]) = oacc[i][ct];
        __syncthreads();
        for (int c = tid; c < 16 * (D / 4); c += 64 * DC_WAVES) {
            const int col = c / (D / 4), dv = (c % (D / 4)) * 4;
            const int r = r0 + 16 * ct + col;
            if (r >= p.rows || (PART && dv >= a.hd)) continue;
            float m = -INFINITY;
#pragma unroll
            for (int w = 0; w < DC_WAVES; ++w) m = fmaxf(m, ml[0][w][16 * ct + col]);
            float l = 0.0f;
            f32x4 o = f32x4{0, 0, 0, 0};
#pragma unroll
            for (int w = 0; w < DC_WAVES; ++w) {
                const float mw = ml[0][w][16 * ct + col];
                const float f = mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mw - m) * UNIT);
                const f32x4 ow = *reinterpret_cast<const f32x4*>(&red[(w * 16 + col) * LDO + dv]);
                l += ml[1][w][16 * ct + col] * f;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] += ow[e] * f;
            }
            if (p.splits > 1) {
                const __amdgpu_buffer_rsrc_t rs = decode_rsrc(p);
                const int64_t row = (int64_t)blockIdx.y * all_rows + (int64_t)bhk * p.rows + r;
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rs, decode_o_at(p, row, dv), 0, kCoherent);
                if (dv == 0)
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2v{m, l}), rs, decode_ml_at(p, row), 0, kCoherent);
            } else {
                int h, qi;
                decode_row(p, r, hk, h, qi);
                const float inv = l > 0.0f ? 1.0f / l : 0.0f;
                decode_store<DT>(a, b, h, qi, dv, f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
                if (dv == 0)
                    a.lse[(int64_t)b * a.sl[0] + (int64_t)h * a.sl[1] + (int64_t)qi * a.sl[2]] =
                        l > 0.0f ? m * (BIAS ? 1.0f : AT_LN2) + logf(l) : INFINITY;
            }
        }
    }
    if (p.splits == 1 || !p.count) return;

    // ---- the last workgroup of the row block merges its splits; none waits for another
    __shared__ int last;
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wave's partials are in memory
    __syncthreads();
    if (tid == 0) {
        unsigned* cnt = p.count + blockIdx.x;
        last = atomicAdd_system(cnt, 1u) + 1 == (unsigned)p.splits;
        if (last) atomicExch_system(cnt, 0u);
    }
    __syncthreads();
    if (!last) return;
    const int block_rows = min(16 * CT, p.rows - r0);
    for (int c = tid; c < block_rows * (D / 4); c += 64 * DC_WAVES) {
        const int dv = (c % (D / 4)) * 4;
        if (!PART || dv < a.hd) decode_merge<DT, BIAS>(p, (int64_t)bhk * p.rows + r0 + c / (D / 4), all_rows, dv);
    }
}

// The merge as a launch of its own: 32 lanes per query row, four columns a lane.
template <int DT, bool BIAS>
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(DecodeArgs p, int64_t all_rows) {
    const int64_t row = (int64_t)blockIdx.x * 8 + threadIdx.x / 32;
    const int dv = (threadIdx.x % 32) * 4;
    if (row >= all_rows || dv >= p.a.hd) return;
    decode_merge<DT, BIAS>(p, row, all_rows, dv);
}

template <int DT, int D, bool PART>
void launch_d(const DecodeArgs& p, bool bias, int ct, dim3 grid, hipStream_t s) {
    const dim3 block(64 * DC_WAVES);
    if (bias) {
        if (ct == 2) hipLaunchKernelGGL((attn_decode_kernel<DT, D, true, 2, PART>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((attn_decode_kernel<DT, D, true, 1, PART>), grid, block, 0, s, p);
    } else {
        if (ct == 2) hipLaunchKernelGGL((attn_decode_kernel<DT, D, false, 2, PART>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((attn_decode_kernel<DT, D, false, 1, PART>), grid, block, 0, s, p);
    }
}

template <int DT>
void launch(const DecodeArgs& p, bool bias, int ct, dim3 grid, int64_t all_rows, hipStream_t s) {
    if (p.a.hd == 64) launch_d<DT, 64, false>(p, bias, ct, grid, s);
    else if (p.a.hd == 128) launch_d<DT, 128, false>(p, bias, ct, grid, s);
    else if (p.a.hd <= 32) launch_d<DT, 32, true>(p, bias, ct, grid, s);
    else if (p.a.hd <= 64) launch_d<DT, 64, true>(p, bias, ct, grid, s);
    else if (p.a.hd <= 96) launch_d<DT, 96, true>(p, bias, ct, grid, s);
    else launch_d<DT, 128, true>(p, bias, ct, grid, s);
    if (p.splits > 1 && !p.count) {
        const dim3 mg((unsigned)((all_rows + 7) / 8));
        if (bias) hipLaunchKernelGGL((attn_decode_merge_kernel<DT, true>), mg, dim3(256), 0, s, p, all_rows);
        else hipLaunchKernelGGL((attn_decode_merge_kernel<DT, false>), mg, dim3(256), 0, s, p, all_rows);
    }
}

// The keys are split until about two workgroups a CU run (their registers let
// two be resident; bfloat16 8 x 32/8 heads x 4001 x 128: 28.0 us for 512, 29.9
// for 256, 30.9 for 768), as long as every wave keeps a tile (32/8 heads x
// 1000 x 64: 6.1 us, 6.5 with two tiles a wave) and into at most 32 parts: the
// last workgroup reads them one after another (1 x 32/8 x 16000 x 128: 17.7 us
// in 32 parts, 21.3 in 63). Two column blocks merge twice the rows: below 16
// tiles one part (64 x 8/2 heads, 5 queries x 256 x 128: 8.9 us, 12.2 in two; 512
// keys 14.2, 12.1 in four), except with a bias, whose loads the parts share out.
constexpr int kTargetGroups = 512, kMaxSplits = 32, kMinTiles2 = 16;

}  // namespace

bool attn_decode_applies(const AttnArgs& a, bool causal, bool bias, int64_t batch, int64_t heads) {
    // row offsets inside a tile are 32-bit
    const auto row_ok = [](int64_t st) { return (DC_BN * st + 128) * 2 < (int64_t)0x7fffffff; };
    // one tile of keys and no head to share them with leaves nothing to split or pack: the tiled forward is as fast
    // (64 x 8 heads x 64 keys of 64, 16 queries: 4.2 us there, 4.5 here; 128 keys: 7.0 there, 6.4 here)
    if (a.group == 1 && a.S <= AT_BN) return false;
    // More than 16 query rows a key/value head are two column blocks a wave: over short sequences, where the tiled
    // forward's workgroup a query head is at most two rounds, the blocks' merge costs more than the shared keys save.
    // Tiled and here, float16 4 x 8/2 heads, 16 queries: of 128, 65 keys 5.7 and 6.9 us, 256 keys 7.6 and 12.4, 512 keys
    // 12.1 and 12.8, 700 keys 16.0 and 14.1; of 64, 128 keys 4.4 and 5.2, 400 keys 8.7 and 8.9 (7.7 in one part), 700
    // keys 12.1 and 9.0. With 1024 heads (64 x 16/1) of 64: 64 keys 5.1 and 6.4, 65 keys 7.3 and 6.4. With a bias, whose
    // values the tiled forward loads a head at a time, only a single tile of keys (4 x 64/8 heads, 5 queries, of 128: 64
    // keys 6.7 and 8.2, 65 keys 8.7 and 8.3).
    if (a.L * a.group > 16) {
        const int64_t bh = batch * heads;
        if (a.S <= AT_BN && bh <= (bias ? 256 : a.hd <= 64 ? 1024 : 512)) return false;
        if (!bias && a.S <= (a.hd <= 96 ? 6 : a.L * a.group <= 32 ? 7 : 8) * AT_BN && bh <= 256) return false;
    }
    return !causal && a.L <= 16 && a.S > 0 && row_ok(a.sk[2]) && row_ok(a.sv[2]) &&
           batch * (heads / a.group) * (((int64_t)a.L * a.group + 15) / 16) <= (int64_t)0x7fffffff;
}

void attn_decode_fwd(int dtype, const AttnArgs& args, bool bias, int64_t batch, int64_t heads, hipStream_t s) {
    DecodeArgs p{};
    p.a = args;
    p.kvh = (int)(heads / args.group);
    p.rows = args.L * args.group;
    const int ct = p.rows > 16 ? 2 : 1;
    p.nrb = (p.rows + 16 * ct - 1) / (16 * ct);
    const int64_t bhk = batch * p.kvh, base = bhk * p.nrb, all_rows = bhk * p.rows;
    const int tiles = (args.S + DC_BN - 1) / DC_BN;
    const int most = ct == 2 && !bias && tiles < kMinTiles2 ? 1 : std::max(1, std::min(kMaxSplits, tiles / DC_WAVES));
    const int want = (int)std::min<int64_t>(std::max<int64_t>(1, kTargetGroups / base), most);
    p.per = ((tiles + want - 1) / want + DC_WAVES - 1) / DC_WAVES * DC_WAVES;
    p.splits = (tiles + p.per - 1) / p.per;
    Scratch scratch;
    if (p.splits > 1) {
        // partials need scratch: a call that gets none takes one split
        const bool can = scratch_usable(s);
        const size_t rows = (size_t)p.splits * all_rows, bytes = rows * (args.hd + 2) * 4;
        float* part = !can || bytes >= (size_t)1 << 31 ? nullptr : static_cast<float*>(scratch.get(bytes, s));
        if (part) {
            p.part_o = part;
            p.part_ml = part + rows * args.hd;
            p.part_bytes = (unsigned)bytes;
            p.count = split_counters(s, base);
        } else {
            clear_error();
            p.splits = 1;
            p.per = tiles;
        }
    }
    const dim3 grid((unsigned)base, (unsigned)p.splits);
    if (dtype == TVK_F16) launch<TVK_F16>(p, bias, ct, grid, all_rows, s);
    else launch<TVK_BF16>(p, bias, ct, grid, all_rows, s);
}

}  // namespace tvk
