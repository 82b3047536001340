// The attention kernels of attention_kernels.h for head dims other than 64 and
// 128: any multiple of 8 up to 128, on the next tile width of 32, 64, 96 or
// 128 columns with zeros past the head dim. They ran on the general VALU
// kernels before (attention_any.hip), whose scores and products are scalar
// fused multiply-adds over float32 LDS tiles: forward and backward of bfloat16
// 8 x 16 heads x 577 x 80 took 4690 us there and take 162 us here. The next
// tile width above the head dim, since a column of zeros costs its products
// and its LDS but no memory traffic.
#include "attention_kernels.h"

namespace tvk {
namespace {

template <int DT>
bool fwd(const AttnArgs& a, bool causal, bool bias, int64_t batch, int64_t heads, int64_t L, hipStream_t s) {
    switch ((a.hd + 31) / 32) {
    case 1: launch_attn<DT, 32, true>(a, causal, bias, batch, heads, L, s); return true;
    case 2: launch_attn<DT, 64, true>(a, causal, bias, batch, heads, L, s); return true;
    case 3: launch_attn<DT, 96, true>(a, causal, bias, batch, heads, L, s); return true;
    case 4: launch_attn<DT, 128, true>(a, causal, bias, batch, heads, L, s); return true;
    default: return false;
    }
}

template <int DT>
bool bwd(const AttnBwdArgs& a, bool causal, bool bias, int64_t batch, int64_t heads, int64_t L, int64_t S, hipStream_t s) {
    switch ((a.hd + 31) / 32) {
    case 1: launch_attn_bwd<DT, 32, true>(a, causal, bias, batch, heads, L, S, s); return true;
    case 2: launch_attn_bwd<DT, 64, true>(a, causal, bias, batch, heads, L, S, s); return true;
    case 3: launch_attn_bwd<DT, 96, true>(a, causal, bias, batch, heads, L, S, s); return true;
    case 4: launch_attn_bwd<DT, 128, true>(a, causal, bias, batch, heads, L, S, s); return true;
    default: return false;
    }
}

}  // namespace

bool attn_part_fwd(int dtype, const AttnArgs& a, bool causal, bool bias, int64_t batch, int64_t heads, int64_t L, hipStream_t s) {
    return dtype == TVK_F16 ? fwd<TVK_F16>(a, causal, bias, batch, heads, L, s)
                            : fwd<TVK_BF16>(a, causal, bias, batch, heads, L, s);
}

bool attn_part_bwd(int dtype, const AttnBwdArgs& a, bool causal, bool bias, int64_t batch, int64_t heads, int64_t L, int64_t S,
                   hipStream_t s) {
    return dtype == TVK_F16 ? bwd<TVK_F16>(a, causal, bias, batch, heads, L, S, s)
                            : bwd<TVK_BF16>(a, causal, bias, batch, heads, L, S, s);
}

}  // namespace tvk
