// Scaled dot-product attention entry points (tvk_attention_fwd,
// tvk_attention_bwd): validation, and the choice between the MFMA kernels
// (attention_kernels.h) and the general ones (attention_any.hip).
#include "attention_any.h"
#include "attention_kernels.h"

using namespace tvk;

namespace {

// Head dims of the MFMA kernels: whole 16-byte chunks up to 128 columns.
bool mfma_dims(const tvk_attention_desc* d) {
    return d->head_dim == d->head_dim_v && d->head_dim >= 8 && d->head_dim <= 128 && d->head_dim % 8 == 0;
}

// The MFMA forward (float16/bfloat16, 16-byte rows); TVK_ERR_UNSUPPORTED when the case is not one it takes.
tvk_status fused_fwd(const tvk_attention_desc* d) {
    if (d->dtype != TVK_F16 && d->dtype != TVK_BF16)
        return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: dtype must be float16 or bfloat16");
    if (d->batch < 0 || d->heads_q < 0 || d->heads_kv <= 0 || d->len_q < 0 || d->len_kv < 0)
        return fail(TVK_ERR_INVALID, "tvk_attention_fwd: negative size");
    if (d->heads_q % d->heads_kv != 0)
        return fail(TVK_ERR_INVALID, "tvk_attention_fwd: heads_q is not a multiple of heads_kv");
    if (!mfma_dims(d))
        return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: head_dim == head_dim_v, a multiple of 8 up to 128, only");
    if (d->len_q > ((int64_t)1 << 30) || d->len_kv > ((int64_t)1 << 30) ||
        d->batch * d->heads_q * ((d->len_q + 63) / 64) > (int64_t)0x7fffffff)
        return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: grid too large");
    if (d->batch == 0 || d->heads_q == 0 || d->len_q == 0) return TVK_OK;
    if (!d->q || !d->k || !d->v || !d->out || !d->lse) return fail(TVK_ERR_INVALID, "tvk_attention_fwd: NULL tensor");
    auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    for (const int64_t* st : {d->q_stride, d->k_stride, d->v_stride}) {
        if (st[3] != 1) return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: q, k, v need unit stride along the head dimension");
        for (int i = 0; i < 3; ++i)
            if (st[i] % 8 != 0) return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: q, k, v rows must be 16-byte aligned");
    }
    if (!al16(d->q) || !al16(d->k) || !al16(d->v)) return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: unaligned q, k or v");
    // a key tile's rows are addressed by 32-bit byte offsets from the tile's first row
    for (const int64_t row : {d->k_stride[2], d->v_stride[2]})
        if (row < 0 || (63 * row + d->head_dim) * 2 > (int64_t)0xffffffff)
            return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: k or v row stride too large");
    AttnArgs a{};
    a.q = static_cast<const uint16_t*>(d->q);
    a.k = static_cast<const uint16_t*>(d->k);
    a.v = static_cast<const uint16_t*>(d->v);
    a.bias = static_cast<const uint16_t*>(d->bias);
    a.out = static_cast<uint16_t*>(d->out);
    a.lse = d->lse;
    for (int i = 0; i < 4; ++i) {
        a.sq[i] = d->q_stride[i];
        a.sk[i] = d->k_stride[i];
        a.sv[i] = d->v_stride[i];
        a.sb[i] = d->bias ? d->bias_stride[i] : 0;
        a.so[i] = d->out_stride[i];
    }
    for (int i = 0; i < 3; ++i) a.sl[i] = d->lse_stride[i];
    a.L = (int)d->len_q;
    a.S = (int)d->len_kv;
    a.Hq = (int)d->heads_q;
    a.group = (int)(d->heads_q / d->heads_kv);
    a.hd = (int)d->head_dim;
    a.scale = (float)d->scale;
    a.c2 = std::fabs(a.scale) * AT_LOG2E;
    a.qflip = a.scale < 0.0f ? 0x80008000u : 0u;
    const bool causal = d->causal != 0;
    a.out_vec = d->out_stride[3] == 1 && (reinterpret_cast<uintptr_t>(d->out) & 7) == 0 && d->out_stride[2] % 4 == 0 &&
                d->out_stride[1] % 4 == 0 && d->out_stride[0] % 4 == 0;
    const hipStream_t s = resolve_stream(d->stream);
    const bool bias = d->bias != nullptr;
    if (attn_decode_applies(a, causal, bias, d->batch, d->heads_q)) {
        attn_decode_fwd(d->dtype, a, bias, d->batch, d->heads_q, s);
    } else if (d->head_dim != 64 && d->head_dim != 128) {
        if (!attn_part_fwd(d->dtype, a, causal, bias, d->batch, d->heads_q, d->len_q, s))
            return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: head dim");
    } else if (d->dtype == TVK_F16) {
        if (d->head_dim == 64) launch_attn<TVK_F16, 64, false>(a, causal, bias, d->batch, d->heads_q, d->len_q, s);
        else launch_attn<TVK_F16, 128, false>(a, causal, bias, d->batch, d->heads_q, d->len_q, s);
    } else {
        if (d->head_dim == 64) launch_attn<TVK_BF16, 64, false>(a, causal, bias, d->batch, d->heads_q, d->len_q, s);
        else launch_attn<TVK_BF16, 128, false>(a, causal, bias, d->batch, d->heads_q, d->len_q, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TVK_ERR_DEVICE, std::string("tvk_attention_fwd: launch failed: ") + hipGetErrorString(e));
    return TVK_OK;
}

tvk_status check_attention(const tvk_attention_desc* d, const char* who) {
    auto bad = [&](tvk_status st, const char* m) { return fail(st, std::string(who) + ": " + m); };
    if (d->dtype != TVK_F16 && d->dtype != TVK_BF16) return bad(TVK_ERR_UNSUPPORTED, "dtype must be float16 or bfloat16");
    if (d->batch < 0 || d->heads_q < 0 || d->heads_kv <= 0 || d->len_q < 0 || d->len_kv < 0) return bad(TVK_ERR_INVALID, "negative size");
    if (d->heads_q % d->heads_kv != 0) return bad(TVK_ERR_INVALID, "heads_q is not a multiple of heads_kv");
    if (!mfma_dims(d)) return bad(TVK_ERR_UNSUPPORTED, "head_dim == head_dim_v, a multiple of 8 up to 128, only");
    if (d->batch > 65535 || d->heads_q > 65535 || d->len_q > ((int64_t)1 << 30) || d->len_kv > ((int64_t)1 << 30) ||
        d->batch * d->heads_q * ((d->len_q + 63) / 64) > (int64_t)0x7fffffff)
        return bad(TVK_ERR_UNSUPPORTED, "grid too large");
    return TVK_OK;
}

bool rows_ok(const void* ptr, const int64_t* st) {
    if ((reinterpret_cast<uintptr_t>(ptr) & 15) != 0 || st[3] != 1) return false;
    for (int i = 0; i < 3; ++i)
        if (st[i] % 8 != 0) return false;
    return true;
}

// The MFMA backward passes; TVK_ERR_UNSUPPORTED when the case is not one they take.
tvk_status fused_bwd(const tvk_attention_bwd_desc* desc) {
    const tvk_attention_desc* d = &desc->fwd;
    tvk_status st = check_attention(d, "tvk_attention_bwd");
    if (st != TVK_OK) return st;
    if (d->batch == 0 || d->heads_q == 0 || (d->len_q == 0 && d->len_kv == 0)) return TVK_OK;
    if (!d->q || !d->k || !d->v || !d->out || !d->lse || !desc->dout || !desc->dq || !desc->dk || !desc->dv)
        return fail(TVK_ERR_INVALID, "tvk_attention_bwd: NULL tensor");
    if (!rows_ok(d->q, d->q_stride) || !rows_ok(d->k, d->k_stride) || !rows_ok(d->v, d->v_stride) ||
        !rows_ok(desc->dout, desc->dout_stride) || !rows_ok(desc->dq, desc->dq_stride) ||
        !rows_ok(desc->dk, desc->dk_stride) || !rows_ok(desc->dv, desc->dv_stride))
        return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_bwd: q, k, v, dout, dq, dk, dv need unit stride along the head dimension and 16-byte aligned rows");
    AttnBwdArgs a{};
    a.q = static_cast<const uint16_t*>(d->q);
    a.k = static_cast<const uint16_t*>(d->k);
    a.v = static_cast<const uint16_t*>(d->v);
    a.bias = static_cast<const uint16_t*>(d->bias);
    a.out = static_cast<const uint16_t*>(d->out);
    a.dout = static_cast<const uint16_t*>(desc->dout);
    a.lse = d->lse;
    a.dq = static_cast<uint16_t*>(desc->dq);
    a.dk = static_cast<uint16_t*>(desc->dk);
    a.dv = static_cast<uint16_t*>(desc->dv);
    for (int i = 0; i < 4; ++i) {
        a.sq[i] = d->q_stride[i];
        a.sk[i] = d->k_stride[i];
        a.sv[i] = d->v_stride[i];
        a.sb[i] = d->bias ? d->bias_stride[i] : 0;
        a.so[i] = d->out_stride[i];
        a.sdo[i] = desc->dout_stride[i];
        a.sdq[i] = desc->dq_stride[i];
        a.sdk[i] = desc->dk_stride[i];
        a.sdv[i] = desc->dv_stride[i];
    }
    for (int i = 0; i < 3; ++i) a.sl[i] = d->lse_stride[i];
    a.L = (int)d->len_q;
    a.S = (int)d->len_kv;
    a.Hq = (int)d->heads_q;
    a.group = (int)(d->heads_q / d->heads_kv);
    a.hd = (int)d->head_dim;
    a.scale = (float)d->scale;
    a.c2 = a.scale * AT_LOG2E;
    a.o_vec = rows_ok(d->out, d->out_stride) ? 1 : 0;
    const hipStream_t s = resolve_stream(d->stream);
    Scratch scratch;
    a.delta = static_cast<float*>(scratch.get((size_t)std::max<int64_t>(1, d->batch * d->heads_q * d->len_q) * 4, s));
    if (!a.delta) return fail(TVK_ERR_OOM, "tvk_attention_bwd: workspace allocation failed");
    const bool bias = d->bias != nullptr;
    if (d->head_dim != 64 && d->head_dim != 128) {
        if (!attn_part_bwd(d->dtype, a, d->causal != 0, bias, d->batch, d->heads_q, d->len_q, d->len_kv, s))
            return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_bwd: head dim");
    } else if (d->dtype == TVK_F16) {
        if (d->head_dim == 64) launch_attn_bwd<TVK_F16, 64, false>(a, d->causal != 0, bias, d->batch, d->heads_q, d->len_q, d->len_kv, s);
        else launch_attn_bwd<TVK_F16, 128, false>(a, d->causal != 0, bias, d->batch, d->heads_q, d->len_q, d->len_kv, s);
    } else {
        if (d->head_dim == 64) launch_attn_bwd<TVK_BF16, 64, false>(a, d->causal != 0, bias, d->batch, d->heads_q, d->len_q, d->len_kv, s);
        else launch_attn_bwd<TVK_BF16, 128, false>(a, d->causal != 0, bias, d->batch, d->heads_q, d->len_q, d->len_kv, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TVK_ERR_DEVICE, std::string("tvk_attention_bwd: launch failed: ") + hipGetErrorString(e));
    return TVK_OK;
}

// Validation shared by both directions: every case that passes runs on the
// device, in the MFMA kernels when they take it, else in the general kernels
// of attention_any.hip.
tvk_status check_any(const tvk_attention_desc* d, const char* who) {
    auto bad = [&](tvk_status st, const std::string& m) { return fail(st, std::string(who) + ": " + m); };
    if (d->dtype != TVK_F32 && d->dtype != TVK_F16 && d->dtype != TVK_BF16)
        return bad(TVK_ERR_UNSUPPORTED, "dtype must be float32, float16 or bfloat16");
    if (d->batch < 0 || d->heads_q < 0 || d->heads_kv <= 0 || d->len_q < 0 || d->len_kv < 0 || d->head_dim < 0 ||
        d->head_dim_v < 0)
        return bad(TVK_ERR_INVALID, "negative size");
    if (d->heads_q % d->heads_kv != 0) return bad(TVK_ERR_INVALID, "heads_q is not a multiple of heads_kv");
    if (!attn_any_applies(d))
        return bad(TVK_ERR_UNSUPPORTED, "head dims above 512, or batch or heads above 65535, or sequences above 2^30");
    return TVK_OK;
}

}  // namespace

extern "C" tvk_status tvk_attention_fwd(const tvk_attention_desc* d) {
    if (!d) return fail(TVK_ERR_INVALID, "tvk_attention_fwd: desc is NULL");
    tvk_status st = check_any(d, "tvk_attention_fwd");
    if (st != TVK_OK) return st;
    if (d->batch == 0 || d->heads_q == 0 || d->len_q == 0) return TVK_OK;
    if (!d->q || !d->k || !d->v || !d->out || !d->lse) return fail(TVK_ERR_INVALID, "tvk_attention_fwd: NULL tensor");
    if (d->head_dim == 0 && d->len_kv > 0) return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_fwd: empty head dim");
    st = fused_fwd(d);
    if (st != TVK_ERR_UNSUPPORTED) return st;
    clear_error();
    return attn_any_fwd(d, resolve_stream(d->stream));
}

extern "C" tvk_status tvk_attention_bwd(const tvk_attention_bwd_desc* desc) {
    if (!desc) return fail(TVK_ERR_INVALID, "tvk_attention_bwd: desc is NULL");
    const tvk_attention_desc* d = &desc->fwd;
    tvk_status st = check_any(d, "tvk_attention_bwd");
    if (st != TVK_OK) return st;
    if (d->batch == 0 || d->heads_q == 0 || (d->len_q == 0 && d->len_kv == 0)) return TVK_OK;
    if (!d->q || !d->k || !d->v || !d->out || !d->lse || !desc->dout || !desc->dq || !desc->dk || !desc->dv)
        return fail(TVK_ERR_INVALID, "tvk_attention_bwd: NULL tensor");
    if (d->head_dim == 0 || d->head_dim_v == 0) return fail(TVK_ERR_UNSUPPORTED, "tvk_attention_bwd: empty head dim");
    if (!desc->dscores) {
        st = fused_bwd(desc);
        if (st != TVK_ERR_UNSUPPORTED) return st;
        clear_error();
    }
    const hipStream_t s = resolve_stream(d->stream);
    Scratch scratch;
    float* delta = static_cast<float*>(scratch.get((size_t)std::max<int64_t>(1, d->batch * d->heads_q * d->len_q) * 4, s));
    if (!delta) return fail(TVK_ERR_OOM, "tvk_attention_bwd: workspace allocation failed");
    return attn_any_bwd(desc, delta, s);
}
