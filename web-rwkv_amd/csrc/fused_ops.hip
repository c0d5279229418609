// Fused forms of the small ops of an RWKV-v6 layer (src/runtime/v6.rs:758-955).  At batch 1 every
// op of a layer is bound by its launch (about 2.3 us under HIP-graph replay, 27 of them per layer
// beside the 8 quantized products); these entry points do the work of 3 - 5 consecutive ops of the
// reference's list in one launch each and bring a layer from 35 launches to 12.  Each computes what the
// op list computes, with the same roundings where the list stores an f16 buffer in between:
//   wrq_v6_pre          (add) + blit + layer_norm + token_shift x 1..2     v6.rs:759-777, :906-933
//   (wrq_fused_pre: the same with up to 6 shifts, for the layers of v7, src/runtime/v7.rs:705-760)
//   wrq_v6_time_mix     transpose + time_mix_w2 + add + token_shift(5)     v6.rs:785-805
//   wrq_v6_decay        time_decay_w2 + add + activate(StableExp)          v6.rs:839-848
//   wrq_v6_wkv_gate     blit + time_mix_v6 + group_norm + blit + mul(Silu) v6.rs:851-887
//   wrq_v6_post_ffn     channel_mix + add (+ affine 0.5)                   v6.rs:942-955
// They have no counterpart among the reference's constructors; buffers are the f16 / f32 tensors of
// `Runtime<f16>` (v6.rs:270-303), contiguous, [C, A, 1, 1].
#include "recurrence.h"

namespace wrq {

namespace {

constexpr int kPreThreads = 256;
constexpr int kPreCache = 8; // 4-element vectors a thread keeps of a row at most: rows up to 8192 elements
constexpr int kPreShifts = 6;
// Runs from here on take the adapters in 16-token tiles: at 8 tokens both forms cost the same (768 channels: time_mix 3.31 against
// 3.35 us, 5120: 3.36 against 3.45), at 16 the tiles win where rows are long (5120 channels: 3.60 against 4.62 us), below they are half empty.
constexpr uint32_t kTileTokens = 8;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

struct ShiftArgs {
    const uint16_t *factor[kPreShifts];
    uint16_t *out[kPreShifts];
};

// One workgroup per token.  row = x[t] (+ add[t]), written to x_out when given; ln = f16(LN(row)) -> ln_out;
// out[s][t] = f16(mix(ln, prev, factor[s])) with prev = the request's state row for its first
// token of the stack, else f16(LN(row t-1)) recomputed here.  NC vectors of a row per thread (the smallest of 1, 2, 4, 8
// that holds it): the six factors of a v7 layer then cost no registers for vectors that a row does not have.
template <int NS, int NC>
__global__ __launch_bounds__(kPreThreads) void pre_kernel(const uint32_t *cursors, const uint16_t *x, const uint16_t *add, uint16_t *x_out,
                                                          const uint16_t *ln_w, const uint16_t *ln_b, float eps, uint32_t C, const float *state, ViewArgs vs,
                                                          uint16_t *ln_out, ShiftArgs sh) {
    __shared__ float red[kPreThreads / 64];
    const uint32_t t = blockIdx.x, nv = C / 4;
    // Everything that does not depend on the row statistics is requested first: a workgroup is a chain of
    // dependent memory round trips otherwise (cursor, row, weights after the reductions, state, factors),
    // and at one token per launch that chain is the kernel's whole time.
    uint2 wq[NC], bq[NC], fq[NS][NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const uint32_t i = threadIdx.x + c * kPreThreads;
        if (i < nv) {
            wq[c] = *reinterpret_cast<const uint2 *>(ln_w + 4 * i);
            bq[c] = *reinterpret_cast<const uint2 *>(ln_b + 4 * i);
#pragma unroll
            for (int s = 0; s < NS; s++) fq[s][c] = *reinterpret_cast<const uint2 *>(sh.factor[s] + 4 * i);
        }
    }
    auto unpack = [](uint2 v) {
        return make_float4(h2f((uint16_t)(v.x & 0xffffu)), h2f((uint16_t)(v.x >> 16)), h2f((uint16_t)(v.y & 0xffffu)), h2f((uint16_t)(v.y >> 16)));
    };
    const Cursor cur = read_cursor(cursors, t, vs);
    const bool first = t == cur.token;
    float4 pst[NC]; // the request's state row, for its first token of the stack
    if (first) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const uint32_t i = threadIdx.x + c * kPreThreads;
            if (i < nv) pst[c] = load_vec4(state + view_elem(vs, cur.batch, 0, 4 * i));
        }
    }
    // rows t (which = 0) and t - 1 (which = 1): normalised, rounded to f16 as the op list stores them
    float4 ln[2][NC];
#pragma unroll
    for (int which = 0; which < 2; which++) {
        if (which == 1 && first) break;
        const uint64_t base = (uint64_t)(t - which) * C;
        float4 row[NC];
        float part = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const uint32_t i = threadIdx.x + c * kPreThreads;
            if (i < nv) {
                float4 v = load_vec4(x + base + 4 * i);
                if (add) {
                    const float4 a = load_vec4(add + base + 4 * i);
                    v = make_float4(round_h(a.x + v.x), round_h(a.y + v.y), round_h(a.z + v.z), round_h(a.w + v.w));
                    if (which == 0) store_vec4(x_out + base + 4 * i, v);
                }
                row[c] = v;
                part += (v.x + v.y) + (v.z + v.w);
            }
        }
        const float mean = block_reduce<false, kPreThreads>(part, red) / (float)C;
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; c++)
            if (threadIdx.x + c * kPreThreads < nv) {
                const float4 v = row[c];
                acc += ((v.x - mean) * (v.x - mean) + (v.y - mean) * (v.y - mean)) + ((v.z - mean) * (v.z - mean) + (v.w - mean) * (v.w - mean));
            }
        const float dev = rsqrtf(block_reduce<false, kPreThreads>(acc, red) / (float)C + eps);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const uint32_t i = threadIdx.x + c * kPreThreads;
            if (i < nv) {
                const float4 v = row[c], w = unpack(wq[c]), b = unpack(bq[c]);
                ln[which][c] = make_float4(round_h(fmaf((v.x - mean) * dev, w.x, b.x)), round_h(fmaf((v.y - mean) * dev, w.y, b.y)),
                                           round_h(fmaf((v.z - mean) * dev, w.z, b.z)), round_h(fmaf((v.w - mean) * dev, w.w, b.w)));
                if (which == 0) store_vec4(ln_out + base + 4 * i, ln[0][c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const uint32_t i = threadIdx.x + c * kPreThreads;
        if (i >= nv) continue;
        const float4 p = first ? pst[c] : ln[1][c];
        const float4 a = ln[0][c];
        auto mix = [](float xx, float pp, float f) { return xx * (1.0f - f) + pp * f; }; // reversed token shift: mix(x, prev, f)
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float4 f = unpack(fq[s][c]);
            store_vec4(sh.out[s] + (uint64_t)t * C + 4 * i, make_float4(mix(a.x, p.x, f.x), mix(a.y, p.y, f.y), mix(a.z, p.z, f.z), mix(a.w, p.w, f.w)));
        }
    }
}

// thread = (token, channel c): f[s] = f16(f16(sum_k w2[s][c][k] lora[t][s][k]) + time_mix[s][c]),
// out[s][t][c] = f16(mix(att_x[t][c], prev[c], f[s])), s = 0..4
template <int KL>
__global__ __launch_bounds__(256) void v6_time_mix_kernel(const uint32_t *cursors, const uint16_t *lora, const uint16_t *w2, const uint16_t *time_mix,
                                                          const float *state, ViewArgs vs, const uint16_t *att_x, uint16_t *out, uint32_t C, uint32_t A) {
    __shared__ __align__(16) uint16_t ls[5 * KL];
    const uint32_t t = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    const uint32_t cc = min(c, C - 1); // threads past the row repeat its last channel and store nothing
    // every operand is requested before the first wait: the rows of w2, the mix vectors, the token and the
    // one before it (the state row needs the cursor: one more round trip, for a request's first token only)
    uint4 wv[5][KL / 8];
    float tm[5];
#pragma unroll
    for (int s = 0; s < 5; s++) {
        const uint16_t *wrow = w2 + ((uint64_t)s * C + cc) * KL;
#pragma unroll
        for (int k8 = 0; k8 < KL / 8; k8++) wv[s][k8] = load128(wrow + 8 * k8);
        tm[s] = h2f(time_mix[(uint64_t)s * C + cc]);
    }
    const Cursor cur = read_cursor(cursors, t, vs);
    const float a = h2f(att_x[(uint64_t)t * C + cc]);
    const float before = h2f(att_x[(uint64_t)(t ? t - 1 : 0) * C + cc]);
    for (uint32_t e = threadIdx.x; e < 5 * KL / 8; e += 256) *reinterpret_cast<uint4 *>(&ls[8 * e]) = load128(lora + (uint64_t)t * 5 * KL + 8 * e);
    const float p = t == cur.token ? state[view_elem(vs, cur.batch, 0, cc)] : before;
    lds_barrier();
    if (c >= C) return;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int s = 0; s < 5; s++) {
        float acc = 0.0f;
#pragma unroll
        for (int k8 = 0; k8 < KL / 8; k8++) {
            const uint4 xv = *reinterpret_cast<const uint4 *>(&ls[s * KL + 8 * k8]);
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[s][k8].x), __builtin_bit_cast(h2, xv.x), acc, false);
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[s][k8].y), __builtin_bit_cast(h2, xv.y), acc, false);
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[s][k8].z), __builtin_bit_cast(h2, xv.z), acc, false);
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[s][k8].w), __builtin_bit_cast(h2, xv.w), acc, false);
        }
        const float f = round_h(round_h(acc) + tm[s]);
        out[((uint64_t)s * A + t) * C + c] = f2h(a * (1.0f - f) + p * f);
    }
}

// The same for runs of kTileTokens and more, as 16 x 16 tiles on the matrix cores: a wave takes 16 channels of 16 tokens, and a
// lane ends up with 4 channels of one token of each of the five products.  The rows of w2 are read once per 16 tokens instead of
// once per token; every operand is requested before the first use.
// 5120 channels, 100 / 255 tokens: 12.7 -> 6.1 / 28.2 -> 10.6 us (the decay below: 9.1 -> 3.5 / 20.2 -> 5.3 us); 2048 channels, 100
// tokens: 7.2 -> 3.7 (5.4 -> 2.4).
template <int KL>
__global__ __launch_bounds__(256) void v6_time_mix_tile_kernel(const uint32_t *cursors, const uint16_t *lora, const uint16_t *w2, const uint16_t *time_mix,
                                                               const float *state, ViewArgs vs, const uint16_t *att_x, uint16_t *out, uint32_t C, uint32_t A) {
    constexpr int NK = KL / 32;
    const uint32_t lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t c0 = 64 * blockIdx.x + 16 * (threadIdx.x >> 6), t = min(16 * blockIdx.y + r16, A - 1); // columns past the run repeat its last token
    if (c0 >= C) return;
    const uint32_t ch = c0 + 4 * g; // the lane's channels after the product
    uint4 wa[5][NK], xb[5][NK];
    float4 tm[5];
#pragma unroll
    for (int s = 0; s < 5; s++) {
#pragma unroll
        for (int k = 0; k < NK; k++) {
            wa[s][k] = load128(w2 + ((uint64_t)s * C + c0 + r16) * KL + 32 * k + 8 * g);
            xb[s][k] = load128(lora + ((uint64_t)t * 5 + s) * KL + 32 * k + 8 * g);
        }
        tm[s] = load_vec4(time_mix + (uint64_t)s * C + ch);
    }
    const Cursor cur = read_cursor(cursors, t, vs);
    const float4 a = load_vec4(att_x + (uint64_t)t * C + ch);
    float4 p = load_vec4(att_x + (uint64_t)(t ? t - 1 : 0) * C + ch);
    if (t == cur.token) p = load_vec4(state + view_elem(vs, cur.batch, 0, ch));
    auto mix = [](float y, float m, float x, float prev) {
        const float f = round_h(round_h(y) + m);
        return x * (1.0f - f) + prev * f;
    };
#pragma unroll
    for (int s = 0; s < 5; s++) {
        float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NK; k++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wa[s][k]), __builtin_bit_cast(half8, xb[s][k]), acc, 0, 0, 0);
        if (16 * blockIdx.y + r16 < A)
            store_vec4(out + ((uint64_t)s * A + t) * C + ch, make_float4(mix(acc[0], tm[s].x, a.x, p.x), mix(acc[1], tm[s].y, a.y, p.y),
                                                                         mix(acc[2], tm[s].z, a.z, p.z), mix(acc[3], tm[s].w, a.w, p.w)));
    }
}

// thread = (token, channel c): out[t][c] = exp(-exp(sum_k w2[c][k] lora[t][k] + time_decay[c])) in f32
template <int KL>
__global__ __launch_bounds__(256) void v6_decay_kernel(const uint16_t *lora, const uint16_t *w2, const uint16_t *time_decay, float *out, uint32_t C) {
    __shared__ __align__(16) uint16_t ls[KL];
    const uint32_t t = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    const uint32_t cc = min(c, C - 1); // threads past the row repeat its last channel and store nothing
    // the row of w2 and the bias are requested together with the token's vector, before the first wait
    const uint16_t *wrow = w2 + (uint64_t)cc * KL;
    uint4 wv[KL / 8];
#pragma unroll
    for (int k8 = 0; k8 < KL / 8; k8++) wv[k8] = load128(wrow + 8 * k8);
    const float bias = h2f(time_decay[cc]);
    for (uint32_t e = threadIdx.x; e < KL / 8; e += 256) *reinterpret_cast<uint4 *>(&ls[8 * e]) = load128(lora + (uint64_t)t * KL + 8 * e);
    lds_barrier();
    if (c >= C) return;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    float acc = 0.0f;
#pragma unroll
    for (int k8 = 0; k8 < KL / 8; k8++) {
        const uint4 xv = *reinterpret_cast<const uint4 *>(&ls[8 * k8]);
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[k8].x), __builtin_bit_cast(h2, xv.x), acc, false);
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[k8].y), __builtin_bit_cast(h2, xv.y), acc, false);
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[k8].z), __builtin_bit_cast(h2, xv.z), acc, false);
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, wv[k8].w), __builtin_bit_cast(h2, xv.w), acc, false);
    }
    out[(uint64_t)t * C + c] = act_one<WRQ_ACT_STABLE_EXP>(bias + acc);
}

// The same in 16 x 16 tiles, as v6_time_mix_tile_kernel.
template <int KL>
__global__ __launch_bounds__(256) void v6_decay_tile_kernel(const uint16_t *lora, const uint16_t *w2, const uint16_t *time_decay, float *out, uint32_t C, uint32_t A) {
    constexpr int NK = KL / 32;
    const uint32_t lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t c0 = 64 * blockIdx.x + 16 * (threadIdx.x >> 6), t = min(16 * blockIdx.y + r16, A - 1);
    if (c0 >= C) return;
    const uint32_t ch = c0 + 4 * g;
    uint4 wa[NK], xb[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        wa[k] = load128(w2 + (uint64_t)(c0 + r16) * KL + 32 * k + 8 * g);
        xb[k] = load128(lora + (uint64_t)t * KL + 32 * k + 8 * g);
    }
    const float4 bias = load_vec4(time_decay + ch);
    float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NK; k++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wa[k]), __builtin_bit_cast(half8, xb[k]), acc, 0, 0, 0);
    auto f = [](float y, float b) { return act_one<WRQ_ACT_STABLE_EXP>(b + y); };
    if (16 * blockIdx.y + r16 < A) store_vec4(out + (uint64_t)t * C + ch, make_float4(f(acc[0], bias.x), f(acc[1], bias.y), f(acc[2], bias.z), f(acc[3], bias.w)));
}

// state[request] <- ffn_x at its last token; x_out = f16(f16(sigmoid(r) v) + x_in) (halved when `rescale`)
__global__ __launch_bounds__(256) void v6_post_ffn_kernel(const uint32_t *cursors, float *state, ViewArgs vs, const uint16_t *r, const uint16_t *v,
                                                          const uint16_t *ffn_x, const uint16_t *x_in, uint16_t *x_out, uint32_t C, int rescale) {
    const uint32_t at = blockIdx.x * 256 + threadIdx.x, index = min(at, C / 4 - 1), t = blockIdx.y;
    const uint64_t bti = (uint64_t)t * C + 4 * index;
    // all loads before the store into the state: the compiler cannot move them across it (the pointers may
    // alias), and behind it they would wait for the cursor's round trip first
    const float4 rr = load_vec4(r + bti), vv = load_vec4(v + bti), xx = load_vec4(x_in + bti), fx = load_vec4(ffn_x + bti);
    const uint32_t ahead = cursor_ahead(cursors, t, gridDim.y);
    const Cursor cur = read_cursor(cursors, t, vs);
    const bool keeps = keeps_row(cursors, t, gridDim.y, cur, vs, ahead);
    if (at >= C / 4) return; // lanes past the row took part in the search
    if (keeps) *reinterpret_cast<float4 *>(state + view_elem(vs, cur.batch, 0, 4 * index)) = fx;
    const float sc = rescale ? 0.5f : 1.0f;
    auto f = [&](float a, float b, float c) { return round_h(round_h(1.0f / (1.0f + expf(-a)) * b) + c) * sc; };
    store_vec4(x_out + bti, make_float4(f(rr.x, vv.x, xx.x), f(rr.y, vv.y, xx.y), f(rr.z, vv.z, xx.z), f(rr.w, vv.w, xx.w)));
}

// `most`: shifts of the entry point
int launch_pre(const char *what, int most, wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const void *x, const void *add, void *x_out, const void *ln_w,
                  const void *ln_b, float eps, const wrq_tensor_view *state, int shifts, const void *const *factors, void *ln_out, void *const *outs) {
    if (C == 0 || A == 0) return WRQ_OK;
    if (C % 4 || C > 4u * kPreThreads * kPreCache) return fail(WRQ_ERR_UNSUPPORTED, "%s: %u channels (a multiple of 4 up to %d is built)", what, C, 4 * kPreThreads * kPreCache);
    if ((shifts != 1 && shifts != 2 && shifts != 6) || shifts > most)
        return fail(WRQ_ERR_UNSUPPORTED, "%s: %d token shifts (%s)", what, shifts, most > 2 ? "1, 2 or 6" : "1 or 2");
    if (!factors || !outs) return fail(WRQ_ERR_NULL, "%s: null pointer", what);
    int s = check_state(state, C, state ? state->view.shape[1] : 0, what);
    for (const void *p : {cursors, x, ln_w, ln_b, (const void *)ln_out})
        if (s == WRQ_OK) s = check_ptr(p, what);
    ShiftArgs sh{};
    for (int i = 0; i < shifts && s == WRQ_OK; i++) {
        sh.factor[i] = static_cast<const uint16_t *>(factors[i]), sh.out[i] = static_cast<uint16_t *>(outs[i]);
        s = check_ptr(factors[i], what);
        if (s == WRQ_OK) s = check_ptr(outs[i], what);
    }
    if (s == WRQ_OK && add) s = check_ptr(x_out, what);
    if (s != WRQ_OK) return s;
    // workgroup t rebuilds row t - 1 from x and add while workgroup t - 1 stores its rows: what is stored may overlap neither
    // (a single token has no neighbour: it may be normalised in place)
    auto overlaps_input = [&](const void *out) {
        const uintptr_t lo = (uintptr_t)out, bytes = (uintptr_t)A * C * 2;
        for (const void *src : {x, add})
            if (src && lo < (uintptr_t)src + bytes && (uintptr_t)src < lo + bytes) return true;
        return false;
    };
    if (add && overlaps_input(x_out))
        return fail(WRQ_ERR_UNSUPPORTED, "%s: the sum must go to a buffer that overlaps neither input (a token's workgroup reads its neighbour's row)", what);
    bool overlap = overlaps_input(ln_out);
    for (int i = 0; i < shifts; i++) overlap = overlap || overlaps_input(outs[i]);
    if (A > 1 && overlap)
        return fail(WRQ_ERR_UNSUPPORTED, "%s: the outputs must go to buffers that overlap no input (a token's workgroup reads its neighbour's row)", what);
    const ViewArgs vs = view_args(state->view);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    auto o16 = [](void *p) { return static_cast<uint16_t *>(p); };
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(A), dim3(kPreThreads), 0, static_cast<hipStream_t>(stream), static_cast<const uint32_t *>(cursors), u16(x), u16(add),
                           o16(x_out), u16(ln_w), u16(ln_b), eps, C, static_cast<const float *>(state->data), vs, o16(ln_out), sh);
    };
    const uint32_t nc = (C / 4 + kPreThreads - 1) / kPreThreads;
#define WRQ_PRE(NS) (nc <= 1 ? go(pre_kernel<NS, 1>) : nc <= 2 ? go(pre_kernel<NS, 2>) : nc <= 4 ? go(pre_kernel<NS, 4>) : go(pre_kernel<NS, 8>))
    shifts == 1 ? WRQ_PRE(1) : shifts == 2 ? WRQ_PRE(2) : WRQ_PRE(6);
#undef WRQ_PRE
    return check_launch(what);
}

} // namespace

} // namespace wrq

using namespace wrq;

extern "C" {

int wrq_fused_pre(wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const void *x, const void *add, void *x_out, const void *ln_w,
                  const void *ln_b, float eps, const wrq_tensor_view *state, int shifts, const void *const *factors, void *ln_out, void *const *outs) {
    return launch_pre("fused_pre", kPreShifts, stream, C, A, cursors, x, add, x_out, ln_w, ln_b, eps, state, shifts, factors, ln_out, outs);
}

int wrq_v6_pre(wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const void *x, const void *add, void *x_out, const void *ln_w,
               const void *ln_b, float eps, const wrq_tensor_view *state, int shifts, const void *factor0, const void *factor1, void *ln_out,
               void *shift0, void *shift1) {
    const void *const factors[2] = {factor0, factor1};
    void *const outs[2] = {shift0, shift1};
    return launch_pre("v6_pre", 2, stream, C, A, cursors, x, add, x_out, ln_w, ln_b, eps, state, shifts, factors, ln_out, outs);
}

int wrq_v6_time_mix(wrq_stream stream, uint32_t C, uint32_t A, uint32_t lora_size, const void *cursors, const void *lora, const void *w2, const void *time_mix,
                    const wrq_tensor_view *state, const void *att_x, void *att_sx) {
    const char *what = "v6_time_mix";
    if (C == 0 || A == 0) return WRQ_OK;
    if (lora_size != 32 && lora_size != 64) return fail(WRQ_ERR_UNSUPPORTED, "%s: adapter size %u (32 or 64 is built)", what, lora_size);
    if (A > 65535u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    int s = check_state(state, C, state ? state->view.shape[1] : 0, what);
    for (const void *p : {cursors, lora, w2, time_mix, att_x, (const void *)att_sx})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s != WRQ_OK) return s;
    const ViewArgs vs = view_args(state->view);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    auto go = [&](auto kern, const dim3 &grid) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, hs, static_cast<const uint32_t *>(cursors), u16(lora), u16(w2), u16(time_mix),
                           static_cast<const float *>(state->data), vs, u16(att_x), static_cast<uint16_t *>(att_sx), C, A);
    };
    if (A >= kTileTokens && C % 16 == 0) {
        const dim3 grid((C + 63) / 64, (A + 15) / 16);
        lora_size == 32 ? go(v6_time_mix_tile_kernel<32>, grid) : go(v6_time_mix_tile_kernel<64>, grid);
    } else {
        const dim3 grid((C + 255) / 256, A);
        lora_size == 32 ? go(v6_time_mix_kernel<32>, grid) : go(v6_time_mix_kernel<64>, grid);
    }
    return check_launch(what);
}

int wrq_v6_decay(wrq_stream stream, uint32_t C, uint32_t A, uint32_t lora_size, const void *lora, const void *w2, const void *time_decay, void *out) {
    const char *what = "v6_decay";
    if (C == 0 || A == 0) return WRQ_OK;
    if (lora_size != 64 && lora_size != 128) return fail(WRQ_ERR_UNSUPPORTED, "%s: adapter size %u (64 or 128 is built)", what, lora_size);
    if (A > 65535u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    int s = WRQ_OK;
    for (const void *p : {lora, w2, time_decay, (const void *)out})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s != WRQ_OK) return s;
    hipStream_t hs = static_cast<hipStream_t>(stream);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    if (A >= kTileTokens && C % 16 == 0) {
        const dim3 grid((C + 63) / 64, (A + 15) / 16);
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, hs, u16(lora), u16(w2), u16(time_decay), static_cast<float *>(out), C, A); };
        lora_size == 64 ? go(v6_decay_tile_kernel<64>) : go(v6_decay_tile_kernel<128>);
    } else {
        const dim3 grid((C + 255) / 256, A);
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, hs, u16(lora), u16(w2), u16(time_decay), static_cast<float *>(out), C); };
        lora_size == 64 ? go(v6_decay_kernel<64>) : go(v6_decay_kernel<128>);
    }
    return check_launch(what);
}

int wrq_v6_wkv_gate(wrq_stream stream, uint32_t S, uint32_t H, uint32_t A, const void *cursors, const void *time_decay, const void *time_first,
                    const wrq_tensor_view *state, const void *k, const void *v, const void *r, const void *g, const void *gn_w, const void *gn_b, float eps,
                    void *att_x) {
    const char *what = "v6_wkv_gate";
    if (H == 0 || A == 0) return WRQ_OK;
    if (S != 64) return fail(WRQ_ERR_UNSUPPORTED, "%s: head size %u (64 is built)", what, S);
    int s = check_state(state, S * H, S + 1, what);
    for (const void *p : {cursors, time_decay, time_first, k, v, r, g, gn_w, gn_b, (const void *)att_x})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s != WRQ_OK) return s;
    const ViewArgs vs = view_args(state->view);
    auto f32 = [](const void *p) { return static_cast<const float *>(p); };
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    const bool wide = wide_walk(vs, H, A);
    auto *kern = wide ? &time_mix_kernel<float, 64, true, true, true> : &time_mix_kernel<float, 64, true, true, false>;
    hipLaunchKernelGGL(kern, dim3(H, slot_grid(vs, A)), dim3(wide ? RecurrenceTile<64, true>::THREADS : RecurrenceTile<64>::THREADS), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint32_t *>(cursors), f32(time_decay), f32(time_first), static_cast<float *>(state->data), f32(k), f32(v), f32(r),
                       static_cast<float *>(nullptr), vs, H, A, GateArgs{u16(g), u16(gn_w), u16(gn_b), static_cast<uint16_t *>(att_x), eps});
    return check_launch(what);
}

int wrq_v6_post_ffn(wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const wrq_tensor_view *state, const void *r, const void *v, const void *ffn_x,
                    const void *x_in, void *x_out, int rescale) {
    const char *what = "v6_post_ffn";
    if (C == 0 || A == 0) return WRQ_OK;
    if (C % 4) return fail(WRQ_ERR_ALIGNMENT, "%s: row length %u not a multiple of 4", what, C);
    if (A > 65535u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    int s = check_state(state, C, 1, what);
    for (const void *p : {cursors, r, v, ffn_x, x_in, (const void *)x_out})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s != WRQ_OK) return s;
    const ViewArgs vs = view_args(state->view);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    hipLaunchKernelGGL(v6_post_ffn_kernel, dim3((C / 4 + 255) / 256, A), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const uint32_t *>(cursors),
                       static_cast<float *>(state->data), vs, u16(r), u16(v), u16(ffn_x), u16(x_in), static_cast<uint16_t *>(x_out), C, rescale);
    return check_launch(what);
}

} // extern "C"
