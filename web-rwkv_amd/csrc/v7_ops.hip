// The ops an RWKV-v7 layer adds to the ones of v5 / v6:
//   l2_norm          src/tensor/ops.rs:642-700,   src/shaders/normalize.wgsl:118-152
//   control_k_v7     src/tensor/ops.rs:1800-1858, src/shaders/control_k_v7.wgsl
//   time_mix_v7      src/tensor/ops.rs:1679-1741, src/shaders/time_mix_v7.wgsl:137-212
//   time_first_v7    src/tensor/ops.rs:1743-1798, src/shaders/time_mix_v7.wgsl:214-255
//   channel_mix_v7   src/tensor/ops.rs:1917-1970, src/shaders/channel_mix.wgsl (V7)
//
// time_mix_v7 is, per head and token, with S[j][i] the head's state, a = -kk, b = kk * a_in and
// w = exp(-exp(-0.5) sigmoid(w_in)):
//   sa[i] = sum_j S[j][i] a[j];   S[j][i] <- S[j][i] w[j] + k[j] v[i] + sa[i] b[j];   y[i] = sum_j r[j] S[j][i]
// The shader walks the state in memory twice per token; recurrence.h keeps it in registers over all tokens of
// a request in the run.
//
// Fused forms of the layer's small ops (src/runtime/v7.rs:704-1006), which are bound by their launches at the run
// lengths of a serving schedule: wrq_adapters_in, wrq_v7_mid, wrq_v7_wkv_gate, wrq_v7_post_ffn (with wrq_fused_pre of
// fused_ops.hip).  A layer takes 10 launches beside the second ones of split products instead of 42.
#include "recurrence.h"

namespace wrq {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kMaxAdapters = 4;
struct AdapterArgs {
    const uint16_t *w[kMaxAdapters], *x[kMaxAdapters];
    uint16_t *out[kMaxAdapters];
    uint32_t rank[kMaxAdapters], tile_begin[kMaxAdapters + 1]; // 16-row tiles of all adapters, one adapter after the other
    int act[kMaxAdapters];
};

// First halves of a layer's low-rank adapters, out[t][r] = f16(act(sum_k w[r][k] x[t][k])): a few dozen rows over K = C
// per adapter, so the product is one short pass over weights that fit in the caches and its time is latency.  One workgroup
// per 16 rows x 16 tokens of any adapter of the layer; its WAVES waves take the steps of 128 elements of K in turn, Q steps in flight,
// and add up through LDS.  LINES: a step comes line-wise from memory (the 256 bytes of a row in 16 adjacent lanes) and gets
// into the operand layout of the 16x16x32 MFMA through LDS of the wave's own; gathered straight into that layout a load touches 16 rows and costs
// the address units three times as much.  Without LINES (K no multiple of 128) steps are 32 elements, gathered.
template <int WAVES, int Q, bool LINES>
__global__ __launch_bounds__(64 * WAVES) void adapters_in_kernel(uint32_t K, uint32_t T, AdapterArgs aa) {
    constexpr int PITCH = 256 + 16; // bytes per staged row: +16 B rotates the banks
    __shared__ __align__(16) uint8_t slots[LINES ? WAVES : 1][LINES ? 32 * PITCH : 16];
    __shared__ float4 red[WAVES - 1][64];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
    uint32_t p = 0;
#pragma unroll
    for (uint32_t i = 1; i < kMaxAdapters; i++)
        if (blockIdx.x >= aa.tile_begin[i]) p = i;
    const uint32_t row0 = 16 * (blockIdx.x - aa.tile_begin[p]), t0 = 16 * blockIdx.y;
    // columns past the run repeat its last token, never stored
    float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
    if constexpr (LINES) {
        const uint32_t steps = K / 128, at = lane / 16, piece = 8 * (lane % 16);
        const uint16_t *wp = aa.w[p] + (uint64_t)(row0 + at) * K + piece, *xp[4];
#pragma unroll
        for (int i = 0; i < 4; i++) xp[i] = aa.x[p] + (uint64_t)min(t0 + 4 * i + at, T - 1) * K + piece;
        uint8_t *const put = slots[wave] + at * PITCH + 2 * piece;
        const uint8_t *const get = slots[wave] + r16 * PITCH + 16 * g;
        for (uint32_t s0 = wave; s0 < steps; s0 += Q * WAVES) {
            uint4 a[Q][4], b[Q][4];
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t k = 128 * min(s0 + q * WAVES, steps - 1);
                    a[q][i] = load128(wp + (uint64_t)(4 * i) * K + k), b[q][i] = load128(xp[i] + k);
                }
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if (s0 + q * WAVES >= steps) break;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    *reinterpret_cast<uint4 *>(put + 4 * i * PITCH) = a[q][i];
                    *reinterpret_cast<uint4 *>(put + (16 + 4 * i) * PITCH) = b[q][i];
                }
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const half8 *>(get + 64 * j), *reinterpret_cast<const half8 *>(get + 16 * PITCH + 64 * j), acc, 0, 0, 0);
            }
        }
    } else {
        const uint32_t steps = K / 32;
        const uint16_t *wp = aa.w[p] + (uint64_t)(row0 + r16) * K + 8 * g, *xp = aa.x[p] + (uint64_t)min(t0 + r16, T - 1) * K + 8 * g;
        for (uint32_t s0 = wave; s0 < steps; s0 += Q * WAVES) {
            uint4 a[Q], b[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const uint32_t at = 32 * min(s0 + q * WAVES, steps - 1);
                a[q] = load128(wp + at), b[q] = load128(xp + at);
            }
#pragma unroll
            for (int q = 0; q < Q; q++)
                if (s0 + q * WAVES < steps) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a[q]), __builtin_bit_cast(half8, b[q]), acc, 0, 0, 0);
        }
    }
    if (wave) red[wave - 1][lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (int w = 0; w < WAVES - 1; w++) {
        const float4 v = red[w][lane];
        acc[0] += v.x, acc[1] += v.y, acc[2] += v.z, acc[3] += v.w;
    }
    // lane: token r16 of the tile, rows 4 g .. 4 g + 3
    if (t0 + r16 < T) {
        const int act = aa.act[p];
        store_vec4(aa.out[p] + (uint64_t)(t0 + r16) * aa.rank[p] + row0 + 4 * g,
                   make_float4(act_apply(act, acc[0]), act_apply(act, acc[1]), act_apply(act, acc[2]), act_apply(act, acc[3])));
    }
}

struct MidArgs {
    const uint16_t *aux_w, *aux_a, *aux_g, *aux_v;                 // [T, rank]
    const uint16_t *w2, *a2, *g2, *v2;                             // [C, rank]
    const uint16_t *w0, *a0, *v0, *k_k, *k_a;                      // [C]
    const uint16_t *k, *v;                                         // [T, C]
    uint16_t *att_v0, *att_w, *att_g, *n;                          // [T, C], n: [4, T, C]
    uint16_t *att_k, *att_v, *att_a, *att_kk, *att_vv;             // [T, C] or null: the list's buffers; att_k and att_v may be k and v
};

// Second halves of the four adapters and what a v7 layer makes of them before the recurrence.  A workgroup takes one head
// (64 channels, 16 per wave) and 16 tokens: nine MFMAs of 32 inner elements per wave, then every lane holds 4 channels of
// one token and finishes them in registers with the roundings to f16 the op list has:
//   w = w0 + w2 aux_w;   a = sigmoid(a0 + a2 aux_a);   g = g2 aux_g;   v <- mix(v, v0, sigmoid(v_0 + v2 aux_v)) (FIRST: v0 <- v);
//   kk = l2_norm(k k_k) over the head;   k <- k (1 + (a - 1) k_a);   n = (k, v, a, kk)
// (src/runtime/v7.rs:780-880).  2048 channels, 32 tokens: 5.0 us (5.6 with the list's buffers) against about 60 us for the 16 launches of the list; bound by one
// round trip to memory, which is why every operand is requested before the first use.
template <int RW, int RA, int RG, int RV, bool FIRST>
__global__ __launch_bounds__(256) void v7_mid_kernel(uint32_t C, uint32_t T, float eps, MidArgs m) {
    __shared__ float part[4][16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const uint32_t t0 = 16 * blockIdx.y, t = min(t0 + r16, T - 1);
    const uint32_t c0 = 64 * blockIdx.x + 16 * wave; // the wave's 16 channels; this lane finishes c0 + 4 g ..
    constexpr int NW = RW / 32, NA = RA / 32, NG = RG / 32, NV = FIRST ? 0 : RV / 32;
    uint4 wa[NW + NA + NG + NV + 1], xb[NW + NA + NG + NV + 1];
    auto fetch = [&](auto rank, const uint16_t *w, const uint16_t *x, int at) {
        constexpr int R = decltype(rank)::value;
#pragma unroll
        for (int s = 0; s < R / 32; s++) {
            wa[at + s] = load128(w + (uint64_t)(c0 + r16) * R + 32 * s + 8 * g);
            xb[at + s] = load128(x + (uint64_t)t * R + 32 * s + 8 * g);
        }
    };
    fetch(std::integral_constant<int, RW>{}, m.w2, m.aux_w, 0);
    fetch(std::integral_constant<int, RA>{}, m.a2, m.aux_a, NW);
    fetch(std::integral_constant<int, RG>{}, m.g2, m.aux_g, NW + NA);
    if constexpr (!FIRST) fetch(std::integral_constant<int, RV>{}, m.v2, m.aux_v, NW + NA + NG);
    const uint32_t ch = c0 + 4 * g;
    const uint64_t at = (uint64_t)t * C + ch, plane = (uint64_t)T * C;
    const float4 w0 = load_vec4(m.w0 + ch), a0 = load_vec4(m.a0 + ch), v0 = FIRST ? make_float4(0.f, 0.f, 0.f, 0.f) : load_vec4(m.v0 + ch), k_k = load_vec4(m.k_k + ch), k_a = load_vec4(m.k_a + ch);
    const float4 k = load_vec4(m.k + at), v = load_vec4(m.v + at);
    const float4 first = FIRST ? v : load_vec4(m.att_v0 + at);
    auto product = [&](int from, int count) {
        float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < count; s++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wa[from + s]), __builtin_bit_cast(half8, xb[from + s]), acc, 0, 0, 0);
        return make_float4(round_h(acc[0]), round_h(acc[1]), round_h(acc[2]), round_h(acc[3]));
    };
    auto each = [](auto f, float4 a, float4 b, float4 c) { return make_float4(f(a.x, b.x, c.x), f(a.y, b.y, c.y), f(a.z, b.z, c.z), f(a.w, b.w, c.w)); };
    auto sigmoid_sum = [](float bias, float y, float) { return round_h(act_one<WRQ_ACT_SIGMOID>(bias + y)); };
    const float4 w = each([](float bias, float y, float) { return bias + y; }, w0, product(0, NW), w0);
    const float4 a = each(sigmoid_sum, a0, product(NW, NA), a0);
    const float4 gate = product(NW + NA, NG);
    float4 vm = v, f = v;
    if constexpr (!FIRST) {
        f = each(sigmoid_sum, v0, product(NW + NA + NG, NV), v0);
        vm = each([](float vv, float ff, float va) { return vv * (1.0f - ff) + va * ff; }, v, f, first);
    }
    const float4 kk = each([](float p, float kv, float) { return round_h(p * kv); }, k_k, k, k);
    float sum = kk.x * kk.x + kk.y * kk.y + kk.z * kk.z + kk.w * kk.w;
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lane < 16) part[wave][lane] = sum;
    __syncthreads();
    const float norm = 1.0f / sqrtf((part[0][r16] + part[1][r16]) + (part[2][r16] + part[3][r16]) + eps);
    if (t0 + r16 >= T) return;
    store_vec4(m.att_w + at, w);
    store_vec4(m.att_g + at, gate);
    if constexpr (FIRST) store_vec4(m.att_v0 + at, v);
    auto keep = [&](uint16_t *buffer, int i, float4 value) {
        store_vec4(m.n + i * plane + at, value);
        if (buffer) store_vec4(buffer + at, value);
    };
    keep(m.att_k, 0, each([](float kv, float av, float p) { return kv * (1.0f + (av - 1.0f) * p); }, k, a, k_a));
    keep(m.att_v, 1, vm);
    keep(m.att_a, 2, a);
    keep(m.att_kk, 3, make_float4(kk.x * norm, kk.y * norm, kk.z * norm, kk.w * norm));
    if constexpr (!FIRST) {
        if (m.att_vv) store_vec4(m.att_vv + at, f);
    }
}

// state[request] <- ffn_x at its last token; x_out = f16(v + x_in) (halved when `rescale`); ffn_out, where given, <- v
__global__ __launch_bounds__(256) void v7_post_ffn_kernel(const uint32_t *cursors, float *state, const uint16_t *v, const uint16_t *ffn_x, const uint16_t *x_in,
                                                          uint16_t *x_out, uint32_t C, int rescale, uint16_t *ffn_out, ViewArgs vs) {
    const uint32_t at = blockIdx.x * 256 + threadIdx.x, index = min(at, C / 4 - 1), t = blockIdx.y;
    const uint64_t bti = (uint64_t)t * C + 4 * index;
    const float4 vv = load_vec4(v + bti), xx = load_vec4(x_in + bti), fx = load_vec4(ffn_x + bti); // before the cursor's round trip and the store into the state
    const uint32_t ahead = cursor_ahead(cursors, t, gridDim.y);
    const Cursor cur = read_cursor(cursors, t, vs);
    const bool keeps = keeps_row(cursors, t, gridDim.y, cur, vs, ahead);
    if (at >= C / 4) return; // lanes past the row took part in the search
    if (keeps) *reinterpret_cast<float4 *>(state + view_elem(vs, cur.batch, 0, 4 * index)) = fx;
    const float sc = rescale ? 0.5f : 1.0f;
    auto f = [&](float a, float b) { return round_h(a + b) * sc; };
    store_vec4(x_out + bti, make_float4(f(vv.x, xx.x), f(vv.y, xx.y), f(vv.z, xx.z), f(vv.w, xx.w)));
    if (ffn_out) store_vec4(ffn_out + bti, vv);
}

template <typename XT>
__global__ __launch_bounds__(64) void l2_norm_kernel(XT *x, uint32_t C, float eps) {
    XT *row = x + (uint64_t)blockIdx.x * C;
    float sum = 0.0f;
    for (uint32_t i = 4 * threadIdx.x; i < C; i += 256) {
        const float4 v = load_vec4(row + i);
        sum += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    const float norm = 1.0f / sqrtf(wave_sum(sum) + eps);
    for (uint32_t i = 4 * threadIdx.x; i < C; i += 256) {
        const float4 v = load_vec4(row + i);
        store_vec4(row + i, make_float4(v.x * norm, v.y * norm, v.z * norm, v.w * norm));
    }
}

// k <- k (1 + (a - 1) p)
template <typename AT, typename KT>
__global__ __launch_bounds__(256) void control_k_kernel(const uint16_t *p, const AT *a, KT *k, ViewArgs va, ViewArgs vk, uint32_t C) {
    const uint32_t index = blockIdx.x * 256 + threadIdx.x, token = blockIdx.y, batch = blockIdx.z;
    if (index >= C / 4) return;
    const float4 pp = load_vec4(p + 4 * index), aa = load_vec4(a + view_elem(va, batch, token, 4 * index));
    KT *kp = k + view_elem(vk, batch, token, 4 * index);
    const float4 kk = load_vec4(kp);
    auto f = [](float kv, float av, float pv) { return kv * (1.0f + (av - 1.0f) * pv); };
    store_vec4(kp, make_float4(f(kk.x, aa.x, pp.x), f(kk.y, aa.y, pp.y), f(kk.z, aa.z, pp.z), f(kk.w, aa.w, pp.w)));
}

// x[i] += (sum_j u[j] k[j] r[j]) v[i] per head and token; one wave per (token, head)
template <typename XT>
__global__ __launch_bounds__(64) void time_first_v7_kernel(const uint16_t *u, const XT *r, const XT *n, XT *x, uint32_t S, uint32_t H, uint32_t A) {
    const uint32_t head = blockIdx.x, t = blockIdx.y;
    const uint32_t C = S * H;
    const uint64_t base = (uint64_t)t * C + head * S, plane = (uint64_t)A * C;
    float sum = 0.0f;
    for (uint32_t j = threadIdx.x; j < S; j += 64) sum += h2f(u[head * S + j]) * load_one(n + base + j) * load_one(r + base + j);
    sum = wave_sum(sum);
    for (uint32_t i = threadIdx.x; i < S; i += 64) {
        const float y = load_one(x + base + i) + sum * load_one(n + plane + base + i);
        if constexpr (sizeof(XT) == 2) x[base + i] = f2h(y);
        else x[base + i] = y;
    }
}

// state[request] <- x at the request's last token of the stack; x <- v
template <typename XT>
__global__ __launch_bounds__(256) void channel_mix_v7_kernel(const uint32_t *cursors, float *state, const XT *v, XT *x, ViewArgs vs, uint32_t C) {
    const uint32_t at = blockIdx.x * 256 + threadIdx.x, index = min(at, C / 4 - 1), stack = blockIdx.y;
    const uint64_t bti = (uint64_t)stack * C + 4 * index;
    const float4 vv = load_vec4(v + bti), xx = load_vec4(x + bti); // both before the cursor's round trip and the store into the state
    const uint32_t ahead = cursor_ahead(cursors, stack, gridDim.y);
    const Cursor cur = read_cursor(cursors, stack, vs);
    const bool keeps = keeps_row(cursors, stack, gridDim.y, cur, vs, ahead);
    if (at >= C / 4) return; // lanes past the row took part in the search
    if (keeps) *reinterpret_cast<float4 *>(state + view_elem(vs, cur.batch, 0, 4 * index)) = xx;
    store_vec4(x + bti, vv);
}

int check_float(wrq_dtype dtype, const char *name) {
    if (dtype != WRQ_F16 && dtype != WRQ_F32) return fail(WRQ_ERR_TYPE, "%s: unsupported element type %d", name, (int)dtype);
    return WRQ_OK;
}

} // namespace

} // namespace wrq

using namespace wrq;

extern "C" {

int wrq_l2_norm(wrq_stream stream, const wrq_tensor *x, wrq_dtype dtype, float eps) {
    int s = check_layer_tensor(x, "l2_norm");
    if (s == WRQ_OK) s = check_float(dtype, "l2_norm");
    if (s != WRQ_OK) return s;
    const uint32_t *sh = x->shape;
    if (sh[3] != 1) return fail(WRQ_ERR_SHAPE, "l2_norm: data shape not match [%u, %u, %u, %u]", sh[0], sh[1], sh[2], sh[3]);
    if (sh[0] % 4) return fail(WRQ_ERR_ALIGNMENT, "l2_norm: row length %u not a multiple of 4", sh[0]);
    const uint64_t rows = (uint64_t)sh[1] * sh[2];
    if (sh[0] == 0 || rows == 0) return WRQ_OK;
    if (rows > 0x7fffffffull) return fail(WRQ_ERR_SIZE, "l2_norm: data size not match");
    hipStream_t hs = static_cast<hipStream_t>(stream);
    if (dtype == WRQ_F16) hipLaunchKernelGGL((l2_norm_kernel<uint16_t>), dim3((uint32_t)rows), dim3(64), 0, hs, static_cast<uint16_t *>(x->data), sh[0], eps);
    else hipLaunchKernelGGL((l2_norm_kernel<float>), dim3((uint32_t)rows), dim3(64), 0, hs, static_cast<float *>(x->data), sh[0], eps);
    return check_launch("l2_norm");
}

int wrq_control_k_v7(wrq_stream stream, const wrq_tensor *p, const wrq_tensor_view *a, const wrq_tensor_view *k) {
    int s = check_layer_tensor(p, "control_k_v7");
    if (s == WRQ_OK) s = check_layer_view(a, "control_k_v7");
    if (s == WRQ_OK) s = check_layer_view(k, "control_k_v7");
    if (s != WRQ_OK) return s;
    const uint32_t *sh = k->view.shape;
    // src/tensor/ops.rs:1812-1815
    const uint32_t ps[4] = {sh[0], 1, 1, 1};
    if (sh[3] != 1 || !same_shape(a->view.shape, sh) || !same_shape(p->shape, ps))
        return fail(WRQ_ERR_SHAPE, "control_k_v7: data shape not match [%u, %u, %u, %u]", sh[0], sh[1], sh[2], sh[3]);
    if (sh[0] == 0 || sh[1] == 0 || sh[2] == 0) return WRQ_OK;
    if (sh[1] > 65535u || sh[2] > 65535u) return fail(WRQ_ERR_SIZE, "control_k_v7: data size not match");
    const dim3 grid((sh[0] / 4 + 255) / 256, sh[1], sh[2]);
    const ViewArgs va = view_args(a->view), vk = view_args(k->view);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const uint16_t *pp = static_cast<const uint16_t *>(p->data);
    const bool a16 = a->dtype == WRQ_F16, k16 = k->dtype == WRQ_F16;
    if (a16 && k16) hipLaunchKernelGGL((control_k_kernel<uint16_t, uint16_t>), grid, dim3(256), 0, hs, pp, static_cast<const uint16_t *>(a->data), static_cast<uint16_t *>(k->data), va, vk, sh[0]);
    else if (a16) hipLaunchKernelGGL((control_k_kernel<uint16_t, float>), grid, dim3(256), 0, hs, pp, static_cast<const uint16_t *>(a->data), static_cast<float *>(k->data), va, vk, sh[0]);
    else if (k16) hipLaunchKernelGGL((control_k_kernel<float, uint16_t>), grid, dim3(256), 0, hs, pp, static_cast<const float *>(a->data), static_cast<uint16_t *>(k->data), va, vk, sh[0]);
    else hipLaunchKernelGGL((control_k_kernel<float, float>), grid, dim3(256), 0, hs, pp, static_cast<const float *>(a->data), static_cast<float *>(k->data), va, vk, sh[0]);
    return check_launch("control_k_v7");
}

int wrq_time_mix_v7(wrq_stream stream, const wrq_tensor *cursors, const wrq_tensor_view *state, const wrq_tensor *r, const wrq_tensor *w, const wrq_tensor *n,
                    const wrq_tensor *x, wrq_dtype dtype) {
    int s = check_layer_tensor(cursors, "time_mix_v7");
    for (const wrq_tensor *t : {r, w, n, x})
        if (s == WRQ_OK) s = check_layer_tensor(t, "time_mix_v7");
    if (s == WRQ_OK) s = check_state_view(state, "time_mix_v7");
    if (s == WRQ_OK) s = check_float(dtype, "time_mix_v7");
    if (s != WRQ_OK) return s;
    if (state->dtype != WRQ_F32) return fail(WRQ_ERR_TYPE, "time_mix_v7: the state is f32");
    const uint32_t *sh = x->shape, *st = state->view.shape; // [S, H, A, 1]
    const uint32_t S = sh[0], H = sh[1], A = sh[2];
    // src/tensor/ops.rs:1695-1698
    const uint32_t ns[4] = {S, H, A, 4};
    if (sh[3] != 1 || !same_shape(r->shape, sh) || !same_shape(w->shape, sh) || !same_shape(n->shape, ns) || st[0] != S * H || st[1] != S + 1 || st[3] != 1)
        return fail(WRQ_ERR_SHAPE, "time_mix_v7: data shape not match [%u, %u, %u, %u]", sh[0], sh[1], sh[2], sh[3]);
    if (cursors->shape[0] < A) return fail(WRQ_ERR_SHAPE, "time_mix_v7: %u cursors for %u tokens", cursors->shape[0], A);
    if (S == 0 || H == 0 || A == 0) return WRQ_OK;
    const ViewArgs vs = view_args(state->view);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const uint32_t *cur = static_cast<const uint32_t *>(cursors->data);
    float *sp = static_cast<float *>(state->data);
    const bool wide = S == 64 && wide_walk(vs, H, A);
#define WRQ_TM7_FORM(XT, SZ, WIDE)                                                                                                                   \
    hipLaunchKernelGGL((time_mix_v7_kernel<XT, SZ, false, WIDE>), dim3(H, slot_grid(vs, A)), dim3(RecurrenceTile<SZ, WIDE>::THREADS), 0, hs, cur, sp,                     \
                       static_cast<const XT *>(r->data), static_cast<const XT *>(w->data), static_cast<const XT *>(n->data), static_cast<XT *>(x->data), \
                       vs, H, A, nullptr, GateArgs{})
#define WRQ_TM7_LAUNCH(XT, SZ)                                                                                                                       \
    if (wide) WRQ_TM7_FORM(XT, SZ, (SZ == 64));                                                                                                      \
    else WRQ_TM7_FORM(XT, SZ, false)
#define WRQ_TM7(SZ)                                                                                                                                  \
    if (S == SZ) {                                                                                                                                   \
        if (dtype == WRQ_F16) { WRQ_TM7_LAUNCH(uint16_t, SZ); }                                                                                      \
        else { WRQ_TM7_LAUNCH(float, SZ); }                                                                                                          \
        return check_launch("time_mix_v7");                                                                                                          \
    }
    WRQ_TM7(32) WRQ_TM7(64) WRQ_TM7(128)
#undef WRQ_TM7
#undef WRQ_TM7_LAUNCH
#undef WRQ_TM7_FORM
    return fail(WRQ_ERR_UNSUPPORTED, "time_mix_v7: head size %u (32, 64 or 128 is built)", S);
}

int wrq_time_first_v7(wrq_stream stream, const wrq_tensor *u, const wrq_tensor *r, const wrq_tensor *n, const wrq_tensor *x, wrq_dtype dtype) {
    int s = WRQ_OK;
    for (const wrq_tensor *t : {u, r, n, x})
        if (s == WRQ_OK) s = check_layer_tensor(t, "time_first_v7");
    if (s == WRQ_OK) s = check_float(dtype, "time_first_v7");
    if (s != WRQ_OK) return s;
    const uint32_t *sh = x->shape;
    const uint32_t S = sh[0], H = sh[1], A = sh[2];
    // src/tensor/ops.rs:1755-1757
    const uint32_t us[4] = {S, H, 1, 1}, ns[4] = {S, H, A, 4};
    if (sh[3] != 1 || !same_shape(r->shape, sh) || !same_shape(u->shape, us) || !same_shape(n->shape, ns))
        return fail(WRQ_ERR_SHAPE, "time_first_v7: data shape not match [%u, %u, %u, %u]", sh[0], sh[1], sh[2], sh[3]);
    if (S == 0 || H == 0 || A == 0) return WRQ_OK;
    if (A > 65535u) return fail(WRQ_ERR_SIZE, "time_first_v7: data size not match");
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const uint16_t *up = static_cast<const uint16_t *>(u->data);
    if (dtype == WRQ_F16)
        hipLaunchKernelGGL((time_first_v7_kernel<uint16_t>), dim3(H, A), dim3(64), 0, hs, up, static_cast<const uint16_t *>(r->data), static_cast<const uint16_t *>(n->data),
                           static_cast<uint16_t *>(x->data), S, H, A);
    else
        hipLaunchKernelGGL((time_first_v7_kernel<float>), dim3(H, A), dim3(64), 0, hs, up, static_cast<const float *>(r->data), static_cast<const float *>(n->data),
                           static_cast<float *>(x->data), S, H, A);
    return check_launch("time_first_v7");
}

int wrq_channel_mix_v7(wrq_stream stream, const wrq_tensor *cursors, const wrq_tensor_view *state, const wrq_tensor *v, const wrq_tensor *x, wrq_dtype dtype) {
    int s = check_layer_tensor(cursors, "channel_mix_v7");
    for (const wrq_tensor *t : {v, x})
        if (s == WRQ_OK) s = check_layer_tensor(t, "channel_mix_v7");
    if (s == WRQ_OK) s = check_state_view(state, "channel_mix_v7");
    if (s == WRQ_OK) s = check_float(dtype, "channel_mix_v7");
    if (s != WRQ_OK) return s;
    if (state->dtype != WRQ_F32) return fail(WRQ_ERR_TYPE, "channel_mix_v7: the state is f32");
    const uint32_t *sh = x->shape, *st = state->view.shape;
    // src/tensor/ops.rs:1929-1930
    if (!same_shape(v->shape, sh) || st[0] != sh[0] || st[1] != 1 || st[3] != 1 || sh[2] != 1 || sh[3] != 1)
        return fail(WRQ_ERR_SHAPE, "channel_mix_v7: data shape not match [%u, %u, %u, %u]", sh[0], sh[1], sh[2], sh[3]);
    if (cursors->shape[0] < sh[1]) return fail(WRQ_ERR_SHAPE, "channel_mix_v7: %u cursors for %u tokens", cursors->shape[0], sh[1]);
    if (sh[0] % 4) return fail(WRQ_ERR_ALIGNMENT, "channel_mix_v7: row length %u not a multiple of 4", sh[0]);
    if (sh[0] == 0 || sh[1] == 0) return WRQ_OK;
    if (sh[1] > 65535u) return fail(WRQ_ERR_SIZE, "channel_mix_v7: data size not match");
    const dim3 grid((sh[0] / 4 + 255) / 256, sh[1]);
    const ViewArgs vs = view_args(state->view);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const uint32_t *cur = static_cast<const uint32_t *>(cursors->data);
    if (dtype == WRQ_F16)
        hipLaunchKernelGGL((channel_mix_v7_kernel<uint16_t>), grid, dim3(256), 0, hs, cur, static_cast<float *>(state->data), static_cast<const uint16_t *>(v->data),
                           static_cast<uint16_t *>(x->data), vs, sh[0]);
    else
        hipLaunchKernelGGL((channel_mix_v7_kernel<float>), grid, dim3(256), 0, hs, cur, static_cast<float *>(state->data), static_cast<const float *>(v->data),
                           static_cast<float *>(x->data), vs, sh[0]);
    return check_launch("channel_mix_v7");
}

int wrq_adapters_in(wrq_stream stream, uint32_t C, uint32_t A, int n, const void *const *w, const uint32_t *ranks, const int *acts, const void *const *x,
                    void *const *out) {
    const char *what = "adapters_in";
    if (n < 0 || n > kMaxAdapters) return fail(WRQ_ERR_UNSUPPORTED, "%s: %d adapters (up to %d)", what, n, kMaxAdapters);
    if (n == 0 || C == 0 || A == 0) return WRQ_OK;
    if (!w || !ranks || !acts || !x || !out) return fail(WRQ_ERR_NULL, "%s: null pointer", what);
    if (C % 32) return fail(WRQ_ERR_ALIGNMENT, "%s: row length %u not a multiple of 32", what, C);
    if (A > 65535u * 16u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    AdapterArgs aa{};
    uint32_t tiles = 0;
    for (int i = 0; i < kMaxAdapters; i++) {
        aa.tile_begin[i] = i < n ? tiles : ~0u;
        if (i >= n) continue;
        if (ranks[i] == 0 || ranks[i] % 16 || ranks[i] > 65536u) return fail(WRQ_ERR_UNSUPPORTED, "%s: adapter size %u (a multiple of 16 up to 65536 is built)", what, ranks[i]);
        if (acts[i] < 0 || acts[i] > WRQ_ACT_SILU) return fail(WRQ_ERR_UNSUPPORTED, "%s: activation %d", what, acts[i]);
        for (const void *p : {w[i], x[i], (const void *)out[i]}) {
            const int s = check_ptr(p, what);
            if (s != WRQ_OK) return s;
        }
        aa.w[i] = static_cast<const uint16_t *>(w[i]), aa.x[i] = static_cast<const uint16_t *>(x[i]), aa.out[i] = static_cast<uint16_t *>(out[i]);
        aa.rank[i] = ranks[i], aa.act[i] = acts[i];
        tiles += ranks[i] / 16;
    }
    auto go = [&](auto kern, int waves) { hipLaunchKernelGGL(kern, dim3(tiles, (A + 15) / 16), dim3(64 * waves), 0, static_cast<hipStream_t>(stream), C, A, aa); };
    // Eight waves, two steps each in flight: 2048 channels in one go.  us, gathered -> line-wise: 160 rows x 100 tokens over 768 / 2048 / 4096 / 5120
    // channels 6.5 / 6.5 / 10.3 / 12.0 -> 3.7 / 4.5 / 6.0 / 6.9; four adapters of a v7 layer, 32 tokens, 6.3 / 6.5 / 10.2 / 12.0 -> 3.5 / 4.5 /
    // 5.8 / 6.8.  Sixteen waves of one step 3.7 / 4.5 / 6.1 / 7.3, four of four 4.0 / 5.3 / 7.7 / 8.8.
    // Gathered, steps of 32: eight waves of eight steps, where their rounds are full.  A second round that would hold less than a quarter of the steps goes into
    // the first one with ten steps, a third one with sixteen waves of ten.  160 rows x 100 tokens, us, eight of eight / the other: 2112 channels 7.2 / 7.4,
    // 2144 6.4 / 6.3, 2240 8.8 / 7.4, 2496 10.1 / 7.4; 4256 9.3 / 9.4, 4320 9.7 / 9.4, 4672 13.5 / 11.7, 5184 13.4 / 12.7, 6112 10.8 / 16.0, 8160 13.2 / 15.8.
    const uint32_t steps = C / 32;
    if (C % 128 == 0) go(adapters_in_kernel<8, 2, true>, 8);
    else if (steps >= 67 && steps <= 80) go(adapters_in_kernel<8, 10, false>, 8);
    else if (steps >= 135 && steps <= 162) go(adapters_in_kernel<16, 10, false>, 16);
    else go(adapters_in_kernel<8, 8, false>, 8);
    return check_launch(what);
}

int wrq_v7_mid(wrq_stream stream, uint32_t S, uint32_t H, uint32_t A, int first, const uint32_t *ranks, const void *const *aux, const void *const *w2,
               const void *const *vectors, float eps, const void *k, const void *v, void *att_v0, void *att_w, void *att_g, void *n) {
    void *const none[5] = {};
    return wrq_v7_mid_buffers(stream, S, H, A, first, ranks, aux, w2, vectors, eps, k, v, att_v0, att_w, att_g, n, none);
}

int wrq_v7_mid_buffers(wrq_stream stream, uint32_t S, uint32_t H, uint32_t A, int first, const uint32_t *ranks, const void *const *aux, const void *const *w2,
                       const void *const *vectors, float eps, const void *k, const void *v, void *att_v0, void *att_w, void *att_g, void *n,
                       void *const *buffers) {
    const char *what = "v7_mid";
    if (H == 0 || A == 0) return WRQ_OK;
    if (S != 64) return fail(WRQ_ERR_UNSUPPORTED, "%s: head size %u (64 is built)", what, S);
    if (!ranks || !aux || !w2 || !vectors || !buffers) return fail(WRQ_ERR_NULL, "%s: null pointer", what);
    if (ranks[0] != 64 || ranks[1] != 64 || ranks[2] != 128 || (!first && ranks[3] != 32))
        return fail(WRQ_ERR_UNSUPPORTED, "%s: adapter sizes %u, %u, %u, %u (64, 64, 128, 32 are built)", what, ranks[0], ranks[1], ranks[2], ranks[3]);
    if (A > 65535u * 16u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    int s = WRQ_OK;
    for (int i = 0; i < (first ? 3 : 4) && s == WRQ_OK; i++) {
        s = check_ptr(aux[i], what);
        if (s == WRQ_OK) s = check_ptr(w2[i], what);
    }
    for (int i = 0; i < 5 && s == WRQ_OK; i++)
        if (!first || i != 2) s = check_ptr(vectors[i], what); // the first layer has no adapter v and so no v0
    for (const void *p : {k, v, (const void *)att_v0, (const void *)att_w, (const void *)att_g, (const void *)n})
        if (s == WRQ_OK) s = check_ptr(p, what);
    for (int i = 0; i < 5 && s == WRQ_OK; i++)
        if (buffers[i]) s = check_ptr(buffers[i], what);
    if (s != WRQ_OK) return s;
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    auto o16 = [](void *p) { return static_cast<uint16_t *>(p); };
    const MidArgs m{u16(aux[0]),     u16(aux[1]),     u16(aux[2]),     u16(aux[3]),     u16(w2[0]), u16(w2[1]), u16(w2[2]),  u16(w2[3]),  u16(vectors[0]),
                    u16(vectors[1]), u16(vectors[2]), u16(vectors[3]), u16(vectors[4]), u16(k),     u16(v),     o16(att_v0), o16(att_w), o16(att_g),
                    o16(n),          o16(buffers[0]), o16(buffers[1]), o16(buffers[2]), o16(buffers[3]), o16(buffers[4])};
    const dim3 grid(H, (A + 15) / 16);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    if (first) hipLaunchKernelGGL((v7_mid_kernel<64, 64, 128, 32, true>), grid, dim3(256), 0, hs, S * H, A, eps, m);
    else hipLaunchKernelGGL((v7_mid_kernel<64, 64, 128, 32, false>), grid, dim3(256), 0, hs, S * H, A, eps, m);
    return check_launch(what);
}

int wrq_v7_wkv_gate(wrq_stream stream, uint32_t S, uint32_t H, uint32_t A, const void *cursors, const wrq_tensor_view *state, const void *r, const void *w,
                    const void *n, const void *r_k, const void *g, const void *gn_w, const void *gn_b, float eps, void *att_x) {
    const char *what = "v7_wkv_gate";
    if (H == 0 || A == 0) return WRQ_OK;
    if (S != 64) return fail(WRQ_ERR_UNSUPPORTED, "%s: head size %u (64 is built)", what, S);
    int s = check_state(state, S * H, S + 1, what);
    for (const void *p : {cursors, r, w, n, r_k, g, gn_w, gn_b, (const void *)att_x})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s != WRQ_OK) return s;
    const ViewArgs vs = view_args(state->view);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    const bool wide = wide_walk(vs, H, A);
    auto *kern = wide ? &time_mix_v7_kernel<uint16_t, 64, true, true> : &time_mix_v7_kernel<uint16_t, 64, true, false>;
    hipLaunchKernelGGL(kern, dim3(H, slot_grid(vs, A)), dim3(wide ? RecurrenceTile<64, true>::THREADS : RecurrenceTile<64>::THREADS), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint32_t *>(cursors), static_cast<float *>(state->data), u16(r), u16(w), u16(n), static_cast<uint16_t *>(nullptr), vs, H, A,
                       u16(r_k), GateArgs{u16(g), u16(gn_w), u16(gn_b), static_cast<uint16_t *>(att_x), eps});
    return check_launch(what);
}

int wrq_v7_post_ffn(wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const wrq_tensor_view *state, const void *v, const void *ffn_x,
                    const void *x_in, void *x_out, int rescale) {
    return wrq_v7_post_ffn_buffers(stream, C, A, cursors, state, v, ffn_x, x_in, x_out, rescale, nullptr);
}

int wrq_v7_post_ffn_buffers(wrq_stream stream, uint32_t C, uint32_t A, const void *cursors, const wrq_tensor_view *state, const void *v, const void *ffn_x,
                            const void *x_in, void *x_out, int rescale, void *ffn_out) {
    const char *what = "v7_post_ffn";
    if (C == 0 || A == 0) return WRQ_OK;
    if (C % 4) return fail(WRQ_ERR_ALIGNMENT, "%s: row length %u not a multiple of 4", what, C);
    if (A > 65535u) return fail(WRQ_ERR_SIZE, "%s: data size not match", what);
    int s = check_state(state, C, 1, what);
    for (const void *p : {cursors, v, ffn_x, x_in, (const void *)x_out})
        if (s == WRQ_OK) s = check_ptr(p, what);
    if (s == WRQ_OK && ffn_out) s = check_ptr(ffn_out, what);
    if (s != WRQ_OK) return s;
    const ViewArgs vs = view_args(state->view);
    auto u16 = [](const void *p) { return static_cast<const uint16_t *>(p); };
    hipLaunchKernelGGL(v7_post_ffn_kernel, dim3((C / 4 + 255) / 256, A), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const uint32_t *>(cursors),
                       static_cast<float *>(state->data), u16(v), u16(ffn_x), u16(x_in), static_cast<uint16_t *>(x_out), C, rescale, static_cast<uint16_t *>(ffn_out), vs);
    return check_launch(what);
}

} // extern "C"
