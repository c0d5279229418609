// The state recurrences of the v5 / v6 / v7 layers (recurrent_ops.hip, v7_ops.hip, fused_ops.hip).
//
// A run is a stack of A tokens from several requests; the state of a request is one 64 x 64 matrix S per head (or
// SZ x SZ).  Requests do not depend on each other, so a workgroup takes one head of ONE state slot and walks that
// slot's tokens only: 32 requests of one token each are 32 workgroups per head instead of a chain of 32 state
// reloads in one.  S stays in registers over the slot's tokens: L = 8 lanes share two columns of S and hold SZ / 8
// of their rows each (SZ = 16: four lanes, one column; long runs of SZ = 64: sixteen lanes, see wide_walk).  What bounds
// a long run is the vector ALU of the one CU a head's state lives on: per element of S three fmas in v5 / v6 (k v, the
// decay, y) and five in v7; the bonus term of v5 / v6, sum_j r[j] u[j] k[j] v[i], does not depend on S and is one number
// per token, formed while the operands are staged.  Sharing two columns halves the LDS reads per token against one
// column per quad, which came out as the second bound.
#pragma once

#include "layer_device.h"

namespace wrq {

constexpr uint32_t kSlotScan = 256; // cursors scanned at a time: one per thread

// The slot a workgroup takes; false: none.  A grid of less than the slots has a workgroup per token (slot_grid): it takes its
// token's slot, unless an earlier token has it.
__device__ __forceinline__ bool own_slot(const uint32_t *cursors, uint32_t A, uint32_t slots, uint32_t *slot) {
    *slot = blockIdx.y;
    if (gridDim.y == A && A < slots) {
        *slot = min(cursors[blockIdx.y] & 0xffu, slots - 1);
        if (blockIdx.y) {
            const bool taken = threadIdx.x < blockIdx.y && min(cursors[min(threadIdx.x, A - 1)] & 0xffu, slots - 1) == *slot;
            return !__syncthreads_or(taken);
        }
    }
    return true;
}

// The tokens of `slot` among cursors[base .. base + 256): their offsets from `base` in stack order, and their number.
// With a single slot (a slot beyond the view counts as the last one) or a single token, `every` token is its own and `list` stays unused.
template <int THREADS>
__device__ __forceinline__ uint32_t slot_tokens(const uint32_t *cursors, uint32_t base, uint32_t A, uint32_t slot, uint32_t slots, bool every, uint8_t *list, uint32_t *count) {
    if (every) return min(kSlotScan, A - base);
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool scans = THREADS == kSlotScan || tid < kSlotScan;
    const bool mine = scans && base + tid < A && min(cursors[min(base + tid, A - 1)] & 0xffu, slots - 1) == slot;
    const uint64_t mask = __ballot(mine);
    if (scans && lane == 0) count[wave] = (uint32_t)__popcll(mask);
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSlotScan / 64; w++) {
        before += w < wave ? count[w] : 0u;
        total += count[w];
    }
    if (mine) list[before + (uint32_t)__popcll(mask & ((1ull << lane) - 1))] = (uint8_t)tid;
    __syncthreads();
    return total;
}

// Sum over groups of LANES adjacent lanes (a power of two), the same value in each of them.
template <int LANES>
__device__ __forceinline__ float lanes_sum(float v) {
    if constexpr (LANES >= 2) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));  // quad_perm [1,0,3,2]
    if constexpr (LANES >= 4) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));  // quad_perm [2,3,0,1]
    if constexpr (LANES >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true)); // row_half_mirror
    if constexpr (LANES >= 16) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true)); // row_mirror
    if constexpr (LANES >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (LANES >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

__device__ __forceinline__ float round_h(float v) { return h2f(f2h(v)); }

template <int SZ, bool WIDE = false>
struct RecurrenceTile {
    static_assert(!WIDE || SZ == 64, "the wide form: head size 64");
    static constexpr int THREADS = WIDE ? 512 : 256;
    static constexpr int L = WIDE ? 16 : SZ >= 32 ? 8 : 4; // lanes that share CPT columns of S
    static constexpr int CPT = SZ >= 32 ? 2 : 1;           // columns of a lane
    static constexpr int JL = SZ / L;           // rows of S a lane holds
    static constexpr int TB = 1024 / SZ;        // tokens per chunk: a 4-element vector of each operand per thread
    static constexpr int TL = SZ / 4;           // threads per token of a chunk, the first 256 of the workgroup
    static constexpr int PARTS = WIDE ? 1 : 2;  // partial sums of a lane's rows: the even and the odd ones, or all of its own
    // Rows first_row(l), first_row(l) + ROW_STEP, .. are lane l's.  In the wide form a pair of lanes has eight adjacent rows, the
    // even lane the even ones: the pair's two sums are then the two partial sums of the narrow form's lane.
    static constexpr int ROW_STEP = WIDE ? 2 : 1;
    static __device__ __forceinline__ uint32_t first_row(uint32_t l) { return WIDE ? 8 * (l >> 1) + (l & 1) : l * JL; }
    // Vector `tid` of a chunk's operand that is indexed by rows; in LDS the rows of a lane lie side by side.
    static __device__ __forceinline__ void put_rows(float *buf, uint32_t tid, float4 v) {
        if constexpr (WIDE) {
            float *p = buf + 4 * (tid & ~1u) + 2 * (tid & 1);
            *reinterpret_cast<float2 *>(p) = make_float2(v.x, v.z), *reinterpret_cast<float2 *>(p + 4) = make_float2(v.y, v.w);
        } else {
            *reinterpret_cast<float4 *>(buf + 4 * tid) = v;
        }
    }
    static __device__ __forceinline__ float4 get_rows(const float *buf, uint32_t tid) {
        if constexpr (WIDE) {
            const float *p = buf + 4 * (tid & ~1u) + 2 * (tid & 1);
            const float2 even = *reinterpret_cast<const float2 *>(p), odd = *reinterpret_cast<const float2 *>(p + 4);
            return make_float4(even.x, odd.x, even.y, odd.y);
        } else {
            return *reinterpret_cast<const float4 *>(buf + 4 * tid);
        }
    }
};

template <int N>
__device__ __forceinline__ void load_cols(float (&d)[N], const float *p) {
    if constexpr (N == 2) {
        const float2 v = *reinterpret_cast<const float2 *>(p);
        d[0] = v.x, d[1] = v.y;
    } else {
        d[0] = *p;
    }
}
template <int N>
__device__ __forceinline__ void store_cols(float *p, const float (&d)[N]) {
    if constexpr (N == 2) *reinterpret_cast<float2 *>(p) = make_float2(d[0], d[1]);
    else *p = d[0];
}

// Row 0 of a slot's state keeps the layer's input at the last token of a request; the tokens of a chunk are finished side by
// side, so where several requests of the slot end among its `count` tokens the latest one's input is the one kept.
__device__ __forceinline__ bool keeps_input(const uint32_t *tokens, const uint32_t *cursors, uint32_t at, uint32_t count) {
    auto ends = [&](uint32_t j) {
        const Cursor cur = unpack_cursor(cursors[j]);
        return tokens[j] - min(cur.token, tokens[j]) + 1 == cur.len; // the first token clamped as in read_cursor
    };
    if (!ends(at)) return false;
    for (uint32_t j = at + 1; j < count; j++)
        if (ends(j)) return false;
    return true;
}

// The tokens of a chunk in groups of L (eight; sixteen, a whole chunk, in the wide form).  A whole group is one piece of straight code:
// the operands of its later tokens are read from LDS while the earlier ones are worked on, where a loop over tokens waits out one LDS
// round trip, the reduction over the lanes and a branch for the store at each of them.  The tokens past the last whole group take
// that loop.  `token(tt, u)` leaves its result in lane u of the L that share the columns, `flush(from, count)` then stores the group
// at once.
// 32 heads of 64, one request: v6 gate form 100 tokens 31.0 -> 27.2 us, 255 tokens 72.5 -> 62.1; v7, whose tokens are a chain through
// sa, 45.4 -> 44.4 and 109.0 -> 106.1.  Reads ahead stop at every second token where a lane holds up to eight rows: over the
// whole group they took up to 250 registers, two waves per SIMD instead of three, and were slower in the end (v6 gate form 27.7 -> 25.6 us, v7
// 45.2 -> 39.1 at 100 tokens; 32 requests of one token 15.7 -> 15.0).  With 16 rows and more per lane they are left as they fall.
template <int L, int JL, typename Token, typename Flush>
__device__ __forceinline__ void walk_tokens(uint32_t tend, Token token, Flush flush) {
    uint32_t tt = 0;
    for (; tt + L <= tend; tt += L) {
#pragma unroll
        for (int u = 0; u < L; u++) {
            token(tt + u, u);
            if (JL <= 8 && u % 2) __builtin_amdgcn_sched_barrier(0);
        }
        flush(tt, (uint32_t)L);
    }
    if (tt == tend) return;
    for (uint32_t u = 0; tt + u < tend; u++) token(tt + u, (int)u);
    flush(tt, tend - tt);
}

// The wide form: 512 threads, sixteen lanes share two columns and hold four rows each.  The same LDS bytes and half the vector work
// per wave and token, by eight waves instead of four: one wave per SIMD issues a vector instruction every 2.3 ns whatever its
// dependences allow, two reach one per 1.15 ns.  Both forms add a column's rows in the same order (of eight rows the even and the odd
// ones, these two, then the eights in pairs, fours, ...), so they give the same bits.  The wide one is taken for head size 64 where
// the stack has 16 tokens and more per slot of the state and the workgroups have a CU each; narrow -> wide in us, v6 gate form / v7
// gate form / v5 (f32):
//   32 heads, one request of 16 tokens  7.4 /  9.4 /  6.7 ->  6.7 /  8.1 /  6.3     64 heads, 4 x 16  8.5 / 10.7 / 7.9 -> 7.8 / 9.5 / 7.5
//                            24 tokens  9.1 / 12.4 /  8.3 ->  8.8 / 11.5 /  8.3               4 x 31  11.9 / 15.8 / 10.9 -> 11.2 / 14.8 / 10.7
//                            31 tokens 10.8 / 14.6 /  9.6 ->  9.9 / 13.3 /  9.3
//                           100 tokens 25.6 / 39.0 / 21.7 -> 23.7 / 34.1 / 20.5
//                           512 tokens  111 /  179 / 91.4 ->  102 /  155 / 85.5
// Not so beyond: 64 heads, 8 x 16 10.9 / 13.4 / 10.3 -> 10.9 / 16.4 / 10.3; 32 heads, 32 x 1 12.7 / 15.0 / 12.2 -> 14.7 / 18.5 / 14.3
// and 32 x 16 20.5 / 25.6 / 16.2 -> 21.8 / 32.6 / 20.4, their time being the state's way in and out.  The launch knows the state's
// slots and not how many of them the stack names: one request of 100 tokens on a state of 32 slots keeps the narrow form (32 heads
// 25.9 / 39.2 / 21.9, where the wide one takes 24.4 / 34.5 / 21.3).
inline bool wide_walk(const ViewArgs &vs, uint32_t H, uint32_t A) { return A >= 16ull * vs.shape[2] && (uint64_t)H * vs.shape[2] <= 256; }

// Sum of the partial sums of a lane's rows.
template <int N>
__device__ __forceinline__ float parts_sum(const float (&v)[N]) {
    if constexpr (N == 2) return v[0] + v[1];
    else return v[0];
}

// Outputs of a group of tokens of one slot, token l in lane l.
template <int N, typename XT>
__device__ __forceinline__ void store_tokens(uint32_t count, uint32_t l, const uint32_t *tokens, const float (&y)[N], XT *x, uint32_t C, uint32_t chan) {
    if (l >= count) return;
    const uint64_t ti = (uint64_t)tokens[l] * C + chan;
#pragma unroll
    for (int c = 0; c < N; c++) {
        if constexpr (sizeof(XT) == 2) x[ti + c] = f2h(y[c]);
        else x[ti + c] = y[c];
    }
}

// What follows the recurrence in the fused forms of a layer (head size 64): the group norm over the head and the gate.
// att_x holds the layer's normalised input before and the gated output after.
struct GateArgs {
    const uint16_t *g, *gn_w, *gn_b;
    uint16_t *att_x;
    float eps;
};

// y4[e] (f32) of 4 elements per thread, 16 threads per token -> group norm over the 64 elements of the head, in f32
__device__ __forceinline__ float4 head_norm(float4 y, uint2 wq, uint2 bq, float eps) {
    const float mean = lanes_sum<16>((y.x + y.y) + (y.z + y.w)) * (1.0f / 64);
    const float4 d = make_float4(y.x - mean, y.y - mean, y.z - mean, y.w - mean);
    const float dev = rsqrtf(lanes_sum<16>((d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w)) * (1.0f / 64) + eps);
    auto w = [](uint2 v, int i) { return h2f((uint16_t)((i < 2 ? v.x : v.y) >> (16 * (i & 1)))); };
    return make_float4(fmaf(d.x * dev, w(wq, 0), w(bq, 0)), fmaf(d.y * dev, w(wq, 1), w(bq, 1)), fmaf(d.z * dev, w(wq, 2), w(bq, 2)),
                       fmaf(d.w * dev, w(wq, 3), w(bq, 3)));
}

// v5 (a decay per channel) and v6 (TOKEN_DECAY: a decay per token):
//   y[i] = sum_j r[j] (u[j] k[j] v[i] + S[j][i]),  S[j][i] <- w[j] S[j][i] + k[j] v[i]
// GATE: the fused form, y then goes through the group norm (rounded to f16) and silu(g) into att_x; otherwise into x.
// grid (heads, slot_grid).  The operands come in chunks of TB tokens of the slot: every thread fetches one 4-element
// vector of each while the previous chunk is worked on and passes it round through LDS (two buffers).
template <typename XT, int SZ, bool TOKEN_DECAY, bool GATE, bool WIDE = false>
__global__ __launch_bounds__((RecurrenceTile<SZ, WIDE>::THREADS)) void time_mix_kernel(const uint32_t *cursors, const float *time_decay, const float *time_first, float *state, const XT *k,
                                                       const XT *v, const XT *r, XT *x, ViewArgs vs, uint32_t H, uint32_t A, GateArgs ga) {
    using G = RecurrenceTile<SZ, WIDE>;
    constexpr int L = G::L, CPT = G::CPT, JL = G::JL, TB = G::TB, TL = G::TL, PARTS = G::PARTS;
    static_assert(!GATE || (SZ == 64 && sizeof(XT) == 4), "the fused form: head size 64, f32 operands");
    __shared__ __align__(16) float ks[2][1024], rs[2][1024], ws[TOKEN_DECAY ? 2 : 1][TOKEN_DECAY ? 1024 : 4], vsh[2][1024], ysh[GATE ? 1024 : 4];
    __shared__ float bonus[2][TB];
    __shared__ uint32_t csh[2][TB], tsh[2][TB]; // cursors and numbers of the chunk's tokens
    __shared__ uint8_t list[kSlotScan];
    __shared__ uint32_t count[kSlotScan / 64];
    const uint32_t head = blockIdx.x, slots = vs.shape[2], tid = threadIdx.x;
    const bool every = slots == 1 || A == 1;
    uint32_t slot;
    if (!own_slot(cursors, A, slots, &slot)) return;
    const uint32_t l = tid % L;
    const uint32_t C = SZ * H;
    // this thread's vector of a chunk: token tid / TL of the chunk, elements 4 (tid % TL) ..
    const uint32_t lt = (tid % 256) / TL, le = 4 * (tid % TL);
    const bool staging = !WIDE || tid < 256;
    const float4 u4 = *reinterpret_cast<const float4 *>(time_first + head * SZ + le);
    uint2 gw = make_uint2(0, 0), gb = make_uint2(0, 0);
    if constexpr (GATE) gw = *reinterpret_cast<const uint2 *>(ga.gn_w + head * SZ + le), gb = *reinterpret_cast<const uint2 *>(ga.gn_b + head * SZ + le);
    float4 fk, fr, fw, fv;
    // the layer's input, which row 0 of the slot's state keeps, comes with the operands of its chunk: read where it is stored it
    // is a round trip to memory at the end of every run (32 heads of 64, one token: v6 5.06 -> 4.72 us, v7 5.49 -> 5.10)
    using IT = std::conditional_t<GATE, uint16_t, XT>;
    using IV = std::conditional_t<sizeof(IT) == 2, uint2, float4>;
    const IT *in;
    if constexpr (GATE) in = ga.att_x;
    else in = x;
    uint2 fg = make_uint2(0, 0);
    IV fx = {};
    bool first_pass = true; // over the columns: the later ones find x overwritten
    uint32_t fc = 0, ft = 0, fct = 0;
    uint32_t base = 0, n = 0;
    auto fetch = [&](uint32_t chunk) {
        if (!staging) return;
        auto token = [&](uint32_t j) { return base + (every ? min(j, n - 1) : (uint32_t)list[min(j, n - 1)]); }; // clamped: past the slot's tokens, never used
        ft = token(chunk * TB + lt);
        const uint64_t g = (uint64_t)ft * C + head * SZ + le;
        fk = load_vec4(k + g), fr = load_vec4(r + g), fv = load_vec4(v + g);
        if constexpr (TOKEN_DECAY) fw = load_vec4(time_decay + g);
        if constexpr (GATE) fg = *reinterpret_cast<const uint2 *>(ga.g + g);
        if (SZ <= 64 || first_pass) fx = *reinterpret_cast<const IV *>(in + g);
        if (GATE) fc = cursors[ft];
        else if (tid < (uint32_t)TB) fct = token(chunk * TB + tid), fc = cursors[fct];
    };
    auto stage = [&](int buf) {
        if (!staging) return;
        G::put_rows(ks[buf], tid, fk);
        G::put_rows(rs[buf], tid, fr);
        if constexpr (TOKEN_DECAY) G::put_rows(ws[buf], tid, fw);
        *reinterpret_cast<float4 *>(&vsh[buf][4 * tid]) = fv;
        const float b = lanes_sum<TL>(fmaf(fr.x, u4.x * fk.x, fr.y * (u4.y * fk.y)) + fmaf(fr.z, u4.z * fk.z, fr.w * (u4.w * fk.w)));
        if (tid % TL == 0) bonus[buf][lt] = b;
        if (GATE && tid % TL == 0) csh[buf][lt] = fc, tsh[buf][lt] = ft;
        if (!GATE && tid < (uint32_t)TB) csh[buf][tid] = fc, tsh[buf][tid] = fct;
    };
    for (uint32_t i0 = 0; i0 < SZ; i0 += 64) {
        const uint32_t i = i0 + CPT * (tid / L);
        const bool live = i < SZ; // head sizes below 64 leave waves without a column
        const uint32_t chan = head * SZ + min(i, (uint32_t)(SZ - CPT));
        float *const rows = state + view_elem(vs, slot, G::first_row(l) + 1, chan); // the lane's rows of S, ROW_STEP rows of the state apart
        float s[JL][CPT], wc[TOKEN_DECAY ? 1 : JL]; // wc: the constant decay of this lane's rows
        if constexpr (!TOKEN_DECAY) {
#pragma unroll
            for (int jj = 0; jj < JL; jj++) wc[jj] = time_decay[head * SZ + G::first_row(l) + G::ROW_STEP * jj];
        }
        bool held = false;
        for (base = 0; base < A; base += kSlotScan) {
            n = slot_tokens<G::THREADS>(cursors, base, A, slot, slots, every, list, count);
            if (n == 0) continue;
            fetch(0);
            if (!held) {
#pragma unroll
                for (int jj = 0; jj < JL; jj++) load_cols(s[jj], rows + (uint64_t)(G::ROW_STEP * jj) * vs.stride[0]);
                held = true;
            }
            const uint32_t nchunk = (n + TB - 1) / TB;
            __syncthreads(); // the buffers may still be read
            stage(0);
            for (uint32_t chunk = 0; chunk < nchunk; chunk++) {
                const int buf = chunk & 1;
                const uint2 cg = fg;
                const IV cx = fx;
                const uint32_t ct = ft;
                if (chunk + 1 < nchunk) fetch(chunk + 1);
                __syncthreads(); // chunk `chunk` is in LDS; buffer buf ^ 1 is free
                const uint32_t tend = min((uint32_t)TB, n - chunk * TB);
                if (!GATE && first_pass && staging && lt < tend && keeps_input(tsh[buf], csh[buf], lt, tend))
                    *reinterpret_cast<float4 *>(state + view_elem(vs, slot, 0, head * SZ + le)) = load_vec4(reinterpret_cast<const IT *>(&cx));
                if (live) {
                    float yo[CPT] = {}; // y of token u of a group of L in lane u of the L that share the columns
                    auto token = [&](uint32_t tt, int u) {
                        float vv[CPT], y[CPT];
                        load_cols(vv, &vsh[buf][tt * SZ + i]);
                        const float *kp = &ks[buf][tt * SZ + l * JL], *rp = &rs[buf][tt * SZ + l * JL], *wp = &ws[TOKEN_DECAY ? buf : 0][TOKEN_DECAY ? tt * SZ + l * JL : 0];
                        float y2[CPT][PARTS] = {};
#pragma unroll
                        for (int q = 0; q < JL / 4; q++) {
                            const float4 k4 = *reinterpret_cast<const float4 *>(kp + 4 * q), r4 = *reinterpret_cast<const float4 *>(rp + 4 * q);
                            const float kk[4] = {k4.x, k4.y, k4.z, k4.w}, rr[4] = {r4.x, r4.y, r4.z, r4.w};
                            float ww[4];
                            if constexpr (TOKEN_DECAY) {
                                const float4 w4 = *reinterpret_cast<const float4 *>(wp + 4 * q);
                                ww[0] = w4.x, ww[1] = w4.y, ww[2] = w4.z, ww[3] = w4.w;
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++) ww[e] = wc[4 * q + e];
                            }
#pragma unroll
                            for (int e = 0; e < 4; e++)
#pragma unroll
                                for (int c = 0; c < CPT; c++) {
                                    float &sv = s[4 * q + e][c];
                                    y2[c][e % PARTS] = fmaf(rr[e], sv, y2[c][e % PARTS]);
                                    sv = fmaf(ww[e], sv, kk[e] * vv[c]);
                                }
                        }
#pragma unroll
                        for (int c = 0; c < CPT; c++) {
                            y[c] = lanes_sum<L>(parts_sum(y2[c]));
                            if (!GATE) y[c] = fmaf(bonus[buf][tt], vv[c], y[c]);
                            yo[c] = l == (uint32_t)u ? y[c] : yo[c];
                        }
                    };
                    walk_tokens<L, JL>(tend, token, [&](uint32_t from, uint32_t count) {
                        if constexpr (GATE) {
                            if (l < count) store_cols(&ysh[(from + l) * SZ + i], yo);
                        } else {
                            store_tokens(count, l, tsh[buf] + from, yo, x, C, chan);
                        }
                    });
                }
                if constexpr (GATE) {
                    __syncthreads(); // the chunk's y are in LDS
                    if (staging && lt < tend) {
                        if (keeps_input(tsh[buf], csh[buf], lt, tend)) *reinterpret_cast<float4 *>(state + view_elem(vs, slot, 0, head * SZ + le)) = load_vec4(reinterpret_cast<const IT *>(&cx));
                        const float4 y0 = *reinterpret_cast<const float4 *>(&ysh[4 * tid]), v4 = *reinterpret_cast<const float4 *>(&vsh[buf][4 * tid]);
                        const float b = bonus[buf][lt];
                        const float4 o = head_norm(make_float4(fmaf(b, v4.x, y0.x), fmaf(b, v4.y, y0.y), fmaf(b, v4.z, y0.z), fmaf(b, v4.w, y0.w)), gw, gb, ga.eps);
                        const float4 g4 = load_vec4(reinterpret_cast<const uint16_t *>(&cg));
                        auto gate = [](float gv, float ov) { return act_one<WRQ_ACT_SILU>(gv) * round_h(ov); };
                        store_vec4(ga.att_x + ((uint64_t)ct * C + head * SZ + le), make_float4(gate(g4.x, o.x), gate(g4.y, o.y), gate(g4.z, o.z), gate(g4.w, o.w)));
                    }
                }
                if (chunk + 1 < nchunk) stage(buf ^ 1); // read two chunks ago, before the barrier above
            }
        }
        if (live && held) {
#pragma unroll
            for (int jj = 0; jj < JL; jj++) store_cols(rows + (uint64_t)(G::ROW_STEP * jj) * vs.stride[0], s[jj]);
        }
        first_pass = false;
    }
}

// v7, with a = -kk, b = kk * a_in and w = exp(-exp(-0.5) sigmoid(w_in)):
//   sa[i] = sum_j S[j][i] a[j];   S[j][i] <- S[j][i] w[j] + k[j] v[i] + sa[i] b[j];   y[i] = sum_j r[j] S[j][i]
// GATE: the fused form; y (rounded to f16) then goes through the group norm, the bonus (sum_j u[j] k[j] r[j]) v[i]
// (u = `first`) and the gate g into att_x, rounded to f16 after each as the op list stores it.
template <typename XT, int SZ, bool GATE, bool WIDE = false>
__global__ __launch_bounds__((RecurrenceTile<SZ, WIDE>::THREADS)) void time_mix_v7_kernel(const uint32_t *cursors, float *state, const XT *r, const XT *w, const XT *n_, XT *x, ViewArgs vs,
                                                          uint32_t H, uint32_t A, const uint16_t *first, GateArgs ga) {
    using G = RecurrenceTile<SZ, WIDE>;
    constexpr int L = G::L, CPT = G::CPT, JL = G::JL, TB = G::TB, TL = G::TL, PARTS = G::PARTS;
    static_assert(!GATE || (SZ == 64 && sizeof(XT) == 2), "the fused form: head size 64, f16 operands");
    __shared__ __align__(16) float rs[2][1024], ws[2][1024], ks[2][1024], as[2][1024], bs[2][1024], vsh[2][1024], ysh[GATE ? 1024 : 4];
    __shared__ uint32_t csh[2][TB], tsh[2][TB]; // cursors and numbers of the chunk's tokens
    __shared__ uint8_t list[kSlotScan];
    __shared__ uint32_t count[kSlotScan / 64];
    const uint32_t head = blockIdx.x, slots = vs.shape[2], tid = threadIdx.x;
    const bool every = slots == 1 || A == 1;
    uint32_t slot;
    if (!own_slot(cursors, A, slots, &slot)) return;
    const uint32_t l = tid % L;
    const uint32_t C = SZ * H;
    const uint64_t plane = (uint64_t)A * C; // n_ holds k, v, a, kk one after the other
    const uint32_t lt = (tid % 256) / TL, le = 4 * (tid % TL);
    const bool staging = !WIDE || tid < 256;
    uint2 gw = make_uint2(0, 0), gb = make_uint2(0, 0);
    float4 u4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (GATE) {
        gw = *reinterpret_cast<const uint2 *>(ga.gn_w + head * SZ + le), gb = *reinterpret_cast<const uint2 *>(ga.gn_b + head * SZ + le);
        u4 = load_vec4(first + head * SZ + le);
    }
    float4 fr, fw, fk, fv, fa, fkk;
    using IT = std::conditional_t<GATE, uint16_t, XT>;
    using IV = std::conditional_t<sizeof(IT) == 2, uint2, float4>;
    const IT *in;
    if constexpr (GATE) in = ga.att_x;
    else in = x;
    uint2 fg = make_uint2(0, 0);
    IV fx = {};
    bool first_pass = true; // over the columns: the later ones find x overwritten
    uint32_t fc = 0, ft = 0, fct = 0;
    uint32_t base = 0, n = 0;
    auto fetch = [&](uint32_t chunk) {
        if (!staging) return;
        auto token = [&](uint32_t j) { return base + (every ? min(j, n - 1) : (uint32_t)list[min(j, n - 1)]); }; // clamped: past the slot's tokens, never used
        ft = token(chunk * TB + lt);
        const uint64_t g = (uint64_t)ft * C + head * SZ + le;
        fr = load_vec4(r + g), fw = load_vec4(w + g), fk = load_vec4(n_ + g), fv = load_vec4(n_ + plane + g);
        fa = load_vec4(n_ + 2 * plane + g), fkk = load_vec4(n_ + 3 * plane + g);
        if constexpr (GATE) fg = *reinterpret_cast<const uint2 *>(ga.g + g);
        if (SZ <= 64 || first_pass) fx = *reinterpret_cast<const IV *>(in + g);
        if (GATE) fc = cursors[ft];
        else if (tid < (uint32_t)TB) fct = token(chunk * TB + tid), fc = cursors[fct];
    };
    auto decay = [](float v) { return expf(-0.606531f / (1.0f + expf(-v))); }; // exp(-exp(-0.5) sigmoid(w))
    auto stage = [&](int buf) {
        if (!staging) return;
        G::put_rows(rs[buf], tid, fr);
        G::put_rows(ws[buf], tid, make_float4(decay(fw.x), decay(fw.y), decay(fw.z), decay(fw.w)));
        G::put_rows(ks[buf], tid, fk);
        G::put_rows(as[buf], tid, make_float4(-fkk.x, -fkk.y, -fkk.z, -fkk.w));
        G::put_rows(bs[buf], tid, make_float4(fkk.x * fa.x, fkk.y * fa.y, fkk.z * fa.z, fkk.w * fa.w));
        *reinterpret_cast<float4 *>(&vsh[buf][4 * tid]) = fv;
        if (GATE && tid % TL == 0) csh[buf][lt] = fc, tsh[buf][lt] = ft;
        if (!GATE && tid < (uint32_t)TB) csh[buf][tid] = fc, tsh[buf][tid] = fct;
    };
    for (uint32_t i0 = 0; i0 < SZ; i0 += 64) {
        const uint32_t i = i0 + CPT * (tid / L);
        const bool live = i < SZ; // head sizes below 64 leave waves without a column
        const uint32_t chan = head * SZ + min(i, (uint32_t)(SZ - CPT));
        float *const rows = state + view_elem(vs, slot, G::first_row(l) + 1, chan); // the lane's rows of S, ROW_STEP rows of the state apart
        float s[JL][CPT];
        bool held = false;
        for (base = 0; base < A; base += kSlotScan) {
            n = slot_tokens<G::THREADS>(cursors, base, A, slot, slots, every, list, count);
            if (n == 0) continue;
            fetch(0);
            if (!held) {
#pragma unroll
                for (int jj = 0; jj < JL; jj++) load_cols(s[jj], rows + (uint64_t)(G::ROW_STEP * jj) * vs.stride[0]);
                held = true;
            }
            const uint32_t nchunk = (n + TB - 1) / TB;
            __syncthreads(); // the buffers may still be read
            stage(0);
            for (uint32_t chunk = 0; chunk < nchunk; chunk++) {
                const int buf = chunk & 1;
                const uint2 cg = fg;
                const IV cx = fx;
                const uint32_t ct = ft;
                if (chunk + 1 < nchunk) fetch(chunk + 1);
                __syncthreads(); // chunk `chunk` is in LDS; buffer buf ^ 1 is free
                const uint32_t tend = min((uint32_t)TB, n - chunk * TB);
                if (!GATE && first_pass && staging && lt < tend && keeps_input(tsh[buf], csh[buf], lt, tend))
                    *reinterpret_cast<float4 *>(state + view_elem(vs, slot, 0, head * SZ + le)) = load_vec4(reinterpret_cast<const IT *>(&cx));
                if (live) {
                    float yo[CPT] = {}; // y of token u of a group of L in lane u of the L that share the columns
                    auto token = [&](uint32_t tt, int u) {
                        float vv[CPT], sa[CPT], za[CPT][PARTS] = {}, acc[CPT][PARTS] = {};
                        load_cols(vv, &vsh[buf][tt * SZ + i]);
                        const uint32_t at = tt * SZ + l * JL;
#pragma unroll
                        for (int q = 0; q < JL / 4; q++) {
                            const float4 a4 = *reinterpret_cast<const float4 *>(&as[buf][at + 4 * q]);
                            const float aa[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
                            for (int e = 0; e < 4; e++)
#pragma unroll
                                for (int c = 0; c < CPT; c++) za[c][e % PARTS] = fmaf(s[4 * q + e][c], aa[e], za[c][e % PARTS]);
                        }
#pragma unroll
                        for (int c = 0; c < CPT; c++) sa[c] = lanes_sum<L>(parts_sum(za[c]));
#pragma unroll
                        for (int q = 0; q < JL / 4; q++) {
                            const float4 w4 = *reinterpret_cast<const float4 *>(&ws[buf][at + 4 * q]), k4 = *reinterpret_cast<const float4 *>(&ks[buf][at + 4 * q]),
                                         b4 = *reinterpret_cast<const float4 *>(&bs[buf][at + 4 * q]), r4 = *reinterpret_cast<const float4 *>(&rs[buf][at + 4 * q]);
                            const float ww[4] = {w4.x, w4.y, w4.z, w4.w}, kk[4] = {k4.x, k4.y, k4.z, k4.w}, bb[4] = {b4.x, b4.y, b4.z, b4.w},
                                        rr[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
                            for (int e = 0; e < 4; e++)
#pragma unroll
                                for (int c = 0; c < CPT; c++) {
                                    float &sv = s[4 * q + e][c];
                                    sv = fmaf(sa[c], bb[e], fmaf(sv, ww[e], kk[e] * vv[c]));
                                    acc[c][e % PARTS] = fmaf(rr[e], sv, acc[c][e % PARTS]);
                                }
                        }
#pragma unroll
                        for (int c = 0; c < CPT; c++) {
                            const float y = lanes_sum<L>(parts_sum(acc[c]));
                            yo[c] = l == (uint32_t)u ? y : yo[c];
                        }
                    };
                    walk_tokens<L, JL>(tend, token, [&](uint32_t from, uint32_t count) {
                        if constexpr (GATE) {
                            if (l < count) store_cols(&ysh[(from + l) * SZ + i], yo);
                        } else {
                            store_tokens(count, l, tsh[buf] + from, yo, x, C, chan);
                        }
                    });
                }
                if constexpr (GATE) {
                    __syncthreads(); // the chunk's y are in LDS
                    if (staging && lt < tend) {
                        if (keeps_input(tsh[buf], csh[buf], lt, tend)) *reinterpret_cast<float4 *>(state + view_elem(vs, slot, 0, head * SZ + le)) = load_vec4(reinterpret_cast<const IT *>(&cx));
                        const float4 y0 = *reinterpret_cast<const float4 *>(&ysh[4 * tid]), v4 = *reinterpret_cast<const float4 *>(&vsh[buf][4 * tid]);
                        const float4 k4 = G::get_rows(ks[buf], tid), r4 = G::get_rows(rs[buf], tid);
                        const float b = lanes_sum<16>((u4.x * k4.x * r4.x + u4.y * k4.y * r4.y) + (u4.z * k4.z * r4.z + u4.w * k4.w * r4.w));
                        const float4 o = head_norm(make_float4(round_h(y0.x), round_h(y0.y), round_h(y0.z), round_h(y0.w)), gw, gb, ga.eps);
                        const float4 g4 = load_vec4(reinterpret_cast<const uint16_t *>(&cg));
                        auto gate = [&](float gv, float ov, float vv) { return gv * round_h(round_h(ov) + b * vv); };
                        store_vec4(ga.att_x + ((uint64_t)ct * C + head * SZ + le),
                                   make_float4(gate(g4.x, o.x, v4.x), gate(g4.y, o.y, v4.y), gate(g4.z, o.z, v4.z), gate(g4.w, o.w, v4.w)));
                    }
                }
                if (chunk + 1 < nchunk) stage(buf ^ 1); // read two chunks ago, before the barrier above
            }
        }
        if (live && held) {
#pragma unroll
            for (int jj = 0; jj < JL; jj++) store_cols(rows + (uint64_t)(G::ROW_STEP * jj) * vs.stride[0], s[jj]);
        }
        first_pass = false;
    }
}

// Workgroups per head: one per state slot a cursor can name (8 bits, the last slot of the view for what lies beyond it), and no
// more than tokens: idle slots are workgroups that look at the cursors and end, and a state holds more slots than a short run
// names (64 heads, one request of one token, v6 gate form: 7.1 -> 4.9 us with 32 slots, 22.9 -> 4.9 with 256; one slot 4.9).
inline uint32_t slot_grid(const ViewArgs &vs, uint32_t A) {
    const uint32_t slots = vs.shape[2] < 256u ? vs.shape[2] : 256u;
    return A < slots ? A : slots;
}

} // namespace wrq
