// Products on packed weights for short runs (a few tokens up to 48, small products up to 256) for gfx950, on the f16 matrix cores:
// the same sums as gemm.hip (src/shaders/matmul_vec_int8.wgsl, matmul_vec_nf4.wgsl, matmul_mat_int8.wgsl,
// matmul_mat_nf4.wgsl), split over the machine in another way.
//
// A short run reads every weight once and has little to do with it, so a launch is a few microseconds long and what counts
// is how soon all its loads are under way and how few times a wave has to wait for another one.  The chunk kernel of gemm.hip
// shares one activation tile between the waves of a workgroup: a barrier per K step or four, narrow grids, and a split of K
// over the grid with a second launch (4.5 us) where rows are few.  Here
//   * a workgroup owns 16 * MRT rows and the whole K; its NW waves take the K steps (128 * SUB elements) in turn and each
//     keeps everything it needs to itself: weights and activations go line-wise from memory into registers (a row's bytes of
//     a step in adjacent lanes) and through a slot of LDS that belongs to the wave into operand layout, while the next step is
//     on its way.  No barrier between the first load and the sum of the waves' partial tiles at the end, no second launch;
//   * activations come first in a step's loads and in the order of their use, so that staging starts on the first of them;
//     buffer loads keep addresses in scalar registers and return zeros for rows and tokens past the end;
//   * the first product's operands are leading scalar arguments (preloaded); what only the end of the kernel needs is
//     fetched before the first step, behind the loads.
// Bound: at 5 .. 16 tokens the stream of weights (with the latency of one launch), from 17 tokens on the activations
// that every workgroup fetches and stages again (2 K T bytes against 16 MRT K or half of that) and, for nf4, the table lookups.
// Scales are applied per block in f32 as in gemm.hip: the f16 operands stay exact.  Lines of the rules below are where the time against the kernels that took these
// launches before crosses 1, on a grid of 18 row counts x 21 K x 23 run lengths and drawn groups of products.
//
// Measured (us per launch in a graph over cold copies, chunk kernel -> here; attention group / att.output / {ffn.key,
// ffn.receptance} / ffn.value): 1.6B nf4 at 5 tokens 8.2 / 5.8 / 10.4 / 10.6 -> 6.2 / 4.1 / 7.5 / 7.8; 3B int8 at 19
// tokens 14.3 / 8.4 / 14.4 / 16.5 -> 9.9 / 5.7 / 10.1 / 13.0; 7B int8 at 8 tokens 18.7 / 10.3 / 23.3 / 19.7 ->
// 14.4 / 6.1 / 18.5 / 14.2; 7B nf4 at 32 tokens 25.7 / 12.7 / 33.0 / 24.0 -> 20.5 / 8.7 / 26.8 / 22.9.
#include "gemm_device.h"
#include "wrq_host.h"

#include <iterator>

namespace wrq {

// Geometry of one instantiation: 16 * MRT rows, up to TOK tokens, NW waves that split K in steps of 128 * SUB elements.
template <int QUANT, int MRT, int TOK, int NW, int SUB>
struct ShortGeometry {
    static constexpr bool N4 = QUANT == kNf4;
    static constexpr int KST = 128 * SUB;
    static constexpr int WB = N4 ? KST / 2 : KST;  // weight bytes per row and step
    static constexpr int NT = (TOK + 15) / 16;     // token tiles; the last may be half full (TOK = 8, 24)
    static constexpr int XL = TOK * KST * 2 / 1024; // 1 KiB activation loads per wave and step
    static constexpr int WL = 16 * MRT * WB / 1024; // 1 KiB weight loads per wave and step
    static constexpr int XPITCH = KST * 2 + 16;     // bytes per staged token: +16 B rotates the banks
    static constexpr int WPITCH = WB + 16;
    // a wave's slot: weights | activations | scales [2 * SUB][16 * MRT] f32 | token sums [SUB][TOK] f32 (int8);
    // the wave's partial tile takes its place at the end
    static constexpr int W_BYTES = MRT * 16 * WPITCH, X_BYTES = TOK * XPITCH, S_BYTES = MRT * 16 * 4 * 2 * SUB;
    static constexpr int STAGED = W_BYTES + X_BYTES + S_BYTES + (N4 ? 0 : TOK * 4 * SUB), PARTIAL = MRT * NT * 1024;
    static constexpr int SLOT = STAGED > PARTIAL ? STAGED : PARTIAL;
    static constexpr int TABLE = N4 ? 256 * 8 : 0;
    static constexpr int LDS = TABLE + SLOT * NW;
    static_assert(LDS <= 160 * 1024 && SLOT % 16 == 0, "a workgroup's slots fit the LDS of a CU");
};

struct ShortArgs {
    uint32_t begin[kMaxGroup]; // first workgroup of every product, unused entries 0xffffffff
    MatmulArgs m[kMaxGroup];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00027000);
}

template <int AUX>
__device__ __forceinline__ uint4 buffer_load128(__amdgpu_buffer_rsrc_t r, uint32_t offset) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, AUX));
    return make_uint4(v.x, v.y, v.z, v.w);
}
constexpr int kStream = 2; // nt: weights are read once (7B int8 at 8 tokens 15.9 against 16.9 us without)

// CENTRED (int8, runs of 2 .. 4 tokens, which the decode kernels took before): codes enter as u - 128 instead of 1024 + u and the step of a block
// is rounded correctly.  The decode kernels cancel 1024 sum_k x over 16 elements, the sums below over 128, which loses more:
// f32 outputs against 64 bits, decode kernels / 1024 + u / u - 128: 7680 x 2560, 3 tokens, normal inputs 1.4e-6 / 2.0e-6 / 1.0e-7, squared relu of them
// 3.9e-6 / 8.5e-6 / 3.0e-7 (with 1 / 255 rounded once, as elsewhere, the last is 3.2e-6: an error of one sign).  Costs 2 % of a launch.
template <int QUANT, int MRT, int TOK, int NW, int SUB, bool CENTRED>
__global__ __launch_bounds__(64 * NW) void gemm_short_kernel(const uint8_t *w0, const uint16_t *scale0, const void *x0, const float *quant0,
                                                             const uint32_t begin1, const uint32_t R0, const uint32_t x_stride0, const uint32_t K,
                                                             const uint32_t T_all, const uint32_t tblocks, const ShortArgs a) {
    using G = ShortGeometry<QUANT, MRT, TOK, NW, SUB>;
    constexpr bool N4 = G::N4;
    constexpr int NT = G::NT, XL = G::XL, WL = G::WL, KST = G::KST, WB = G::WB;
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15, g = lane >> 4;
    const uint8_t *w = w0;
    const uint16_t *scale = scale0;
    const void *x = x0;
    const float *quant = quant0;
    uint32_t R = R0, x_stride = x_stride0, pi = 0, wg = blockIdx.x;
    if (blockIdx.x >= begin1) {
        pi = 1;
#pragma unroll
        for (uint32_t i = 2; i < (uint32_t)kMaxGroup; i++)
            if (blockIdx.x >= a.begin[i]) pi = i;
        const MatmulArgs &m = a.m[pi];
        w = m.w, scale = m.scale, x = m.x, quant = m.quant, R = m.R, x_stride = (uint32_t)m.x_token_stride;
        wg -= a.begin[pi];
    }
    uint32_t t0 = 0;
    if (tblocks > 1) { // the token blocks of one row tile run on one XCD one after the other: its L2 serves their weights
        const uint32_t slot = wg >> 3;
        t0 = slot % tblocks * TOK;
        wg = slot / tblocks * 8 + (wg & 7);
        if (wg * (16 * MRT) >= R) return; // padding to eight row tiles
        x = static_cast<const uint16_t *>(x) + (uint64_t)t0 * x_stride;
    }
    const uint32_t T = min(T_all - t0, (uint32_t)TOK); // of this workgroup
    const uint32_t row0 = wg * (16 * MRT);
    uint2 *pair = reinterpret_cast<uint2 *>(smem);
    uint8_t *const slot = smem + G::TABLE + wv * G::SLOT;
    uint8_t *const ws = slot, *const xs = slot + G::W_BYTES;
    float *const scl = reinterpret_cast<float *>(xs + G::X_BYTES); // nf4: absmax of block b at [b][row]; int8: (s, min - 1024 s) of step u at [2 u][row], [2 u + 1][row]
    float *const sxs = scl + MRT * 16 * 2 * SUB;                   // int8: token sums at [u][token]
    // nf4: requested before everything else, so that the table is written while the weights are on their way
    float tq0 = 0.0f, tq1 = 0.0f;
    if (N4) tq0 = quant[tid & 15], tq1 = quant[(tid >> 4) & 15];

    const uint32_t rows = min((uint32_t)(16 * MRT), R - row0);
    const uint32_t row_bytes = N4 ? K / 2 : K, scale_bytes = K / 128 * 4; // one 32-bit scale word per row and 128 elements in both formats
    const auto rw = buffer_of(w + (size_t)row0 * row_bytes, rows * row_bytes);
    const auto rs = buffer_of(reinterpret_cast<const uint8_t *>(scale) + (size_t)row0 * scale_bytes, rows * scale_bytes);
    const auto rx = buffer_of(x, ((T - 1) * x_stride + K) * 2);
    constexpr int LPR = WB / 16, RPL = 64 / LPR; // lanes per row and rows per weight load
    constexpr int LPT = KST / 8, TPL = 64 / LPT; // lanes per token and tokens per activation load
    const uint32_t w_lane = (lane / LPR) * row_bytes + 16 * (lane % LPR), x_lane = (lane / LPT) * (x_stride * 2) + 16 * (lane % LPT);
    const uint32_t s_lane = lane * scale_bytes; // lane = row of the workgroup; rows past the end read zeros

    // The waves take the steps in turn.  Rows a multiple of 4 KiB apart lie on the same memory channels: there every workgroup
    // starts at another step (7B int8 at 8 tokens, attention group: 15.6 -> 14.6 us; other row lengths lose 1 % from it).
    const uint32_t nsteps = K / KST, count = (nsteps + NW - 1 - wv) / NW;
    const uint32_t turn = row_bytes % 4096 == 0 ? (wg * 5) % nsteps : 0;

    struct Step {
        uint4 x[XL], w[WL];
        uint32_t s[SUB];
    } st;
    auto load = [&](uint32_t m) {
        uint32_t s = min(wv + m * NW, nsteps - 1) + turn;
        s = s >= nsteps ? s - nsteps : s;
#pragma unroll
        for (int i = 0; i < XL; i++) st.x[i] = buffer_load128<0>(rx, x_lane + (i * TPL * x_stride * 2 + s * (KST * 2)));
        if constexpr (SUB == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, s_lane + s * 8, 0, 0);
            st.s[0] = v[0], st.s[SUB - 1] = v[1];
        } else {
            st.s[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, s_lane + s * 4, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < WL; i++) st.w[i] = buffer_load128<kStream>(rw, w_lane + (i * RPL * row_bytes + s * WB));
    };
    // nf4 rows as long as a single row tile may have them: even and odd blocks are summed apart, which halves the longest chain
    // of f32 additions (14336 x 4096, f32 outputs against 64 bits: 1.33e-7 in one chain, the chunk kernel's K split 1.20e-7)
    constexpr int CHAINS = N4 && MRT == 1 ? 2 : 1;
    float4v out[CHAINS][MRT][NT];
    const float4v zero4 = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < CHAINS; c++)
#pragma unroll
        for (int i = 0; i < MRT; i++)
#pragma unroll
            for (int n = 0; n < NT; n++) out[c][i][n] = zero4;

    load(0);
    __builtin_amdgcn_sched_barrier(0); // the order of these loads is the order of the loop's
    if (N4) {
        // entry for byte v: (hi(q[v & 15]), hi(q[v >> 4])), (lo(..), lo(..)); lo scaled by 2^11
        const float h0 = h2f(f2h(tq0)), h1 = h2f(f2h(tq1));
        if (tid < 256) pair[tid] = make_uint2(pack_h2(tq0, tq1), pack_h2((tq0 - h0) * 2048.0f, (tq1 - h1) * 2048.0f));
        lds_barrier();
    }
    // scalar loads of cold argument memory, waited for here rather than in front of the stores (0.1 us per launch)
    void *const o_ptr = a.m[pi].out;
    const uint64_t o_stride = a.m[pi].out_token_stride;
    const int o_f16 = a.m[pi].out_f16, o_act = a.m[pi].act;
    asm volatile("" ::"s"(o_ptr), "s"(o_stride), "s"(o_f16), "s"(o_act));

    uint32_t token[NT]; // staged token of this lane's column; of a half tile the upper columns repeat the lower ones and are not stored
    const uint8_t *xb[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        token[n] = 16 * n + (TOK - 16 * n < 16 ? (r16 & 7) : r16);
        xb[n] = xs + token[n] * G::XPITCH + 32 * g;
    }
    // B operands of 64 elements: lane (token, g) holds elements 16 g .. + 8 and 16 g + 8 .. + 16
    auto read_b = [&](int half, HalfPack (&b)[NT][2]) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint4 v = *reinterpret_cast<const uint4 *>(xb[n] + 128 * half + 16 * j);
                b[n][j].u[0] = v.x, b[n][j].u[1] = v.y, b[n][j].u[2] = v.z, b[n][j].u[3] = v.w;
            }
    };
#pragma unroll 1
    for (uint32_t m = 0; m < count; m++) {
        // registers -> the wave's slot (one wave writes and reads it, in program order: no barrier)
#pragma unroll
        for (int i = 0; i < XL; i++) {
            *reinterpret_cast<uint4 *>(xs + (i * TPL + lane / LPT) * G::XPITCH + 16 * (lane % LPT)) = st.x[i];
            if (!N4) { // the 16 pieces of a token and 128 elements sit in one DPP row
                float q = dot2_ones(st.x[i].x, 0.0f);
                q = dot2_ones(st.x[i].y, q);
                q = dot2_ones(st.x[i].z, q);
                q = dot2_ones(st.x[i].w, q);
                q = row16_sum(q);
                if ((lane & 15) == 0) sxs[((lane % LPT) / 16) * TOK + i * TPL + lane / LPT] = q;
            }
        }
#pragma unroll
        for (int i = 0; i < WL; i++) *reinterpret_cast<uint4 *>(ws + (RPL * i + lane / LPR) * G::WPITCH + 16 * (lane % LPR)) = st.w[i];
        if (lane < 16 * MRT) {
#pragma unroll
            for (int u = 0; u < SUB; u++) {
                const float lo = h2f((uint16_t)st.s[u]), hi = h2f((uint16_t)(st.s[u] >> 16));
                constexpr float kInv = 1.0f / 255.0f, kInvRest = (float)(1.0 / 255.0 - (double)kInv);
                const float s = CENTRED ? fmaf(hi - lo, kInv, (hi - lo) * kInvRest) : (hi - lo) * kInv; // (min, max) -> (s, min - 1024 s)
                scl[(2 * u) * 16 * MRT + lane] = N4 ? lo : s;
                scl[(2 * u + 1) * 16 * MRT + lane] = N4 ? hi : fmaf(CENTRED ? 128.0f : -1024.0f, s, lo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (m + 1 < count) load(m + 1);
        __builtin_amdgcn_sched_barrier(0);
        // Work items of a step: (64 elements, row tile), row tiles first.  Weights are read two items ahead, an item's table
        // lookups are issued in front of the matrix work of the item before it, whose sums are taken in behind the next one's.
        constexpr int ITEMS = 2 * SUB * MRT;
        HalfPack B[2][NT][2];
        auto scale_of = [&](int word, int i) { return *reinterpret_cast<const float4 *>(scl + word * 16 * MRT + 16 * i + 4 * g); };
        if constexpr (N4) {
            uint2 wq[2];
            HalfPack Ah[2][2], Al[2][2];
            float4 am[2];
            float4v Dh[2][NT], Dl[2][NT];
            auto read_w = [&](int it) { return *reinterpret_cast<const uint2 *>(ws + (16 * (it % MRT) + r16) * G::WPITCH + 32 * (it / MRT) + 8 * g); };
            auto lookup = [&](int it) {
                const int q = it & 1, blk = it / MRT;
                if (it % MRT == 0) read_b(blk, B[blk & 1]);
                const uint32_t ww[2] = {wq[q].x, wq[q].y};
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const uint2 e = pair[(ww[j] >> (8 * c)) & 0xffu];
                        Ah[q][j].u[c] = e.x;
                        Al[q][j].u[c] = e.y;
                    }
                am[q] = scale_of(blk, it % MRT);
                if (it + 2 < ITEMS) wq[q] = read_w(it + 2);
            };
            auto take_in = [&](int it) { // out += absmax * (D_hi + 2^-11 D_lo)
                const int q = it & 1, i = it % MRT, c = it / MRT % CHAINS;
                const float s[4] = {am[q].x, am[q].y, am[q].z, am[q].w};
#pragma unroll
                for (int n = 0; n < NT; n++)
#pragma unroll
                    for (int d = 0; d < 4; d++) out[c][i][n][d] = fmaf(s[d], fmaf(Dl[q][n][d], 1.0f / 2048.0f, Dh[q][n][d]), out[c][i][n][d]);
            };
            wq[0] = read_w(0);
            wq[1] = read_w(1);
            lookup(0);
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const int q = it & 1, blk = it / MRT;
                __builtin_amdgcn_sched_barrier(0);
                if (it > 0) take_in(it - 1);
                __builtin_amdgcn_sched_barrier(0);
                if (it + 1 < ITEMS) lookup(it + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    Dh[q][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah[q][0].h, B[blk & 1][n][0].h, zero4, 0, 0, 0);
                    Dl[q][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Al[q][0].h, B[blk & 1][n][0].h, zero4, 0, 0, 0);
                }
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    Dh[q][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah[q][1].h, B[blk & 1][n][1].h, Dh[q][n], 0, 0, 0);
                    Dl[q][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Al[q][1].h, B[blk & 1][n][1].h, Dl[q][n], 0, 0, 0);
                }
            }
            take_in(ITEMS - 1);
        } else {
            uint4 wq[2];
            float4v D[MRT][NT];
            auto read_w = [&](int it) { return *reinterpret_cast<const uint4 *>(ws + (16 * (it % MRT) + r16) * G::WPITCH + 64 * (it / MRT) + 16 * g); };
            read_b(0, B[0]);
            wq[0] = read_w(0);
            wq[1] = read_w(1);
#pragma unroll
            for (int it = 0; it < ITEMS; it++) {
                const int q = it & 1, half = it / MRT, i = it % MRT;
                __builtin_amdgcn_sched_barrier(0);
                const uint32_t ww[4] = {wq[q].x, wq[q].y, wq[q].z, wq[q].w};
                HalfPack A[2];
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int c = 0; c < 2; c++) { // 4 codes of one dword -> f16 pairs 1024 + u
                        A[j].u[2 * c] = __builtin_amdgcn_perm(0x64646464u, ww[2 * j + c], 0x04010400u);
                        A[j].u[2 * c + 1] = __builtin_amdgcn_perm(0x64646464u, ww[2 * j + c], 0x04030402u);
                        if constexpr (CENTRED) {
                            const half2v centre{(_Float16)1152.0f, (_Float16)1152.0f};
                            A[j].u[2 * c] = as_u32(as_h2(A[j].u[2 * c]) - centre);
                            A[j].u[2 * c + 1] = as_u32(as_h2(A[j].u[2 * c + 1]) - centre);
                        }
                    }
                if (it + 2 < ITEMS) wq[q] = read_w(it + 2);
                if (i == 0 && half + 1 < 2 * SUB) read_b(half + 1, B[(half + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < NT; n++)
                    D[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0].h, B[half & 1][n][0].h, (half & 1) == 0 ? zero4 : D[i][n], 0, 0, 0);
#pragma unroll
                for (int n = 0; n < NT; n++) D[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[1].h, B[half & 1][n][1].h, D[i][n], 0, 0, 0);
                if ((half & 1) && i == MRT - 1) { // a 128-block is complete: out += s * D + (min - 1024 s) * sum_k x
                    const int u = half >> 1;
#pragma unroll
                    for (int k = 0; k < MRT; k++) {
                        const float4 sv = scale_of(2 * u, k), cv = scale_of(2 * u + 1, k);
                        const float s[4] = {sv.x, sv.y, sv.z, sv.w}, c[4] = {cv.x, cv.y, cv.z, cv.w};
#pragma unroll
                        for (int n = 0; n < NT; n++) {
                            const float sx = sxs[u * TOK + token[n]];
#pragma unroll
                            for (int d = 0; d < 4; d++) out[0][k][n][d] = fmaf(s[d], D[k][n][d], fmaf(c[d], sx, out[0][k][n][d]));
                        }
                    }
                }
            }
        }
    }

    // The partial tiles of the waves, each in the wave's own slot, summed pairwise.  D layout of a 16 x 16 tile: lane holds
    // token column (lane & 15), rows 4 g .. 4 g + 3.
    float4 *const part = reinterpret_cast<float4 *>(slot);
#pragma unroll
    for (int i = 0; i < MRT; i++)
#pragma unroll
        for (int n = 0; n < NT; n++) {
            float4v o = out[0][i][n];
            if constexpr (CHAINS == 2) o += out[CHAINS - 1][i][n];
            part[(i * NT + n) * 64 + lane] = make_float4(o[0], o[1], o[2], o[3]);
        }
    lds_barrier();
    for (uint32_t q = tid; q < MRT * NT * 64; q += 64 * NW) {
        float4 e[NW];
#pragma unroll
        for (int u = 0; u < NW; u++) e[u] = *reinterpret_cast<const float4 *>(smem + G::TABLE + u * G::SLOT + 16 * q);
#pragma unroll
        for (int d = 1; d < NW; d *= 2)
#pragma unroll
            for (int u = 0; u < NW; u += 2 * d) e[u].x += e[u + d].x, e[u].y += e[u + d].y, e[u].z += e[u + d].z, e[u].w += e[u + d].w;
        const float4 v = e[0];
        const uint32_t tile = q >> 6, l = q & 63, i = tile / NT, n = tile % NT;
        const uint32_t row = row0 + 16 * i + 4 * (l >> 4), t = 16 * n + (l & 15);
        if (t >= T || row >= R) continue;
        const float o[4] = {act_apply(o_act, v.x), act_apply(o_act, v.y), act_apply(o_act, v.z), act_apply(o_act, v.w)};
        const uint64_t idx = (uint64_t)(t0 + t) * o_stride + row;
        if (o_f16)
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(o_ptr) + idx) = make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
        else
            *reinterpret_cast<float4 *>(reinterpret_cast<float *>(o_ptr) + idx) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

namespace {

template <int QUANT, int MRT, int TOK, int NW, int SUB, bool CENTRED = false>
int launch_one(hipStream_t stream, const MatmulArgs *args, int n) {
    using G = ShortGeometry<QUANT, MRT, TOK, NW, SUB>;
    auto *kern = &gemm_short_kernel<QUANT, MRT, TOK, NW, SUB, CENTRED>;
    if (G::LDS > 48 * 1024) {
        // one-time opt-in to more than the default dynamic LDS limit
        static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
        (void)once;
    }
    ShortArgs a;
    uint32_t total = 0;
    const uint32_t tblocks = (args[0].T + TOK - 1) / TOK;
    for (int i = 0; i < kMaxGroup; i++) {
        a.begin[i] = 0xffffffffu;
        if (i >= n) continue;
        a.m[i] = args[i];
        a.begin[i] = total;
        const uint32_t tiles = (args[i].R + 16 * MRT - 1) / (16 * MRT);
        total += tblocks > 1 ? (tiles + 7) / 8 * 8 * tblocks : tiles;
    }
    const MatmulArgs &m = args[0];
    hipLaunchKernelGGL(kern, dim3(total), dim3(64 * NW), G::LDS, stream, m.w, m.scale, m.x, m.quant, a.begin[1], m.R, (uint32_t)m.x_token_stride,
                       m.K, m.T, tblocks, a);
    return check_launch("matmul (short run)");
}

// Tile of a launch: row tiles, tokens, waves and 128-element pieces of a step; mrt 0: the chunk kernel is the faster one.
struct ShortTile {
    int mrt, tok, nw, sub;
};
constexpr ShortTile kNoTile{0, 0, 0, 0};

// Runs of up to 48 tokens in one token block.  Row tiles per workgroup: one up to 4096 rows (256 workgroups), then the fewest that
// leave one workgroup per CU; beyond 16384 rows no number does, and three keep the last round short (18432 x 4096 at 16 tokens: int8
// 21.0 us with 3, 24.8 with 4; nf4 20.1, 24.3).  Workgroups have eight waves, two per SIMD.  Where two rounds of workgroups with three row tiles run, and
// where the activations of 33 tokens and more leave no room for eight slots, they have four (18432 x 4096 at 24 / 32 tokens, four waves / eight: int8 24.2 / 24.6 and
// 26.1 / 27.0 us, nf4 25.3 / 27.1 and 26.3 / 28.6; 20480 x 5120 int8 31.9 / 31.2 and 34.5 / 33.6, nf4 31.6 / 33.6 and 33.5 / 35.3).
ShortTile one_block(Quant quant, uint64_t rows, uint32_t K, uint32_t T) {
    const uint64_t tiles = (rows + 15) / 16;
    const bool rounds = tiles > 1024;
    const int tok = T <= 8 ? 8 : T <= 16 ? 16 : T <= 24 ? 24 : T <= 32 ? 32 : 48;
    // up to 8 tokens activations are cheap: steps of 256 elements keep twice the bytes in flight.  One row tile of long
    // int8 rows (4096 x 14336: 14.2 against 14.8 us), and every grid of several rounds (nf4 18432 x 4096 17.8 against 19.2 us,
    // 20480 x 5120 22.0 against 24.7; int8 20480 x 5120 24.2 against 25.4)
    if (tok == 8 && K % 256 == 0 && (rounds || (quant == kInt8 && tiles <= 256 && K >= 7168))) return {1, tok, 8, 2};
    if (tiles <= 256) return {1, tok, 8, 1};
    if (tiles <= 512) return {2, tok, 8, 1};
    if (tok <= 32 && tiles <= 768) return {3, tok, 8, 1};
    if (tiles > 768 && !rounds) return {4, tok, tok <= 32 ? 8 : 4, 1};
    return {3, tok, tok <= 16 ? 8 : 4, 1};
}

// Most rows for which one block was measured the faster one: with more, its workgroups come in rounds that each begin with the
// latency of a whole K, while the chunk kernel's wide tiles read the activations less often.  Share of the chunk kernel's time, single
// products of 16384 .. 65536 rows, K of 768 .. 5120: int8 up to 8 tokens, K 1024: 20480 rows 0.97, 24576 1.06, 65536 1.45; K 2560 and more: 49152 rows
// 0.73 .. 0.88, 65536 up to 1.08; 9 .. 48 tokens, K from 2048: 24576 rows 0.79 .. 0.97, 32768 0.90 .. 1.26, 65536 up to 1.7.  nf4 up to 8 tokens, K below
// 2048: 16384 rows 0.83 .. 0.86, 20480 1.02 .. 1.10; up to 16 tokens otherwise: 49152 rows 0.61 .. 0.87, 65536 up to 1.04; up to 48 tokens: 24576 rows
// 0.58 .. 0.88, 32768 0.82 .. 1.19, 65536 1.06 .. 1.35.
uint64_t one_block_rows(Quant quant, uint32_t K, uint32_t T) {
    if (K < 512) return 16384; // K 256: int8 16620 rows, 5 tokens 1.05; nf4 29128 rows, 11 tokens 1.21
    if (quant == kNf4) return T > 16 ? 24576 : K < (T <= 8 ? 2048 : 768) ? 16384 : 49152;
    if (K < 2048) return T > 32 && K < 1024 ? 16384 : 20480; // 18664 x 512, 39 tokens 1.07
    return T <= 8 && K >= 2560 ? 49152 : 24576;
}

// Where one block is the faster split than the chunk kernel's (measured over the layer shapes of the
// 0.1B .. 14B models and 128 .. 6144 rows x 896 .. 14336, 5 .. 64 tokens).  With few rows most CUs have no workgroup and a
// long K is a long chain: there the chunk kernel's split of K over the grid wins, the sooner the more activations a
// workgroup has to fetch for its rows.
bool one_block_pays(Quant quant, uint64_t rows, uint32_t K, uint32_t T) {
    if (rows > one_block_rows(quant, K, T)) return false;
    const bool nf4 = quant == kNf4;
    if (T <= 8) return nf4 || rows >= 2048 || K <= 10240; // int8 1024 rows: K 8192 0.89 of the chunk kernel's time, 14336 1.01
    // int8 1024 rows: 4096 0.81, 8192 1.07; nf4 0.78, 0.95.  2048 rows, which the chunk kernel splits eight ways: int8 8960 0.97, 10240 1.08, 14336
    // 1.26; nf4 12288 1.00, 14336 1.07; 2560 rows of 14336 0.95, 0.82
    if (T <= 16) return rows > 2048 || K <= (nf4 ? (rows < 2048 ? 10240u : 12288u) : rows < 2048 ? 5120u : 8960u);
    if (T <= 24) return nf4 || K <= 10240 || (T <= 20 && rows >= 2048 && (rows > 4096 || K <= 14336)); // int8 4096 x 14336 at 19 / 24 tokens 0.92 / 1.04, 17920 at 20 1.04, 11260 x 15488 0.78; nf4 0.85
    if (T <= 32) {
        if (rows >= 2560) return nf4 ? rows > 4096 || K <= 15360 : K <= 8192; // 4096 x 14336 0.96 .. 1.02 (nf4), 1.18 (int8), 16384 nf4 1.03 .. 1.06, 5120 x 17920 1.02
        // 2048 x 7168 1.04 (nf4), 1.13 (int8); 1024 x 4096 int8 1.10 (its measured chunk tile serves up to 7 % around), 768 and 1280 rows 0.84 and 0.77
        return K <= 4096 && (nf4 || K < 3810 || rows < 953 || rows > 1095);
    }
    // 1.6B / 3B / 7B groups 0.7 .. 0.9, 2048 x 7168 1.02 .. 1.14; one K step: 16384 x 128 1.07 (int8), 1.20 (nf4)
    return T <= 48 && rows >= 2560 && K <= 8192 && (K >= 256 || rows <= 8192);
}

// Runs of 33 .. 256 tokens in several token blocks: where the smallest tile that gives every workgroup a CU of its own is the chunk
// kernel's better.  That is single products with few rows (att.output, ffn.value) and the groups of small models; as a share of the chunk
// kernel's time, int8 / nf4: att.output 1.6B 64 tokens 0.78 / 0.80, 128 0.70 / 0.78, 256 0.79 / 0.81, 7B 64 0.72 / 0.70, 128 0.79 / 0.72, 192 0.81 / 0.85;
// ffn.value 1.6B 128 tokens 0.90 / 0.74, 3B 128 0.90 / 0.83; attention group 0.4B 128 tokens 0.82 / 0.90, 1.6B 96 0.81 / 0.82.  In two rounds the
// chunk kernel is the faster one (1.6B attention group int8 192 tokens 1.05, 7B 128 1.14).
ShortTile several_blocks(Quant quant, const MatmulArgs *args, int n, uint64_t rows, uint32_t K, uint32_t T) {
    // long K: the chunk kernel splits it over the grid.  2560 x 8960 int8 64 tokens 1.04, 96 0.92; 4096 x 14336 int8 1.07 .. 1.28,
    // nf4 64 / 96 / 128 tokens 0.96 / 0.85 / 1.04
    if (T > 256 || K > (quant == kInt8 ? (T > 64 ? 10240u : 8192u) : T <= 96 ? 17920u : 10240u) || (K > 4096 && rows < 2048)) return kNoTile;
    // ... and where four row tiles are needed for one round: 4096 x 8960 at 112 and 128 tokens int8 1.12, nf4 1.00, 10240 1.27, 1.05; nf4 8192 x 8960 .. 17920 at 64
    // tokens 1.04 .. 1.11 (two row tiles, 48 tokens: 0.81 .. 0.91)
    if (K > 8192 && ((T > 96 && rows > 3072) || (T > 48 && T <= 64 && rows > 6144))) return kNoTile;
    // int8 10240: 2560 .. 4096 rows at 80 .. 128 tokens 1.02 .. 1.08, 2048 from 160 tokens on 1.04 .. 1.16; 5120 rows 0.94, 3072 at 160 tokens 0.89
    // (8960: 2048 rows at 224 and 256 tokens 1.04)
    if (quant == kInt8 && (K > 8960 ? rows <= (T > 128 ? 2560 : 4096) : K > 8192 && T > 192)) return kNoTile;
    // padding included: a launch is dealt to the XCDs round-robin, and 256 live workgroups among more are not 32 on each of them
    // (588 + 548 + 2804 + 1040 rows, 148 tokens, counted without: 1.42 of the chunk kernel's time)
    auto workgroups = [&](int mrt, int tok) {
        uint64_t w = 0;
        for (int i = 0; i < n; i++) w += ((args[i].R + 16 * mrt - 1) / (16 * mrt) + 7) / 8 * 8;
        return w * ((T + tok - 1) / tok);
    };
    constexpr uint64_t kOneRound = 256;
    constexpr ShortTile int8_tiles[] = {{1, 32, 8, 1}, {2, 32, 8, 1}, {3, 32, 8, 1}, {2, 48, 8, 1}, {4, 32, 8, 1}, {3, 48, 4, 1}, {4, 48, 4, 1}};
    constexpr ShortTile nf4_tiles[] = {{1, 32, 8, 1}, {1, 48, 8, 1}, {2, 32, 8, 1}, {2, 48, 8, 1}, {3, 32, 8, 1}, {4, 32, 8, 1}, {3, 48, 4, 1}, {4, 48, 4, 1}};
    const ShortTile *tile = quant == kInt8 ? std::begin(int8_tiles) : std::begin(nf4_tiles), *const end = quant == kInt8 ? std::end(int8_tiles) : std::end(nf4_tiles);
    for (; tile != end; tile++) // in the order of their size, near ties as measured
        if (workgroups(tile->mrt, tile->tok) <= kOneRound) break;
    // four waves instead of eight: long K loses what the wide tile saves (nf4 3036 x 7936, 214 tokens 1.06; 16296 x 9344, 34 tokens 1.16)
    // one K step keeps one wave busy: there wide tiles lose as well (K of 128, int8 3 and 4 x 48 1.01 .. 1.16; nf4 4 x 32 1.02 .. 1.14, 3 and 4 x 48 1.09 .. 1.31;
    // nf4 3 x 32 0.95 .. 1.07 from one run to another)
    if (tile != end && K < 256 && (tile->nw == 4 || (quant == kNf4 && tile->mrt == 4))) return kNoTile;
    if (tile != end) return tile->nw == 8 || K <= 5120 ? *tile : kNoTile;
    // int8, 64 x 64: from 2048 channels on (1.6B group 128 tokens 0.93, 3B and 7B 64 tokens 0.87 .. 0.90; 0.1B 256 tokens 1.08, 8040 x 7936,
    // 57 tokens 1.20; 3072 .. 5120 rows at 160 .. 256 tokens: K 4096 0.97 .. 1.04, 5120 1.04 .. 1.09)
    if (quant == kInt8 && K >= 2048 && K <= (T > 128 ? 4096 : 5120) && workgroups(4, 64) <= kOneRound) return {4, 64, 4, 1};
    // nf4, 64 x 48: two workgroups fit a CU.  Where they fill most of them and the last block is nearly full (3B 96 and 128 tokens 0.73,
    // 1.6B group 192 tokens 0.79, 7B 96 tokens 0.77; one block, 32768 rows, 0.82 .. 0.99, K of 5120 1.03; 288 .. 384 workgroups 0.95 .. 1.12, 64 tokens in two blocks 1.05 .. 1.20, K of 256 1.14)
    const uint64_t w = workgroups(4, 48);
    if (quant == kNf4 && K >= 1024 && K <= (T > 48 ? 5120 : 4096) && w >= 400 && w <= 2 * kOneRound && T * 8 >= (T + 47) / 48 * 48 * 7) return {4, 48, 4, 1};
    return kNoTile;
}

uint64_t rows_of(const MatmulArgs *args, int n) {
    uint64_t rows = 0;
    for (int i = 0; i < n; i++) rows += args[i].R;
    return rows;
}

// The tile of a launch, kNoTile where the chunk kernel takes it: the one place that decides.
ShortTile short_tile(Quant quant, const MatmulArgs *args, int n) {
    const uint32_t K = args[0].K, T = args[0].T;
    if (quant == kFp16 || T > 256 || K < 128 || !tune(kTuneGemmShort, 1)) return kNoTile;
    // a pinned tile of the chunk kernel means that kernel
    if (tune_is_set(kTuneGemmNtile) || tune_is_set(kTuneGemmMrt) || tune_is_set(kTuneGemmKg) || tune_is_set(kTuneGemmKsplit)) return kNoTile;
    // 32-bit byte offsets into a workgroup's rows and into the activations of its tokens
    for (int i = 0; i < n; i++)
        if (args[i].B != 1 || K > (1u << 24) || ((uint64_t)((T < 64 ? T : 64) - 1) * args[i].x_token_stride + K) * 2 > 0x7fffffffull) return kNoTile;
    const uint64_t rows = rows_of(args, n);
    return one_block_pays(quant, rows, K, T) ? one_block(quant, rows, K, T) : T > 32 ? several_blocks(quant, args, n, rows, K, T) : kNoTile;
}

template <int QUANT>
int launch_tile(hipStream_t stream, const MatmulArgs *args, int n, const ShortTile &t) {
    if constexpr (QUANT == kInt8) {
        if (args[0].T <= 4 && t.tok == 8) {
#define WRQ_SHORT(M, SUB) \
    if (t.mrt == M && t.nw == 8 && t.sub == SUB) return launch_one<QUANT, M, 8, 8, SUB, true>(stream, args, n);
            WRQ_SHORT(1, 2) WRQ_SHORT(1, 1) WRQ_SHORT(2, 1) WRQ_SHORT(3, 1) WRQ_SHORT(4, 1)
#undef WRQ_SHORT
        }
    }
#define WRQ_SHORT(M, TOK, NW, SUB) \
    if (t.mrt == M && t.tok == TOK && t.nw == NW && t.sub == SUB) return launch_one<QUANT, M, TOK, NW, SUB>(stream, args, n);
#define WRQ_SHORT_TOK(TOK) WRQ_SHORT(1, TOK, 8, 1) WRQ_SHORT(2, TOK, 8, 1) WRQ_SHORT(3, TOK, 8, 1) WRQ_SHORT(4, TOK, 8, 1)
    WRQ_SHORT(1, 8, 8, 2) WRQ_SHORT_TOK(8) WRQ_SHORT_TOK(16) WRQ_SHORT_TOK(24) WRQ_SHORT_TOK(32)
    WRQ_SHORT(3, 24, 4, 1) WRQ_SHORT(3, 32, 4, 1)
    WRQ_SHORT(1, 48, 8, 1) WRQ_SHORT(2, 48, 8, 1) WRQ_SHORT(3, 48, 4, 1) WRQ_SHORT(4, 48, 4, 1)
    if constexpr (QUANT == kInt8) { WRQ_SHORT(4, 64, 4, 1) }
#undef WRQ_SHORT_TOK
#undef WRQ_SHORT
    return fail(WRQ_ERR_UNSUPPORTED, "no short-run kernel for tile (%d, %d, %d, %d)", t.mrt, t.tok, t.nw, t.sub);
}

} // namespace

// Decode runs of 2 .. 4 tokens: where this kernel is faster than the decode kernels, which share a pass of the vector ALU between the
// tokens.  Those are at their best for int8 where whole waves own rows (K a multiple of 1024) and anywhere with long K and few rows.  Their
// time against this kernel's as 1, 600 drawn launches and the model shapes: int8, K < 1024: 2 tokens 0.84 .. 0.99, 3 and 4 0.59 .. 0.75;
// K up to 2560 from 1024 rows on, up to 10240 from 2560 rows on, 3 and 4 tokens 0.49 .. 0.85 (fewer rows 0.83 .. 1.6, beyond 10240 0.78 .. 1.7); whole waves,
// 4 tokens from 4096 rows on 0.75 .. 1.0, otherwise 0.95 .. 1.35.  nf4, K up to 1024: 2 tokens 0.66 .. 0.99, 3 0.52 .. 0.71; K up to 2560 0.67 .. 1.0
// (2 tokens: 9216 x 2048 1.06); K up to 5120 beyond 1024 rows, 3 tokens, 0.69 .. 1.04 (1024 rows,
// one task of the decode kernel per CU: K 4096 1.13, 5120 1.27), 2 tokens 0.84 .. 1.07; longer K 0.9 .. 1.8.
// Many rows, single products: int8, 4 tokens, K 1024: 16384 rows 0.88, 20480 1.12, 65536 1.23; K 2048: 20480 1.01, 32768 1.07; K 4096 and 5120 up to 65536 rows
// 0.83 .. 0.98; K 768, 3 and 4 tokens: 20480 rows 0.87, 65536 1.00; K 2560 up to 65536 rows 0.64 .. 0.76.  nf4, K 1024, 2 tokens: 16384 rows 0.83, 20480 1.03,
// 65536 1.11; 3 tokens, K of 768 .. 5120, up to 65536 rows 0.58 .. 0.97, but K 1792 19092 rows 1.08, 24876 1.16.
// nf4, f32 outputs against 64 bits: 0.85 .. 0.91 of the decode kernels' error for symmetric inputs, 1.00 .. 1.16 for inputs of one sign (of a layer's products ffn.value
// alone has those, and its K keeps it on the decode kernels).
// nf4 runs of 4 tokens through these entries are on the matrix cores anyway, so their launches were compared with the chunk kernel.
// Four products of K x K in one launch, before and now, us: int8 K 2560 3 tokens 10.7 -> 7.6, 4 tokens 10.7 -> 7.7; K 4096 4 tokens
// 15.9 -> 13.8; nf4 K 2048 2 tokens 6.5 -> 6.2, 3 tokens 7.7 -> 6.1; K 2560 3 tokens 11.8 -> 8.5; K 4096 3 tokens 17.0 -> 14.6.
bool short_run_pays(Quant quant, const MatmulArgs *args, int n) {
    const uint32_t K = args[0].K, T = args[0].T;
    if (T < 2 || T > 4 || !short_tile(quant, args, n).mrt) return false; // what `launch_gemm_short` hands on stays on the decode kernels
    // a pinned choice among the decode kernels means those
    for (const TuneKey key : {kTuneGemvOneshot, kTuneGemvRows, kTuneGemvSl, kTuneGemvNt, kTuneGemvGrid, kTuneGemvWaveRows, kTuneGemvRowsTokens})
        if (tune_is_set(key)) return false;
    const uint64_t rows = rows_of(args, n);
    if (quant == kInt8) {
        if (K % 1024 == 0) return T == 4 && rows >= 4096 && rows <= (K < 2048 ? 16384 : K < 4096 ? 20480 : 49152);
        if (K < 1024) return T > 2 || rows <= 8192; // 2 tokens, 16428 x 512 1.39
        return T > 2 && (K <= 2560 ? rows >= 1024 : K <= 10240 && rows >= 2560);
    }
    if (T == 2) return K <= 1024 || (K <= 2560 && rows >= 1024 && rows <= 8192);
    return K <= 2560 || (K <= 5120 && rows > 1024);
}

uint32_t short_run_tile(Quant quant, const MatmulArgs *args, int n) {
    const ShortTile t = short_tile(quant, args, n);
    return (uint32_t)(t.mrt | t.tok << 8 | t.nw << 16 | t.sub << 24);
}

// Takes the `n` products of a launch (one K and token count, f16 activations, one batch, K % 128 == 0 and the
// alignments of the chunk kernel) if this kernel is the faster one for them; false leaves them to the caller.
bool launch_gemm_short(hipStream_t stream, Quant quant, const MatmulArgs *args, int n, int &status) {
    const ShortTile t = short_tile(quant, args, n);
    if (!t.mrt) return false;
    status = quant == kNf4 ? launch_tile<kNf4>(stream, args, n, t) : launch_tile<kInt8>(stream, args, n, t);
    return true;
}

} // namespace wrq
