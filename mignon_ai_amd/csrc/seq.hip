// The model body over whole sequences in one kernel.
//
// The layered forward passes every token's rows through memory between its kernels (eight to nine launches per block,
// 0.4 to 1.5 KB per token each way) and is bound by that traffic and, for small batches, by the launches. For state
// sizes up to 128 a 16-token tile of the state is 32 registers per lane, so here a wave keeps its tile from the
// embedding to the head's operand and nothing but token ids, weights and the final rows touches memory.
//
// Layout. A workgroup is eight waves; wave w holds one 16-token tile of one sequence (floor(8 / tiles) sequences per
// workgroup). Every matrix product is v_mfma_i32_16x16x64_i8 with the weights as row operand, so lane L of a result
// tile holds token L & 15 and channels 4 * (L >> 4) + r. The operand of the next product wants 16 bytes of K per lane.
// The sum over K is exact in any order, so K is permuted inside each block of 64 instead of moving data between lanes:
// byte 4j + r of lane group g is channel 16j + 4g + r, which is what that lane already holds. The weights are stored
// in that order once (seq_pack). A row's maxima and sums combine four lanes (two shuffles).
//
// Activations are expanded to three base-256 digits with one scale per row (scale = amax / 127, digits of
// round(x * 127 * 65536 / amax), off by at most 0.75 / 8323072 of the row's maximum and without a mean: digits23_4).
//
// Weights are read by the workgroup as a stream of units of UF fragments (1 KiB each) in the order of use (a block's rule
// steps read the same units again, so that the stream is no longer than the weights whatever the step count), moved
// straight from memory into four LDS slots: while unit u is used, units u + 1 to u + 3 are on their way, one barrier a
// unit. A unit takes 1 to 2 thousand cycles and a load that misses the L2 about two thousand, so with only one unit
// between a request and its use (through registers, two slots) every unit waited some 500 cycles: 1024 x 128 tokens of
// the D128 model 756 -> 733 us, a call on 45 tokens 85.1 -> 81.8 us, scoring 60 documents 1486 -> 1432 us (a slower card
// than that of the comparison below).
//
// The latch recurrence g = lambda g + (1 - lambda) n runs over the tile's tokens as a scan over the 16 lanes of a DPP
// row (pairs (a, b) composed in four steps), then over the tiles through LDS (each tile's composed pair).
//
// Bound by the matrix cores and the vector units together, which two waves per SIMD only partly overlap: per sequence
// of 128 tokens of the D128 H256 two-block model about 95k matrix-core and 105k vector cycles per SIMD in 205k cycles.
// Measured against the layered body, whole calls in turn on one card: 1024 x 128 tokens of that model with logits and
// log-probabilities 1278 -> 709 us (about 200 of them the head's); 300 x 100 tokens of D96 H160 465 -> 277 us; 64 x 128
// of D32 H64 123 -> 40.5 us; the next-token call on 45 tokens of D96 H160, its head over one row instead of 45, 245 ->
// 82 us; scoring 60 documents with the D128 model, its last block only where a scored position depends on it, 3144 ->
// 1423 us. Where it is not the faster body: seq_pays.
#include <cmath>
#include <cstring>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"
#include "model_file.hpp"
#include "seq.hpp"

namespace mg {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// Units of the weight stream in LDS: the one in use and three on their way.
constexpr int kSlots = 4;

template <int DT, int HT, int ND>
struct Cfg {
    static constexpr int Dp = 64 * DT, Hp = 64 * HT;
    static constexpr int HW = HT <= 3 ? 2 : 1;  // highway channel tiles per unit
    static constexpr int UF = cmax(cmax(6 * DT, 2 * HW * HT), cmax(4 * DT, 3 * ND * DT));
    static constexpr int XS = Dp + 4;        // row stride of the normalised rows in LDS (floats)
    static constexpr int KS = 16 * ND + 4;   // row stride of a head's keys
    static constexpr int VS = kSeqMaxT + 4;  // row stride of a head's transposed values
    static constexpr int NV = Dp + 2 * Hp + 4 * Dp;  // vector floats in LDS: latch base, b1, b2, gamma, attention gamma
    static constexpr int o_x = kSlots * UF * 1024;
    static constexpr int o_k = o_x + kSeqMaxT * XS * 4;
    static constexpr int o_v = o_k + (ND ? kSeqMaxT * KS * 4 : 0);
    // The tiles' composed pairs. With attention they lie on the keys: a rule step is over, and the units of its products
    // lie between, when a head's keys are written, and the output product's units when the next block's pairs are.
    static constexpr int o_carry = ND ? o_k : o_v;
    static constexpr int carry = 8 * Dp * 8;
    static_assert(ND == 0 || carry <= kSeqMaxT * KS * 4 + 16 * ND * VS * 4, "");
    static constexpr int o_nmax = ND ? o_v + 16 * ND * VS * 4 : o_carry + carry;
    static constexpr int o_vec = o_nmax + kSeqMaxT * 4;
    static constexpr int lds = o_vec + NV * 4;
    // Waves per SIMD: four (two workgroups per CU, 128 registers) where a 64-channel state without attention leaves the
    // room, two (256 registers) otherwise.
    static constexpr int waves = DT == 1 && ND == 0 ? 4 : 2;
};

__device__ __forceinline__ void wg_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One 16-byte load per lane from global memory straight into LDS: lane L reads base + off and its bytes land at LDS offset
// lds + 16 L. Inline assembly, with the waits written out (vm_wait), because the compiler would wait for all such loads
// before any LDS read. The LDS address goes through M0. The base is a scalar register pair: a vector instruction may have
// written it (the compiler keeps spilled scalars in vector lanes), which takes five wait states before a memory instruction
// reads it, and one between the write of M0 and its use: the move counts one, the s_nop four. No register receives anything.
__device__ __forceinline__ void lds_load16(const int8_t* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "m0", "memory");
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// At most N of this wave's memory operations are outstanding (they complete in order).
template <int N>
__device__ __forceinline__ void vm_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// A value computed at this point: without it the compiler moves the last steps of each output to its use, units later,
// and keeps (spills) their several inputs until then.
__device__ __forceinline__ float here(float v) {
    asm volatile("" : "+v"(v));
    return v;
}

// sigmoid_epi without compares: beyond |x| = 15 the exponent is pushed to +-1e24 and more, so that 2^t is 0 or infinite
// and the result exactly 1 or 0.
__device__ __forceinline__ float sigmoid_med(float x) {
    const float lim = 15.0f * 1.4426950408889634f;
    const float t = x * -1.4426950408889634f;
    const float e = __builtin_amdgcn_exp2f(fmaf(t - __builtin_amdgcn_fmed3f(t, -lim, lim), 1e30f, t));
    return __builtin_amdgcn_rcpf(1.0f + e);
}

// Over the four lanes that hold a token.
__device__ __forceinline__ float row_max4(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float row_sum4(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

template <int N>
__device__ __forceinline__ float abs_max(const float (&v)[N]) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < N; i++) m = fmaxf(m, fabsf(v[i]));
    return m;
}

// Operand registers of NK K steps from a lane's 16 values per step (value 4j + r of step k: channel 64k + 16j + 4g + r).
template <int NK, int N>
__device__ __forceinline__ void expand(const float (&v)[N], float inv, v4i (*d)[3]) {
#pragma unroll
    for (int k = 0; k < NK; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int w0, w1, w2;
            const int i = 16 * k + 4 * j;
            digits23_4(v[i], v[i + 1], v[i + 2], v[i + 3], inv, w0, w1, w2);
            d[k][0][j] = w0;
            d[k][1][j] = w1;
            d[k][2][j] = w2;
        }
}

// NT result tiles over NK K steps; fragments at wl + (k * LD + t) KiB.
template <int NT, int NK, int LD = NT>
__device__ __forceinline__ void products(const int8_t* wl, const v4i (*d)[3], v4i (&acc)[NT][3]) {
#pragma unroll
    for (int k = 0; k < NK; k++) {
        v4i wf[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) wf[t] = *(const v4i*)(wl + (k * LD + t) * 1024);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int l = 0; l < 3; l++)
                acc[t][l] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[t], d[k][l], k == 0 ? v4i{0, 0, 0, 0} : acc[t][l], 0, 0, 0);
    }
}

// The same with `outputs(e0, e1)` called after each K step, for the previous unit's NE outputs in NK shares: a wave then
// alternates between 3 * NT matrix instructions and a share of vector instructions, so that two waves of a SIMD, which
// meet at every unit's barrier, fill each other's gaps instead of both running all products and then all outputs.
template <int NT, int NK, int NE, class F>
__device__ __forceinline__ void products_with(const int8_t* wl, const v4i (*d)[3], v4i (&acc)[NT][3], F&& outputs) {
    v4i wf[2][NT];
#pragma unroll
    for (int t = 0; t < NT; t++) wf[0][t] = *(const v4i*)(wl + t * 1024);
#pragma unroll
    for (int k = 0; k < NK; k++) {
        if (k + 1 < NK)
#pragma unroll
            for (int t = 0; t < NT; t++) wf[(k + 1) & 1][t] = *(const v4i*)(wl + ((k + 1) * NT + t) * 1024);
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int l = 0; l < 3; l++)
                acc[t][l] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[k & 1][t], d[k][l], k == 0 ? v4i{0, 0, 0, 0} : acc[t][l], 0, 0, 0);
        outputs(NE * k / NK, NE * (k + 1) / NK);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The three digit sums joined, times 65536 / scale: the two lower ones exactly in integers first
// (|256 p1 + p2| < 2^31 for K up to 512).
__device__ __forceinline__ float dot3(const v4i (&acc)[3], int r) {
    return fmaf((float)((acc[1][r] << 8) + acc[2][r]), kInvLimb256_2, (float)acc[0][r]);
}

__device__ __forceinline__ int vswz(int r) { return 4 * ((r >> 3) & 3); }

// The scan over the 16 tokens of a DPP row for four channels: (a, b) of each lane composed with the pairs of the lanes
// before it, b = a * b' + b (fused), a = a * a', over 1, 2, 4 and 8 lanes. Lanes without a partner keep a (a DPP
// instruction writes nothing there without bound_ctrl) and add zero to b. The DPP operands were written at least
// seven instructions earlier inside the block; the leading s_nop covers the two wait states after the inputs.
__device__ __forceinline__ void scan16(float* a, float* b) {
#define MG_SCAN(S)                                                                  \
    "v_fmac_f32_dpp %4, %4, %0 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"       \
    "v_fmac_f32_dpp %5, %5, %1 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"       \
    "v_fmac_f32_dpp %6, %6, %2 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"       \
    "v_fmac_f32_dpp %7, %7, %3 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"       \
    "v_mul_f32_dpp %0, %0, %0 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"        \
    "v_mul_f32_dpp %1, %1, %1 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"        \
    "v_mul_f32_dpp %2, %2, %2 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"        \
    "v_mul_f32_dpp %3, %3, %3 row_shr:" #S " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" MG_SCAN(1) MG_SCAN(2) MG_SCAN(4) MG_SCAN(8)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
#undef MG_SCAN
}

// One token's key or value row of a head into its session's ring (fp32, or packed as kv_pack describes).
template <int ND>
__device__ __forceinline__ void keep_row(const v4f (&y)[ND], int kg, int dh, long long row, float* ring, uint32_t* pack,
                                         float* scale) {
    if (pack) {
        float m = 0.0f;
#pragma unroll
        for (int g = 0; g < ND; g++)
#pragma unroll
            for (int r = 0; r < 4; r++) m = fmaxf(m, fabsf(y[g][r]));
        const int e = kv_exp(row_max4(m));
#pragma unroll
        for (int g = 0; g < ND; g++)
            if (16 * g + 4 * kg < dh)
                stg_pk3((Pk3*)pack + row * (dh / 4) + 4 * g + kg, kv_pack(make_float4(y[g][0], y[g][1], y[g][2], y[g][3]), e));
        if (kg == 0) stg(scale + row, ldexpf(1.0f, e));
    } else {
#pragma unroll
        for (int g = 0; g < ND; g++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (16 * g + 4 * kg + r < dh) stg(ring + row * dh + 16 * g + 4 * kg + r, y[g][r]);
    }
}

// KEEP: also writes the session state.
template <int DT, int HT, int ND, bool KEEP>
__global__ __launch_bounds__(512)
    __attribute__((amdgpu_waves_per_eu(Cfg<DT, HT, ND>::waves, Cfg<DT, HT, ND>::waves))) void seq_kernel(SeqArgs a) {
    using C = Cfg<DT, HT, ND>;
    constexpr int Dp = C::Dp, Hp = C::Hp, NC = 16 * DT;  // NC: channels of a lane
    extern __shared__ __align__(16) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = lane & 15, kg = lane >> 4;

    // the wave's tile
    const int tiles = (a.T + 15) >> 4, spw = 8 / tiles;
    const int slot = w / tiles, tile = w - slot * tiles;
    const int b = blockIdx.x * spw + slot;
    const bool mine = slot < spw && b < a.B;
    const int len = mine ? (a.lens ? min(a.lens[b], a.T) : a.T) : 0;
    const int t = 16 * tile + qi;
    const int lrow = 16 * w + qi;  // the token's row in LDS
    int4 rows = make_int4(0, a.T, (mine ? b : 0) * a.T, 0);
    if (a.rows && mine) rows = a.rows[b];
    if (a.last_only) rows = make_int4(len - 1, 1, b, 0);
    const int span = a.window > 0 ? min(a.window, a.cap) : a.cap;
    // which tiles of the last block are read: its output by the head's rows, its input to the attention also by the
    // keys those rows attend
    const bool in_rows = 16 * tile < rows.x + rows.y;
    const bool out_act = in_rows && 16 * tile + 15 >= rows.x;
    const bool key_act = in_rows && 16 * tile + 15 >= rows.x - span + 1;

    // The weight stream: wave w moves fragments w and w + 8 of every unit, unit u to LDS slot u & 3.
    const int8_t* wp = a.stream + w * 1024;
    const uint32_t wlane = lane * 16;
    const uint32_t slots = lds_offset(smem) + w * 1024;
    auto request = [&](int u) {
        const uint32_t d = slots + (u & (kSlots - 1)) * (C::UF * 1024);
        if (C::UF >= 8 || w < C::UF) lds_load16(wp, wlane, d);
        if (C::UF > 8 && w + 8 < C::UF) lds_load16(wp + 8192, wlane, d + 8192);
        wp += C::UF * 1024;
    };
    // this wave's fragments of all units but the `newer` last requested have arrived
    auto arrived = [&](auto newer) {
        constexpr int N = decltype(newer)::value;
        if (C::UF > 8 && w + 8 < C::UF) vm_wait<2 * N>();
        else vm_wait<N>();
    };
    int u = 0;
    // a unit: `begin` requests the unit three later into the slot that the last `end` freed, `end` makes the next unit
    // readable
    auto begin = [&]() -> const int8_t* {
        request(u + kSlots - 1);
        __builtin_amdgcn_sched_barrier(0);
        return smem + (u & (kSlots - 1)) * C::UF * 1024 + lane * 16;
    };
    auto end = [&]() {
        arrived(std::integral_constant<int, kSlots - 2>{});
        wg_barrier();
        u++;
    };
    auto vec_load = [&](int blk) {
        const float* src = a.vec + Dp + (long long)blk * (C::NV - Dp);
        static_assert((C::NV - Dp) / 4 <= 512, "one float4 per thread");
        if (tid < (C::NV - Dp) / 4) *(float4*)(smem + C::o_vec + 4 * Dp + 16 * tid) = *(const float4*)(src + 4 * tid);
    };
    // A wave without work from here on only carries its share of the weights: n units of the current block.
    auto idle_units = [&](int n) {
        for (int i = 0; i < n; i++) {
            begin();
            end();
        }
    };
    auto idle_attention = [&]() {
        for (int i = 0; i < a.heads; i++) {
            begin();
            end();
            wg_barrier();
        }
        idle_units(DT);
    };
    constexpr int RULE2 = 4 * HT + 4 * DT / C::HW;  // units of a rule step after the latch's DT
    constexpr int RULE = DT + RULE2;
    // A block's rule steps share one copy of their units: before the request of the unit past a step's last (made three
    // units ahead, at the step's unit RULE - 3), the stream goes back to the step's first unit if another step follows.
    constexpr int TURN = RULE - (kSlots - 1);
    static_assert(TURN >= DT, "the turn lies among the units after the latch's");
    auto turn = [&](bool again) { wp -= again ? RULE * C::UF * 1024 : 0; };

    // out-of-range ids are token 0, as are the positions past the sequence
    int id = mine && t < a.T ? a.ids[(long long)b * a.T + t] : 0;
    for (int i = 0; i < kSlots - 1; i++) request(i);
    if (tid < Dp / 4) *(float4*)(smem + C::o_vec + 16 * tid) = *(const float4*)(a.vec + 4 * tid);
    vec_load(0);
    if (16 * tile >= len) {
        arrived(std::integral_constant<int, kSlots - 2>{});
        wg_barrier();
        for (int blk = 0; blk < a.nblocks; blk++) {
            for (int st = 1; st <= a.blocks[blk].steps; st++) {
                idle_units(TURN);
                turn(st < a.blocks[blk].steps);
                idle_units(RULE - TURN);
            }
            if (ND > 0 && a.blocks[blk].attn) idle_attention();
            if (blk + 1 < a.nblocks) {
                vec_load(blk + 1);
                wg_barrier();
            }
        }
        vm_wait<0>();
        return;
    }

    // LDS offsets (bytes) of this lane; opaque, so that every access is one of these registers plus a constant
    auto opaque = [](int x) {
        asm volatile("" : "+v"(x));
        return x;
    };
    const int x_off = opaque(C::o_x + 4 * (lrow * C::XS + 4 * kg));
    const int v_off = opaque(C::o_vec + 16 * kg);
    const int c_off = opaque(C::o_carry + 16 * kg);
    auto ld4 = [&](int off) -> float4 { return *(const float4*)(smem + off); };
    auto st4 = [&](int off, float x, float y, float z, float w_) { *(float4*)(smem + off) = make_float4(x, y, z, w_); };
    constexpr int V_B1 = 4 * Dp, V_B2 = V_B1 + 8 * Hp, V_G = V_B2 + 8 * Dp, V_AG = V_G + 4 * Dp;

    const long long m = (long long)b * a.T + min(t, a.T - 1);
    if (id < 0 || id >= a.V) id = 0;
    auto embed = [&](int row, int ti, float (&e)[4]) {
        const int c = 16 * ti + 4 * kg;
        const uint32_t x = c < a.D ? ldg((const uint32_t*)(a.emb + (long long)row * a.D + c)) : 0u;
#pragma unroll
        for (int r = 0; r < 4; r++) e[r] = (float)(int8_t)(x >> (8 * r)) * a.emb_scale;
    };
    float cur[NC];
#pragma unroll
    for (int ti = 0; ti < 4 * DT; ti++) {
        float e[4];
        embed(id, ti, e);
#pragma unroll
        for (int r = 0; r < 4; r++) cur[4 * ti + r] = e[r];
    }
    arrived(std::integral_constant<int, kSlots - 2>{});
    wg_barrier();

    // RMSNorm of the state rows (nn.RMSNormForwardF32): 1/rms from the mean square, then times gamma
    auto rms_inv = [&]() -> float {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NC; i++) ss = fmaf(cur[i], cur[i], ss);
        ss = row_sum4(ss);
        const float rms = (float)sqrt((double)(ss / (float)a.D + 1e-5f));
        return 1.0f / rms;
    };
    auto scale_by = [&](float inv, int ti, float4 g, float (&n)[NC]) {
        n[4 * ti] = (cur[4 * ti] * inv) * g.x;
        n[4 * ti + 1] = (cur[4 * ti + 1] * inv) * g.y;
        n[4 * ti + 2] = (cur[4 * ti + 2] * inv) * g.z;
        n[4 * ti + 3] = (cur[4 * ti + 3] * inv) * g.w;
    };

    const bool keeps = KEEP && t < len;  // a position whose state the session may keep
    int bs = 0, ab = 0;                                    // rule steps and attention blocks so far
    for (int blk = 0; blk < a.nblocks; blk++) {
        const SeqBlock& B = a.blocks[blk];
        const int steps = B.steps;
        const bool last_blk = blk + 1 == a.nblocks;
        int dil = B.init_dil;
        for (int st = 0; st < steps; st++) {
            const int dl = min(dil, 32);
            if (dil < 32) dil *= B.dil_base;
            // n, its digits, lambda, and the scan within the tile
            float n[NC], sa[NC], sb[NC];
            if (B.norm) {
                const float inv = rms_inv();
#pragma unroll
                for (int ti = 0; ti < 4 * DT; ti++) scale_by(inv, ti, ld4(v_off + V_G + 64 * ti), n);
            } else {
#pragma unroll
                for (int i = 0; i < NC; i++) n[i] = cur[i];
            }
            const float nm = row_max4(abs_max(n));
#pragma unroll
            for (int ti = 0; ti < 4 * DT; ti++) st4(x_off + 64 * ti, n[4 * ti], n[4 * ti + 1], n[4 * ti + 2], n[4 * ti + 3]);
            if (kg == 0) *(float*)(smem + C::o_nmax + 4 * lrow) = nm;
            if (KEEP && keeps && t >= len - a.ring) {
                float* d = a.norm_ring + (((long long)bs * a.B + b) * a.ring + t % a.ring) * Dp + 4 * kg;
#pragma unroll
                for (int ti = 0; ti < 4 * DT; ti++) stg((float4*)(d + 16 * ti), make_float4(n[4 * ti], n[4 * ti + 1], n[4 * ti + 2], n[4 * ti + 3]));
            }
            {
                const DigitScale sc = digit_scale(nm);
                v4i nd[DT][3];
                expand<DT>(n, sc.inv, nd);
                const float sw = sc.s * B.ssel;
#pragma unroll
                for (int un = 0; un < DT; un++) {
                    const int8_t* wl = begin();
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v4i acc[1][3];
                        products<1, DT, 4>(wl + q * 1024, nd, acc);
                        const int ti = 4 * un + q;
                        const float4 bs = ld4(v_off + 64 * ti);
                        const float bb[4] = {bs.x, bs.y, bs.z, bs.w};
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int i = 4 * ti + r;
                            const float lam = sigmoid_med(fmaf(dot3(acc[0], r), sw, bb[r]));
                            sa[i] = lam;
                            sb[i] = (1.0f - lam) * n[i];
                        }
                        scan16(sa + 4 * ti, sb + 4 * ti);
                        if (qi == 15) {
                            st4(c_off + 4 * w * Dp + 64 * ti, sa[4 * ti], sa[4 * ti + 1], sa[4 * ti + 2], sa[4 * ti + 3]);
                            st4(c_off + 4 * (w + 8) * Dp + 64 * ti, sb[4 * ti], sb[4 * ti + 1], sb[4 * ti + 2], sb[4 * ti + 3]);
                        }
                    }
                    end();
                }
            }
            if (last_blk && st + 1 == steps && !(B.attn ? key_act : out_act)) {
                idle_units(RULE2);
                if (ND > 0 && B.attn) idle_attention();
                vm_wait<0>();
                return;
            }
            v4i xd[3 * DT][3];
            float xsw;
            {
                // g: the tiles before this one composed in order, then the tile's own scan applied to their state
                float gm = 0.0f;
                float c[NC];
#pragma unroll
                for (int i = 0; i < NC; i++) c[i] = 0.0f;
#pragma unroll 1
                for (int j = w - tile; j < w; j++) {
                    const int o = c_off + 4 * j * Dp;
#pragma unroll
                    for (int ti = 0; ti < 4 * DT; ti++) {
                        const float4 ca = ld4(o + 64 * ti), cb = ld4(o + 32 * Dp + 64 * ti);
                        c[4 * ti] = fmaf(ca.x, c[4 * ti], cb.x);
                        c[4 * ti + 1] = fmaf(ca.y, c[4 * ti + 1], cb.y);
                        c[4 * ti + 2] = fmaf(ca.z, c[4 * ti + 2], cb.z);
                        c[4 * ti + 3] = fmaf(ca.w, c[4 * ti + 3], cb.w);
                    }
                }
#pragma unroll
                for (int i = 0; i < NC; i++) {
                    sb[i] = fmaf(sa[i], c[i], sb[i]);
                    gm = fmaxf(gm, fabsf(sb[i]));
                }
                if (KEEP && keeps && t == len - 1) {
                    float* d = a.g + ((long long)bs * a.B + b) * Dp + 4 * kg;
#pragma unroll
                    for (int ti = 0; ti < 4 * DT; ti++) stg((float4*)(d + 16 * ti), make_float4(sb[4 * ti], sb[4 * ti + 1], sb[4 * ti + 2], sb[4 * ti + 3]));
                }
                bs++;
                // the rule input [n | n of dl positions earlier | g], one scale per row
                const bool hasl = t >= dl;
                const int back = hasl ? dl : 0;
                const float lm = hasl ? *(const float*)(smem + C::o_nmax + 4 * (lrow - back)) : 0.0f;
                const DigitScale sc = digit_scale(fmaxf(fmaxf(nm, lm), row_max4(gm)));
                xsw = sc.s * B.s1;
                expand<DT>(n, sc.inv, xd);
                expand<DT>(sb, sc.inv, xd + 2 * DT);
                const float linv = hasl ? sc.inv : 0.0f;
                const int l_off = x_off - 4 * back * C::XS;
                float lf[NC];
#pragma unroll
                for (int ti = 0; ti < 4 * DT; ti++) {
                    const float4 v = ld4(l_off + 64 * ti);
                    lf[4 * ti] = v.x; lf[4 * ti + 1] = v.y; lf[4 * ti + 2] = v.z; lf[4 * ti + 3] = v.w;
                }
                expand<DT>(lf, linv, xd + DT);
            }
            // h = (x W1v + b1v) * sigmoid(x W1g + b1g), 16 outputs a unit. Each unit's products are issued between the
            // previous unit's outputs: the matrix cores and the vector units then work side by side in one wave.
            float h[16 * HT];
            v4i acc[2][2][3];
            auto glu_vecs = [&](int p, float (&bv)[4], float (&bg)[4]) {
                const float4 x = ld4(v_off + V_B1 + 128 * p), y = ld4(v_off + V_B1 + 128 * p + 64);
                bv[0] = x.x; bv[1] = x.y; bv[2] = x.z; bv[3] = x.w;
                bg[0] = y.x; bg[1] = y.y; bg[2] = y.z; bg[3] = y.w;
            };
            auto glu_out = [&](int p, int r, const v4i (&ac)[2][3], const float (&bv)[4], const float (&bg)[4]) {
                h[4 * p + r] = here(fmaf(dot3(ac[0], r), xsw, bv[r]) * sigmoid_med(fmaf(dot3(ac[1], r), xsw, bg[r])));
            };
#pragma unroll
            for (int p = 0; p < 4 * HT; p++) {
                if (DT + p == TURN) turn(st + 1 < steps);
                const int8_t* wl = begin();
                if (p > 0) {
                    float bv[4], bg[4];
                    glu_vecs(p - 1, bv, bg);
                    products_with<2, 3 * DT, 4>(wl, xd, acc[p & 1], [&](int e0, int e1) {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (e >= e0 && e < e1) glu_out(p - 1, e, acc[(p - 1) & 1], bv, bg);
                    });
                } else {
                    products<2, 3 * DT>(wl, xd, acc[0]);
                }
                end();
                if (p == 0) {
                    // every wave has read its left neighbours: the state waits in the tile's own rows there (each lane
                    // reads back what it wrote) instead of in registers beside x and h
#pragma unroll
                    for (int ti = 0; ti < 4 * DT; ti++) st4(x_off + 64 * ti, cur[4 * ti], cur[4 * ti + 1], cur[4 * ti + 2], cur[4 * ti + 3]);
                }
            }
            {
                float bv[4], bg[4];
                glu_vecs(4 * HT - 1, bv, bg);
#pragma unroll
                for (int e = 0; e < 4; e++) glu_out(4 * HT - 1, e, acc[1], bv, bg);
            }
            // cur = (1 - g) cur + g o, in the same manner
            v4i hd[HT][3];
            const DigitScale sc = digit_scale(row_max4(abs_max(h)));
            const float hsw = sc.s * B.s2;
            expand<HT>(h, sc.inv, hd);
            constexpr int NU = 4 * DT / C::HW;
            v4i ho[2][2 * C::HW][3];
            struct Vecs {
                float bv[4], bg[4], c[4];
            };
            auto hw_vecs = [&](int ti, Vecs& v) {
                const float4 x = ld4(v_off + V_B2 + 128 * ti), y = ld4(v_off + V_B2 + 128 * ti + 64), z = ld4(x_off + 64 * ti);
                v.bv[0] = x.x; v.bv[1] = x.y; v.bv[2] = x.z; v.bv[3] = x.w;
                v.bg[0] = y.x; v.bg[1] = y.y; v.bg[2] = y.z; v.bg[3] = y.w;
                v.c[0] = z.x; v.c[1] = z.y; v.c[2] = z.z; v.c[3] = z.w;
            };
            auto hw_out = [&](int ti, int r, const v4i (&av)[3], const v4i (&ag)[3], const Vecs& v) {
                const float o = fmaf(dot3(av, r), hsw, v.bv[r]);
                const float gt = sigmoid_med(fmaf(dot3(ag, r), hsw, v.bg[r]));
                const float x = (1.0f - gt) * v.c[r], y = gt * o;
                cur[4 * ti + r] = here(x + y);
            };
            Vecs vlast[C::HW];
#pragma unroll
            for (int un = 0; un < NU; un++) {
                if (DT + 4 * HT + un == TURN) turn(st + 1 < steps);
                const int8_t* wl = begin();
                if (un > 0) {
                    Vecs vs[C::HW];
#pragma unroll
                    for (int q = 0; q < C::HW; q++) hw_vecs(C::HW * (un - 1) + q, vs[q]);
                    products_with<2 * C::HW, HT, 4 * C::HW>(wl, hd, ho[un & 1], [&](int e0, int e1) {
#pragma unroll
                        for (int e = 0; e < 4 * C::HW; e++)
                            if (e >= e0 && e < e1)
                                hw_out(C::HW * (un - 1) + e / 4, e % 4, ho[(un - 1) & 1][2 * (e / 4)], ho[(un - 1) & 1][2 * (e / 4) + 1], vs[e / 4]);
                    });
                } else {
                    products<2 * C::HW, HT>(wl, hd, ho[0]);
                }
                // the last unit's vectors are read before its barrier: past it another wave may store the next block's
                if (un == NU - 1)
#pragma unroll
                    for (int q = 0; q < C::HW; q++) hw_vecs(C::HW * un + q, vlast[q]);
                end();
            }
#pragma unroll
            for (int q = 0; q < C::HW; q++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    hw_out(C::HW * (NU - 1) + q, e, ho[(NU - 1) & 1][2 * q], ho[(NU - 1) & 1][2 * q + 1], vlast[q]);
        }
        if constexpr (ND > 0) {
            if (B.attn) {
                const bool qo = !last_blk || out_act;
                if (last_blk && !key_act) {  // (a last block without rule steps)
                    idle_attention();
                    vm_wait<0>();
                    return;
                }
                v4i nd[DT][3];
                float sw;
                {
                    float n[NC];
                    const float inv = rms_inv();
#pragma unroll
                    for (int ti = 0; ti < 4 * DT; ti++) scale_by(inv, ti, ld4(v_off + V_AG + 64 * ti), n);
                    const DigitScale sc = digit_scale(row_max4(abs_max(n)));
                    sw = sc.s * B.sqkv;
                    expand<DT>(n, sc.inv, nd);
                }
                // scores in units of ln 2, for the hardware 2^x
                const float scale2 = (float)(1.0 / sqrt((double)a.dh)) * 1.4426950408889634f;
                const int k_off = opaque(C::o_k + 4 * (lrow * C::KS + 4 * kg));  // this token's key row
                int vw[ND], vr[ND];  // its value columns; the lane's value operands of its own key block
#pragma unroll
                for (int g = 0; g < ND; g++) {
                    vw[g] = opaque(C::o_v + 4 * ((16 * g + 4 * kg) * C::VS + (lrow ^ vswz(16 * g + 4 * kg))));
                    vr[g] = opaque(C::o_v + 4 * ((16 * g + qi) * C::VS + 16 * w + ((4 * kg) ^ vswz(16 * g + qi))));
                }
                // the heads' outputs collect in the tile's rows of the LDS (the rule's reads of them are over)
                for (int i = a.heads * ND; i < 4 * DT; i++) st4(x_off + 64 * i, 0.0f, 0.0f, 0.0f, 0.0f);
                // first tile whose keys are computed and can be attended
                const int first = last_blk ? max(rows.x - span + 1, 0) >> 4 : 0;
                // One head's attention of the tile over NB 16-key blocks, its own last: S^T = K Q^T (lane L: query L & 15,
                // keys 4 * (L >> 4) + r of each block), softmax, V^T P^T (dimensions 16g + 4 * (L >> 4) + r). Blocks
                // before the first tile are computed with the others, so that the blocks' chains run side by side, and
                // masked.
                auto attend = [&](const v4f (&q)[ND], auto nb, int hh) {
                    constexpr int NB = decltype(nb)::value, K0 = 5 - NB;
                    v4f s[5], kv[5][ND];
                    int at[5];  // the block read: blocks that hold no key of this tile repeat the first one that does
#pragma unroll
                    for (int kb = K0; kb < 5; kb++) {
                        at[kb] = kb < 4 ? max(kb - 4, first - tile) : 0;
                        s[kb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int g = 0; g < ND; g++) kv[kb][g] = *(const v4f*)(smem + k_off + 64 * at[kb] * C::KS + 64 * g);
                    }
#pragma unroll
                    for (int g = 0; g < ND; g++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
#pragma unroll
                            for (int kb = K0; kb < 5; kb++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[kb][g][e], q[g][e], s[kb], 0, 0, 0);
                    v4f vv[5][ND];
#pragma unroll
                    for (int kb = K0; kb < 5; kb++)
#pragma unroll
                        for (int g = 0; g < ND; g++) vv[kb][g] = *(const v4f*)(smem + vr[g] + 64 * at[kb]);
                    // masked to the attended keys: only the own block can hold later ones; only the first block (or, for
                    // spans under 64, any) keys before the span; blocks before the sequence are left out whole
                    float mx = -3.40282347e38f;
#pragma unroll
                    for (int kb = K0; kb < 5; kb++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int j = 4 * kg + r;
                            float x = s[kb][r] * scale2;
                            if (kb == 4) x = j <= qi ? x : -INFINITY;
                            if (kb == 0 || span < 64) x = 16 * kb + j - 64 >= qi - span + 1 ? x : -INFINITY;
                            if (kb < 4) x = tile - 4 + kb >= first ? x : -INFINITY;
                            s[kb][r] = x;
                            mx = fmaxf(mx, x);
                        }
                    mx = row_max4(mx);
                    float sum = 0.0f;
#pragma unroll
                    for (int kb = K0; kb < 5; kb++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            s[kb][r] = __builtin_amdgcn_exp2f(s[kb][r] - mx);
                            sum += s[kb][r];
                        }
                    const float inv = 1.0f / row_sum4(sum);
                    // two chains per dimension tile
                    v4f o[ND][2];
#pragma unroll
                    for (int g = 0; g < ND; g++) o[g][0] = o[g][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int kb = K0; kb < 5; kb++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
#pragma unroll
                            for (int g = 0; g < ND; g++)
                                o[g][r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[kb][g][r], s[kb][r], o[g][r & 1], 0, 0, 0);
#pragma unroll
                    for (int g = 0; g < ND; g++) *(v4f*)(smem + x_off + 64 * (hh * ND + g)) = (o[g][0] + o[g][1]) * inv;
                };
#pragma unroll 1
                for (int hh = 0; hh < a.heads; hh++) {
                    const int8_t* wl = begin();
                    v4f k[ND], v[ND], q[ND];  // rows of this lane's token
                    auto project = [&](int part, v4f (&y)[ND]) {
                        v4i acc[ND][3];
                        products<ND, DT>(wl + part * ND * DT * 1024, nd, acc);
#pragma unroll
                        for (int g = 0; g < ND; g++)
#pragma unroll
                            for (int r = 0; r < 4; r++) y[g][r] = dot3(acc[g], r) * sw;
                    };
                    project(0, k);
                    project(1, v);
                    project(2, q);
                    end();  // every wave is past the previous head's attention
                    if (KEEP && keeps && t >= len - a.cap) {
                        const long long row = (((long long)ab * a.B + b) * a.heads + hh) * a.cap + t % a.cap;
                        keep_row<ND>(k, kg, a.dh, row, a.kring, a.kpack, a.kscale);
                        keep_row<ND>(v, kg, a.dh, row, a.vring, a.vpack, a.vscale);
                    }
#pragma unroll
                    for (int g = 0; g < ND; g++) {
                        *(v4f*)(smem + k_off + 64 * g) = k[g];
#pragma unroll
                        for (int r = 0; r < 4; r++) *(float*)(smem + vw[g] + 4 * r * C::VS) = v[g][r];
                    }
                    wg_barrier();
                    if (qo) {
                        if (tile < 3) attend(q, std::integral_constant<int, 3>{}, hh);
                        else attend(q, std::integral_constant<int, 5>{}, hh);
                    }
                }
                ab++;
                if (!qo) {
                    idle_units(DT);
                    vm_wait<0>();
                    return;
                }
                float osw;
                {
                    float att[NC];
#pragma unroll
                    for (int ti = 0; ti < 4 * DT; ti++) {
                        const float4 x = ld4(x_off + 64 * ti);
                        att[4 * ti] = x.x; att[4 * ti + 1] = x.y; att[4 * ti + 2] = x.z; att[4 * ti + 3] = x.w;
                    }
                    const DigitScale sc = digit_scale(row_max4(abs_max(att)));
                    osw = sc.s * B.so;
                    expand<DT>(att, sc.inv, nd);
                }
#pragma unroll
                for (int un = 0; un < DT; un++) {
                    const int8_t* wl = begin();
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v4i acc[1][3];
                        products<1, DT, 4>(wl + q * 1024, nd, acc);
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int i = 4 * (4 * un + q) + r;
                            cur[i] = cur[i] + dot3(acc[0], r) * osw;
                        }
                    }
                    end();
                }
            }
        }
        if (!last_blk) {
            // blockIn += cur; cur = blockIn. The first block's input is the embedding, read again; later ones' go
            // through memory (each lane reads back what it wrote).
            vec_load(blk + 1);
            float* brow = a.bin + m * Dp;
            int row = id;
            asm volatile("" : "+v"(row));
#pragma unroll
            for (int ti = 0; ti < 4 * DT; ti++) {
                const int c = 16 * ti + 4 * kg;
                float e[4];
                if (blk == 0) {
                    embed(row, ti, e);
                } else {
                    const float4 x = *(const float4*)(brow + c);
                    e[0] = x.x; e[1] = x.y; e[2] = x.z; e[3] = x.w;
                }
#pragma unroll
                for (int r = 0; r < 4; r++) cur[4 * ti + r] = e[r] + cur[4 * ti + r];
                if (blk + 2 < a.nblocks && t < a.T)
                    *(float4*)(brow + c) = make_float4(cur[4 * ti], cur[4 * ti + 1], cur[4 * ti + 2], cur[4 * ti + 3]);
            }
            wg_barrier();
        }
    }
    vm_wait<0>();  // nothing lands in LDS after the workgroup's end
    if (!out_act) return;

    // the head's operand: final RMSNorm, limb planes in the GEMM's own channel order
    float n[NC];
    if (a.final_norm) {
        const float inv = rms_inv();
#pragma unroll
        for (int ti = 0; ti < 4 * DT; ti++) scale_by(inv, ti, *(const float4*)(a.final_norm + 16 * ti + 4 * kg), n);
    } else {
#pragma unroll
        for (int i = 0; i < NC; i++) n[i] = cur[i];
    }
    float s, inv;
    limb_scale(row_max4(abs_max(n)), s, inv);
    if (t >= rows.x && t < rows.x + rows.y && t < len) {
        const int mo = rows.z + t - rows.x;
        int8_t* d = a.limbs + (((long long)(mo >> 4) * DT * 3) << 10) + ((mo & 15) << 4) + 4 * kg;
#pragma unroll
        for (int ti = 0; ti < 4 * DT; ti++) {
            uint32_t w0, w1, w2;
            split4_pack(make_float4(n[4 * ti], n[4 * ti + 1], n[4 * ti + 2], n[4 * ti + 3]), inv, w0, w1, w2);
            int8_t* p = d + (((ti >> 2) * 3) << 10) + (ti & 3) * 256;
            *(uint32_t*)p = w0;
            *(uint32_t*)(p + 1024) = w1;
            *(uint32_t*)(p + 2048) = w2;
        }
        if (kg == 0) a.lscale[mo] = s;
    }
}

template <int DT, int HT, int ND, bool KEEP>
hipError_t launch_t(const SeqArgs& a, hipStream_t s) {
    using C = Cfg<DT, HT, ND>;
    static const hipError_t attr =
        hipFuncSetAttribute((const void*)seq_kernel<DT, HT, ND, KEEP>, hipFuncAttributeMaxDynamicSharedMemorySize, C::lds);
    if (attr != hipSuccess) return attr;
    const int spw = 8 / ((a.T + 15) / 16);
    hipLaunchKernelGGL((seq_kernel<DT, HT, ND, KEEP>), dim3((a.B + spw - 1) / spw), dim3(512), C::lds, s, a);
    return hipGetLastError();
}

// f(Cfg) of the compiled variant, or `none`.
template <class R, class F>
R with_shape(SeqShape sh, R none, F&& f) {
    const int key = sh.dt * 100 + sh.ht * 10 + sh.nd;
    switch (key) {
        case 110: return f(Cfg<1, 1, 0>{});
        case 120: return f(Cfg<1, 2, 0>{});
        case 220: return f(Cfg<2, 2, 0>{});
        case 230: return f(Cfg<2, 3, 0>{});
        case 240: return f(Cfg<2, 4, 0>{});
        case 112: return f(Cfg<1, 1, 2>{});
        case 122: return f(Cfg<1, 2, 2>{});
        case 222: return f(Cfg<2, 2, 2>{});
        case 232: return f(Cfg<2, 3, 2>{});
        case 242: return f(Cfg<2, 4, 2>{});
        default: return none;
    }
}

}  // namespace

SeqShape seq_shape(const HostModel& hm, int span) {
    SeqShape sh;
    sh.dt = round_up(hm.D, 64) / 64;
    sh.ht = round_up(hm.H, 64) / 64;
    bool attn = false;
    for (const HostBlock& b : hm.blocks) attn |= b.has_attn;
    if (attn) {
        const int dh = hm.D / std::max(hm.attn_heads, 1);
        sh.nd = 2;
        if (dh > 32 || hm.attn_heads * 32 > 64 * sh.dt || span > kSeqMaxSpan) return SeqShape{};
    }
    if (hm.D % 4 || hm.blocks.empty() || !with_shape(sh, false, [](auto) { return true; })) return SeqShape{};
    return sh;
}

SeqPack seq_pack(const HostModel& hm, SeqShape sh, const std::vector<float>& latch_base) {
    SeqPack p;
    const int D = hm.D, H = hm.H, DT = sh.dt, HT = sh.ht, ND = sh.nd, Dp = 64 * DT, Hp = 64 * HT;
    const int UF = with_shape(sh, 0, [](auto c) { return decltype(c)::UF; });
    const int HW = HT <= 3 ? 2 : 1;
    const int dh = ND ? D / hm.attn_heads : 0;
    // fragments: row i of a fragment comes from row(i) (or -1), byte 4j + r of lane group g from column col(16j + 4g + r)
    size_t unit = 0;
    int f = 0;
    auto open = [&]() {
        unit = p.stream.size();
        p.stream.resize(unit + (size_t)UF * 1024, 0);
        f = 0;
    };
    auto frag = [&](const std::vector<int8_t>& w, int ld, auto row, auto col) {
        int8_t* d = p.stream.data() + unit + (size_t)f++ * 1024;
        for (int i = 0; i < 16; i++) {
            const int rr = row(i);
            if (rr < 0) continue;
            for (int g = 0; g < 4; g++)
                for (int j = 0; j < 4; j++)
                    for (int r = 0; r < 4; r++) {
                        const int c = col(16 * j + 4 * g + r);
                        if (c >= 0) d[(i + 16 * g) * 16 + 4 * j + r] = w[(size_t)rr * ld + c];
                    }
        }
    };
    auto within = [](int v, int n) { return v < n ? v : -1; };
    p.vec = latch_base;
    p.vec.resize(Dp, 0.0f);
    for (const HostBlock& hb : hm.blocks) {
        SeqBlock b;
        b.steps = hb.steps; b.dil_base = hb.dilation_base; b.init_dil = hb.initial_dilation;
        b.attn = hb.has_attn ? 1 : 0; b.norm = (int)hb.gamma.size() == D ? 1 : 0;
        b.ssel = hb.ssel; b.s1 = hb.s1; b.s2 = hb.s2; b.sqkv = hb.sqkv; b.so = hb.so;
        p.blocks.push_back(b);
        if (hb.steps > 0) {  // one copy, read again by every step
            for (int un = 0; un < DT; un++) {
                open();
                for (int ks = 0; ks < DT; ks++)
                    for (int q = 0; q < 4; q++)
                        frag(hb.wsel, D, [&](int i) { return within(16 * (4 * un + q) + i, D); }, [&](int k) { return within(64 * ks + k, D); });
            }
            for (int u = 0; u < 4 * HT; u++) {
                open();
                for (int ks = 0; ks < 3 * DT; ks++)
                    for (int q = 0; q < 2; q++)
                        frag(hb.w1, 3 * D, [&](int i) { return 16 * u + i < H ? q * H + 16 * u + i : -1; },
                             [&](int k) { const int c = 64 * (ks % DT) + k; return c < D ? (ks / DT) * D + c : -1; });
            }
            for (int un = 0; un < 4 * DT / HW; un++) {
                open();
                for (int ks = 0; ks < HT; ks++)
                    for (int q = 0; q < 2 * HW; q++)
                        frag(hb.w2, H, [&](int i) { const int c = 16 * (HW * un + q / 2) + i; return c < D ? (q & 1) * D + c : -1; },
                             [&](int k) { return within(64 * ks + k, H); });
            }
        }
        if (hb.has_attn) {
            for (int h = 0; h < hm.attn_heads; h++) {
                open();
                for (int part = 0; part < 3; part++)  // k, v, q
                    for (int ks = 0; ks < DT; ks++)
                        for (int g = 0; g < ND; g++)
                            frag(hb.qkv, D, [&](int i) { return 16 * g + i < dh ? (part + 1) % 3 * D + h * dh + 16 * g + i : -1; },
                                 [&](int k) { return within(64 * ks + k, D); });
            }
            for (int un = 0; un < DT; un++) {
                open();
                for (int ks = 0; ks < DT; ks++)
                    for (int q = 0; q < 4; q++)
                        frag(hb.wo, D, [&](int i) { return within(16 * (4 * un + q) + i, D); },
                             [&](int k) {
                                 const int h = (64 * ks + k) / (16 * ND), d = (64 * ks + k) % (16 * ND);
                                 return h < hm.attn_heads && d < dh ? h * dh + d : -1;
                             });
            }
        }
        // vectors: b1 and b2 with the rows' pairing (16 values, then their 16 gates), zero padding
        for (int r = 0; r < 2 * Hp; r++) {
            const int j = 16 * (r / 32) + r % 16;
            p.vec.push_back(j < H ? hb.b1[r % 32 < 16 ? j : H + j] : 0.0f);
        }
        for (int r = 0; r < 2 * Dp; r++) {
            const int c = 16 * (r / 32) + r % 16;
            p.vec.push_back(c < D ? hb.b2[r % 32 < 16 ? c : D + c] : 0.0f);
        }
        for (int c = 0; c < Dp; c++) p.vec.push_back(b.norm && c < D ? hb.gamma[c] : 0.0f);
        for (int c = 0; c < Dp; c++) p.vec.push_back(hb.has_attn && c < D ? hb.attn_norm[c] : 0.0f);
    }
    p.stream.resize(p.stream.size() + (size_t)(kSlots - 1) * UF * 1024, 0);  // the units requested past the last one
    return p;
}

// The kernel's time goes with its workgroups, whose eight tiles of 16 tokens cost the same however full they are; the
// layered kernels' time goes with the rows, the sequences (attention) and their launches. So many sequences of a few tokens
// are the layered body's: 65536 of one token, D128 H256, two blocks without attention, 1878 us in the kernel and 538
// layered, of four tokens 1966 and 1437, of six 2023 and 2143; with attention and three blocks, of one token 4548 and 3516,
// of two 4586 and 4165, of three 4622 and 4864. With 256 workgroups (2048 such sequences) the launches decide and the
// kernel is the faster one at one token too (78 and 101, 171 and 301). From six tokens on it is always the faster one, also
// where a workgroup is filled worst (131072 tokens of D128 H128 without attention: T = 8 582 and 881 us, T = 17 589 and
// 901, T = 33 582 and 914, T = 65 580 and 917). The two estimates are nanoseconds on the whole chip without the head, fitted
// to forwards and prefills of 20 models, T 1 to 128, 1 to 524288 sequences: the body they take was the faster one or within
// 1 % of it in 99.6 % of 2805 measurements and never more than 9 % behind.
bool seq_pays(SeqShape sh, int B, int T, int steps, int attns, int heads) {
    if (T > 8) return true;
    const int seqs = 8 / ((T + 15) / 16), slots = sh.dt == 1 && sh.nd == 0 ? 512 : 256;  // workgroups at once
    const double wgs = (double)round_up((B + seqs - 1) / seqs, slots);
    const double step = sh.dt == 2 ? (sh.ht == 2 ? 82 : sh.ht == 3 ? 94 : 111)
                        : sh.nd    ? (sh.ht == 1 ? 33 : 42)
                                   : (sh.ht == 1 ? 28 : 57);
    const double kernel = wgs * (steps * step + attns * heads * 18.4);
    const double row = 0.5 + steps * (sh.dt == 2 ? 1.4 + 0.2 * sh.ht : 1.05) + attns * (0.6 + 0.6 * sh.dt);
    const double layered = 35000.0 * steps + 25000.0 * attns + B * (attns * heads * 3.1 + T * row);
    return kernel <= layered;
}

bool seq_fits(const SeqArgs& a) { return a.shape.dt > 0 && a.T >= 1 && a.T <= kSeqMaxT && a.B >= 1; }

hipError_t launch_seq(const SeqArgs& a, hipStream_t s) {
    if (!seq_fits(a) || !a.stream || !a.vec || !a.blocks || !a.limbs || !a.lscale) return hipErrorInvalidValue;
    if (a.nblocks > 2 && !a.bin) return hipErrorInvalidValue;
    // packed rows are whole groups of four
    if (a.norm_ring && (!a.g || (a.heads > 0 && !(a.kring && a.vring) && !(a.kpack && a.vpack && a.kscale && a.vscale && a.dh % 4 == 0))))
        return hipErrorInvalidValue;
    return with_shape(a.shape, hipErrorInvalidValue, [&](auto c) {
        using K = decltype(c);
        if (a.norm_ring) return launch_t<K::Dp / 64, K::Hp / 64, (K::KS - 4) / 16, true>(a, s);
        return launch_t<K::Dp / 64, K::Hp / 64, (K::KS - 4) / 16, false>(a, s);
    });
}

}  // namespace mg
