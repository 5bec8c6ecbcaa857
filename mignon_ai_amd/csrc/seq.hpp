// The model body over whole sequences in one kernel (see seq.hip), for models small enough that a sequence's
// state stays in one workgroup's registers from the embedding to the head's operand.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace mg {

struct HostModel;

// Longest sequence: one 16-token tile per wave, eight waves.
constexpr int kSeqMaxT = 128;
// Longest attended span: the query's own 16-key block and the four before it.
constexpr int kSeqMaxSpan = 65;

struct SeqBlock {
    int steps = 0, dil_base = 2, init_dil = 1, attn = 0, norm = 0;
    float ssel = 0, s1 = 0, s2 = 0, sqkv = 0, so = 0;
};

// Kernel variant of a model: padded state and hidden size in units of 64 channels, 16-dimension tiles per
// attention head (0: no attention). dt == 0: the kernel does not take the model.
struct SeqShape {
    int dt = 0, ht = 0, nd = 0;
};
// span: keys a position attends at most.
SeqShape seq_shape(const HostModel& hm, int span);

// The weights in the order the kernel reads them (each block's rule units once), and the vectors [latch base | per block b1 | b2 | gamma |
// attention gamma] it copies to LDS block by block.
struct SeqPack {
    std::vector<int8_t> stream;
    std::vector<float> vec;
    std::vector<SeqBlock> blocks;
};
SeqPack seq_pack(const HostModel& hm, SeqShape sh, const std::vector<float>& latch_base);

struct SeqArgs {
    SeqShape shape;
    int B = 0, T = 0, D = 0, heads = 0, dh = 0, window = 0, cap = 0, nblocks = 0, V = 0;
    const int32_t* ids = nullptr;    // [B][T]
    const int8_t* emb = nullptr;     // [V][D]
    float emb_scale = 0;
    const int8_t* stream = nullptr;  // SeqPack, on the device
    const float* vec = nullptr;
    const SeqBlock* blocks = nullptr;
    const float* final_norm = nullptr;  // [Dp], or null: no normalisation
    float* bin = nullptr;               // [B * T][Dp]: blockIn between blocks, used with three blocks or more
    // The rows the head reads: sequence b gives its positions rows[b].x .. rows[b].x + rows[b].y - 1, as output
    // rows rows[b].z on. Null: every position, row b * T + t; or with last_only, each sequence's last position, row b.
    const int4* rows = nullptr;
    bool last_only = false;
    // Valid positions of each sequence, or null: T. Positions past them are not computed.
    const int32_t* lens = nullptr;
    // Session state after each sequence's last position (null: not wanted), in the session set's layout: normalised rows
    // [block step][B][ring][Dp], latch states [block step][B][Dp] and K/V rings [attention block][B][heads][cap], fp32
    // rows (kring, vring) or packed ones (kpack, vpack and their scales).
    float* norm_ring = nullptr;
    float* g = nullptr;
    int ring = 1;
    float* kring = nullptr;
    float* vring = nullptr;
    uint32_t* kpack = nullptr;
    uint32_t* vpack = nullptr;
    float* kscale = nullptr;
    float* vscale = nullptr;
    int8_t* limbs = nullptr;   // normalised final rows, limb-expanded (GEMM fragment layout, K = Dp)
    float* lscale = nullptr;
};
// Whether the kernel takes sequences of this length of a model whose shape it takes.
bool seq_fits(const SeqArgs& a);
// Whether it is the faster body there, for B sequences through `steps` rule steps and `attns` attention blocks in all.
bool seq_pays(SeqShape sh, int B, int T, int steps, int attns, int heads);
hipError_t launch_seq(const SeqArgs& a, hipStream_t s);

}  // namespace mg
