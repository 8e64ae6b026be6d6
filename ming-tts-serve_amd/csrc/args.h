// Plain argument blocks shared by the host glue and the kernels (no device
// code, so host-only translation units can include it).
#pragma once

#include <stdint.h>

namespace ming {

// Weights of one linear as the kernels see them.
struct LinearDev {
    int32_t kind;  // 0 bf16, 1 affine 4-bit / group 64
    int32_t N, K;
    float gscale;
    const uint32_t* w;   // affine: u32 [N, K/8]; bf16: bf16 [N, K] viewed as u32 pairs
    const uint16_t* s;   // bf16 [N, K/64]
    const uint16_t* b;   // bf16 [N, K/64]
};

// fused.LmLayer (src/ming_fused.zig:576-589) as the kernels see it.
struct LayerDev {
    const uint16_t *ln1, *ln2;
    LinearDev q, k, v, o, g, u, d;
    const uint16_t *bq, *bk, *bv;
};

// Everything one decode step touches.  Activations of every layer are kept
// (x[l] is layer l's input, x[n_layers] the stack output), which also lets
// tests read any intermediate.
struct StepArgs {
    const LayerDev* layers;   // device array [n_layers] (persistent schedule)
    int n_layers, H, heads, kvh, hd, I;
    float eps, log2_theta;
    const uint16_t* final_norm;
    LinearDev head;           // tied LM head [V, H]
    LinearDev embed;          // embedding table [V, H]
    uint16_t* kc;             // [n_layers][kvh][cap][hd]
    uint16_t* vc;
    int cap;
    int pos;                  // position of this token (= cached length before the step)
    const int32_t* token_in;  // device id, or null: x[0] already holds the input row
    int32_t* argmax_out;      // device i32, or null
    // Activations of layer l: input x + l*sx, output xo + l*sx, x1 + l*sx,
    // att + l*sx, qkv + l*sq, hh + l*sh.  The stack uses one buffer per layer
    // (xo = x + H, so x[l + 1] is layer l's output); a single-layer call
    // passes caller buffers with zero strides.
    uint16_t* x;
    uint16_t* xo;
    uint16_t* x1;
    uint16_t* att;
    uint16_t* qkv;
    uint16_t* hh;
    int64_t sx, sq, sh;
    float* part;              // attention partials [kvh][nsplit][grp][hd + 2]
    int split_len;            // positions per attention split (multiple of 64)
    uint16_t* hidden;         // [H] final-normed hidden (bf16)
    float* logits;            // [V] f32, or null
    float* amax_v;            // [kMaxParts] argmax partials
    int32_t* amax_i;
    int32_t* flags;           // [0] error flag, [1] grid barrier counter
    // Tagged hand-off buffers of the persistent schedule: u64 words holding a
    // pair of bf16 values (low half) and the step's epoch (high half).
    uint64_t* tx;             // [n_layers + 1][H/2]   layer inputs / stack output
    uint64_t* tq;             // [n_layers][(H + 2*kvh*hd)/2]
    uint64_t* ta;             // [n_layers][H/2]       merged attention
    uint64_t* tx1;            // [n_layers][H/2]
    uint64_t* th;             // [n_layers][I/2]
    int32_t* counters;        // [n_layers * kvh] attention arrivals, [1] head arrivals, [n_layers * kvh] attention
                              // arrivals of XCD-local splits (L2 atomics)
    uint32_t epoch;
    uint64_t* tstamp;         // optional [n_stamps][grid] wall-clock stamps per stage boundary
    // Hubs of the persistent schedule (one workgroup per XCD): each publishes
    // the staged GEMV input of every stage into memory that the other
    // workgroups of its XCD read through their shared L2.
    int nhubs;                // 0: every workgroup stages its own inputs
    int hub_stages;           // stages whose inputs come from the hubs (HUB_* bits); the others stage their own
    uint32_t* img;            // [kMaxHubs][kImgSlots][img_stride] stage images
    int img_stride;           // u32 words per image slot
    uint32_t* hflag;          // [kMaxHubs][nflag] epoch of each published image
    int nflag;                // flag words per hub (>= 4 * n_layers + 1)
    uint64_t* hubtab;         // [kMaxHubs] tagged XCC id of each hub, then [kAttXlSlots] of attention workers
    // Attention splits grouped by XCD (1): worker W-1-(8 sp + g) runs split sp of kv
    // head g, so a kv head's splits share an XCD when workgroup b runs on XCD b % 8
    // (checked per launch); they then meet through that XCD's L2.  0: splits in
    // unit order across the grid, meeting device-coherently.
    int att_xl;
    // XCD-local schedule: o_proj partials of each kv head and down partials of
    // each XCD slot, f32 whose lowest mantissa bit carries the epoch's parity
    // (the reader clears it); xslots = slots that hold SwiGLU groups (and so
    // down partials).  Every word is written at every step of this schedule,
    // and consecutive steps of it use epochs of opposite parity.
    uint32_t* tpo;            // [n_layers][kvh][H]
    uint32_t* tpd;            // [n_layers][8][H]
    int xslots;
    uint64_t* tpa;            // [n_layers][kvh][xnsm][grp][hd + 2] attention split partials, tagged words
    int xnsm;                 // split slots per (layer, kv head) in tpa
    int xloc;                 // 1: hand-offs inside an XCD slot use plain stores where the slot is on one XCD
};

constexpr int kAttXlBase = 32;    // hubtab index of the attention workers' XCC ids
constexpr int kAttXlSlots = 256;
constexpr int kXcdBase = kAttXlBase + kAttXlSlots;  // hubtab index of every workgroup's XCC id (XCD-local schedule)
constexpr int kXcdSlots = 1024;

// Stages of the persistent schedule, as bits of StepArgs::hub_stages.
enum : int { HUB_QKV = 1, HUB_O = 2, HUB_UP = 4, HUB_DOWN = 8, HUB_HEAD = 16 };

// One DiT block (fused.Block, src/ming_fused.zig:482-500): bf16 [out, in]
// linears with biases, two RMSNorm weights; D = hidden, F = feed-forward.
struct DitBlockDev {
    int D, F, heads, hd;
    float eps;
    const uint16_t *norm1, *norm2;
    const uint16_t *wq, *wk, *wv, *wo, *w1, *w2;
    const uint16_t *bq, *bk, *bv, *bo, *b1, *b2;
};

constexpr int kMaxHubs = 8;
constexpr int kImgSlots = 5;  // q/k/v, o_proj, gate/up, down, LM head

constexpr int kMaxParts = 4096;

// ---- VAE decoder (vae_gemm.hip, vae.hip) ----
enum VWf : int { VW_BF16 = 0, VW_Q4 = 1 };
enum VEpi : int {
    VE_PLAIN = 0,   // y = acc (+ bias)
    VE_QKV = 1,     // y = acc + bias, rotary on the segments that ask for it (heads of 64, position = row)
    VE_RES = 2,     // y [ks][M][ldy] = the K slices' sums (launch_vrow adds them to the residual)
    VE_SWIGLU = 3,  // planes yp = (g * sigmoid(g)) * u, g from seg[0], u from up
};

// One weight of the decoder's linears: bf16 [n][K] or MLX affine 4-bit (u32
// [n][K/8] + bf16 scales/biases [n][K/64]).
struct VSeg {
    const void* w;
    const uint16_t *s, *b;
    float gs;               // affine global scale
    const uint16_t* bias;   // bf16 [n] or null (VE_PLAIN, VE_QKV)
    int n;                  // output columns (a multiple of 64 except in the last segment)
    int rope;               // VE_QKV: 1 = rotary on these columns
};

// C [M][N] = A [M][K] x W^T in f32; the output columns are the segments'
// columns one after another (N = sum of seg[i].n).
// Rows up to which the unstaged kernel runs.  A decode of 24 layers (896, ff 4864) in us, this kernel / LDS tiles, 4-bit
// and bf16: 4 rows 791 / 1821 and 1067 / 1675, 36 rows 1164 / 1898 and 1432 / 1736, 64 rows 1274 / 1940 and
// 1510 / 1765.  The line could lie higher: 96 rows 1424 / 1985 and 1658 / 1770, 128 rows 1727 / 2012 and 1986 / 1791.
constexpr int kV3SmallRows = 64;
struct V3Gemm {
    // np = 3: bf16 planes whose sum is A, in operand order (vae_gemm.hip), rows padded to 16;
    // np = 1: bf16 [M][K]
    const uint16_t* a;
    size_t aps;             // values between planes
    int np, M, K;
    VSeg seg[3];
    int nseg;
    VSeg up;                // VE_SWIGLU
    float* y;
    int ldy;
    uint16_t* yp;           // VE_SWIGLU: the output's planes (ldyp columns)
    size_t yps;
    int ldyp, ypair;        // ypair: the planes' consumer has 4-bit weights
    const float* rope_cs;   // VE_QKV: f32 [rows][32][2] (cos, sin)
    int ks;                 // VE_RES: K slices
};

// The rows between the decoder's linears (launch_vrow): x = res + sum of the K
// slices part [ks][M][N], or the upsampled rows of the fc1 sums part [T][N]
// (+ bias, rounded to bf16); h = planes of rms_norm(x) with weight w.
struct VRowArgs {
    const float* part;
    int ks;
    const float* res;       // f32 [M][N]
    float* x;               // f32 [M][N]
    int M, N;
    const uint16_t* w;      // bf16 [N]
    float eps;
    uint16_t* h;            // planes of N columns
    size_t hps;
    int hpair;              // the planes' consumer has 4-bit weights
    const uint16_t* bias;   // upsample: fc1's bias (bf16 [N] or null), format, latents, factor
    int q4, T, scale;
};

// Inverse real FFT of n = 2 h points per frame by passes of the given radices
// over h complex points (launch_virfft).
constexpr int kFftMaxHalf = 4096, kFftMaxPasses = 12;
struct VFftPlan {
    int h, passes;
    int radix[kFftMaxPasses];
};

// C [M][n] = A [M][K] (f32) x W^T (f32 [n][K]) * win[col], for the transforms
// whose length has a prime factor above 7.  ks > 1 splits K into ks slices whose
// partials [ks][M][n] a reduce kernel sums in slice order.
struct VBasis {
    const float* a;
    const float* w;
    int M, K, n;
    const float* win;
    float* y;
    int ks;
    float* part;
};

}  // namespace ming
