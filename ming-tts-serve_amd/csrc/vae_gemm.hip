// The VAE decoder's linears (Model.vaeDecode, src/ming_model.zig:1257-1309) on
// the bf16 matrix cores at f32 precision.  Every activation after the upsample
// is f32 in the reference graph, but the weights are bf16 or MLX affine 4-bit,
// so only the activation needs more than one bf16 operand: an f32 value is the
// exact sum of three bf16 ones (its 24 mantissa bits in three truncations of 8,
// split3 below), the products of two bf16 values are exact in f32, and three
// v_mfma_f32_16x16x32_bf16 per tile do what eight v_mfma_f32_16x16x4f32 did at
// a fifth of their cost (dense bf16 against f32: 1213 against 154 TFLOP/s for
// a library product on this card).  The high plane's sum and the two low
// planes' sum are kept apart and added once, so the low planes' roundings fall
// below the last bit.  4-bit weights enter as the exact values 2^-12 (16 + q) (a
// nibble OR-ed into bits 3..6 of bf16(2^-8): two instructions a pair, where
// converting q - 8 took five); each group of 64 is folded in f32 from its sums
// with them and of 2^-12 x (the same MFMAs against a column of 2^-12), the high
// plane's and the low planes' apart (q16_fold).
//
// Activations therefore travel between the kernels as planes, written by the
// kernel that produces them in the MFMA A operand's order: bf16 [3][M / 16]
// [K / 32][lane][8], lane = 16 (k % 32 / 8) + m % 16 (plane_at), so that a
// wave's operand is one contiguous KiB.  (Row-major planes made each operand
// load 16 half-used cache lines.)  For 4-bit weights the 8 values lie in the
// unpacked word's pair order (0, 4), (1, 5), (2, 6), (3, 7).  fc1's bf16 input
// stays row-major in natural order, one plane.
//
// Two kernels.  vsmall_kernel (few rows): no LDS staging, the waves of a
// workgroup split K and stream their operands straight into registers, which
// is what a launch of a few microseconds needs (T = 7, 28 rows: the time is
// one workgroup's chain of loads).  vtile_kernel (many rows): LDS tiles of
// 64-k stages.  Both write K-slice partials for the residual projections; the
// next norm's kernel (vrow_kernel) sums them.
#include "args.h"
#include "common.h"
#include "internal.h"

namespace ming {

namespace {

__device__ __forceinline__ int v3_total_n(const V3Gemm& g) {
    return g.seg[0].n + (g.nseg > 1 ? g.seg[1].n : 0) + (g.nseg > 2 ? g.seg[2].n : 0);
}

// x = p[0] + p[1] + p[2] exactly, each a bf16 (as f32 bits with a zero low half): truncations
// leave 16, then 8 significant bits, so both differences are exact.  An infinity is its own
// first plane (the others 0) and a NaN stays one.
__device__ __forceinline__ void split3(float x, uint32_t (&p)[3]) {
    p[0] = __float_as_uint(x) & 0xffff0000u;
    const float h = __uint_as_float(p[0]), r = h == x ? 0.0f : x - h;
    p[1] = __float_as_uint(r) & 0xffff0000u;
    p[2] = __float_as_uint(r - __uint_as_float(p[1]));
}

// The high halves of two words as a bf16 pair (lo in the low half).
__device__ __forceinline__ uint32_t hi_pair(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

// 8 nibbles of a packed word as the bf16 values 2^-12 (16 + q) (exact) in pair order: nibble i and
// i + 4 are one pair.  The power of two keeps a group's sums finite for any finite x (64 values of
// 2^-8 (1 + q / 16) < 2^-7, where 64 of 16 + q overflowed from 2^118 on) and changes no bit.
__device__ __forceinline__ uint4 unpack_q16(uint32_t w, uint32_t mask, uint32_t magic) {
    return make_uint4(((w << 3) & mask) | magic, ((w >> 1) & mask) | magic, ((w >> 5) & mask) | magic,
                      ((w >> 9) & mask) | magic);
}
constexpr uint32_t kQ16Mask = 0x00780078u, kQ16Magic = 0x3b803b80u, kQ16One = 0x39803980u;  // bf16(2^-12)
constexpr float kQ16Scale = 4096.0f;  // what the sums lack (into the global scale: load_view)

// acc + s sum q x + b sum x of one group, all over 2^12, from the sums with 2^-12 (16 + q) (h: high
// plane, l: low planes) and of 2^-12 x (xh, xl); off = b + 8 s.  sum (16 + q) x and 24 sum x are five
// times the size of their difference sum (q - 8) x; the high plane's are sums of short mantissas (13
// and 8 bits), all but exact in f32, so the difference is taken plane by plane and rounds at its own
// size.  (Folding s (h + l) + (b - 16 s) sum x instead left up to 1.2e-6 at 28 rows where the f32
// MFMA path had 8e-7.)  An infinite x gives NaN where s q + b times it is infinite: the norm of the
// row makes NaN of both.
__device__ __forceinline__ float q16_fold(float s, float off, float h, float l, float xh, float xl, float acc) {
    const float d = fmaf(-24.0f, xh, h) + fmaf(-24.0f, xl, l);
    return fmaf(s, d, fmaf(off, xh + xl, acc));
}

// A value the compiler must keep in a register: mask and magic then make one v_and_or_b32
// (which takes no literal operands).
__device__ __forceinline__ uint32_t in_reg(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The operand of 8 natural-order values in pair order.
__device__ __forceinline__ uint4 pair_order(uint4 e) {
    return make_uint4(__builtin_amdgcn_perm(e.z, e.x, 0x05040100u), hi_pair(e.x, e.z),
                      __builtin_amdgcn_perm(e.w, e.y, 0x05040100u), hi_pair(e.y, e.w));
}

// Place of value (row m, column k) in a plane of K columns; pair: the consumer's weights are 4-bit.
__device__ __forceinline__ size_t plane_at(int m, int k, int K, int pair) {
    const int e = k % 8;
    return ((size_t)(m / 16) * (K / 32) + k / 32) * 512 + (16 * (k % 32 / 8) + m % 16) * 8 +
           (pair ? 2 * (e % 4) + e / 4 : e);
}

__device__ __forceinline__ f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(a), as_bf8(b), c, 0, 0, 0);
}

constexpr f32x4_t kZero4 = {0.0f, 0.0f, 0.0f, 0.0f};

// What a workgroup needs of its arguments, read in one go (load_view): the argument block's
// scalar loads are a chain of cold misses (0.3 - 0.7 us each) when a kernel picks its segment
// by index and reads each field where it is used.
template <int WF, int EPI>
struct V3View {
    const char *w, *wu;              // weights: the block's segment, up
    const uint16_t *s, *b, *su, *bu;  // affine scales and biases
    const uint16_t* bias;
    float gs, gu;                    // global scales, times kQ16Scale for affine weights
    int n, start, rope;  // the segment's columns, its first column, rotary
    int M, K, ks, ldy, ldyp, ypair;
    const uint16_t* a;
    size_t aps, yps;
    float* y;
    uint16_t* yp;
    const float* rope_cs;
};

#define MING_PIN(...) asm volatile("" : __VA_ARGS__)
#define MING_S(x) "+s"(x)

// The view of the segment that holds output column c0 (segments start at multiples of 64).
template <int WF, int EPI>
__device__ __forceinline__ V3View<WF, EPI> load_view(const V3Gemm& g, int c0) {
    V3View<WF, EPI> v;
    VSeg s0 = g.seg[0], s1 = EPI == VE_SWIGLU ? g.up : g.seg[1], s2 = g.seg[2];
    v.M = g.M;
    v.K = g.K;
    v.ks = g.ks;
    v.a = g.a;
    v.aps = g.aps;
    v.y = g.y;
    v.ldy = g.ldy;
    v.yp = g.yp;
    v.yps = g.yps;
    v.ldyp = g.ldyp;
    v.ypair = g.ypair;
    v.rope_cs = g.rope_cs;
    // all that this kernel reads in registers here, before anything depends on any of it
    if constexpr (EPI == VE_SWIGLU) {
        if constexpr (WF == VW_Q4)
            MING_PIN(MING_S(s0.w), MING_S(s0.gs), MING_S(s0.n), MING_S(v.M), MING_S(v.K), MING_S(v.a), MING_S(s0.s),
                     MING_S(s0.b), MING_S(s1.w), MING_S(s1.gs), MING_S(v.yp), MING_S(v.ldyp), MING_S(v.ypair),
                     MING_S(s1.s), MING_S(s1.b));
        else
            MING_PIN(MING_S(s0.w), MING_S(s0.gs), MING_S(s0.n), MING_S(v.M), MING_S(v.K), MING_S(v.a), MING_S(s1.w),
                     MING_S(s1.gs), MING_S(v.yp), MING_S(v.ldyp), MING_S(v.ypair));
        MING_PIN(MING_S(v.yps), MING_S(v.aps));
    } else if constexpr (EPI == VE_QKV) {
        MING_PIN(MING_S(s0.w), MING_S(s0.n), MING_S(s1.w), MING_S(s1.n), MING_S(s2.w), MING_S(s2.n), MING_S(v.M),
                 MING_S(v.K), MING_S(v.a), MING_S(v.aps), MING_S(v.y), MING_S(v.ldy), MING_S(v.rope_cs));
        if constexpr (WF == VW_Q4)
            MING_PIN(MING_S(s0.s), MING_S(s0.b), MING_S(s1.s), MING_S(s1.b), MING_S(s2.s), MING_S(s2.b));
        MING_PIN(MING_S(s0.gs), MING_S(s0.bias), MING_S(s0.rope), MING_S(s1.gs), MING_S(s1.bias), MING_S(s1.rope),
                 MING_S(s2.gs), MING_S(s2.bias), MING_S(s2.rope));
    } else {
        MING_PIN(MING_S(s0.w), MING_S(s0.gs), MING_S(s0.n), MING_S(v.M), MING_S(v.K), MING_S(v.a), MING_S(v.aps),
                 MING_S(v.y), MING_S(v.ldy), MING_S(v.ks), MING_S(s0.bias), MING_S(s0.s), MING_S(s0.b));
    }
    v.start = 0;
    if (EPI == VE_QKV) {
        const int e0 = s0.n, e1 = s0.n + s1.n;
        if (c0 >= e1) {
            s0 = s2;
            v.start = e1;
        } else if (c0 >= e0) {
            s0 = s1;
            v.start = e0;
        }
        v.rope = s0.rope;
    }
    v.w = static_cast<const char*>(s0.w);
    constexpr float kGs = WF == VW_Q4 ? kQ16Scale : 1.0f;
    v.gs = kGs * s0.gs;
    v.n = s0.n;
    v.bias = s0.bias;
    v.s = s0.s;
    v.b = s0.b;
    if (EPI == VE_SWIGLU) {
        v.wu = static_cast<const char*>(s1.w);
        v.su = s1.s;
        v.bu = s1.b;
        v.gu = kGs * s1.gs;
    }
    return v;
}

// MLX fast::rope of the pair (d, d + 32) of a 64-column head from the table's (cos, sin).
__device__ __forceinline__ void v3_rope(const float* rope_cs, int row, int d, float& x1, float& x2) {
    const float2 cs = *reinterpret_cast<const float2*>(rope_cs + ((size_t)row * 32 + d) * 2);
    const float a = x1, b = x2;
    x1 = a * cs.x - b * cs.y;
    x2 = a * cs.y + b * cs.x;
}

__device__ __forceinline__ float v3_swiglu(float g, float u) { return (g * (1.0f / (1.0f + expf(-g)))) * u; }

// The epilogue of one row: x[t] are the sums of this lane's columns col[t]; QKV holds rotary
// pairs in (t, t + NT / 2), SWIGLU gate and up likewise.
template <int WF, int EPI, int NT>
__device__ __forceinline__ void v3_epi(const V3View<WF, EPI>& v, int row, const int (&col)[NT], float (&x)[NT], int z) {
    if constexpr (EPI == VE_SWIGLU) {
#pragma unroll
        for (int t = 0; t < NT / 2; t++) {  // into the planes of the next linear's input
            uint32_t p[3];
            split3(v3_swiglu(x[t] * v.gs, x[t + NT / 2] * v.gu), p);
            uint16_t* y = v.yp + plane_at(row, col[t], v.ldyp, v.ypair);
#pragma unroll
            for (int k = 0; k < 3; k++) gst(y + k * v.yps, (uint16_t)(p[k] >> 16));
        }
    } else if constexpr (EPI == VE_RES) {  // this K slice's sums; the row kernel adds them to the residual
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (col[t] < v.n) gst(v.y + ((size_t)z * v.M + row) * v.ldy + col[t], x[t] * v.gs);
    } else {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            x[t] *= v.gs;
            if (v.bias) x[t] += bf2f(gld(v.bias + min(col[t] - v.start, v.n - 1)));
        }
        if constexpr (EPI == VE_QKV)
            if (v.rope)
#pragma unroll
                for (int t = 0; t < NT / 2; t++) v3_rope(v.rope_cs, row, col[t] % 64, x[t], x[t + NT / 2]);
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (col[t] - v.start < v.n) gst(v.y + (size_t)row * v.ldy + col[t], x[t]);
    }
}

// ---- few rows -----------------------------------------------------------------------
// Workgroup (column block x, row block of 16 MT rows y, K slice z); its waves split the
// slice's units (32 k for bf16 weights, one group of 64 for affine ones) in chunks of CH
// whose loads are all issued before the chunk's MFMAs, and their sums meet in LDS in wave
// order.  Columns of a block: 16 (PLAIN, RES), 32 gate + 32 up (SWIGLU), or 16 and the 16
// that are 32 further in the same head (QKV: rotary pairs meet in one lane).
template <int WF>
constexpr int kUnitK = WF == VW_Q4 ? 64 : 32;
// 4-bit: the two groups of one load.  bf16: units whose loads are all issued together; a decode of 24 layers in us with
// chunks of 1, 2, 4 and 8: 4 rows 945, 1063, 1067, 1308, 28 rows 1034, 1136, 1203, 2122, 64 rows 1223, 1394, 1510, 2778
// (the longest ones spill; shorter ones split K over more waves, another order of the sum).
template <int WF>
constexpr int kSmallCh = WF == VW_Q4 ? 2 : 4;
template <int EPI>
constexpr int kSmallNT = EPI == VE_SWIGLU ? 4 : (EPI == VE_QKV ? 2 : 1);
// most waves of a workgroup: what their registers allow (one column tile: three a SIMD)
template <int EPI>
constexpr int kSmallWaves = kSmallNT<EPI> == 1 ? 10 : 8;

// The weights of a chunk come by quads of lanes (lane l: 16 bytes of row l / 4; bf16: the 64
// bytes of a 32-k step, 4-bit: the 64 bytes of two groups) and each wave turns them round in LDS
// of its own: a load of 16 rows in the operand's order (16 consecutive lanes on 16 rows) takes the
// address unit four times as long, and a 4-bit group took four of them a tile (two words, scale,
// bias), more than all the activations.  The scales and biases of two groups are one load: lane
// 16 x + c the value x of column c, (s, s', b, b').
constexpr int kQRow = 20;  // dwords of a 4-bit row's two groups in LDS (16, padded: no bank conflicts)
template <int WF, int MT, int NT>
constexpr int kSmallLds() {  // bytes a wave: its turned weights, and after the loop its sums
    const int turn = WF == VW_Q4 ? NT * (16 * kQRow + 64) * 4 : 2 * NT * 1024, sums = MT * NT * 1024;
    return turn > sums ? turn : sums;
}

template <int WF, int NP, int MT, int NT>
struct V3Chunk {
    uint4 a[kSmallCh<WF>][kUnitK<WF> / 32][NP][MT];
    uint4 w[WF == VW_Q4 ? 1 : kSmallCh<WF>][NT];
    uint16_t sb[NT];
};

template <int WF, int EPI, int NP, int MT>
__global__ __launch_bounds__(64 * kSmallWaves<EPI>) void vsmall_kernel(V3Gemm g) {
    constexpr int NT = kSmallNT<EPI>;
    constexpr int UK = kUnitK<WF>, UH = UK / 32, CH = kSmallCh<WF>;
    extern __shared__ __align__(16) float vs_lds[];  // [waves][kSmallLds]
    constexpr int LW = kSmallLds<WF, MT, NT>() / 4;
    const int W = blockDim.x / kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave, c = lane % 16, j = lane / 16;
    const int m0 = blockIdx.y * 16 * MT, z = blockIdx.z;
    const int c0 = EPI == VE_QKV ? (blockIdx.x / 2) * 64 + (blockIdx.x % 2) * 16 : blockIdx.x * (EPI == VE_SWIGLU ? 32 : 16);
    int col[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) col[t] = c0 + (EPI == VE_QKV ? 32 * t : 16 * (t % 2)) + c;
    const V3View<WF, EPI> v = load_view<WF, EPI>(g, c0);
    const int U = v.K / UK, per = (U + v.ks - 1) / v.ks, u0 = z * per, u1 = min(U, u0 + per);
    // 32-bit byte offsets per lane from uniform bases (operands: row tile; weights: row lane / 4)
    uint32_t ao[MT], wo[NT], so[NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        ao[mt] = NP == 1 ? (uint32_t)min(m0 + 16 * mt + c, v.M - 1) * v.K * 2u + 16u * j
                         : (uint32_t)min(m0 / 16 + mt, (v.M - 1) / 16) * (v.K / 32) * 1024u + 16u * lane;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        wo[t] = (uint32_t)min(col[t] - c - v.start + lane / 4, v.n - 1) * (WF == VW_Q4 ? v.K / 2 : v.K * 2) + 16u * (lane % 4);
        so[t] = (uint32_t)min(col[t] - v.start, v.n - 1) * (v.K / 64) * 2u;
    }
    auto at = [](const void* base, uint32_t off) { return static_cast<const char*>(base) + off; };
    f32x4_t hi[MT][NT], lo[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) hi[mt][t] = lo[mt][t] = kZero4;
    float* mine = vs_lds + wave * LW;
    auto load = [&](int u, V3Chunk<WF, NP, MT, NT>& in) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const bool up = EPI == VE_SWIGLU && t >= NT / 2;
            const char* w = up ? v.wu : v.w;
            if (WF == VW_Q4) {
                const bool two = u + 1 < u1;  // a last single group is read twice
                in.w[0][t] = ldg4(at(w + 32 * (size_t)u, wo[t] - (!two && lane % 4 >= 2 ? 32u : 0u)));
                const uint16_t* sv = up ? v.su : v.s;
                const uint16_t* bv = up ? v.bu : v.b;
                const char* p = at(j < 2 ? sv : bv, so[t]);
                in.sb[t] = gld(reinterpret_cast<const uint16_t*>(p) + u + (two ? j % 2 : 0));
            } else {
#pragma unroll
                for (int k = 0; k < CH; k++)
                    if (u + k < u1) in.w[k][t] = ldg4(at(w + 64 * (size_t)(u + k), wo[t]));
            }
        }
#pragma unroll
        for (int k = 0; k < CH; k++)
            if (u + k < u1)
#pragma unroll
                for (int h = 0; h < UH; h++)
#pragma unroll
                    for (int p = 0; p < NP; p++)
#pragma unroll
                        for (int mt = 0; mt < MT; mt++)
                            in.a[k][h][p][mt] =
                                ldg4(at(v.a + p * v.aps + ((size_t)(u + k) * UH + h) * (NP == 1 ? 32 : 512), ao[mt]));
    };
    const uint4 ones = make_uint4(kQ16One, kQ16One, kQ16One, kQ16One);
    const uint32_t mask = in_reg(kQ16Mask), magic = in_reg(kQ16Magic);
    auto work = [&](const V3Chunk<WF, NP, MT, NT>& in, int n) {  // n units
        if constexpr (WF == VW_Q4) {
            uint32_t* q = reinterpret_cast<uint32_t*>(mine);  // [tile][16 rows][kQRow], [tile][s, s', b, b'][16]
            uint32_t* sc = q + NT * 16 * kQRow;
            wave_lds_order();
#pragma unroll
            for (int t = 0; t < NT; t++) {
                *reinterpret_cast<uint4*>(q + (16 * t + lane / 4) * kQRow + 4 * (lane % 4)) = in.w[0][t];
                sc[64 * t + lane] = (uint32_t)in.sb[t] << 16;
            }
            wave_lds_order();
#pragma unroll
            for (int k = 0; k < CH; k++) {
                if (k >= n) break;
                // the group sums of x, in every column's place: the high plane's, and the low planes'
                f32x4_t xh[MT], xl[MT];
                uint4 x[2][NP][MT];
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int p = 0; p < NP; p++)
#pragma unroll
                        for (int mt = 0; mt < MT; mt++)
                            x[h][p][mt] = NP == 1 ? pair_order(in.a[k][h][p][mt]) : in.a[k][h][p][mt];
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    xl[mt] = kZero4;
#pragma unroll
                    for (int p = NP - 1; p > 0; p--) xl[mt] = mma(x[1][p][mt], ones, mma(x[0][p][mt], ones, xl[mt]));
                    xh[mt] = mma(x[1][0][mt], ones, mma(x[0][0][mt], ones, kZero4));
                }
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const uint32_t* qr = q + (16 * t + c) * kQRow + 8 * k + j;
                    const uint4 b0 = unpack_q16(qr[0], mask, magic), b1 = unpack_q16(qr[4], mask, magic);
                    const float s = __uint_as_float(sc[64 * t + 16 * k + c]),
                                off = fmaf(8.0f, s, __uint_as_float(sc[64 * t + 32 + 16 * k + c]));
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        f32x4_t l = kZero4;
#pragma unroll
                        for (int p = NP - 1; p > 0; p--) l = mma(x[1][p][mt], b1, mma(x[0][p][mt], b0, l));
                        const f32x4_t h = mma(x[1][0][mt], b1, mma(x[0][0][mt], b0, kZero4));
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            hi[mt][t][r] = q16_fold(s, off, h[r], l[r], xh[mt][r], xl[mt][r], hi[mt][t][r]);
                    }
                }
            }
        } else {
            // 16 rows of 4 blocks of 16 bytes, the block permuted by the row: no bank conflicts either way
            uint4* wt = reinterpret_cast<uint4*>(mine);
#pragma unroll
            for (int k = 0; k < CH; k++) {
                if (k >= n) break;
                uint4 w[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) wt[(k % 2 * NT + t) * 64 + 4 * (lane / 4) + (lane % 4 ^ lane / 16)] = in.w[k][t];
                wave_lds_order();  // and the loads of step k - 1 before the stores of k + 1
#pragma unroll
                for (int t = 0; t < NT; t++) w[t] = wt[(k % 2 * NT + t) * 64 + 4 * c + (j ^ c / 4)];
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            f32x4_t& acc = p == 0 ? hi[mt][t] : lo[mt][t];
                            acc = mma(in.a[k][0][p][mt], w[t], acc);
                        }
            }
        }
    };
    for (int ub = u0 + wave * CH; ub < u1; ub += W * CH) {
        // a fresh scalar each time round: the loads keep their uniform base + lane offset form
        const int u = __builtin_amdgcn_readfirstlane(ub);
        V3Chunk<WF, NP, MT, NT> in;
        load(u, in);
        work(in, u1 - u);
    }
    wave_lds_order();
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < NT; t++) mine[((mt * 4 + r) * NT + t) * kWave + lane] = hi[mt][t][r] + lo[mt][t][r];
    __syncthreads();
    for (int u = wave; u < MT * 4; u += W) {  // row slot u = 4 mt + r
        const int row = m0 + 16 * (u / 4) + 4 * j + u % 4;
        if (row >= v.M) continue;
        float x[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float s = vs_lds[(u * NT + t) * kWave + lane];
            for (int w = 1; w < W; w++) s += vs_lds[w * LW + (u * NT + t) * kWave + lane];
            x[t] = s;
        }
        v3_epi<WF, EPI, NT>(v, row, col, x, z);
    }
}

// ---- many rows ------------------------------------------------------------------------
// Workgroup tile of BM rows x 16 WN NT weight columns, K in stages of 64 through one LDS
// buffer (the next AHEAD stages' global loads are in registers while this one computes; two or
// three workgroups share a CU and cover each other's barriers).  4 waves in a WM x WN grid;
// wave (wm, wn) owns the rows BM / WM of wm and the column tiles wn, wn + WN, ..., so that a
// rotary pair (32 columns apart) and a gate / up pair lie in one lane.  The activations keep
// their operand order in LDS; a weight row is 64 values (128 bytes) with its 16-byte chunks
// permuted by the row (chunk ^ row % 8): the 16 rows of a fragment read then fall in distinct
// banks without padding.
template <int WF, int EPI, int BM, int WM, int NT>
__global__ __launch_bounds__(256, 2) void vtile_kernel(V3Gemm g) {
    constexpr int WN = 4 / WM, MT = BM / WM / 16, BN = 16 * WN * NT;
    constexpr bool DUAL = EPI == VE_SWIGLU;
    constexpr int AHEAD = NT > 2 ? 1 : 2;   // stages in flight in registers (the wide tile has room for one)
    constexpr int CB = DUAL ? BN / 2 : BN;  // output columns per workgroup
    constexpr int AL = 3 * BM * 8 / 256, WL = WF == VW_Q4 ? (BN * 2 + 255) / 256 : BN * 8 / 256;
    static_assert(AL * 256 == 3 * BM * 8 && BN % 32 == 0, "whole chunks per thread");
    __shared__ uint4 As[3 * BM * 8];
    __shared__ uint4 Ws[BN * 8];
    __shared__ float2 Ss[WF == VW_Q4 ? BN : 1];
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, c = lane % 16, j = lane / 16;
    const int wm = wave / WN, wn = wave % WN;
    const int N = v3_total_n(g), gx = (N + CB - 1) / CB, gy = (g.M + BM - 1) / BM;
    // workgroup id -> (K slice, row block, column block): the ids of one XCD (id mod 8) share
    // column blocks (whole columns of W are read by one XCD's L2), or K slices when K is split
    const int id = blockIdx.x, z = id % g.ks, tile = id / g.ks;
    int bx, by;
    if (g.ks > 1) {
        bx = tile / gy;
        by = tile % gy;
    } else {
        bx = tile % 8 + 8 * (tile / 8 / gy);
        by = tile / 8 % gy;
    }
    if (bx >= gx) return;
    const int n0 = bx * CB, m0 = by * BM;
    const V3View<WF, EPI> v = load_view<WF, EPI>(g, n0);
    const int G = v.K / 64, per = (G + g.ks - 1) / g.ks, s0 = z * per, S = min(G, s0 + per) - s0;
    const uint16_t* ag[AL];
#pragma unroll
    for (int i = 0; i < AL; i++) {
        // chunk q = [plane][row tile][k32 of the stage][lane]
        const int q = tid + 256 * i, p = q / (BM * 8), mt = q / 128 % (BM / 16);
        ag[i] = v.a + p * v.aps + (size_t)min(m0 / 16 + mt, (v.M - 1) / 16) * (v.K / 32) * 512 + 8 * (q % 128);
    }
    // weight column k of the tile: its row in the segment (DUAL: the second half is the up weight)
    auto wrow = [&](int k, bool& up) {
        up = DUAL && k >= CB;
        return (size_t)min(n0 - v.start + (DUAL ? k % CB : k), v.n - 1);
    };
    const char* wg[WL];
    const uint16_t *sr = nullptr, *br = nullptr;
    const bool wload = WF != VW_Q4 || tid < 2 * BN, sload = tid < BN;
#pragma unroll
    for (int i = 0; i < WL; i++) {
        bool up;
        const int q = tid + 256 * i;
        const size_t n = wrow(WF == VW_Q4 ? min(q / 2, BN - 1) : q / 8, up);
        wg[i] = (up ? v.wu : v.w) + (WF == VW_Q4 ? n * (v.K / 2) + 16 * (q % 2) : n * v.K * 2 + 16 * (q % 8));
    }
    if (WF == VW_Q4) {
        bool up;
        const size_t n = wrow(min(tid, BN - 1), up);
        sr = (up ? v.su : v.s) + n * G;
        br = (up ? v.bu : v.b) + n * G;
    }
    struct Stage {
        uint4 a[AL], w[WL];
        uint16_t s, b;
    };
    auto gload = [&](int s, Stage& r) {
        const int u = s0 + s;
#pragma unroll
        for (int i = 0; i < AL; i++) r.a[i] = ldg4(ag[i] + 1024 * (size_t)u);
        if (wload)
#pragma unroll
            for (int i = 0; i < WL; i++) r.w[i] = ldg4(wg[i] + (WF == VW_Q4 ? 32 : 128) * (size_t)u);
        if (WF == VW_Q4 && sload) {
            r.s = gld(sr + u);
            r.b = gld(br + u);
        }
    };
    const uint32_t mask = in_reg(kQ16Mask), magic = in_reg(kQ16Magic);
    auto lstore = [&](const Stage& r) {
#pragma unroll
        for (int i = 0; i < AL; i++) As[tid + 256 * i] = r.a[i];
        if (WF == VW_Q4) {
            if (wload)
#pragma unroll
                for (int i = 0; i < WL; i++) {
                    const int q = tid + 256 * i, k = q / 2;
                    const uint32_t e[4] = {r.w[i].x, r.w[i].y, r.w[i].z, r.w[i].w};
#pragma unroll
                    for (int w = 0; w < 4; w++) Ws[k * 8 + ((4 * (q % 2) + w) ^ (k % 8))] = unpack_q16(e[w], mask, magic);
                }
            if (sload) {
                const float s = bf2f(r.s);
                Ss[tid] = make_float2(s, fmaf(8.0f, s, bf2f(r.b)));
            }
        } else {
#pragma unroll
            for (int i = 0; i < WL; i++) {
                const int q = tid + 256 * i, k = q / 8;
                Ws[k * 8 + ((q % 8) ^ (k % 8))] = r.w[i];
            }
        }
    };
    f32x4_t hi[MT][NT], lo[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) hi[mt][t] = lo[mt][t] = kZero4;
    const uint4 ones = make_uint4(kQ16One, kQ16One, kQ16One, kQ16One);
    auto afrag = [&](int p, int mt, int h) { return As[((p * (BM / 16) + wm * MT + mt) * 2 + h) * 64 + lane]; };
    auto wfrag = [&](int t, int h) {
        const int k = 16 * (t * WN + wn) + c;
        return Ws[k * 8 + ((4 * h + j) ^ (k % 8))];
    };
    auto compute = [&]() {
        if constexpr (WF == VW_Q4) {
            f32x4_t th[MT][NT], tl[MT][NT], xh[MT], xl[MT];  // high plane, low planes
            uint4 w[2][NT];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < NT; t++) w[h][t] = wfrag(t, h);
#pragma unroll
            for (int p = 2; p >= 0; p--)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        const uint4 a = afrag(p, mt, h);
                        const bool first = p != 1 && h == 0;
                        f32x4_t& xs = p == 0 ? xh[mt] : xl[mt];
                        xs = mma(a, ones, first ? kZero4 : xs);
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            f32x4_t& acc = p == 0 ? th[mt][t] : tl[mt][t];
                            acc = mma(a, w[h][t], first ? kZero4 : acc);
                        }
                    }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float2 f = Ss[16 * (t * WN + wn) + c];
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        hi[mt][t][r] = q16_fold(f.x, f.y, th[mt][t][r], tl[mt][t][r], xh[mt][r], xl[mt][r], hi[mt][t][r]);
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint4 w[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) w[t] = wfrag(t, h);
#pragma unroll
                for (int p = 0; p < 3; p++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        const uint4 a = afrag(p, mt, h);
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            f32x4_t& acc = p == 0 ? hi[mt][t] : lo[mt][t];
                            acc = mma(a, w[t], acc);
                        }
                    }
            }
        }
    };
    Stage r0{};
    if (S > 0) gload(0, r0);
    if constexpr (AHEAD == 1) {
        for (int s = 0; s < S; s++) {
            lstore(r0);
            lds_sync();
            if (s + 1 < S) gload(s + 1, r0);
            compute();
            lds_sync();
        }
    } else {
        Stage r1{};
        if (S > 1) gload(1, r1);
        for (int s = 0; s < S; s += 2) {
            lstore(r0);
            lds_sync();
            if (s + 2 < S) gload(s + 2, r0);
            compute();
            lds_sync();
            if (s + 1 >= S) break;
            lstore(r1);
            lds_sync();
            if (s + 3 < S) gload(s + 3, r1);
            compute();
            lds_sync();
        }
    }
    int col[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) col[t] = n0 + (16 * (t * WN + wn)) % CB + c;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = m0 + wm * (BM / WM) + 16 * mt + 4 * j + r;
            if (row >= v.M) continue;
            float x[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) x[t] = hi[mt][t][r] + lo[mt][t][r];
            v3_epi<WF, EPI, NT>(v, row, col, x, z);
        }
}

// ---- rows between the linears -----------------------------------------------------------
// One workgroup per row: the row's values (SRC 0: the residual plus the K-slice partials in
// slice order; SRC 1: the upsampled fc1 rows), stored as the next layer input, then
// fast::rms_norm (w * (x * rsqrt(mean x^2 + eps))) into the planes of the next linear's
// input.  NC = 8-value chunks a thread holds in registers (0: any width, the row read back).
__device__ __forceinline__ float fc1_value(const VRowArgs& a, int r, int c) {
    // the fc1 row is bf16(acc + bias) for bf16 weights (addmm, one rounding) and
    // bf16(bf16(acc) + bias) for 4-bit ones (quantized_matmul, then the bias add)
    const float v = gld(a.part + (size_t)r * a.N + c), b = a.bias ? bf2f(gld(a.bias + c)) : 0.0f;
    return a.q4 ? rb(rb(v) + b) : rb(v + b);
}

template <int SRC, int NC>
__global__ __launch_bounds__(128) void vrow_kernel(VRowArgs a) {
    __shared__ float red[2];
    const int m = blockIdx.x, N = a.N, n8 = N / 8, t = threadIdx.x;
    struct V8 {
        float e[8];
    };
    auto load8 = [&](const float* p) {
        const float4 x = reinterpret_cast<const float4*>(p)[0], y = reinterpret_cast<const float4*>(p)[1];
        return V8{{x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w}};
    };
    // Decoder._linear_upsample_1d (align_corners=False, f32)
    const float pos = ((float)m + 0.5f) / (float)a.scale - 0.5f;
    const int left = (int)floorf(pos);
    const float wr = pos - (float)left, wl = 1.0f - wr;
    const int l = min(max(left, 0), a.T - 1), r = min(max(left + 1, 0), a.T - 1);
    auto value = [&](int i) {
        V8 x;
        if constexpr (SRC == 1) {
#pragma unroll
            for (int k = 0; k < 8; k++) x.e[k] = fc1_value(a, l, 8 * i + k) * wl + fc1_value(a, r, 8 * i + k) * wr;
        } else {
            x = load8(a.res + (size_t)m * N + 8 * i);
            V8 s{};
            for (int z = 0; z < a.ks; z++) {
                const V8 p = load8(a.part + ((size_t)z * a.M + m) * N + 8 * i);
#pragma unroll
                for (int k = 0; k < 8; k++) s.e[k] += p.e[k];
            }
#pragma unroll
            for (int k = 0; k < 8; k++) x.e[k] += s.e[k];
        }
        float4* o = reinterpret_cast<float4*>(a.x + (size_t)m * N + 8 * i);
        o[0] = make_float4(x.e[0], x.e[1], x.e[2], x.e[3]);
        o[1] = make_float4(x.e[4], x.e[5], x.e[6], x.e[7]);
        return x;
    };
    V8 xv[NC > 0 ? NC : 1];
    float ss = 0.0f;
    auto sq = [&](const V8& x) {
#pragma unroll
        for (int k = 0; k < 8; k += 4)
            ss += (x.e[k] * x.e[k] + x.e[k + 1] * x.e[k + 1]) + (x.e[k + 2] * x.e[k + 2] + x.e[k + 3] * x.e[k + 3]);
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (t + 128 * k < n8) {
                xv[k] = value(t + 128 * k);
                sq(xv[k]);
            }
    } else {
        for (int i = t; i < n8; i += 128) sq(value(i));
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)N + a.eps);
    auto put = [&](int i, const V8& x) {
        uint32_t p[8][3];
#pragma unroll
        for (int k = 0; k < 8; k++) split3(bf2f(gld(a.w + 8 * i + k)) * (x.e[k] * inv), p[k]);
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const uint4 v = make_uint4(hi_pair(p[0][q], p[1][q]), hi_pair(p[2][q], p[3][q]), hi_pair(p[4][q], p[5][q]),
                                       hi_pair(p[6][q], p[7][q]));
            *reinterpret_cast<uint4*>(a.h + q * a.hps + plane_at(m, 8 * i, N, 0)) = a.hpair ? pair_order(v) : v;
        }
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (t + 128 * k < n8) put(t + 128 * k, xv[k]);
    } else {
        for (int i = t; i < n8; i += 128) put(i, load8(a.x + (size_t)m * N + 8 * i));
    }
}

// Sliding-window attention (mask of src/ming_model.zig:618-636: key j is
// visible to query i when i - window < j <= i, window <= 64), with the
// window's K and V rows of one kv head staged in LDS once for the q heads that
// share them: one workgroup per (row i, kv head), wave w = q head kh * grp + w
// (grp <= 16): lane j scores key j0 + j, then lane = dim for P.V.  K rows are
// padded to 68 floats so the lanes' 16-byte reads of 64 different rows spread
// over the banks.  The row leaves as the planes of the o projection's input.
constexpr int kVKs = 68;
__global__ __launch_bounds__(1024) void vattn_gqa_kernel(const float* qkv, int M, int ldq, int H, int heads, int kvh,
                                                         int window, float scale, uint16_t* att, size_t aps, int pair) {
    __shared__ __align__(16) float ks[64 * kVKs];
    __shared__ __align__(16) float vs[64 * 64];
    const int i = blockIdx.x / kvh, kh = blockIdx.x % kvh, grp = heads / kvh;
    const int j0 = max(0, i - window + 1), n = i - j0 + 1;
    for (int f = threadIdx.x; f < 64 * 16; f += blockDim.x) {
        const int r = f / 16, c4 = f % 16;
        const float* base = qkv + (size_t)min(j0 + r, i) * ldq + H + kh * 64 + 4 * c4;
        *reinterpret_cast<float4*>(ks + r * kVKs + 4 * c4) = *reinterpret_cast<const float4*>(base);
        *reinterpret_cast<float4*>(vs + r * 64 + 4 * c4) = *reinterpret_cast<const float4*>(base + kvh * 64);
    }
    __syncthreads();
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave, h = kh * grp + w;
    const float* q = qkv + (size_t)i * ldq + h * 64;
    const float* kr = ks + lane * kVKs;
    float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < 64; d += 4) {
        const float4 qa = *reinterpret_cast<const float4*>(q + d), ka = *reinterpret_cast<const float4*>(kr + d);
        p[0] = fmaf(qa.x, ka.x, p[0]);
        p[1] = fmaf(qa.y, ka.y, p[1]);
        p[2] = fmaf(qa.z, ka.z, p[2]);
        p[3] = fmaf(qa.w, ka.w, p[3]);
    }
    const float s = lane < n ? ((p[0] + p[1]) + (p[2] + p[3])) * scale : -INFINITY;
    const float m = team_max<kWave>(s);
    const float e = lane < n ? expf(s - m) : 0.0f;
    const float l = team_sum<kWave>(e);
    float o = 0.0f;
#pragma unroll
    for (int jj = 0; jj < 64; jj++) {
        const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), jj));
        o = fmaf(pj, vs[jj * 64 + lane], o);
    }
    uint32_t pl[3];
    split3(o / l, pl);
    uint16_t* y = att + plane_at(i, h * 64 + lane, H, pair);
#pragma unroll
    for (int k = 0; k < 3; k++) gst(y + k * aps, (uint16_t)(pl[k] >> 16));
}

// Column blocks (times K slices) from which a workgroup takes two row tiles.  A decode of 24 layers in us with two tiles
// from 1, 128 and 256 blocks on: bf16, 20..32 rows 1259, 1203, 1297, 36..48 rows 1495, 1441, 1397, 64 rows 1566, 1510,
// 1584; 4-bit, 28 rows 1007, 929, 928, 36 rows 1241, 1164, 1005, 64 rows 1354, 1274, 1196 (there one tile each is better
// at every row count: 256 and never measure the same).
constexpr int kSmallTwoTiles = 128;

template <int WF, int EPI, int NP>
hipError_t launch_small(hipStream_t st, const V3Gemm& g, int N) {
    constexpr int NT = kSmallNT<EPI>;
    const int per = (g.K / kUnitK<WF> + g.ks - 1) / g.ks;
    const int W = min(kSmallWaves<EPI>, (per + kSmallCh<WF> - 1) / kSmallCh<WF>);
    const int gx = EPI == VE_QKV ? N / 32 : (EPI == VE_SWIGLU ? N / 32 : (N + 15) / 16);
    // two row tiles per workgroup share its weights; with few column blocks one each, so that
    // twice the CUs pull the activations
    const int mt = g.M > 16 && gx * g.ks >= kSmallTwoTiles ? 2 : 1;
    const dim3 grid(gx, (g.M + 16 * mt - 1) / (16 * mt), g.ks);
    if (mt == 2)
        hipLaunchKernelGGL((vsmall_kernel<WF, EPI, NP, 2>), grid, dim3(64 * W), (size_t)W * (kSmallLds<WF, 2, NT>()), st, g);
    else
        hipLaunchKernelGGL((vsmall_kernel<WF, EPI, NP, 1>), grid, dim3(64 * W), (size_t)W * (kSmallLds<WF, 1, NT>()), st, g);
    return hipGetLastError();
}

template <int WF, int EPI, int BM, int WM, int NT>
hipError_t launch_tile(hipStream_t st, const V3Gemm& g, int N) {
    constexpr int BN = 16 * (4 / WM) * NT, CB = EPI == VE_SWIGLU ? BN / 2 : BN;
    const int gx = (N + CB - 1) / CB, gy = (g.M + BM - 1) / BM;
    const int grid = g.ks > 1 ? g.ks * gx * gy : (gx + 7) / 8 * 8 * gy;
    hipLaunchKernelGGL((vtile_kernel<WF, EPI, BM, WM, NT>), dim3(grid), dim3(256), 0, st, g);
    return hipGetLastError();
}

template <int WF>
hipError_t v3_wf(hipStream_t st, const V3Gemm& g, int epi, int N) {
    if (epi == VE_PLAIN && g.np == 1) return launch_small<WF, VE_PLAIN, 1>(st, g, N);
    if (g.np != 3) return hipErrorInvalidValue;
    const bool small = g.M <= kV3SmallRows;
    switch (epi) {
        case VE_PLAIN:
            return small ? launch_small<WF, VE_PLAIN, 3>(st, g, N) : launch_tile<WF, VE_PLAIN, 64, 2, 2>(st, g, N);
        case VE_QKV:
            return small ? launch_small<WF, VE_QKV, 3>(st, g, N) : launch_tile<WF, VE_QKV, 32, 2, 2>(st, g, N);
        case VE_RES:
            if (small) return launch_small<WF, VE_RES, 3>(st, g, N);
            return g.ks > 1 ? launch_tile<WF, VE_RES, 64, 2, 2>(st, g, N) : launch_tile<WF, VE_RES, 32, 2, 2>(st, g, N);
        case VE_SWIGLU:
            return small ? launch_small<WF, VE_SWIGLU, 3>(st, g, N) : launch_tile<WF, VE_SWIGLU, 64, 2, 4>(st, g, N);
        default:
            return hipErrorInvalidValue;
    }
}

}  // namespace

// Host checks: whole units of K, whole heads of q/k/v, segments that start at
// multiples of 64.
hipError_t launch_v3gemm(hipStream_t st, const V3Gemm& g, int wf, int epi) {
    if (g.nseg < 1 || g.nseg > 3 || g.ks < 1 || g.M < 1 || g.K < 32) return hipErrorInvalidValue;
    // a wave's unit: 32 k of bf16 weights (64 in the tiles), a group of 64 of affine ones
    if (g.K % (wf == VW_BF16 && g.np == 1 ? 32 : 64)) return hipErrorInvalidValue;
    if (g.ks > 1 && epi != VE_RES) return hipErrorInvalidValue;
    int N = 0;
    for (int i = 0; i < g.nseg; i++) {
        if ((i + 1 < g.nseg || epi == VE_QKV || epi == VE_SWIGLU) && g.seg[i].n % 64) return hipErrorInvalidValue;
        N += g.seg[i].n;
    }
    if (N < 1 || (epi != VE_QKV && g.nseg != 1)) return hipErrorInvalidValue;
    if (wf == VW_BF16) return v3_wf<VW_BF16>(st, g, epi, N);
    if (wf == VW_Q4) return v3_wf<VW_Q4>(st, g, epi, N);
    return hipErrorInvalidValue;
}

hipError_t launch_vrow(hipStream_t st, const VRowArgs& a, bool upsample) {
    if (a.N % 32 || a.N < 32 || a.M < 1) return hipErrorInvalidValue;
    const bool one = a.N <= 1024;
    if (upsample) {
        if (one)
            hipLaunchKernelGGL((vrow_kernel<1, 1>), dim3(a.M), dim3(128), 0, st, a);
        else
            hipLaunchKernelGGL((vrow_kernel<1, 0>), dim3(a.M), dim3(128), 0, st, a);
    } else {
        if (one)
            hipLaunchKernelGGL((vrow_kernel<0, 1>), dim3(a.M), dim3(128), 0, st, a);
        else
            hipLaunchKernelGGL((vrow_kernel<0, 0>), dim3(a.M), dim3(128), 0, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_vattn(hipStream_t st, const float* qkv, int M, int ldq, int H, int heads, int kvh, int window,
                        float scale, uint16_t* att, size_t aps, int pair) {
    if (window < 1 || window > 64 || kvh < 1 || heads % kvh) return hipErrorInvalidValue;
    const int grp = heads / kvh;
    if (grp > 16) return hipErrorInvalidValue;  // rejected at model creation
    hipLaunchKernelGGL(vattn_gqa_kernel, dim3(M * kvh), dim3(64 * grp), 0, st, qkv, M, ldq, H, heads, kvh, window,
                       scale, att, aps, pair);
    return hipGetLastError();
}

}  // namespace ming
