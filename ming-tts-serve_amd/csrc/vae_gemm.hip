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
// below the last bit.  4-bit weights enter as the exact integers q - 8; each
// group of 64 is folded in f32 as s * sum (q - 8) x + (b + 8 s) * sum x, the
// group sums of x coming from the same MFMAs against a column of ones.
//
// Activations therefore travel between the kernels as planes: bf16 [3][M][K]
// (fc1's bf16 input is one plane), written by the kernel that produces them.
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

// The segment holding output column c (segments start at multiples of 64) and its first column.
__device__ __forceinline__ int v3_seg_of(const V3Gemm& g, int c, int& start) {
    start = 0;
    int i = 0;
    while (i + 1 < g.nseg && c >= start + g.seg[i].n) {
        start += g.seg[i].n;
        i++;
    }
    return i;
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

// 8 nibbles of a packed word as the bf16 values q - 8 in natural order (exact integers).
__device__ __forceinline__ uint4 unpack_q8(uint32_t w) {
    const int32_t x = (int32_t)(w ^ 0x88888888u);  // q - 8 as a signed 4-bit field
    uint32_t f[8];
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = __float_as_uint((float)((int32_t)((uint32_t)x << (28 - 4 * i)) >> 28));
    return make_uint4(hi_pair(f[0], f[1]), hi_pair(f[2], f[3]), hi_pair(f[4], f[5]), hi_pair(f[6], f[7]));
}

__device__ __forceinline__ f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(a), as_bf8(b), c, 0, 0, 0);
}

constexpr f32x4_t kZero4 = {0.0f, 0.0f, 0.0f, 0.0f};

// MLX fast::rope of the pair (d, d + 32) of a 64-column head from the table's (cos, sin).
__device__ __forceinline__ void v3_rope(const V3Gemm& g, int row, int d, float& x1, float& x2) {
    const float2 cs = *reinterpret_cast<const float2*>(g.rope_cs + ((size_t)row * 32 + d) * 2);
    const float a = x1, b = x2;
    x1 = a * cs.x - b * cs.y;
    x2 = a * cs.y + b * cs.x;
}

__device__ __forceinline__ float v3_swiglu(float g, float u) { return (g * (1.0f / (1.0f + expf(-g)))) * u; }

// One value of the swiglu product into the three planes of the next linear's input.
__device__ __forceinline__ void store_planes(const V3Gemm& g, int row, int col, float o) {
    uint32_t p[3];
    split3(o, p);
    uint16_t* y = g.yp + (size_t)row * g.ldyp + col;
#pragma unroll
    for (int k = 0; k < 3; k++) gst(y + k * g.yps, (uint16_t)(p[k] >> 16));
}

// The epilogue of one row: v[t] are the sums of this lane's columns col[t] (of segment sg that
// starts at sstart); QKV holds rotary pairs in (t, t + NT / 2), SWIGLU gate and up likewise.
template <int EPI, int NT>
__device__ __forceinline__ void v3_epi(const V3Gemm& g, const VSeg& sg, int sstart, int row, const int (&col)[NT],
                                       float (&v)[NT], int z) {
    if constexpr (EPI == VE_SWIGLU) {
#pragma unroll
        for (int t = 0; t < NT / 2; t++)
            store_planes(g, row, col[t], v3_swiglu(v[t] * sg.gs, v[t + NT / 2] * g.up.gs));
    } else if constexpr (EPI == VE_RES) {  // this K slice's sums; the row kernel adds them to the residual
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (col[t] < sg.n) gst(g.y + ((size_t)z * g.M + row) * g.ldy + col[t], v[t] * sg.gs);
    } else {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            v[t] *= sg.gs;
            if (sg.bias) v[t] += bf2f(gld(sg.bias + min(col[t] - sstart, sg.n - 1)));
        }
        if constexpr (EPI == VE_QKV)
            if (sg.rope)
#pragma unroll
                for (int t = 0; t < NT / 2; t++) v3_rope(g, row, col[t] % 64, v[t], v[t + NT / 2]);
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (col[t] - sstart < sg.n) gst(g.y + (size_t)row * g.ldy + col[t], v[t]);
    }
}

// ---- few rows -----------------------------------------------------------------------
// Workgroup (column block x, row block of 16 MT rows y, K slice z); its waves split the
// slice's units (32 k for bf16 weights, one group of 64 for affine ones) in chunks of CH
// whose loads are all issued before the chunk's MFMAs, and their sums meet in LDS in wave
// order.  Columns of a block: 16 (PLAIN, RES), 16 gate + 16 up (SWIGLU), or 16 and the 16
// that are 32 further in the same head (QKV: rotary pairs meet in one lane).
template <int WF>
constexpr int kUnitK = WF == VW_Q4 ? 64 : 32;
template <int WF>
constexpr int kSmallCh = WF == VW_Q4 ? 2 : 4;
constexpr int kSmallWaves = 8;

template <int WF, int NP, int MT, int NT>
struct V3Unit {
    uint4 a[kUnitK<WF> / 32][NP][MT];
    uint4 w[WF == VW_Q4 ? 1 : NT];
    uint2 q[WF == VW_Q4 ? NT : 1];
    uint16_t s[NT], b[NT];
};

template <int WF, int EPI, int NP, int MT>
__global__ __launch_bounds__(64 * kSmallWaves) void vsmall_kernel(V3Gemm g) {
    constexpr int NT = EPI == VE_QKV || EPI == VE_SWIGLU ? 2 : 1;
    constexpr int UK = kUnitK<WF>, UH = UK / 32, CH = kSmallCh<WF>;
    extern __shared__ float red[];  // [waves][MT * 4][NT][64]
    const int W = blockDim.x / kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave, c = lane % 16, j = lane / 16;
    const int m0 = blockIdx.y * 16 * MT, z = blockIdx.z;
    int col[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
        col[t] = EPI == VE_QKV ? (blockIdx.x / 2) * 64 + (blockIdx.x % 2) * 16 + 32 * t + c : blockIdx.x * 16 + c;
    int sstart;
    const VSeg& sg = g.seg[v3_seg_of(g, EPI == VE_QKV ? (blockIdx.x / 2) * 64 : blockIdx.x * 16, sstart)];
    const int U = g.K / UK, per = (U + g.ks - 1) / g.ks, u0 = z * per, u1 = min(U, u0 + per);
    const uint16_t* ar[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        ar[mt] = g.a + (size_t)min(m0 + 16 * mt + c, g.M - 1) * g.K + (WF == VW_Q4 ? 16 : 8) * j;
    const char* wr[NT];
    const uint16_t *sr[NT], *br[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const VSeg& s = EPI == VE_SWIGLU && t == 1 ? g.up : sg;
        const int n = min(col[t] - sstart, s.n - 1);
        if (WF == VW_Q4) {
            wr[t] = static_cast<const char*>(s.w) + (size_t)n * (g.K / 2) + 8 * j;
            sr[t] = s.s + (size_t)n * (g.K / 64);
            br[t] = s.b + (size_t)n * (g.K / 64);
        } else {
            wr[t] = static_cast<const char*>(s.w) + (size_t)n * g.K * 2 + 16 * j;
        }
    }
    f32x4_t hi[MT][NT], lo[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) hi[mt][t] = lo[mt][t] = kZero4;
    auto load = [&](int u, V3Unit<WF, NP, MT, NT>& in) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (WF == VW_Q4) {
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 v = *(const MING_GLOBAL u32x2*)(wr[t] + 32 * (size_t)u);
                in.q[t] = make_uint2(v.x, v.y);
                in.s[t] = gld(sr[t] + u);
                in.b[t] = gld(br[t] + u);
            } else {
                in.w[t] = ldg4(wr[t] + 64 * (size_t)u);
            }
        }
#pragma unroll
        for (int h = 0; h < UH; h++)
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) in.a[h][p][mt] = ldg4(ar[mt] + p * g.aps + (size_t)u * UK + 8 * h);
    };
    const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    auto work = [&](const V3Unit<WF, NP, MT, NT>& in) {
        if constexpr (WF == VW_Q4) {
            f32x4_t xs[MT];  // group sums of x, in every column's place
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                f32x4_t h = mma(in.a[1][0][mt], ones, mma(in.a[0][0][mt], ones, kZero4)), l = kZero4;
#pragma unroll
                for (int p = 1; p < NP; p++) l = mma(in.a[1][p][mt], ones, mma(in.a[0][p][mt], ones, l));
                xs[mt] = h + l;
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint4 b0 = unpack_q8(in.q[t].x), b1 = unpack_q8(in.q[t].y);
                const float s = bf2f(in.s[t]), off = fmaf(8.0f, s, bf2f(in.b[t]));
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    f32x4_t h = mma(in.a[1][0][mt], b1, mma(in.a[0][0][mt], b0, kZero4)), l = kZero4;
#pragma unroll
                    for (int p = 1; p < NP; p++) l = mma(in.a[1][p][mt], b1, mma(in.a[0][p][mt], b0, l));
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        hi[mt][t][r] = fmaf(s, h[r] + l[r], fmaf(off, xs[mt][r], hi[mt][t][r]));
                }
            }
        } else {
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        f32x4_t& acc = p == 0 ? hi[mt][t] : lo[mt][t];
                        acc = mma(in.a[0][p][mt], in.w[t], acc);
                    }
        }
    };
    for (int u = u0 + wave * CH; u < u1; u += W * CH) {
        V3Unit<WF, NP, MT, NT> in[CH];
#pragma unroll
        for (int k = 0; k < CH; k++)
            if (u + k < u1) load(u + k, in[k]);
#pragma unroll
        for (int k = 0; k < CH; k++)
            if (u + k < u1) work(in[k]);
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                red[(((wave * MT + mt) * 4 + r) * NT + t) * kWave + lane] = hi[mt][t][r] + lo[mt][t][r];
    __syncthreads();
    for (int u = wave; u < MT * 4; u += W) {  // row slot u = 4 mt + r
        const int row = m0 + 16 * (u / 4) + 4 * j + u % 4;
        if (row >= g.M) continue;
        float v[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float s = red[(u * NT + t) * kWave + lane];
            for (int w = 1; w < W; w++) s += red[((w * MT * 4 + u) * NT + t) * kWave + lane];
            v[t] = s;
        }
        v3_epi<EPI, NT>(g, sg, sstart, row, col, v, z);
    }
}

// ---- many rows ------------------------------------------------------------------------
// Workgroup tile of BM rows x 16 WN NT weight columns, K in stages of 64 through one LDS
// buffer (the next stage's global loads are in registers while this one computes; two or
// three workgroups share a CU and cover each other's barriers).  4 waves in a WM x WN grid;
// wave (wm, wn) owns the rows BM / WM of wm and the column tiles wn, wn + WN, ..., so that a
// rotary pair (32 columns apart) and a gate / up pair lie in one lane.  LDS rows are 64
// values (128 bytes) with their 16-byte chunks permuted by the row (chunk ^ row % 8): the 16
// rows of a fragment read then fall in distinct banks without padding.
template <int WF, int EPI, int BM, int WM, int NT>
__global__ __launch_bounds__(256) void vtile_kernel(V3Gemm g) {
    constexpr int WN = 4 / WM, MT = BM / WM / 16, BN = 16 * WN * NT;
    constexpr bool DUAL = EPI == VE_SWIGLU;
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
    int sstart;
    const VSeg& sg = g.seg[v3_seg_of(g, n0, sstart)];
    const int G = g.K / 64, per = (G + g.ks - 1) / g.ks, s0 = z * per, S = min(G, s0 + per) - s0;
    const uint16_t* ag[AL];
#pragma unroll
    for (int i = 0; i < AL; i++) {
        const int q = tid + 256 * i, p = q / (BM * 8), row = q / 8 % BM;
        ag[i] = g.a + p * g.aps + (size_t)min(m0 + row, g.M - 1) * g.K + 8 * (q % 8);
    }
    // weight column k of the tile: its row in the segment (DUAL: the second half is the up weight)
    auto wrow = [&](int k, const VSeg*& s) {
        s = DUAL && k >= CB ? &g.up : &sg;
        return (size_t)min(n0 - sstart + (DUAL ? k % CB : k), s->n - 1);
    };
    const char* wg[WL];
    const uint16_t *sr = nullptr, *br = nullptr;
    const bool wload = WF != VW_Q4 || tid < 2 * BN, sload = tid < BN;
#pragma unroll
    for (int i = 0; i < WL; i++) {
        const VSeg* s;
        const int q = tid + 256 * i;
        if (WF == VW_Q4) {
            const size_t n = wrow(min(q / 2, BN - 1), s);
            wg[i] = static_cast<const char*>(s->w) + n * (g.K / 2) + 16 * (q % 2);
        } else {
            const size_t n = wrow(q / 8, s);
            wg[i] = static_cast<const char*>(s->w) + n * g.K * 2 + 16 * (q % 8);
        }
    }
    if (WF == VW_Q4) {
        const VSeg* s;
        const size_t n = wrow(min(tid, BN - 1), s);
        sr = s->s + n * G;
        br = s->b + n * G;
    }
    uint4 ra[AL], rw[WL];
    uint16_t rs = 0, rbi = 0;
    auto gload = [&](int s) {
        const int u = s0 + s;
#pragma unroll
        for (int i = 0; i < AL; i++) ra[i] = ldg4(ag[i] + 64 * (size_t)u);
        if (wload)
#pragma unroll
            for (int i = 0; i < WL; i++) rw[i] = ldg4(wg[i] + (WF == VW_Q4 ? 32 : 128) * (size_t)u);
        if (WF == VW_Q4 && sload) {
            rs = gld(sr + u);
            rbi = gld(br + u);
        }
    };
    auto lstore = [&]() {
#pragma unroll
        for (int i = 0; i < AL; i++) {
            const int q = tid + 256 * i, r = q / 8;  // r % BM = row: BM is a multiple of 8
            As[r * 8 + ((q % 8) ^ (r % 8))] = ra[i];
        }
        if (WF == VW_Q4) {
            if (wload)
#pragma unroll
                for (int i = 0; i < WL; i++) {
                    const int q = tid + 256 * i, k = q / 2;
                    const uint32_t e[4] = {rw[i].x, rw[i].y, rw[i].z, rw[i].w};
#pragma unroll
                    for (int w = 0; w < 4; w++) Ws[k * 8 + ((4 * (q % 2) + w) ^ (k % 8))] = unpack_q8(e[w]);
                }
            if (sload) {
                const float s = bf2f(rs);
                Ss[tid] = make_float2(s, fmaf(8.0f, s, bf2f(rbi)));
            }
        } else {
#pragma unroll
            for (int i = 0; i < WL; i++) {
                const int q = tid + 256 * i, k = q / 8;
                Ws[k * 8 + ((q % 8) ^ (k % 8))] = rw[i];
            }
        }
    };
    f32x4_t hi[MT][NT], lo[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) hi[mt][t] = lo[mt][t] = kZero4;
    const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    auto afrag = [&](int p, int mt, int h) {
        const int r = p * BM + wm * (BM / WM) + 16 * mt + c;
        return As[r * 8 + ((4 * h + j) ^ (r % 8))];
    };
    auto wfrag = [&](int t, int h) {
        const int k = 16 * (t * WN + wn) + c;
        return Ws[k * 8 + ((4 * h + j) ^ (k % 8))];
    };
    auto compute = [&]() {
        if constexpr (WF == VW_Q4) {
            f32x4_t th[MT][NT], tl[MT][NT], xh[MT], xl[MT];
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
                        f32x4_t& x = p == 0 ? xh[mt] : xl[mt];
                        x = mma(a, ones, h == 0 && p < 2 ? kZero4 : x);
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            f32x4_t& acc = p == 0 ? th[mt][t] : tl[mt][t];
                            acc = mma(a, w[t], h == 0 && p < 2 ? kZero4 : acc);
                        }
                    }
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float2 f = Ss[16 * (t * WN + wn) + c];
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        hi[mt][t][r] = fmaf(f.x, th[mt][t][r] + tl[mt][t][r],
                                            fmaf(f.y, xh[mt][r] + xl[mt][r], hi[mt][t][r]));
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
    if (S > 0) gload(0);
    for (int s = 0; s < S; s++) {
        lstore();
        lds_sync();
        if (s + 1 < S) gload(s + 1);
        compute();
        lds_sync();
    }
    int col[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) col[t] = n0 + (16 * (t * WN + wn)) % CB + c;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = m0 + wm * (BM / WM) + 16 * mt + 4 * j + r;
            if (row >= g.M) continue;
            float v[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) v[t] = hi[mt][t][r] + lo[mt][t][r];
            v3_epi<EPI, NT>(g, sg, sstart, row, col, v, z);
        }
}

// ---- rows between the linears -----------------------------------------------------------
// One workgroup per row: the row's values (SRC 0: the residual plus the K-slice partials in
// slice order; SRC 1: the upsampled fc1 rows), stored as the next layer input, then
// fast::rms_norm (w * (x * rsqrt(mean x^2 + eps))) into the planes of the next linear's
// input.  NC = 16-byte chunks a thread holds in registers (0: any width, the row read back).
__device__ __forceinline__ float fc1_value(const VRowArgs& a, int r, int c) {
    // the fc1 row is bf16(acc + bias) for bf16 weights (addmm, one rounding) and
    // bf16(bf16(acc) + bias) for 4-bit ones (quantized_matmul, then the bias add)
    const float v = gld(a.part + (size_t)r * a.N + c), b = a.bias ? bf2f(gld(a.bias + c)) : 0.0f;
    return a.q4 ? rb(rb(v) + b) : rb(v + b);
}

template <int SRC, int NC>
__global__ __launch_bounds__(256) void vrow_kernel(VRowArgs a) {
    __shared__ float red[4];
    const int m = blockIdx.x, N = a.N, n4 = N / 4, t = threadIdx.x;
    // Decoder._linear_upsample_1d (align_corners=False, f32)
    const float pos = ((float)m + 0.5f) / (float)a.scale - 0.5f;
    const int left = (int)floorf(pos);
    const float wr = pos - (float)left, wl = 1.0f - wr;
    const int l = min(max(left, 0), a.T - 1), r = min(max(left + 1, 0), a.T - 1);
    auto value = [&](int i) {
        float4 x;
        if constexpr (SRC == 1) {
            float e[4];
#pragma unroll
            for (int k = 0; k < 4; k++) e[k] = fc1_value(a, l, 4 * i + k) * wl + fc1_value(a, r, 4 * i + k) * wr;
            x = make_float4(e[0], e[1], e[2], e[3]);
        } else {
            float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int z = 0; z < a.ks; z++) {
                const float4 p = reinterpret_cast<const float4*>(a.part + ((size_t)z * a.M + m) * N)[i];
                s = make_float4(s.x + p.x, s.y + p.y, s.z + p.z, s.w + p.w);
            }
            const float4 q = reinterpret_cast<const float4*>(a.res + (size_t)m * N)[i];
            x = make_float4(q.x + s.x, q.y + s.y, q.z + s.z, q.w + s.w);
        }
        reinterpret_cast<float4*>(a.x + (size_t)m * N)[i] = x;
        return x;
    };
    float4 xv[NC > 0 ? NC : 1];
    float ss = 0.0f;
    auto sq = [&](const float4& x) { ss += (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w); };
    if constexpr (NC > 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (t + 256 * k < n4) {
                xv[k] = value(t + 256 * k);
                sq(xv[k]);
            }
    } else {
        for (int i = t; i < n4; i += 256) sq(value(i));
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)N + a.eps);
    auto put = [&](int i, const float4& x) {
        const float e[4] = {x.x, x.y, x.z, x.w};
        uint32_t p[4][3];
#pragma unroll
        for (int k = 0; k < 4; k++) split3(bf2f(gld(a.w + 4 * i + k)) * (e[k] * inv), p[k]);
#pragma unroll
        for (int q = 0; q < 3; q++)
            *reinterpret_cast<uint2*>(a.h + q * a.hps + (size_t)m * N + 4 * i) =
                make_uint2(hi_pair(p[0][q], p[1][q]), hi_pair(p[2][q], p[3][q]));
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (t + 256 * k < n4) put(t + 256 * k, xv[k]);
    } else {
        for (int i = t; i < n4; i += 256) put(i, reinterpret_cast<const float4*>(a.x + (size_t)m * N)[i]);
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
                                                         int window, float scale, uint16_t* att, size_t aps) {
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
    uint16_t* y = att + (size_t)i * H + h * 64 + lane;
#pragma unroll
    for (int k = 0; k < 3; k++) gst(y + k * aps, (uint16_t)(pl[k] >> 16));
}

template <int WF, int EPI, int NP>
hipError_t launch_small(hipStream_t st, const V3Gemm& g, int N) {
    constexpr int NT = EPI == VE_QKV || EPI == VE_SWIGLU ? 2 : 1;
    const int per = (g.K / kUnitK<WF> + g.ks - 1) / g.ks;
    const int W = min(kSmallWaves, (per + kSmallCh<WF> - 1) / kSmallCh<WF>);
    const int gx = EPI == VE_QKV ? N / 32 : (N + 15) / 16;
    const int mt = g.M > 16 ? 2 : 1;
    const dim3 grid(gx, (g.M + 16 * mt - 1) / (16 * mt), g.ks);
    const size_t lds = sizeof(float) * (size_t)W * mt * 4 * NT * kWave;
    if (mt == 2)
        hipLaunchKernelGGL((vsmall_kernel<WF, EPI, NP, 2>), grid, dim3(64 * W), lds, st, g);
    else
        hipLaunchKernelGGL((vsmall_kernel<WF, EPI, NP, 1>), grid, dim3(64 * W), lds, st, g);
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
    if (a.N % 4 || a.N < 4 || a.M < 1) return hipErrorInvalidValue;
    const bool one = a.N <= 1024;
    if (upsample) {
        if (one)
            hipLaunchKernelGGL((vrow_kernel<1, 1>), dim3(a.M), dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((vrow_kernel<1, 0>), dim3(a.M), dim3(256), 0, st, a);
    } else {
        if (one)
            hipLaunchKernelGGL((vrow_kernel<0, 1>), dim3(a.M), dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((vrow_kernel<0, 0>), dim3(a.M), dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_vattn(hipStream_t st, const float* qkv, int M, int ldq, int H, int heads, int kvh, int window,
                        float scale, uint16_t* att, size_t aps) {
    if (window < 1 || window > 64 || kvh < 1 || heads % kvh) return hipErrorInvalidValue;
    const int grp = heads / kvh;
    if (grp > 16) return hipErrorInvalidValue;  // rejected at model creation
    hipLaunchKernelGGL(vattn_gqa_kernel, dim3(M * kvh), dim3(64 * grp), 0, st, qkv, M, ldq, H, heads, kvh, window,
                       scale, att, aps);
    return hipGetLastError();
}

}  // namespace ming
