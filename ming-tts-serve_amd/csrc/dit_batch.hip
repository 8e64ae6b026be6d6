// The flow head for many sequences at once (config 5's DiT head per step):
// cfmSample (src/ming_model.zig:1143-1151, :1161-1203) over R = 6 n rows
// (n sequences x 2 CFG halves x 3 positions), every DiT linear one bf16 GEMM
// on the matrix cores.  Per sequence the arithmetic is the fused DiT path's
// (src/ming_fused.zig:145-289): bias adds rounded once with the product
// (addmm), residuals rounded, gelu with every op rounded, interleaved rotary
// as four f32 products, CFG + Euler (+ SDE) with every op rounded.
//
// GEMM: Y [R][N] = X [R][K] W^T, bf16 in, f32 accumulate.  MFMA 16x16x32 bf16
// lane layout (gfx950): A lane l = row l % 16, k-block l / 16 (8 values); B
// lane l = column l % 16, same k-block; C[r] = (row 4 (l / 16) + r, column
// l % 16).  A rows and W rows are both K-contiguous: the workgroup stages
// 64-k slices of both through LDS (dgemm_kernel below) and each lane reads
// its 16-byte fragments from there.
#include "args.h"
#include "common.h"
#include "dit_attn.h"
#include "flow_steps.h"
#include "internal.h"
#include "tanh_tab.h"

namespace ming {

namespace {


enum DEpi : int { DE_BIAS = 0, DE_RES = 1, DE_GELU = 2, DE_QKV = 3, DE_CFM = 4 };

struct DGemm {
    const uint16_t* x;     // A rows [R][ldx]
    int ldx, R, N, K;
    const uint16_t* w[3];  // [N][K] (DE_QKV: q, k, v of N / 3 rows each)
    const uint16_t* b[3];
    uint16_t* out;         // [R][ldo] (DE_QKV: [3][R][N / 3])
    int ldo;
    const uint16_t* res;   // DE_RES: [R][ldo]
    // DE_QKV
    const float *cos_t, *sin_t;
    int L, hd;
    // DE_CFM: rows 2b (cond) and 2b + 1 (uncond) of sequence b
    const uint16_t *y, *dt, *sq, *sde;  // y [n][N], sde [n][steps][N]
    int step, steps;
    float cfg, shift;
    uint16_t* y_out;       // [n][N]
    uint16_t* y_steps;     // optional [n][steps][N]
    // split K: grid z = ks slices of K / ks; f32 partials [ks][R][N] (bias and
    // epilogue applied by dreduce_kernel).  vs: the slices a row's sum is taken
    // over (a function of K alone); a workgroup that covers several of them (ks <
    // vs) sums each slice from zero and adds the slice sums in slice order, as
    // dreduce_kernel adds the partials, so the bits do not depend on ks
    float* part;
    int ks, vs;
};

__device__ __forceinline__ bf16x8_t as8(uint4 v) { return __builtin_bit_cast(bf16x8_t, u32x4_t{v.x, v.y, v.z, v.w}); }

// this file's copy of the tanh table (tanh_tab.h), filled at context creation
__device__ float dit_batch_tanh_tab[kTanhTabN];

// gelu (approximate) with every op rounded, as gelu_chain (dit.hip): the tanh's argument, then the result.
__device__ __forceinline__ float gelu_arg(float x) {
    const float c0 = rb(0.044715f), c1 = rb(0.7978845608f);
    const float x3 = rb((float)((double)x * (double)x * (double)x));
    const float inner = rb(x + rb(c0 * x3));
    return rb(c1 * inner);
}
__device__ __forceinline__ float gelu_end(float x, float th) { return rb(rb(0.5f * x) * rb(1.0f + rb(th))); }

__device__ __forceinline__ float gelu_chain_b(float x) {
    return gelu_end(x, tanh_bf16(dit_batch_tanh_tab, gelu_arg(x)));
}

// LDS-tiled GEMM: workgroup tile BM rows x 64 columns, K staged kBK (128 where
// K allows, else 64) at a time through two LDS buffers (rows padded by 8
// values: the 16 rows a fragment read touches fall in distinct banks).  256 threads load each stage
// cooperatively (16 bytes each, coalesced) while the previous stage's MFMAs
// run; wave w owns rows 32 (w / 2) .. + 32 and columns 32 (w % 2) .. + 32 of
// a 64-row tile (BM = 64), or rows 0 .. 32 and columns 16 w .. + 16 (BM = 32).
constexpr int kBN = 64;

template <int BM, int kBK>
struct DTile {
    static constexpr int NT = BM == 64 ? 2 : 1;       // 16-column tiles per wave
    static constexpr int AL = BM * kBK / 8 / 256;    // A chunks (16 B) per thread per stage
    static constexpr int BL = kBN * kBK / 8 / 256;   // B chunks per thread per stage
};

template <int BM, int kBK, int E>
__global__ __launch_bounds__(256) void dgemm_kernel(DGemm a) {
    constexpr int kPad = kBK + 8, kCPR = kBK / 8;
    using T = DTile<BM, kBK>;
    constexpr int NT = T::NT;
    __shared__ __align__(16) uint16_t As[2][BM * kPad];
    __shared__ __align__(16) uint16_t Bs[2][kBN * kPad];
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, c = lane % 16, j = lane / 16;
    const int NS = E == DE_QKV ? a.N / 3 : a.N;  // columns per segment (a tile never straddles two)
    const int n0 = blockIdx.x * kBN, si = E == DE_QKV ? n0 / NS : 0, ns0 = n0 - si * NS;
    const uint16_t* W = si == 0 ? a.w[0] : (si == 1 ? a.w[1] : a.w[2]);
    const uint16_t* B = si == 0 ? a.b[0] : (si == 1 ? a.b[1] : a.b[2]);
    const int m0 = blockIdx.y * BM, S = a.K / kBK / a.ks, s0 = blockIdx.z * S;
    const int wm = BM == 64 ? wave / 2 : 0, wn = BM == 64 ? wave % 2 : wave;
    // this thread's global chunks: chunk q -> (row q / kCPR, k 8 (q % kCPR))
    const uint16_t* ag[T::AL];
    const uint16_t* bg[T::BL];
#pragma unroll
    for (int i = 0; i < T::AL; i++) {
        const int q = tid + 256 * i, r = min(m0 + q / kCPR, a.R - 1);
        ag[i] = a.x + (size_t)r * a.ldx + 8 * (q % kCPR);
    }
#pragma unroll
    for (int i = 0; i < T::BL; i++) {
        const int q = tid + 256 * i, n = min(ns0 + q / kCPR, NS - 1);
        bg[i] = W + (size_t)n * a.K + 8 * (q % kCPR);
    }
    // two register sets: the stage about to be stored to LDS and the one after it, in flight
    uint4 ar[2][T::AL], br[2][T::BL];
    auto gload = [&](int s, int set) {
#pragma unroll
        for (int i = 0; i < T::AL; i++) ar[set][i] = ldg4(ag[i] + kBK * (s0 + s));
#pragma unroll
        for (int i = 0; i < T::BL; i++) br[set][i] = ldg4(bg[i] + kBK * (s0 + s));
    };
    auto lstore = [&](int buf, int set) {
#pragma unroll
        for (int i = 0; i < T::AL; i++) {
            const int q = tid + 256 * i;
            *reinterpret_cast<uint4*>(&As[buf][(q / kCPR) * kPad + 8 * (q % kCPR)]) = ar[set][i];
        }
#pragma unroll
        for (int i = 0; i < T::BL; i++) {
            const int q = tid + 256 * i;
            *reinterpret_cast<uint4*>(&Bs[buf][(q / kCPR) * kPad + 8 * (q % kCPR)]) = br[set][i];
        }
    };
    f32x4_t acc[2][NT], tot[2][NT];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[mt][t] = tot[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // after stage s: at the end of a K slice (not the last one of this workgroup), add the
    // slice's sum to the total and start the next slice from zero
    const int Sv = a.K / kBK / a.vs;
    const bool fold = a.ks < a.vs;
    auto slice_end = [&](int s) {
        if (fold && (s + 1) % Sv == 0 && s + 1 < S) {
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    tot[mt][t] = tot[mt][t] + acc[mt][t];
                    acc[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < kBK / 32; ks++) {
            uint4 af[2], bfr[NT];
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
                af[mt] = *reinterpret_cast<const uint4*>(&As[buf][(32 * wm + 16 * mt + c) * kPad + 32 * ks + 8 * j]);
#pragma unroll
            for (int t = 0; t < NT; t++)
                bfr[t] = *reinterpret_cast<const uint4*>(
                    &Bs[buf][((BM == 64 ? 32 : 16) * wn + 16 * t + c) * kPad + 32 * ks + 8 * j]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as8(af[mt]), as8(bfr[t]), acc[mt][t], 0, 0, 0);
        }
    };
    // stages in pairs so that every register-set and LDS-buffer index is a constant:
    // stage s computes from buffer s & 1 while stage s + 1 waits in set (s + 1) & 1
    // and stage s + 2 loads into set s & 1
    gload(0, 0);
    if (S > 1) gload(1, 1);
    lstore(0, 0);
    __syncthreads();
    for (int s = 0; s < S; s += 2) {
        if (s + 2 < S) gload(s + 2, 0);
        compute(0);
        slice_end(s);
        if (s + 1 < S) lstore(1, 1);
        __syncthreads();
        if (s + 1 >= S) break;
        if (s + 3 < S) gload(s + 3, 1);
        compute(1);
        slice_end(s + 1);
        if (s + 2 < S) lstore(0, 0);
        __syncthreads();
    }
    if (fold) {
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[mt][t] = tot[mt][t] + acc[mt][t];
    }
    if (a.ks > 1) {  // split K: f32 partials of this slice; dreduce_kernel finishes
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 32 * wm + 16 * mt + 4 * j + r;
                if (m >= a.R) continue;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int n = ns0 + (BM == 64 ? 32 : 16) * wn + 16 * t + c;
                    if (n < NS) gst(a.part + ((size_t)blockIdx.z * a.R + m) * a.N + n, acc[mt][t][r]);
                }
            }
        return;
    }
    const int cb = ns0 + (BM == 64 ? 32 : 16) * wn;  // this wave's first column within the segment
    if constexpr (E == DE_CFM) {
        // lane rows 4j + {0,1} and 4j + {2,3}: (cond, uncond) of two sequences
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int pr = 0; pr < 2; pr++) {
                const int m = m0 + 32 * wm + 16 * mt + 4 * j + 2 * pr;
                if (m + 1 >= a.R) continue;
                const int sb = m / 2;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int n = cb + 16 * t + c;
                    if (n >= a.N) continue;
                    const float bb = bf2f(gld(B + n));
                    const float pc = rb(acc[mt][t][2 * pr] + bb), pn = rb(acc[mt][t][2 * pr + 1] + bb);
                    const float f0 = rb(pc + rb(rb(pc - pn) * rb(a.cfg)));
                    float y = rb(bf2f(gld(a.y + (size_t)sb * a.N + n)) + rb(bf2f(gld(a.dt + a.step)) * f0));
                    if (a.shift != 0.0f)
                        y = rb(y + rb(rb(rb(a.shift) * bf2f(gld(a.sq + a.step))) *
                                      bf2f(gld(a.sde + ((size_t)sb * a.steps + a.step) * a.N + n))));
                    gst(a.y_out + (size_t)sb * a.N + n, f2bf(y));
                    if (a.y_steps) gst(a.y_steps + ((size_t)sb * a.steps + a.step) * a.N + n, f2bf(y));
                }
            }
        return;
    }
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + 32 * wm + 16 * mt + 4 * j + r;
            const bool row_ok = m < a.R;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int nn = cb + 16 * t + c;  // column within the segment
                const float e = rb(acc[mt][t][r] + bf2f(gld(B + min(nn, NS - 1))));
                if constexpr (E == DE_QKV) {
                    // interleaved rotary on q, k: the pair (2i, 2i+1) is lanes (c, c ^ 1)
                    const float other = __shfl_xor(e, 1, kWave);
                    if (!row_ok) continue;
                    float o = e;
                    if (si < 2) {
                        const int half = a.hd / 2, i = (nn % a.hd) / 2, l = m % a.L;
                        const float cs = gld(a.cos_t + l * half + i), sn = gld(a.sin_t + l * half + i);
                        const float ev = (c & 1) == 0 ? e : other, od = (c & 1) == 0 ? other : e;
                        const float p = ev * cs, q = od * sn, s2 = ev * sn, u = od * cs;
                        o = (c & 1) == 0 ? p - q : s2 + u;
                    }
                    gst(a.out + ((size_t)si * a.R + m) * NS + nn, f2bf(o));
                } else {
                    if (!row_ok || nn >= NS) continue;
                    const size_t off = (size_t)m * a.ldo + nn;
                    if constexpr (E == DE_BIAS) gst(a.out + off, f2bf(e));
                    if constexpr (E == DE_RES) gst(a.out + off, f2bf(bf2f(gld(a.res + off)) + e));
                    if constexpr (E == DE_GELU) gst(a.out + off, f2bf(gelu_chain_b(e)));
                }
            }
        }
}

// Rows rms-normalised (MLX fast::rms_norm: bf16(w * bf16(x * rsqrt(mean x^2 + eps)))),
// one workgroup per output row o; gather > 0: output row o = 2b + h is input
// row (2b + h) * gather + gather - 1 (the last position of each CFG half).
__global__ __launch_bounds__(256) void drms_kernel(const uint16_t* __restrict__ x, int K, int gather,
                                                   const uint16_t* __restrict__ w, float eps,
                                                   uint16_t* __restrict__ out) {
    __shared__ float red[4];
    const int o = blockIdx.x, src = gather > 0 ? o * gather + gather - 1 : o;
    const uint16_t* row = x + (size_t)src * K;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < K / 8; i += 256) {
        const uint4 v = ldg4(row + 8 * i);
        const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const float lo = bf_lo(e[p]), hi = bf_hi(e[p]);
            ss += lo * lo;
            ss += hi * hi;
        }
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)K + eps);
    for (int i = threadIdx.x; i < K / 8; i += 256) {
        const uint4 v = ldg4(row + 8 * i), wv = ldg4(w + 8 * i);
        const uint32_t e[4] = {v.x, v.y, v.z, v.w}, we[4] = {wv.x, wv.y, wv.z, wv.w};
        uint32_t r4[4];
#pragma unroll
        for (int p = 0; p < 4; p++)
            r4[p] = pack_bf2(bf_lo(we[p]) * rb(bf_lo(e[p]) * inv), bf_hi(we[p]) * rb(bf_hi(e[p]) * inv));
        gst(reinterpret_cast<uint4*>(out + (size_t)o * K) + i, make_uint4(r4[0], r4[1], r4[2], r4[3]));
    }
}

// The CFM input rows of every sequence b (cfm `embed`, src/ming_fused.zig:559-561):
// rows (2b + h) * 3 + {0, 1, 2} = [te[h] + ce[b][h], xh[b], xe[b]].
__global__ __launch_bounds__(256) void cfm_rows_kernel(const uint16_t* __restrict__ te, const uint16_t* __restrict__ ce,
                                                       const uint16_t* __restrict__ bc, const uint16_t* __restrict__ xh,
                                                       const uint16_t* __restrict__ xe, int n, int D,
                                                       uint16_t* __restrict__ rows) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n * D) return;
    const int b = k / D, d = k % D;
    const uint16_t xv = gld(xh + k), ev = gld(xe + k);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        // c_emb([z, 0]): the unconditional half is the bias alone
        const float cev = h == 0 ? bf2f(gld(ce + k)) : bf2f(gld(bc + d));
        uint16_t* r = rows + (size_t)(2 * b + h) * 3 * D + d;
        gst(r, f2bf(bf2f(gld(te + (size_t)h * D + d)) + cev));
        gst(r + D, xv);
        gst(r + 2 * D, ev);
    }
}

// Split-K epilogue: sum the ks partials in slice order, then bias and the epilogue.
template <int E>
__global__ __launch_bounds__(256) void dreduce_kernel(DGemm a) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= a.R * a.N) return;
    const int m = k / a.N, n = k % a.N;
    float sum = 0.0f;
    for (int z = 0; z < a.ks; z++) sum += gld(a.part + (size_t)z * a.R * a.N + k);
    const float e = rb(sum + bf2f(gld(a.b[0] + n)));
    const size_t off = (size_t)m * a.ldo + n;
    if constexpr (E == DE_BIAS) gst(a.out + off, f2bf(e));
    if constexpr (E == DE_RES) gst(a.out + off, f2bf(bf2f(gld(a.res + off)) + e));
    if constexpr (E == DE_GELU) gst(a.out + off, f2bf(gelu_chain_b(e)));
}

// Split-K reduce with the residual epilogue (dreduce_kernel<DE_RES>'s arithmetic) followed
// by the row norm of the result (drms_kernel's): one workgroup per row m, thread t holding
// the 8-column chunks t, t + 256; writes the row to a.out and its normalised form to hn.
// The same bits as the two kernels back to back, one launch fewer.
__global__ __launch_bounds__(256) void dreduce_res_rms_kernel(DGemm a, const uint16_t* __restrict__ w, float eps,
                                                              uint16_t* __restrict__ hn) {
    __shared__ float red[4];
    const int m = blockIdx.x, N = a.N;
    constexpr int kMaxC = 2;  // chunks per thread: N <= 4096
    uint32_t xv[kMaxC][4];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < kMaxC; k++) {
        const int i = threadIdx.x + 256 * k;
        if (i >= N / 8) break;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            float v[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int n = 8 * i + 2 * p + h;
                float sum = 0.0f;
                for (int z = 0; z < a.ks; z++) sum += gld(a.part + ((size_t)z * a.R + m) * a.N + n);
                const float e = rb(sum + bf2f(gld(a.b[0] + n)));
                v[h] = rb(bf2f(gld(a.res + (size_t)m * a.ldo + n)) + e);
            }
            xv[k][p] = pack_bf2(v[0], v[1]);
            ss += v[0] * v[0];
            ss += v[1] * v[1];
        }
        gst(reinterpret_cast<uint4*>(a.out + (size_t)m * a.ldo) + i, make_uint4(xv[k][0], xv[k][1], xv[k][2], xv[k][3]));
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
    for (int k = 0; k < kMaxC; k++) {
        const int i = threadIdx.x + 256 * k;
        if (i >= N / 8) break;
        const uint4 wv = ldg4(w + 8 * i);
        const uint32_t we[4] = {wv.x, wv.y, wv.z, wv.w};
        uint32_t r4[4];
#pragma unroll
        for (int p = 0; p < 4; p++)
            r4[p] = pack_bf2(bf_lo(we[p]) * rb(bf_lo(xv[k][p]) * inv), bf_hi(we[p]) * rb(bf_hi(xv[k][p]) * inv));
        gst(reinterpret_cast<uint4*>(hn + (size_t)m * N) + i, make_uint4(r4[0], r4[1], r4[2], r4[3]));
    }
}

// ---- the flow head's block in four launches -------------------------------------------------
// Rows of three positions.  What bounded the general path above at 78 and 384 rows was its eight
// launches a block (split-K partials and their reduce, the norm and the attention between the
// GEMMs: 52 and 70 us a block) and a stage loop with two barriers per 128 k; these kernels take
// the norm into the GEMM that reads it, the attention into the q/k/v GEMM, and keep the K slices
// of a sum in the waves of one workgroup: 33 and 45 us a block, ten steps 4270 -> 2930 us (13
// sequences) and 5720 -> 3780 us (64).  The rounding points and the order of every sum are the
// general path's.  What bounds them now: the redundant norm (each column block normalises its
// rows: 3.4 of ff1's 7.8 us at 78 rows, 4.5 of 12.8 at 384), then the weight stream.
//
// Activations come from LDS (the normalised rows, staged once per workgroup) or from memory in
// the A operand's order: bf16 [row tile][K / 32][lane][8], lane = 16 (k % 32 / 8) + row % 16
// (frag_pos), one contiguous KiB per operand, as the kernel that produced them wrote them.

__device__ __forceinline__ f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as8(a), as8(b), c, 0, 0, 0);
}

__device__ __forceinline__ size_t frag_pos(int m, int k, int K) {
    return ((size_t)(m / 16) * (K / 32) + k / 32) * 512 + (16 * (k % 32 / 8) + m % 16) * 8 + k % 8;
}

// Workgroup id -> (column block, row block): the row blocks of a column block go to ids of one
// XCD (id mod 8), so each XCD's L2 reads its share of the weights once.
__device__ __forceinline__ void col_row(int id, int rb, int& bx, int& by) {
    bx = id % 8 + 8 * (id / 8 / rb);
    by = id / 8 % rb;
}

// Normalised rows (drms_kernel's arithmetic) r0 .. r0 + 16 MT into LDS in operand order, the
// row's place permuted by the chunk so that the writes of a row and the reads of an operand both
// spread over the banks.  A wave takes four rows at a time, 16 lanes a row: lane i holds the
// chunks 4 i .. 4 i + 3 of each 512 values, whose sums meet in the tree that one chunk a lane
// over 64 lanes makes (the same bits), in a loop: straight-line code for every row was 20 KB that
// a launch of ten microseconds fetched cold (13.6 us for ff1 at 78 rows).  gather > 0: row o is
// row o * gather + gather - 1 of x.
template <int D, int MT, int WAVES>
struct NormRows {
    static constexpr int H = D / 512, C = 4 * H;  // 512-value parts, chunks a lane
    uint4 v[C];
    __device__ __forceinline__ static int chunk(int k) { return 64 * (k / 4) + 4 * (threadIdx.x % 16) + k % 4; }
    __device__ __forceinline__ void load(uint4 (&d)[C], const uint16_t* __restrict__ x, int q, int r0, int R,
                                         int gather) {
        const int o = min(r0 + 4 * q + (int)(threadIdx.x % kWave) / 16, R - 1);
        const uint16_t* row = x + (size_t)(gather > 0 ? o * gather + gather - 1 : o) * D;
#pragma unroll
        for (int k = 0; k < C; k++) d[k] = ldg4(row + 8 * chunk(k));
    }
    __device__ __forceinline__ void stage(const uint16_t* __restrict__ x, int r0, int R, int gather,
                                          const uint16_t* __restrict__ nw, float eps, uint4* As) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        uint4 wv[C];
#pragma unroll
        for (int k = 0; k < C; k++) wv[k] = ldg4(nw + 8 * chunk(k));
#pragma unroll 1
        for (int q = wave; q < 4 * MT; q += WAVES) {
            uint4 e[C];
#pragma unroll
            for (int k = 0; k < C; k++) e[k] = v[k];
            if (q + WAVES < 4 * MT) load(v, x, q + WAVES, r0, R, gather);
            float ss = 0.0f;
#pragma unroll
            for (int h = 0; h < H; h++) {
                float t[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t p[4] = {e[4 * h + k].x, e[4 * h + k].y, e[4 * h + k].z, e[4 * h + k].w};
                    t[k] = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        t[k] += bf_lo(p[i]) * bf_lo(p[i]);
                        t[k] += bf_hi(p[i]) * bf_hi(p[i]);
                    }
                }
                ss += team_sum<16>((t[0] + t[1]) + (t[2] + t[3]));
            }
            const float inv = 1.0f / sqrtf(ss / (float)D + eps);
            const int m = 4 * q + (int)(threadIdx.x % kWave) / 16;
#pragma unroll
            for (int k = 0; k < C; k++) {
                const int ch = chunk(k);
                const uint32_t p[4] = {e[k].x, e[k].y, e[k].z, e[k].w};
                const uint32_t we[4] = {wv[k].x, wv[k].y, wv[k].z, wv[k].w};
                uint32_t r[4];
#pragma unroll
                for (int i = 0; i < 4; i++)
                    r[i] = pack_bf2(bf_lo(we[i]) * rb(bf_lo(p[i]) * inv), bf_hi(we[i]) * rb(bf_hi(p[i]) * inv));
                As[((m / 16) * (D / 32) + ch / 4) * 64 + 16 * (ch % 4) + ((m ^ ch) & 15)] =
                    make_uint4(r[0], r[1], r[2], r[3]);
            }
        }
    }
};

// A wave's weight stream: NT column tiles of 16 rows, two register sets of CH 32-k steps in
// flight.  A load of the B operand itself (lane 16 j + c: row c, k block j) puts each of 16
// consecutive lanes on another row, and the address unit takes such a load lane by lane: 35 GB/s
// a CU from the L2 where four lanes to a row's 64 bytes reach 72 and contiguous lanes 75.  So
// lane l loads row l / 4, block l % 4, and the wave turns the set round through 1 KB a step of
// LDS of its own (blocks permuted by the row: no bank conflicts either way).  The order of a
// turn's stores and loads needs no fence: lane 0 loads the word that it stores, of the same type, in
// every block, so no load can be moved past a store of its block.  (A wavefront fence on either side
// of put() also orders what need not be: 64 sequences 3735 -> 3762 us, 13 2920 -> 2944.)
template <int NT, int CH>
struct WStream {
    static constexpr int kLds = CH * NT * 64;  // uint4s a wave
    uint4 r[2][CH][NT];
    const uint16_t* p[NT];
    uint4* wr;
    const uint4* rd;
    // rows: the first weight row of each tile (a pointer to its first k); lds: the wave's area
    __device__ __forceinline__ void init(uint4* lds) {
        const int l = threadIdx.x % kWave, row = l / 4, c = l % 16, j = l / 16;
        wr = lds + 4 * row + (l % 4 ^ row / 4);
        rd = lds + 4 * c + (j ^ c / 4);
    }
    __device__ __forceinline__ void tile(int t, const uint16_t* w, int K) {
        const int l = threadIdx.x % kWave;
        p[t] = w + (size_t)(l / 4) * K + 8 * (l % 4);
    }
    __device__ __forceinline__ void load(int set, int s) {
#pragma unroll
        for (int k = 0; k < CH; k++)
#pragma unroll
            for (int t = 0; t < NT; t++) r[set][k][t] = ldg4(p[t] + 32 * (s + k));
    }
    __device__ __forceinline__ void put(int set) {
#pragma unroll
        for (int k = 0; k < CH; k++)
#pragma unroll
            for (int t = 0; t < NT; t++) wr[64 * (NT * k + t)] = r[set][k][t];
    }
    __device__ __forceinline__ uint4 get(int k, int t) const { return rd[64 * (NT * k + t)]; }
};

// CH steps from step s of activations in LDS (S steps a row tile).
template <int MT, int NT, int CH>
__device__ __forceinline__ void lds_mma(const WStream<NT, CH>& w, const uint4* As, int S, int s, f32x4_t (&acc)[MT][NT]) {
    static_assert(CH % 4 == 0, "the rows' permutation by the step is a constant");
    const int lane = threadIdx.x % kWave, c = lane % 16, j = lane / 16;
#pragma unroll
    for (int k = 0; k < CH; k++) {
        uint4 a[MT], b[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) b[t] = w.get(k, t);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) a[mt] = As[(mt * S + s + k) * 64 + 16 * j + (c ^ j ^ (4 * (k % 4)))];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[mt][t] = mma(a[mt], b[t], acc[mt][t]);
    }
}

struct FlowQkv {
    const uint16_t* x;     // [R][D]
    int R, rb;             // rb: row blocks
    const uint16_t *norm, *w[3], *b[3];
    float eps;
    const float *cos_t, *sin_t;  // [3][32]
    uint16_t* att;         // operand order, D columns
};

// norm1, q/k/v with rotary and the attention of one head (64 columns of each) over 16 MT / 3
// groups of three rows; wave w owns the column tiles w, w + WAVES, ... of the twelve.  One
// workgroup reads a head's 384 KB of weights, so the groups of a workgroup trade weight reads
// against workgroups in flight: 5 groups while that gives at most one workgroup a CU, else 10.
template <int D, int MT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void flow_qkv_kernel(FlowQkv a) {
    constexpr int NT = 12 / WAVES, CH = NT > 1 ? 4 : 8, GR = 16 * MT / 3, LD = 192 + 8, S = D / 32;
    __shared__ uint4 As[MT * S * 64];
    __shared__ uint4 Ws[WAVES * WStream<NT, CH>::kLds];
    static_assert(16 * MT * LD * 2 <= (int)sizeof(As), "the q/k/v tile reuses the rows' buffer");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, c = lane % 16,
              j = lane / 16;
    int head, by;
    col_row(blockIdx.x, a.rb, head, by);
    const int r0 = 3 * GR * by;
    if (64 * head >= D) return;
    NormRows<D, MT, WAVES> rows;
    if (wave < 4 * MT) rows.load(rows.v, a.x, wave, r0, a.R, 0);
    WStream<NT, CH> w;
    w.init(Ws + wave * w.kLds);
    float bias[NT], cs[NT][3], sn[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tile = wave + WAVES * t, col = 64 * head + 16 * (tile % 4) + c;
        const uint16_t* W = tile / 4 == 0 ? a.w[0] : (tile / 4 == 1 ? a.w[1] : a.w[2]);
        const uint16_t* B = tile / 4 == 0 ? a.b[0] : (tile / 4 == 1 ? a.b[1] : a.b[2]);
        w.tile(t, W + (size_t)(col - c) * D, D);
        bias[t] = bf2f(gld(B + col));
#pragma unroll
        for (int l = 0; l < 3; l++) {
            // position of row 16 mt + 4 j + r, (mt + j + r) % 3, at [(mt + r) % 3]
            cs[t][l] = gld(a.cos_t + 32 * ((l + j) % 3) + col % 64 / 2);
            sn[t][l] = gld(a.sin_t + 32 * ((l + j) % 3) + col % 64 / 2);
        }
    }
    w.load(0, 0);
    w.load(1, CH);
    rows.stage(a.x, r0, a.R, 0, a.norm, a.eps, As);
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    lds_sync();
#pragma unroll 1
    for (int s = 0; s < S; s += 2 * CH) {
        w.put(0);
        if (s + 2 * CH < S) w.load(0, s + 2 * CH);
        lds_mma<MT, NT, CH>(w, As, S, s, acc);
        w.put(1);
        if (s + 3 * CH < S) w.load(1, s + 3 * CH);
        lds_mma<MT, NT, CH>(w, As, S, s + CH, acc);
    }
    lds_sync();
    uint16_t* tile = reinterpret_cast<uint16_t*>(As);  // [16 MT][LD]: q | k | v of the head
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 16 * mt + 4 * j + r;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int tl = wave + WAVES * t;
                const float e = rb(acc[mt][t][r] + bias[t]), other = lane_xor1(e);
                // interleaved rotary on q, k: the pair (2i, 2i + 1) is lanes c, c ^ 1
                const float cv = cs[t][(mt + r) % 3], sv = sn[t][(mt + r) % 3];
                const float p = e * cv, q = other * sv;
                const float o = tl < 8 ? ((c & 1) == 0 ? p - q : q + p) : e;
                tile[m * LD + 16 * tl + c] = f2bf(o);
            }
        }
    lds_sync();
    for (int g = wave; g < GR; g += WAVES) {
        const int row = r0 + 3 * g;
        if (row + 2 >= a.R) break;
        float q[kMaxL], k[kMaxL], v[kMaxL], o[kMaxL];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            q[i] = bf2f(tile[(3 * g + i) * LD + lane]);
            k[i] = bf2f(tile[(3 * g + i) * LD + 64 + lane]);
            v[i] = bf2f(tile[(3 * g + i) * LD + 128 + lane]);
        }
        attn_math(q, k, v, 3, true, o);
#pragma unroll
        for (int i = 0; i < 3; i++) gst(a.att + frag_pos(row + i, 64 * head + lane, D), f2bf(o[i]));
    }
}

struct FlowNorm {
    const uint16_t* x;      // [R][K], or gathered rows of it
    int R, N, rb, gather;
    const uint16_t *norm, *w, *b;
    float eps;
    uint16_t* out;          // DE_GELU: operand order, N columns
    // DE_CFM: as DGemm
    const uint16_t *y, *dt, *sq, *sde;
    int step, steps;
    float cfg, shift;
    uint16_t *y_out, *y_steps;
};

// Norm + linear over 16 MT rows x 16 NT W columns, W waves of NT column tiles each: ff1 with gelu
// (DE_GELU) and the final layer with CFG + Euler (DE_CFM).
template <int D, int E, int MT, int NT, int W>
__global__ __launch_bounds__(64 * W, 1) void flow_norm_kernel(FlowNorm a) {
    constexpr int S = D / 32, VS = E == DE_GELU ? k_slices(D) : 1, CH = NT > 1 ? 4 : 8;
    __shared__ uint4 As[MT * S * 64];
    __shared__ uint4 Ws[W * WStream<NT, CH>::kLds];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, c = lane % 16,
              j = lane / 16;
    int bx, by;
    col_row(blockIdx.x, a.rb, bx, by);
    const int r0 = 16 * MT * by, n0 = 16 * W * NT * bx;
    if (n0 >= a.N) return;
    NormRows<D, MT, W> rows;
    if (wave < 4 * MT) rows.load(rows.v, a.x, wave, r0, a.R, a.gather);
    WStream<NT, CH> w;
    w.init(Ws + wave * w.kLds);
    float bias[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int col = n0 + 16 * (NT * wave + t) + c;
        w.tile(t, a.w + (size_t)(col - c) * D, D);
        bias[t] = bf2f(gld(a.b + col));
    }
    w.load(0, 0);
    w.load(1, CH);
    rows.stage(a.x, r0, a.R, a.gather, a.norm, a.eps, As);
    f32x4_t acc[MT][NT], tot[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[mt][t] = tot[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    lds_sync();
#pragma unroll 1
    for (int s = 0; s < S; s += 2 * CH) {
        w.put(0);
        if (s + 2 * CH < S) w.load(0, s + 2 * CH);
        lds_mma<MT, NT, CH>(w, As, S, s, acc);
        w.put(1);
        if (s + 3 * CH < S) w.load(1, s + 3 * CH);
        lds_mma<MT, NT, CH>(w, As, S, s + CH, acc);
        if (VS > 1 && (s + 2 * CH) % (S / VS) == 0)  // the end of a slice
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    tot[mt][t] = tot[mt][t] + acc[mt][t];
                    acc[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
    }
    if constexpr (E == DE_CFM) {
        // lane rows 4j + {0,1} and 4j + {2,3}: (cond, uncond) of two sequences
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int pr = 0; pr < 2; pr++) {
                const int m = r0 + 16 * mt + 4 * j + 2 * pr;
                if (m + 1 >= a.R) continue;
                const int sb = m / 2;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int n = n0 + 16 * (NT * wave + t) + c;
                    const float pc = rb(acc[mt][t][2 * pr] + bias[t]), pn = rb(acc[mt][t][2 * pr + 1] + bias[t]);
                    const float f0 = rb(pc + rb(rb(pc - pn) * rb(a.cfg)));
                    float y = rb(bf2f(gld(a.y + (size_t)sb * a.N + n)) + rb(bf2f(gld(a.dt + a.step)) * f0));
                    if (a.shift != 0.0f)
                        y = rb(y + rb(rb(rb(a.shift) * bf2f(gld(a.sq + a.step))) *
                                      bf2f(gld(a.sde + ((size_t)sb * a.steps + a.step) * a.N + n))));
                    gst(a.y_out + (size_t)sb * a.N + n, f2bf(y));
                    if (a.y_steps) gst(a.y_steps + ((size_t)sb * a.steps + a.step) * a.N + n, f2bf(y));
                }
            }
    } else {
        lds_sync();
        uint16_t* tile = reinterpret_cast<uint16_t*>(As);  // [MT][W NT / 2][lane][8]: the output in operand order
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    tile[frag_pos(16 * mt + 4 * j + r, 16 * (NT * wave + t) + c, 16 * W * NT)] =
                        f2bf((VS > 1 ? tot[mt][t][r] : acc[mt][t][r]) + bias[t]);
        lds_sync();
        // gelu on 8 values a turn, the tanh table's loads in one go (not one round trip a value)
#pragma unroll 1
        for (int q = threadIdx.x; q < MT * NT * W * 32; q += 64 * W) {
            const int rt = r0 / 16 + q / (32 * W * NT);
            if (16 * rt >= a.R) break;
            const uint4 p = As[q];
            const uint32_t e[4] = {p.x, p.y, p.z, p.w};
            float x[8], u[8], th[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                x[i] = i % 2 ? bf_hi(e[i / 2]) : bf_lo(e[i / 2]);
                u[i] = gelu_arg(x[i]);
                th[i] = gld(dit_batch_tanh_tab + min(__float_as_uint(u[i]) >> 16 & 0x7fffu, (uint32_t)kTanhTabN - 1));
            }
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                o[i] = pack_bf2(gelu_end(x[2 * i], tanh_bf16_of(th[2 * i], u[2 * i])),
                                gelu_end(x[2 * i + 1], tanh_bf16_of(th[2 * i + 1], u[2 * i + 1])));
            gst(reinterpret_cast<uint4*>(a.out) + ((size_t)rt * (a.N / 32) + n0 / 32) * 64 + q % (32 * W * NT),
                make_uint4(o[0], o[1], o[2], o[3]));
        }
    }
}

struct FlowRes {
    const uint16_t* a;      // operand order, K columns
    int R, N, K, rb;
    const uint16_t *w, *b, *res;
    uint16_t* out;          // [R][N]
};

// out = res + bf16(a W^T + b) (out_proj, ff2): VS x CW waves, wave (v, cw) sums the K slice v of
// NT column tiles over 16 MT rows; the slices of a value meet in LDS and are added in slice order.
template <int MT, int NT, int VS, int CW>
__global__ __launch_bounds__(64 * VS * CW, 1) void flow_res_kernel(FlowRes a) {
    constexpr int TH = 64 * VS * CW, CB = 16 * NT * CW, CH = flow_set_steps(MT, NT);
    static_assert(kFlowSetSteps % CH == 0, "flow_k_fits: whole register sets");
    constexpr int IT = (MT * 16 * CB / 4 + TH - 1) / TH;  // values (4 columns of a row) per thread at the end
    __shared__ __align__(16) float red[VS * CW * MT * 4 * NT * 64];
    __shared__ uint4 Ws[VS * CW * WStream<NT, CH>::kLds];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, c = lane % 16,
              j = lane / 16;
    const int v = wave % VS, cw = wave / VS;
    int bx, by;
    col_row(blockIdx.x, a.rb, bx, by);
    const int S = a.K / 32 / VS, r0 = 16 * MT * by, n0 = CB * bx;
    if (n0 >= a.N) return;
    const uint16_t* ap[MT];
    WStream<NT, CH> w;
    w.init(Ws + wave * w.kLds);
#pragma unroll
    for (int t = 0; t < NT; t++) w.tile(t, a.w + (size_t)(n0 + 16 * (NT * cw + t)) * a.K + 32 * S * v, a.K);
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        ap[mt] = a.a + ((size_t)min(r0 / 16 + mt, (a.R - 1) / 16) * (a.K / 32) + S * v) * 512 + 8 * lane;
    uint4 ar[2][CH][MT];
    auto load = [&](int set, int s) __attribute__((always_inline)) {
        w.load(set, s);
#pragma unroll
        for (int k = 0; k < CH; k++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) ar[set][k][mt] = ldg4(ap[mt] + 512 * (s + k));
    };
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto work = [&](int set) __attribute__((always_inline)) {
        w.put(set);
#pragma unroll
        for (int k = 0; k < CH; k++) {
            uint4 b[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) b[t] = w.get(k, t);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int t = 0; t < NT; t++) acc[mt][t] = mma(ar[set][k][mt], b[t], acc[mt][t]);
        }
    };
    flow_first<CH>(S, load);
    // the epilogue's operands, in flight behind the first sets
    uint2 rv[IT], bv[IT];
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int it = threadIdx.x + TH * i, row = min(r0 + it / (CB / 4), a.R - 1), n = n0 + 4 * (it % (CB / 4));
        const uint16_t *rp = a.res + (size_t)row * a.N + n, *bp = a.b + n;
        rv[i] = make_uint2(gld(reinterpret_cast<const uint32_t*>(rp)), gld(reinterpret_cast<const uint32_t*>(rp) + 1));
        bv[i] = make_uint2(gld(bp) | (uint32_t)gld(bp + 1) << 16, gld(bp + 2) | (uint32_t)gld(bp + 3) << 16);
    }
    flow_turns<CH>(S, load, work);
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                red[((((v * CW + cw) * MT + mt) * 4 + r) * NT + t) * 64 + lane] = acc[mt][t][r];
    lds_sync();
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int it = threadIdx.x + TH * i, m = it / (CB / 4), col = 4 * (it % (CB / 4));
        if (m >= 16 * MT || r0 + m >= a.R) continue;
        const float* p = red + ((((col / (16 * NT)) * MT + m / 16) * 4 + m % 4) * NT + col / 16 % NT) * 64 +
                         16 * (m % 16 / 4) + col % 16;
        float4 sum = VS > 1 ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *reinterpret_cast<const float4*>(p);
#pragma unroll
        for (int z = 0; z < (VS > 1 ? VS : 0); z++) {
            const float4 q = *reinterpret_cast<const float4*>(p + z * (CW * MT * 4 * NT * 64));
            sum = make_float4(sum.x + q.x, sum.y + q.y, sum.z + q.z, sum.w + q.w);
        }
        const uint32_t lo = pack_bf2(bf_lo(rv[i].x) + rb(sum.x + bf_lo(bv[i].x)), bf_hi(rv[i].x) + rb(sum.y + bf_hi(bv[i].x)));
        const uint32_t hi = pack_bf2(bf_lo(rv[i].y) + rb(sum.z + bf_lo(bv[i].y)), bf_hi(rv[i].y) + rb(sum.w + bf_hi(bv[i].y)));
        uint32_t* op = reinterpret_cast<uint32_t*>(a.out + (size_t)(r0 + m) * a.N + n0 + col);
        gst(op, lo);
        gst(op + 1, hi);
    }
}

// cfm_rows_kernel with x_emb(y) (K = latent, one slice) computed here: 16 sequences x 64
// columns a workgroup, a wave per 16 columns.
__global__ __launch_bounds__(256) void flow_rows_kernel(const uint16_t* __restrict__ y, int lat,
                                                        const uint16_t* __restrict__ wx, const uint16_t* __restrict__ bx,
                                                        const uint16_t* __restrict__ te, const uint16_t* __restrict__ ce,
                                                        const uint16_t* __restrict__ bc, const uint16_t* __restrict__ xh,
                                                        int n, int D, uint16_t* __restrict__ rows) {
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, c = lane % 16, j = lane / 16;
    const int col = 64 * blockIdx.x + 16 * wave + c, b0 = 16 * blockIdx.y;
    const uint16_t *ap = y + (size_t)min(b0 + c, n - 1) * lat + 8 * j, *wp = wx + (size_t)col * lat + 8 * j;
    const float bias = bf2f(gld(bx + col)), t0 = bf2f(gld(te + col)), t1 = bf2f(gld(te + D + col)),
                uc = bf2f(gld(bc + col));
    uint16_t cv[4], xv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const size_t o = (size_t)min(b0 + 4 * j + r, n - 1) * D + col;
        cv[r] = gld(ce + o);
        xv[r] = gld(xh + o);
    }
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k = 0; k < lat; k += 64) {
        const uint4 a0 = ldg4(ap + k), a1 = ldg4(ap + k + 32), w0 = ldg4(wp + k), w1 = ldg4(wp + k + 32);
        acc = mma(a1, w1, mma(a0, w0, acc));
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int b = b0 + 4 * j + r;
        if (b >= n) continue;
        const uint16_t e = f2bf(acc[r] + bias);
        uint16_t* p = rows + (size_t)b * 6 * D + col;
        gst(p, f2bf(t0 + bf2f(cv[r])));
        gst(p + D, xv[r]);
        gst(p + 2 * D, e);
        gst(p + 3 * D, f2bf(t1 + uc));  // c_emb([z, 0]): the unconditional half is the bias alone
        gst(p + 4 * D, xv[r]);
        gst(p + 5 * D, e);
    }
}

int xcd_grid(int cb, int rb) { return (cb + 7) / 8 * 8 * rb; }

// Row and column tiles of a workgroup (columns in units; ff1's second one is four more waves, which
// cover each other's norm and loads: 384 rows 14.5 -> 13.6 us against two tiles a wave): the
// smallest of the list with at most one workgroup a CU (a second one on some CUs doubles the
// launch's time; larger tiles than needed leave CUs idle).
template <class F>
hipError_t pick_tile(int R, int N, int unit, F launch) {
    const int rt = (R + 15) / 16, cus = device_cus();
    const int cand[5][2] = {{1, 1}, {2, 1}, {3, 1}, {2, 2}, {3, 2}};
    for (int i = 0; i < 5; i++) {
        const int rb = (rt + cand[i][0] - 1) / cand[i][0], cb = (N + unit * cand[i][1] - 1) / (unit * cand[i][1]);
        if (N % (unit * cand[i][1])) continue;
        const int alt = i + 1 < 5 && N % (2 * unit) == 0;
        if (rb * cb <= cus || i == 4 || (i == 2 && !alt)) return launch(i, rb, xcd_grid(cb, rb));
    }
    return hipErrorInvalidValue;
}

template <int D>
hipError_t launch_flow_ff1(hipStream_t st, FlowNorm a) {
    return pick_tile(a.R, a.N, 64, [&](int i, int rb, int grid) {
        a.rb = rb;
        void (*k)(FlowNorm) = i == 0   ? flow_norm_kernel<D, DE_GELU, 1, 1, 4>
                              : i == 1 ? flow_norm_kernel<D, DE_GELU, 2, 1, 4>
                              : i == 2 ? flow_norm_kernel<D, DE_GELU, 3, 1, 4>
                              : i == 3 ? flow_norm_kernel<D, DE_GELU, 2, 1, 8>
                                       : flow_norm_kernel<D, DE_GELU, 3, 1, 8>;
        hipLaunchKernelGGL(k, dim3(grid), dim3(i < 3 ? 256 : 512), 0, st, a);
        return hipGetLastError();
    });
}

template <int VS, int CW>
hipError_t launch_flow_res_vs(hipStream_t st, FlowRes a) {
    return pick_tile(a.R, a.N, 16 * CW, [&](int i, int rb, int grid) {
        a.rb = rb;
        void (*k)(FlowRes) = i == 0   ? flow_res_kernel<1, 1, VS, CW>
                             : i == 1 ? flow_res_kernel<2, 1, VS, CW>
                             : i == 2 ? flow_res_kernel<3, 1, VS, CW>
                             : i == 3 ? flow_res_kernel<2, 2, VS, CW>
                                      : flow_res_kernel<3, 2, VS, CW>;
        hipLaunchKernelGGL(k, dim3(grid), dim3(64 * VS * CW), 0, st, a);
        return hipGetLastError();
    });
}

hipError_t launch_flow_res(hipStream_t st, const FlowRes& a) {
    if (!flow_k_fits(a.K)) return hipErrorInvalidValue;
    const int vs = k_slices(a.K);
    return vs == 4 ? launch_flow_res_vs<4, 1>(st, a) : (vs == 2 ? launch_flow_res_vs<2, 2>(st, a) : launch_flow_res_vs<1, 4>(st, a));
}

template <int D>
hipError_t flow_block(hipStream_t st, const DitBlockDev& w, const uint16_t* x, int R, const float* cos_t,
                      const float* sin_t, uint16_t* att, uint16_t* x1, uint16_t* hh, uint16_t* out) {
    const int F = w.F, groups = R / 3, heads = D / 64;
    FlowQkv q{x, R, (groups + 4) / 5, w.norm1, {w.wq, w.wk, w.wv}, {w.bq, w.bk, w.bv}, w.eps, cos_t, sin_t, att};
    if (q.rb * heads <= device_cus()) {
        hipLaunchKernelGGL((flow_qkv_kernel<D, 1, 12>), dim3(xcd_grid(heads, q.rb)), dim3(768), 0, st, q);
    } else {
        q.rb = (groups + 9) / 10;
        hipLaunchKernelGGL((flow_qkv_kernel<D, 2, 4>), dim3(xcd_grid(heads, q.rb)), dim3(256), 0, st, q);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = launch_flow_res(st, FlowRes{att, R, D, D, 0, w.wo, w.bo, x, x1});
    if (e != hipSuccess) return e;
    if ((e = launch_flow_ff1<D>(st, FlowNorm{x1, R, F, 0, 0, w.norm2, w.w1, w.b1, w.eps, hh})) != hipSuccess) return e;
    return launch_flow_res(st, FlowRes{hh, R, D, F, 0, w.w2, w.b2, x1, out});
}

// ---- launches --------------------------------------------------------------------------------
// 64-row tiles when they still give >= 128 workgroups, else 32-row tiles.
// K >= 2048 (plain epilogues, with a partials buffer) splits four ways across
// workgroups; the split depends on K alone, so a row's arithmetic does not
// depend on how many rows are batched.
template <int E>
void dsplit(DGemm& a) {
    constexpr bool SPLIT = E == DE_BIAS || E == DE_RES || E == DE_GELU;
    const int gx = (a.N + kBN - 1) / kBN, tiles = gx * ((a.R + 31) / 32);
    a.vs = SPLIT ? k_slices(a.K) : 1;
    a.ks = !a.part ? 1 : (a.vs == 4 ? 4 : (a.vs == 2 && tiles < 512 ? 2 : 1));
}

template <int E>
hipError_t dpick(hipStream_t st, DGemm a, const uint16_t* rms_w = nullptr, float rms_eps = 0.0f,
                 uint16_t* rms_out = nullptr) {
    const int gx = (a.N + kBN - 1) / kBN;
    // The sum over K is taken in vs slices fixed by K alone (4 from K = 2048, 2 from K = 1024,
    // for the epilogues the reduce kernel applies), so a sequence's bits do not depend on the
    // batch it is in.  How many workgroups share a row's K (ks) is a launch choice: latency
    // bound at these sizes, K split over workgroups keeps more of them per CU in flight
    // (measured on the 16- and 64-sequence server step: +9-11 %), except where the grid
    // already has >= 512 workgroups (splitting one at 768 loses 5 %); with ks < vs each
    // workgroup folds its slices in the reduce kernel's order.
    dsplit<E>(a);
    if (a.K % (64 * a.vs)) return hipErrorInvalidValue;
    // 128-wide K stages put twice the bytes of each stage in flight (measured: +10 % at 96 rows);
    // slices are whole stages
    if (a.K % (128 * a.vs) == 0)
        hipLaunchKernelGGL((dgemm_kernel<32, 128, E>), dim3(gx, (a.R + 31) / 32, a.ks), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((dgemm_kernel<32, 64, E>), dim3(gx, (a.R + 31) / 32, a.ks), dim3(256), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // rms_out: the caller wants the rows' norm next (DE_RES only); with split K the reduce does it
    if (a.ks == 1) {
        if (rms_out) {
            hipLaunchKernelGGL(drms_kernel, dim3(a.R), dim3(256), 0, st, a.out, a.N, 0, rms_w, rms_eps, rms_out);
            e = hipGetLastError();
        }
        return e;
    }
    if constexpr (E == DE_RES) {
        if (rms_out) {
            if (a.N % 8 || a.N > 4096 || a.ldo != a.N) return hipErrorInvalidValue;
            hipLaunchKernelGGL(dreduce_res_rms_kernel, dim3(a.R), dim3(256), 0, st, a, rms_w, rms_eps, rms_out);
            return hipGetLastError();
        }
    }
    if constexpr (E == DE_BIAS || E == DE_RES || E == DE_GELU) {
        hipLaunchKernelGGL(dreduce_kernel<E>, dim3((a.R * a.N + 255) / 256), dim3(256), 0, st, a);
        e = hipGetLastError();
    }
    return e;
}

DGemm gemm_args(const uint16_t* x, int R, int N, int K, const uint16_t* w, const uint16_t* b, uint16_t* out) {
    DGemm a{};
    a.x = x;
    a.ldx = K;
    a.R = R;
    a.N = N;
    a.K = K;
    a.w[0] = a.w[1] = a.w[2] = w;
    a.b[0] = a.b[1] = a.b[2] = b;
    a.out = out;
    a.ldo = N;
    a.ks = a.vs = 1;
    return a;
}

}  // namespace

// One DiT block over R rows of L positions: rms1 -> q/k/v (+ rotary) -> attention
// -> out_proj + residual -> rms2 -> ff1 + gelu -> ff2 + residual.  x and out may
// not alias; hn [R][D], qkv [3][R][D], att [R][D], x1 [R][D], hh [R][F] and
// part f32 scratch of max(4 R D, 2 R F) floats (split-K partials).  hn_ready: hn
// already holds rms1(x) (the block before wrote it); next: the following block,
// whose rms1 of this block's output is left in hn.  A residual projection with
// split K takes the norm after it into its reduce kernel (dreduce_res_rms_kernel).
hipError_t launch_dit_block_gemm(hipStream_t st, const DitBlockDev& w, const uint16_t* x, int R, int L,
                                 const float* cos_t, const float* sin_t, uint16_t* hn, uint16_t* qkv, uint16_t* att,
                                 uint16_t* x1, uint16_t* hh, uint16_t* out, float* part, bool hn_ready,
                                 const DitBlockDev* next) {
    const int D = w.D, F = w.F;
    hipError_t e;
    if (!hn_ready) {
        hipLaunchKernelGGL(drms_kernel, dim3(R), dim3(256), 0, st, x, D, 0, w.norm1, w.eps, hn);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    DGemm a = gemm_args(hn, R, 3 * D, D, w.wq, w.bq, qkv);
    a.w[1] = w.wk;
    a.w[2] = w.wv;
    a.b[1] = w.bk;
    a.b[2] = w.bv;
    a.cos_t = cos_t;
    a.sin_t = sin_t;
    a.L = L;
    a.hd = w.hd;
    if ((e = dpick<DE_QKV>(st, a)) != hipSuccess) return e;
    if ((e = launch_dit_attn(st, qkv, R / L, L, D, w.heads, w.hd, att)) != hipSuccess) return e;
    a = gemm_args(att, R, D, D, w.wo, w.bo, x1);
    a.res = x;
    a.part = part;  // [2][R][D] of the [4][R][D] scratch
    if ((e = dpick<DE_RES>(st, a, w.norm2, w.eps, hn)) != hipSuccess) return e;  // x1, then rms2(x1) into hn
    a = gemm_args(hn, R, F, D, w.w1, w.b1, hh);
    a.part = part;  // [2][R][F]
    if ((e = dpick<DE_GELU>(st, a)) != hipSuccess) return e;
    a = gemm_args(hh, R, D, F, w.w2, w.b2, out);
    a.res = x1;
    a.part = part;  // [4][R][D] f32: ff2's K = F splits
    return next ? dpick<DE_RES>(st, a, next->norm1, next->eps, hn) : dpick<DE_RES>(st, a);
}

// out [R][N] = bf16(x W^T + b) (x [R][K]).
hipError_t launch_dit_linear_gemm(hipStream_t st, const uint16_t* x, int R, const uint16_t* w, int N, int K,
                                  const uint16_t* b, uint16_t* out) {
    return dpick<DE_BIAS>(st, gemm_args(x, R, N, K, w, b, out));
}

hipError_t launch_cfm_rows_batch(hipStream_t st, const uint16_t* te, const uint16_t* ce, const uint16_t* bc,
                                 const uint16_t* xh, const uint16_t* xe, int n, int D, uint16_t* rows) {
    hipLaunchKernelGGL(cfm_rows_kernel, dim3((n * D + 255) / 256), dim3(256), 0, st, te, ce, bc, xh, xe, n, D, rows);
    return hipGetLastError();
}

// The final layer of n sequences at Euler step `step`: rms(norm) of the last
// position of both CFG halves (rows of L positions in h [2n L][D]) -> linear
// [latent, D] + bias -> CFG + Euler (+ SDE) -> y_out [n][latent].
hipError_t launch_cfm_final_batch(hipStream_t st, const uint16_t* h, int n, int L, int D, const uint16_t* norm,
                                  float eps, const uint16_t* wf, const uint16_t* bf, int latent, const uint16_t* y,
                                  const uint16_t* dt, const uint16_t* sq, const uint16_t* sde, int step, int steps,
                                  float cfg, float shift, uint16_t* hn, uint16_t* y_out, uint16_t* y_steps) {
    hipLaunchKernelGGL(drms_kernel, dim3(2 * n), dim3(256), 0, st, h, D, L, norm, eps, hn);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    DGemm a = gemm_args(hn, 2 * n, latent, D, wf, bf, nullptr);
    a.y = y;
    a.dt = dt;
    a.sq = sq;
    a.sde = sde;
    a.step = step;
    a.steps = steps;
    a.cfg = cfg;
    a.shift = shift;
    a.y_out = y_out;
    a.y_steps = y_steps;
    return dpick<DE_CFM>(st, a);
}

// Shapes the four-launch block takes (launch_flow_block): heads of 64 over rows of three
// positions, K slices of whole register sets (flow_k_fits), and a normalised row of one or two
// 16-byte chunks a lane.  Others run launch_dit_block_gemm.
bool flow_block_fits(int D, int F, int hd, int latent) {
    return hd == 64 && (D == 512 || D == 1024) && flow_k_fits(F) && latent % 64 == 0 &&
           k_slices(latent) == 1;
}

// One block over R = 3 * groups rows x [R][D] -> out [R][D]; att [R up to 16s][D] and hh [..][F] in operand
// order, x1 [R][D].  The bits of launch_dit_block_gemm.
hipError_t launch_flow_block(hipStream_t st, const DitBlockDev& w, const uint16_t* x, int R, const float* cos_t,
                             const float* sin_t, uint16_t* att, uint16_t* x1, uint16_t* hh, uint16_t* out) {
    return w.D == 512 ? flow_block<512>(st, w, x, R, cos_t, sin_t, att, x1, hh, out)
                      : flow_block<1024>(st, w, x, R, cos_t, sin_t, att, x1, hh, out);
}

hipError_t launch_flow_rows(hipStream_t st, const uint16_t* y, int lat, const uint16_t* wx, const uint16_t* bx,
                            const uint16_t* te, const uint16_t* ce, const uint16_t* bc, const uint16_t* xh, int n,
                            int D, uint16_t* rows) {
    hipLaunchKernelGGL(flow_rows_kernel, dim3(D / 64, (n + 15) / 16), dim3(256), 0, st, y, lat, wx, bx, te, ce, bc, xh,
                       n, D, rows);
    return hipGetLastError();
}

// launch_cfm_final_batch in one launch (three positions a row group).
hipError_t launch_flow_final(hipStream_t st, const uint16_t* h, int n, int D, const uint16_t* norm, float eps,
                             const uint16_t* wf, const uint16_t* bf, int latent, const uint16_t* y, const uint16_t* dt,
                             const uint16_t* sq, const uint16_t* sde, int step, int steps, float cfg, float shift,
                             uint16_t* y_out, uint16_t* y_steps) {
    const int rb = (2 * n + 15) / 16;
    const FlowNorm f{h, 2 * n, latent, rb, 3, norm, wf, bf, eps, nullptr, y, dt, sq, sde, step, steps, cfg, shift, y_out, y_steps};
    void (*k)(FlowNorm) = D == 512 ? flow_norm_kernel<512, DE_CFM, 1, 1, 4> : flow_norm_kernel<1024, DE_CFM, 1, 1, 4>;
    hipLaunchKernelGGL(k, dim3(xcd_grid(latent / 64, rb)), dim3(256), 0, st, f);
    return hipGetLastError();
}

hipError_t tanh_upload_dit_batch(const float* host) {
    return hipMemcpyToSymbol(HIP_SYMBOL(dit_batch_tanh_tab), host, sizeof(float) * kTanhTabN);
}

}  // namespace ming
