// VAE decoder, the ISTFT head (Model.vaeDecode, src/ming_model.zig:1257-1309):
// spectrum, inverse real FFT, synthesis window, overlap-add.  The decoder's
// linears are in vae_gemm.hip.
//
// The inverse transform is an FFT of n_fft / 2 complex points per frame in LDS
// when n_fft / 2 factors into 2, 3, 5 and 7 (the reference's 3528 = 2 * 1764 =
// 2 * 7 * 7 * 6 * 6 does), else a GEMM against an f32 basis of cos/sin rows
// built at load time.
#include "args.h"
#include "common.h"
#include "internal.h"

namespace ming {

namespace {

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}

// One Stockham pass of radix R over h points (ns: the product of the radices before it):
// butterfly b takes src[b + r h / R], turns them by e^{2 pi i (b % ns) r / (ns R)} and writes
// their R-point transform (sign +) to (b / ns) ns R + b % ns + r ns.
template <int R>
__device__ __forceinline__ void fft_pass(const float2* src, float2* dst, int h, int ns, const float2* tw) {
    const int n = 2 * h, q = h / R, step = n / (ns * R);
    float2 root[R];
#pragma unroll
    for (int k = 1; k < R; k++) root[k] = tw[k * (n / R)];
    for (int b = threadIdx.x; b < q; b += blockDim.x) {
        const int k0 = b % ns;
        float2 v[R], o[R];
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = src[b + r * q];
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = cmul(v[r], tw[k0 * r * step]);
#pragma unroll
        for (int k = 0; k < R; k++) {
            o[k] = v[0];
#pragma unroll
            for (int r = 1; r < R; r++) {
                if ((k * r) % R == 0) {
                    o[k].x += v[r].x;
                    o[k].y += v[r].y;
                } else {
                    const float2 w = root[(k * r) % R];
                    o[k].x = fmaf(v[r].x, w.x, fmaf(-v[r].y, w.y, o[k].x));
                    o[k].y = fmaf(v[r].x, w.y, fmaf(v[r].y, w.x, o[k].y));
                }
            }
        }
        float2* d = dst + (b - k0) * R + k0;
#pragma unroll
        for (int k = 0; k < R; k++) d[k * ns] = o[k];
    }
}

// One workgroup per frame: the head's row p [n_fft + 2] (log-magnitudes | phases) -> windowed
// time samples.  mag = min(exp(.), 100); the imaginary parts of bins 0 and n_fft / 2 are
// ignored.  Real output of n = 2 h points from h complex ones: with X the half spectrum,
// Z[k] = (X[k] + conj X[h - k]) + i e^{2 pi i k / n} (X[k] - conj X[h - k]) has the inverse
// transform n (x[2 m] + i x[2 m + 1]).
// Bound: a chain of passes over 2 h values in LDS (n_fft 3528: 28 frames took 38 us and 400
// frames 145 us as a GEMM against the basis, whose 50 MB alone are 10 us of HBM time).
__global__ __launch_bounds__(256) void virfft_kernel(VFftPlan pl, const float* __restrict__ p,
                                                     const float2* __restrict__ tw, const float* __restrict__ win,
                                                     float* __restrict__ frames) {
    extern __shared__ float2 fb[];  // two buffers of h
    const int f = blockIdx.x, h = pl.h, n = 2 * h;
    const float* pr = p + (size_t)f * (n + 2);
    float2 *src = fb, *dst = fb + h;
    auto bin = [&](int k) {
        const float mag = fminf(expf(pr[k]), 100.0f), ph = pr[h + 1 + k];
        return make_float2(mag * cosf(ph), k == 0 || k == h ? 0.0f : mag * sinf(ph));
    };
    for (int k = threadIdx.x; 2 * k <= h; k += blockDim.x) {
        const int m = h - k;
        const float2 a = bin(k), b = bin(m);
        const float2 e = make_float2(a.x + b.x, a.y - b.y), d = make_float2(a.x - b.x, a.y + b.y);
        // i e^{i t} d at k; at m the roles swap: conj d -> -conj d, e^{i t} -> -e^{-i t}
        const float2 t = cmul(d, tw[k]);
        src[k] = make_float2(e.x - t.y, e.y + t.x);
        if (k > 0 && m != k) src[m] = make_float2(e.x + t.y, -e.y + t.x);
    }
    __syncthreads();
    int ns = 1;
    for (int i = 0; i < pl.passes; i++) {
        switch (pl.radix[i]) {
            case 2: fft_pass<2>(src, dst, h, ns, tw); break;
            case 3: fft_pass<3>(src, dst, h, ns, tw); break;
            case 4: fft_pass<4>(src, dst, h, ns, tw); break;
            case 5: fft_pass<5>(src, dst, h, ns, tw); break;
            case 6: fft_pass<6>(src, dst, h, ns, tw); break;
            default: fft_pass<7>(src, dst, h, ns, tw); break;
        }
        ns *= pl.radix[i];
        __syncthreads();
        float2* s = src;
        src = dst;
        dst = s;
    }
    const float inv = 1.0f / (float)n;
    for (int k = threadIdx.x; k < h; k += blockDim.x) {
        const float2 v = src[k];
        *reinterpret_cast<float2*>(frames + (size_t)f * n + 2 * k) =
            make_float2(v.x * inv * win[2 * k], v.y * inv * win[2 * k + 1]);
    }
}

constexpr int kVBM = 64, kVBN = 64, kVBK = 32, kVT = 256;
constexpr int kVLd = kVBK + 4;  // f32 per LDS row: k permuted so a lane's 8 k-steps are contiguous

// Position of k (0..31 within a stage) in an LDS row: k = 4 kk + j -> j * 8 + kk,
// so lane group j = lane / 16 reads its 8 values (k-steps kk = 0..7) as two 16-byte words.
__device__ __forceinline__ int vperm(int k) { return (k & 3) * 8 + (k >> 2); }

// The basis GEMM: workgroup = 64 x 64 outputs, wave w = rows 16w .. 16w + 15, all
// 64 columns; K (or its slice blockIdx.z of ks) in stages of 32 through
// double-buffered LDS (the next stage's global loads are in flight during the
// current stage's v_mfma_f32_16x16x4f32).
__global__ __launch_bounds__(kVT) void vbasis_kernel(VBasis g) {
    __shared__ __align__(16) float la[2][kVBM * kVLd];
    __shared__ __align__(16) float lw[2][kVBN * kVLd];
    const int t = threadIdx.x, wave = t / kWave, lane = t % kWave, c = lane % 16, j = lane / 16;
    const int n0 = blockIdx.x * kVBN, m0 = blockIdx.y * kVBM, z = blockIdx.z;
    const int Ks = g.K / g.ks, S = Ks / kVBK, kb = z * Ks;
    float4 ra[2], rw[2];
    auto gload = [&](int s) {
        const int k0 = kb + s * kVBK;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int f = t + kVT * p, row = f / 8, kq = f % 8;
            ra[p] = *reinterpret_cast<const float4*>(g.a + (size_t)min(m0 + row, g.M - 1) * g.K + k0 + 4 * kq);
            rw[p] = *reinterpret_cast<const float4*>(g.w + (size_t)min(n0 + row, g.n - 1) * g.K + k0 + 4 * kq);
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int f = t + kVT * p, row = f / 8, kq = f % 8;
            const float e[4] = {ra[p].x, ra[p].y, ra[p].z, ra[p].w}, w[4] = {rw[p].x, rw[p].y, rw[p].z, rw[p].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                la[buf][row * kVLd + vperm(4 * kq + i)] = e[i];
                lw[buf][row * kVLd + vperm(4 * kq + i)] = w[i];
            }
        }
    };
    f32x4_t acc[4];
#pragma unroll
    for (int b = 0; b < 4; b++) acc[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    gload(0);
    lstore(0);
    __syncthreads();
    for (int s = 0; s < S; s++) {
        const int buf = s & 1;
        if (s + 1 < S) gload(s + 1);
        const float* ar = &la[buf][(16 * wave + c) * kVLd + 8 * j];
        const float4 a0 = *reinterpret_cast<const float4*>(ar), a1 = *reinterpret_cast<const float4*>(ar + 4);
        const float av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float* wr = &lw[buf][(16 * b + c) * kVLd + 8 * j];
            const float4 w0 = *reinterpret_cast<const float4*>(wr), w1 = *reinterpret_cast<const float4*>(wr + 4);
            const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
            for (int kk = 0; kk < 8; kk++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[kk], wv[kk], acc[b], 0, 0, 0);
        }
        if (s + 1 < S) lstore(buf ^ 1);
        __syncthreads();
    }
    // lane (c, j): acc[b][i] = C[row 16 wave + 4 j + i][col 16 b + c]
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int col = n0 + 16 * b + c;
        if (col >= g.n) continue;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = m0 + 16 * wave + 4 * j + i;
            if (row >= g.M) continue;
            if (g.ks > 1)  // raw sums of this K slice
                g.part[((size_t)z * g.M + row) * g.n + col] = acc[b][i];
            else
                g.y[(size_t)row * g.n + col] = acc[b][i] * g.win[col];
        }
    }
}

// The ks partials summed in slice order, then the window.
__global__ __launch_bounds__(256) void vbasis_reduce_kernel(VBasis g) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = (int64_t)g.M * g.n;
    if (i >= n) return;
    float sum = 0.0f;
    for (int z = 0; z < g.ks; z++) sum += g.part[z * n + i];
    g.y[i] = sum * g.win[i % g.n];
}

// ISTFT spectrum: p [F][n_fft + 2] (log-magnitudes | phases) -> the GEMM's
// A rows [F][ld]: mag cos(ph) for bins 0 .. nb-1, mag sin(ph) after them,
// zeros to ld; mag = min(exp(.), 100).
__global__ __launch_bounds__(256) void vspec_kernel(const float* p, int F, int nfft, int ld, float* spec) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)F * ld) return;
    const int f = (int)(idx / ld), k = (int)(idx % ld), nb = nfft / 2 + 1;
    const float* pr = p + (size_t)f * (nfft + 2);
    float v = 0.0f;
    if (k < 2 * nb) {
        const int b = k < nb ? k : k - nb;
        const float mag = fminf(expf(pr[b]), 100.0f);
        const float ph = pr[nb + b];
        v = k < nb ? mag * cosf(ph) : mag * sinf(ph);
    }
    spec[idx] = v;
}

// Overlap-add of the windowed frames [F][n_fft] (n_fft = 4 hop), divided by
// the window envelope, "same" trim: block b sums ((frame b-3 part 3 + frame
// b-2 part 2) + frame b-1 part 1) + frame b part 0, in the graph's order.
__global__ __launch_bounds__(256) void vola_kernel(const float* fr, int F, int nfft, int hop, const float* win,
                                                   float* wave) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int pad = (nfft - hop) / 2, n_out = (F + 3) * hop - 2 * pad;
    if (i >= n_out) return;
    const int s = pad + i, b = s / hop, k = s % hop;
    float acc = 0.0f, env = 0.0f;
#pragma unroll
    for (int j = 3; j >= 0; j--) {
        const int t = b - j;
        const bool ok = t >= 0 && t < F;
        const float fv = ok ? fr[(size_t)t * nfft + j * hop + k] : 0.0f;
        const float wv = win[j * hop + k];
        acc = j == 3 ? fv : acc + fv;
        env = env + (ok ? wv * wv : 0.0f);
    }
    wave[i] = acc / fmaxf(env, 1e-11f);
}

// bf16 -> f32 (exact): a checkpoint's bf16 window, which the inverse transform reads as f32.
__global__ __launch_bounds__(256) void vwiden_kernel(const uint16_t* x, int64_t n, float* y) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = bf2f(x[i]);
}

}  // namespace

bool vfft_plan(int n_fft, VFftPlan& p) {
    p = VFftPlan{};
    p.h = n_fft / 2;
    if (n_fft % 2 || p.h < 2 || p.h > kFftMaxHalf) return false;
    int r = p.h;
    // fewest passes: 7s, 6s, 5s, then what is left of 4s, 3s and 2s
    for (int f : {7, 6, 5, 4, 3, 2})
        while (r % f == 0) {
            if (p.passes == kFftMaxPasses) return false;
            p.radix[p.passes++] = f;
            r /= f;
        }
    return r == 1;
}

hipError_t launch_virfft(hipStream_t st, const VFftPlan& pl, const float* p, int F, const float* tw, const float* win,
                         float* frames) {
    if (pl.h < 2 || pl.h > kFftMaxHalf || F < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(virfft_kernel, dim3(F), dim3(256), 2 * sizeof(float2) * pl.h, st, pl, p,
                       reinterpret_cast<const float2*>(tw), win, frames);
    return hipGetLastError();
}

hipError_t launch_vbasis(hipStream_t st, const VBasis& g) {
    if (g.ks < 1 || g.K % (kVBK * g.ks) || g.M < 1 || g.n < 1 || (g.ks > 1 && !g.part)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(vbasis_kernel, dim3((g.n + kVBN - 1) / kVBN, (g.M + kVBM - 1) / kVBM, g.ks), dim3(kVT), 0, st, g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || g.ks == 1) return e;
    hipLaunchKernelGGL(vbasis_reduce_kernel, dim3((unsigned)(((int64_t)g.M * g.n + 255) / 256)), dim3(256), 0, st, g);
    return hipGetLastError();
}

hipError_t launch_vspec(hipStream_t st, const float* p, int F, int nfft, int ld, float* spec) {
    const int64_t n = (int64_t)F * ld;
    hipLaunchKernelGGL(vspec_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, F, nfft, ld, spec);
    return hipGetLastError();
}

hipError_t launch_vola(hipStream_t st, const float* fr, int F, int nfft, int hop, const float* win, float* wave) {
    const int n_out = (F + 3) * hop - (nfft - hop);
    hipLaunchKernelGGL(vola_kernel, dim3((n_out + 255) / 256), dim3(256), 0, st, fr, F, nfft, hop, win, wave);
    return hipGetLastError();
}

hipError_t launch_vwiden(hipStream_t st, const uint16_t* x, int64_t n, float* y) {
    hipLaunchKernelGGL(vwiden_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, n, y);
    return hipGetLastError();
}

}  // namespace ming
