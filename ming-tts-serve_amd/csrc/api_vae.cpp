// C-ABI glue of the VAE decoder (include/ming_hip.h, "VAE decoder";
// Model.vaeDecode, src/ming_model.zig:1257-1309): the model handle with the
// ISTFT tables built at load time, and the per-fragment decode.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "internal.h"

using namespace ming;

struct ming_vae_model {
    ming_ctx* ctx = nullptr;
    ming_vae_cfg cfg{};
    int max_t = 0, ldspec = 0;
    ming_linear fc1{}, head{};
    const uint16_t *fc1_bias = nullptr, *head_bias = nullptr, *norm = nullptr;
    const float* window = nullptr;
    std::vector<ming_lm_layer_w> layers;
    // inverse transform: the FFT's passes and (cos, sin) table, or (lengths the passes do not
    // cover, fft.passes == 0) the irfft basis f32 [n_fft][ldspec] and its spectrum rows
    VFftPlan fft{};
    DevBuf tw, basis, spec;
    DevBuf rope;                                      // f32 [F][32][2] (cos, sin)
    // h, att, hh: bf16 planes; part: K-slice partials (and fc1's sums)
    DevBuf lat, xs, h, qkv, att, x1, hh, p, frames, part;
    int last_f = 0;
};

namespace {

constexpr int kMaxSlices = 8;

int vae_err(ming_ctx* ctx, int st, const std::string& m) { return set_err(ctx, st, "vae: " + m); }

int is_q4(const ming_linear& l) { return linear_dev(l).kind == 1; }

// The weight of a linear as a GEMM segment; wf receives its format.
VSeg seg_of(const ming_linear& l, const void* bias, int rope, int& wf) {
    const LinearDev d = linear_dev(l);
    wf = d.kind == 1 ? VW_Q4 : VW_BF16;
    VSeg s{};
    s.w = d.w;
    s.s = d.s;
    s.b = d.b;
    s.gs = d.kind == 1 ? d.gscale : 1.0f;
    s.bias = static_cast<const uint16_t*>(bias);
    s.n = l.out_features;
    s.rope = rope;
    return s;
}

// K slices of a residual projection: the row kernel after it adds the partials
// either way, so a split costs only their traffic.  Few rows: slices of at most
// ten waves' chunks of 128 (K = 4864: 4), so that no wave loops and N / 16 = 56
// workgroups become 224.  Many rows: enough 64 x 64 tiles to cover the 256 CUs.
int split_k(int M, int N, int K) {
    if (M <= kV3SmallRows) return std::min(kMaxSlices, (K + 1279) / 1280);
    if (K <= 1024) return 1;  // 32 x 64 tiles
    const int tiles = ((N + 63) / 64) * ((M + 63) / 64);
    int ks = 1;
    while (2 * ks <= kMaxSlices && tiles * ks < 256) ks *= 2;
    return ks;
}

// K slices of the basis GEMM: enough 64 x 64 workgroups (with the slices) to cover the 256 CUs.
int split_basis(int M, int N, int K) {
    const int tiles = ((N + 63) / 64) * ((M + 63) / 64);
    int best = 1;
    for (int ks = 1; ks <= kMaxSlices; ks++)
        if (K % (32 * ks) == 0) {
            best = ks;
            if (tiles * ks >= 256) break;
        }
    return best;
}

int check_cfg(ming_ctx* ctx, const ming_vae_cfg* c) {
    if (!c) return vae_err(ctx, MING_E_ARG, "null cfg");
    if (c->head_dim != 64) return vae_err(ctx, MING_E_UNSUPPORTED, "head_dim must be 64");
    if (c->kv_heads < 1 || c->heads % c->kv_heads || c->hidden != c->heads * c->head_dim)
        return vae_err(ctx, MING_E_SHAPE, "heads / kv_heads / hidden inconsistent");
    if (c->hidden % 64 || c->inter % 64 || c->latent % 32 || c->latent < 32)
        return vae_err(ctx, MING_E_UNSUPPORTED, "hidden and inter must be multiples of 64, latent of 32");
    if (c->window < 1 || c->window > 64) return vae_err(ctx, MING_E_UNSUPPORTED, "window must be in [1, 64]");
    if (c->heads / c->kv_heads > 16)
        return vae_err(ctx, MING_E_UNSUPPORTED, "at most 16 q heads per kv head (one workgroup of waves per kv head)");
    if (c->hop < 1 || c->n_fft != 4 * c->hop || c->n_fft % 2)
        return vae_err(ctx, MING_E_UNSUPPORTED, "n_fft must be 4 * hop and even");
    if (c->patch < 1 || c->n_layers < 1) return vae_err(ctx, MING_E_ARG, "patch and n_layers must be >= 1");
    return MING_OK;
}

}  // namespace

extern "C" {

int ming_vae_model_create(ming_ctx* ctx, const ming_vae_cfg* cfg, const ming_vae_w* w, int32_t max_latents,
                          ming_vae_model** out) {
    if (!ctx || !ctx->alive) return MING_E_NOT_INIT;
    if (!w || !out || max_latents < 1) return vae_err(ctx, MING_E_ARG, "bad arguments");
    int st;
    if ((st = check_cfg(ctx, cfg))) return st;
    const int H = cfg->hidden, kvd = cfg->kv_heads * cfg->head_dim, I = cfg->inter, P = cfg->n_fft + 2;
    if (!w->layers || !w->norm || !w->window) return vae_err(ctx, MING_E_ARG, "null layers, norm or window");
    if ((st = check_linear_w(ctx, w->fc1, H, cfg->latent, "fc1")) ||
        (st = check_linear_w(ctx, w->head, P, H, "head")))
        return st;
    for (int i = 0; i < cfg->n_layers; i++) {
        const ming_lm_layer_w& l = w->layers[i];
        if (!l.ln1 || !l.ln2) return vae_err(ctx, MING_E_ARG, "null layer norm");
        if ((st = check_linear_w(ctx, l.wq, H, H, "wq")) || (st = check_linear_w(ctx, l.wk, kvd, H, "wk")) ||
            (st = check_linear_w(ctx, l.wv, kvd, H, "wv")) || (st = check_linear_w(ctx, l.wo, H, H, "wo")) ||
            (st = check_linear_w(ctx, l.wg, I, H, "wg")) || (st = check_linear_w(ctx, l.wu, I, H, "wu")) ||
            (st = check_linear_w(ctx, l.wd, H, I, "wd")))
            return st;
    }
    ming_vae_model* m = new ming_vae_model();
    m->ctx = ctx;
    m->cfg = *cfg;
    m->max_t = max_latents;
    m->fc1 = w->fc1;
    m->head = w->head;
    m->fc1_bias = static_cast<const uint16_t*>(w->fc1_bias);
    m->head_bias = static_cast<const uint16_t*>(w->head_bias);
    m->norm = static_cast<const uint16_t*>(w->norm);
    m->window = static_cast<const float*>(w->window);
    m->layers.assign(w->layers, w->layers + cfg->n_layers);
    const int N = cfg->n_fft, nb = N / 2 + 1;
    const size_t F = (size_t)max_latents * cfg->patch, nq = H + 2 * kvd;
    std::vector<float> tab;  // evaluated in double, rounded once
    hipError_t e;
    if (vfft_plan(N, m->fft)) {
        tab.resize(2 * (size_t)N);
        for (int k = 0; k < N; k++) {
            const double th = 2.0 * M_PI * k / N;
            tab[2 * k] = (float)std::cos(th);
            tab[2 * k + 1] = (float)std::sin(th);
        }
        e = m->tw.ensure(tab.size() * sizeof(float));
        if (e == hipSuccess) e = hipMemcpy(m->tw.p, tab.data(), tab.size() * sizeof(float), hipMemcpyHostToDevice);
    } else {
        m->fft = VFftPlan{};
        m->ldspec = (2 * nb + 31) / 32 * 32;
        // irfft (backward norm) as rows of a matrix: frame[n] = sum_k spec[k] basis[n][k] with
        // spec = [re_0 .. re_{nb-1} | im_0 .. im_{nb-1} | 0 pad]; bins 1 .. N/2-1 count twice and
        // the imaginary parts of bins 0 and N/2 are ignored
        tab.assign((size_t)N * m->ldspec, 0.0f);
        for (int n = 0; n < N; n++) {
            float* row = tab.data() + (size_t)n * m->ldspec;
            for (int k = 0; k < nb; k++) {
                const double c = (k == 0 || 2 * k == N) ? 1.0 : 2.0;
                const double th = 2.0 * M_PI * (double)(((int64_t)k * n) % N) / (double)N;
                row[k] = (float)(c * std::cos(th) / N);
                row[nb + k] = (k == 0 || 2 * k == N) ? 0.0f : (float)(-c * std::sin(th) / N);
            }
        }
        e = m->basis.ensure(tab.size() * sizeof(float));
        if (e == hipSuccess) e = hipMemcpy(m->basis.p, tab.data(), tab.size() * sizeof(float), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = m->spec.ensure(F * m->ldspec * sizeof(float));
    }
    const size_t Fp = (F + 15) / 16 * 16;  // rows of a plane
    const size_t part_cols = m->ldspec ? std::max((size_t)H, (size_t)N) : (size_t)H;
    const std::pair<DevBuf*, size_t> bufs[] = {  // bytes
        {&m->lat, (size_t)max_latents * cfg->latent * 2}, {&m->xs, (cfg->n_layers + 1) * F * H * 4},
        {&m->h, 3 * Fp * H * 2},                          {&m->qkv, F * nq * 4},
        {&m->att, 3 * Fp * H * 2},                        {&m->x1, F * H * 4},
        {&m->hh, 3 * Fp * I * 2},                         {&m->p, F * P * 4},
        {&m->frames, F * N * 4},                          {&m->part, kMaxSlices * F * part_cols * 4},
        {&m->rope, F * 64 * 4}};
    for (const auto& b : bufs)
        if (e == hipSuccess) e = b.first->ensure(b.second);
    if (e == hipSuccess)
        e = launch_rope_table(ctx->stream, static_cast<float*>(m->rope.p), (int)F, 32, cfg->log2_theta);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        ming_vae_model_destroy(m);
        return hip_check(ctx, e, "vae workspace");
    }
    *out = m;
    return MING_OK;
}

int ming_vae_model_destroy(ming_vae_model* m) {
    if (!m) return MING_E_NOT_INIT;
    for (DevBuf* b : {&m->tw, &m->basis, &m->spec, &m->rope, &m->lat, &m->xs, &m->h, &m->qkv, &m->att, &m->x1, &m->hh,
                      &m->p, &m->frames, &m->part})
        b->release();
    delete m;
    return MING_OK;
}

int ming_vae_decode(ming_ctx* ctx, ming_vae_model* m, int32_t T, const void* latents, float* wave_out) {
    if (!ctx || !ctx->alive || !m) return MING_E_NOT_INIT;
    if (!latents || !wave_out) return vae_err(ctx, MING_E_ARG, "null latents or output");
    if (T < 1 || T > m->max_t)
        return vae_err(ctx, MING_E_SHAPE, "T = " + std::to_string(T) + " outside [1, " + std::to_string(m->max_t) + "]");
    const ming_vae_cfg& c = m->cfg;
    const int H = c.hidden, kvd = c.kv_heads * c.head_dim, I = c.inter, nq = H + 2 * kvd, P = c.n_fft + 2;
    const int F = T * c.patch;
    const size_t Fp = (size_t)(F + 15) / 16 * 16;  // rows of a plane
    hipStream_t st = ctx->stream;
    float *xs = static_cast<float*>(m->xs.p), *qkv = static_cast<float*>(m->qkv.p), *x1 = static_cast<float*>(m->x1.p);
    float* part = static_cast<float*>(m->part.p);
    uint16_t *h = static_cast<uint16_t*>(m->h.p), *att = static_cast<uint16_t*>(m->att.p);
    uint16_t* hh = static_cast<uint16_t*>(m->hh.p);
    hipError_t e = hipSuccess;
    int wf = 0;
    auto gemm = [&](const uint16_t* a, int M, int K, float* y, int ldy) {
        V3Gemm g{};
        g.a = a;
        g.aps = Fp * K;
        g.np = 3;
        g.M = M;
        g.K = K;
        g.y = y;
        g.ldy = ldy;
        g.nseg = 1;
        g.ks = 1;
        g.rope_cs = static_cast<const float*>(m->rope.p);
        return g;
    };
    {  // fc1 on the bf16 latents: bias and the bf16 rounding are applied by the row kernel
        const void* lat = latents;
        if (reinterpret_cast<uintptr_t>(latents) % 16) {  // the GEMM reads 16-byte words
            lat = m->lat.p;
            e = hipMemcpyAsync(m->lat.p, latents, (size_t)T * c.latent * 2, hipMemcpyDeviceToDevice, st);
        }
        V3Gemm g = gemm(static_cast<const uint16_t*>(lat), T, c.latent, part, H);
        g.np = 1;
        g.seg[0] = seg_of(m->fc1, nullptr, 0, wf);
        if (e == hipSuccess) e = launch_v3gemm(st, g, wf, VE_PLAIN);
    }
    // x = (res + the partials) or the upsampled rows, and h = rms_norm(x) for the next linear
    auto row = [&](const float* res, float* x, int ks, const void* norm, bool up, const ming_linear& next) {
        VRowArgs a{};
        a.part = part;
        a.ks = ks;
        a.res = res;
        a.x = x;
        a.M = F;
        a.N = H;
        a.w = static_cast<const uint16_t*>(norm);
        a.eps = c.eps;
        a.h = h;
        a.hps = Fp * H;
        a.hpair = is_q4(next);
        a.bias = m->fc1_bias;
        a.q4 = wf == VW_Q4;
        a.T = T;
        a.scale = c.patch;
        return launch_vrow(st, a, up);
    };
    if (e == hipSuccess) e = row(nullptr, xs, 0, m->layers[0].ln1, true, m->layers[0].wq);
    const float scale = 1.0f / std::sqrt((float)c.head_dim);
    const int ks_o = split_k(F, H, H), ks_d = split_k(F, H, I);
    for (int l = 0; l < c.n_layers && e == hipSuccess; l++) {
        const ming_lm_layer_w& L = m->layers[l];
        float* x = xs + (size_t)l * F * H;
        float* xo = xs + (size_t)(l + 1) * F * H;
        {  // q | k | v in one launch, rotary on q and k
            V3Gemm g = gemm(h, F, H, qkv, nq);
            g.seg[0] = seg_of(L.wq, L.bq, 1, wf);
            g.seg[1] = seg_of(L.wk, L.bk, 1, wf);
            g.seg[2] = seg_of(L.wv, L.bv, 0, wf);
            g.nseg = 3;
            e = launch_v3gemm(st, g, wf, VE_QKV);
        }
        if (e == hipSuccess)
            e = launch_vattn(st, qkv, F, nq, H, c.heads, c.kv_heads, c.window, scale, att, Fp * H, is_q4(L.wo));
        if (e == hipSuccess) {
            V3Gemm g = gemm(att, F, H, part, H);
            g.seg[0] = seg_of(L.wo, nullptr, 0, wf);
            g.ks = ks_o;
            e = launch_v3gemm(st, g, wf, VE_RES);
        }
        if (e == hipSuccess) e = row(x, x1, ks_o, L.ln2, false, L.wg);
        if (e == hipSuccess) {
            V3Gemm g = gemm(h, F, H, nullptr, 0);
            g.seg[0] = seg_of(L.wg, nullptr, 0, wf);
            g.up = seg_of(L.wu, nullptr, 0, wf);
            g.yp = hh;
            g.yps = Fp * I;
            g.ldyp = I;
            g.ypair = is_q4(L.wd);
            e = launch_v3gemm(st, g, wf, VE_SWIGLU);
        }
        if (e == hipSuccess) {
            V3Gemm g = gemm(hh, F, I, part, H);
            g.seg[0] = seg_of(L.wd, nullptr, 0, wf);
            g.ks = ks_d;
            e = launch_v3gemm(st, g, wf, VE_RES);
        }
        const bool last = l + 1 == c.n_layers;
        if (e == hipSuccess)
            e = row(x1, xo, ks_d, last ? m->norm : m->layers[l + 1].ln1, false, last ? m->head : m->layers[l + 1].wq);
    }
    float *p = static_cast<float*>(m->p.p), *frames = static_cast<float*>(m->frames.p);
    if (e == hipSuccess) {
        V3Gemm g = gemm(h, F, H, p, P);
        g.seg[0] = seg_of(m->head, m->head_bias, 0, wf);
        e = launch_v3gemm(st, g, wf, VE_PLAIN);
    }
    if (e == hipSuccess && m->fft.passes) {
        e = launch_virfft(st, m->fft, p, F, static_cast<const float*>(m->tw.p), m->window, frames);
    } else if (e == hipSuccess) {
        float* spec = static_cast<float*>(m->spec.p);
        e = launch_vspec(st, p, F, c.n_fft, m->ldspec, spec);
        const VBasis g{spec,   static_cast<const float*>(m->basis.p), F, m->ldspec, c.n_fft, m->window, frames,
                       split_basis(F, c.n_fft, m->ldspec), part};
        if (e == hipSuccess) e = launch_vbasis(st, g);
    }
    if (e == hipSuccess) e = launch_vola(st, frames, F, c.n_fft, c.hop, m->window, wave_out);
    if (e == hipSuccess) m->last_f = F;
    return hip_check(ctx, e, "vae_decode launch");
}

int ming_vae_trace(ming_vae_model* m, float* xs, float* head_out) {
    if (!m || !m->ctx || !m->ctx->alive) return MING_E_NOT_INIT;
    if (!m->last_f) return vae_err(m->ctx, MING_E_ARG, "no decode yet");
    const ming_vae_cfg& c = m->cfg;
    const size_t F = m->last_f, H = c.hidden;
    hipError_t e = hipSuccess;
    if (xs)
        for (int l = 0; l <= c.n_layers && e == hipSuccess; l++)
            e = hipMemcpyAsync(xs + l * F * H, static_cast<float*>(m->xs.p) + l * F * H, F * H * sizeof(float),
                               hipMemcpyDeviceToDevice, m->ctx->stream);
    if (head_out && e == hipSuccess)
        e = hipMemcpyAsync(head_out, m->p.p, F * (c.n_fft + 2) * sizeof(float), hipMemcpyDeviceToDevice,
                           m->ctx->stream);
    return hip_check(m->ctx, e, "vae_trace copy");
}

}  // extern "C"
