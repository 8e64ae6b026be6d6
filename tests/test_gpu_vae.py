"""VAE decoder on the GPU (ming_vae_decode; Model.vaeDecode,
src/ming_model.zig:1257-1309) against the oracle (oracle/oracle_vae.c).

The graph after the upsample is f32, so the bar is f32 summation order:
every layer teacher forced on the GPU's own input (1e-5 of max|ref|), the
head on the GPU's final hidden, the ISTFT on the GPU's head output (f32
basis vs the oracle's double irfft: 2e-5), and end to end (2e-4).  fc1 runs
in bf16 as in the graph, so the upsampled rows may differ by one bf16 ulp
where the two summation orders round differently (2^-7 of max|ref|)."""
import numpy as np
import pytest
import torch

import oracle
from vaekit import assert_close_f32, oracle_vae

pytestmark = pytest.mark.gpu

SMALL = dict(hidden=128, heads=2, kv_heads=1, head_dim=64, inter=256, n_layers=2, window=8, latent=64, patch=4,
             n_fft=64, hop=16)


def syn_mod():
    import importlib

    return importlib.import_module("ming-tts-serve_amd.synthetic")


def run(ming, ctx, syn, T, seed=3, max_latents=None):
    spec = syn.spec
    m = syn.model(max_latents or T)
    lat_h = ming.synth_normal_bf16(seed, "vae.lat", T * spec.latent).reshape(T, spec.latent)
    lat = torch.from_numpy(lat_h.view(np.int16)).cuda().view(torch.bfloat16)
    F = T * spec.patch
    wave = torch.empty(F * spec.hop, dtype=torch.float32, device="cuda")
    m.decode(T, lat, wave)
    xs = torch.empty((spec.n_layers + 1, F, spec.hidden), dtype=torch.float32, device="cuda")
    ho = torch.empty((F, spec.n_fft + 2), dtype=torch.float32, device="cuda")
    m.trace(xs, ho)
    ctx.sync()
    m.close()
    return lat_h, wave.cpu().numpy(), xs.cpu().numpy(), ho.cpu().numpy()


def check(ming, ctx, syn, T, end_to_end=True):
    S = syn_mod()
    spec = syn.spec
    om = oracle_vae(syn)
    c = om.cfg
    lat, wave, xs, ho = run(ming, ctx, syn, T)
    x0 = oracle.linear_upsample(oracle.linear(om.fc1, lat, om.keep[0]), spec.patch)
    assert_close_f32(xs[0], x0, "fc1 + upsample", 2.0 ** -7)
    for l in range(spec.n_layers):
        assert_close_f32(xs[l + 1], oracle.vae_layer(c, om.layers[l], xs[l]), f"layer {l} (teacher forced)", 1e-5)
    p = oracle.linear_f32(om.head, oracle.rms_f32(xs[-1], om.keep[1]), om.keep[2])
    assert_close_f32(ho, p, "final norm + head (teacher forced)", 1e-5)
    assert_close_f32(wave, oracle.vae_istft(ho, spec.n_fft, spec.hop, om.keep[3]), "ISTFT (teacher forced)", 2e-5)
    if end_to_end:
        assert_close_f32(wave, oracle.vae_decode(om, lat), "wave (end to end)", 2e-4)
    assert np.isfinite(wave).all()


@pytest.mark.parametrize("T", [1, 5, 17])
def test_vae_small_bf16(ming, ctx, T):
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=21, std=0.05, norm_std=0.1)
    check(ming, ctx, syn, T)


def test_vae_small_4bit(ming, ctx):
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=22, quant=True, std=0.05, norm_std=0.1)
    check(ming, ctx, syn, 9)


def test_vae_window_covers_all_rows(ming, ctx):
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**dict(SMALL, window=64)), seed=23, std=0.05)
    check(ming, ctx, syn, 3)  # F = 12 rows < 64: plain causal attention


def test_vae_reference_shape(ming, ctx):
    """The reference decoder (24 layers, 896, n_fft 3528) on 6 latents."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.MING_VAE, seed=24)
    check(ming, ctx, syn, 6, end_to_end=False)


def test_vae_decode_independent_of_capacity(ming, ctx):
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=25, std=0.05)
    a = run(ming, ctx, syn, 7)
    b = run(ming, ctx, syn, 7, max_latents=40)
    assert np.array_equal(a[1], b[1])


def test_vae_rejects(ming, ctx):
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=26, std=0.05)
    m = syn.model(4)
    lat = torch.zeros((5, 64), dtype=torch.bfloat16, device="cuda")
    wave = torch.empty(5 * 4 * 16, dtype=torch.float32, device="cuda")
    with pytest.raises(ming.MingError) as e:
        m.decode(5, lat, wave)
    assert e.value.status == ming.MING_E_SHAPE
    m.close()
    bad = S.VaeSpec(**dict(SMALL, window=65)).cfg()
    with pytest.raises(ming.MingError) as e:
        ming.VaeModel(ctx, bad, syn.w, 4)
    assert e.value.status == ming.MING_E_UNSUPPORTED
    # more than 16 q heads per kv head (the attention runs one workgroup of q-head waves per kv head)
    c = S.VaeSpec(**SMALL).cfg()
    c.heads, c.kv_heads, c.hidden = 34, 2, 34 * 64
    with pytest.raises(ming.MingError) as e:
        ming.VaeModel(ctx, c, syn.w, 4)
    assert e.value.status == ming.MING_E_UNSUPPORTED


@pytest.mark.parametrize("rows, quant, over", [
    (16, False, {}), (17, True, {}), (64, False, dict(inter=1152)),  # unstaged kernel: one tile, a remainder, K slices
    (65, True, dict(inter=1152)), (133, False, dict(inter=2176)),    # LDS tiles: a remainder, K slices of unequal length
    (257, True, dict(hidden=256, heads=4, kv_heads=2)),
])
def test_vae_row_counts(ming, ctx, rows, quant, over):
    """Either side of the row-count rules of the linears (16, 32, 64 rows) and of their K slices; the bars
    are those of check()."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**dict(SMALL, patch=1, **over)), seed=27, quant=quant, std=0.05, norm_std=0.1)
    check(ming, ctx, syn, rows)


@pytest.mark.parametrize("rows", [1, 17, 64, 65, 130])
@pytest.mark.parametrize("quant", [False, True])
def test_vae_wide_rows(ming, ctx, rows, quant):
    """Hidden 1152 (18 heads on 2): rows too wide for the row kernel's registers are written and read back for the norm,
    on either side of the linears' 64 rows; the bars are those of check()."""
    S = syn_mod()
    spec = S.VaeSpec(**dict(SMALL, patch=1, hidden=1152, heads=18, kv_heads=2))
    syn = S.SyntheticVae(ctx, spec, seed=33, quant=quant, norm_std=0.1)
    check(ming, ctx, syn, rows)


@pytest.mark.parametrize("hop", [1, 6, 35, 11, 13 * 5])
def test_vae_transform_lengths(ming, ctx, hop):
    """ISTFT by FFT passes (n_fft / 2 = 2, 12, 70: every radix, an odd one last) and by the basis GEMM (a prime
    factor above 7)."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**dict(SMALL, n_fft=4 * hop, hop=hop)), seed=28, std=0.05, norm_std=0.1)
    check(ming, ctx, syn, 5)


@pytest.mark.parametrize("hop", [2048, 2058])
def test_vae_longest_transforms(ming, ctx, hop):
    """The longest transform that the FFT's LDS holds (4096 complex points, 64 KB) and the next one that factors (4116,
    by the basis GEMM)."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**dict(SMALL, n_layers=1, patch=2, n_fft=4 * hop, hop=hop)), seed=34, std=0.05,
                         norm_std=0.1)
    check(ming, ctx, syn, 1)


@pytest.mark.parametrize("four", [("fc1", "o_proj", "gate_proj", "up_proj"),
                                  ("q_proj", "k_proj", "v_proj", "down_proj", "head.out")])
@pytest.mark.parametrize("T", [9, 23])
def test_vae_mixed_formats(ming, ctx, four, T):
    """Some linears in 4 bits and the others in bf16, either way round: each kernel writes the planes in the order that
    the next linear's format reads; on either side of 64 rows."""
    S = syn_mod()
    syn, bf = (S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=35, quant=q, std=0.05, norm_std=0.1) for q in (True, False))
    for name in syn.tensors:
        if not name.endswith(four):
            syn.tensors[name] = bf.tensors[name]
    syn._build_views()
    check(ming, ctx, syn, T)


@pytest.mark.parametrize("T", [9, 23])
def test_vae_global_scale(ming, ctx, T):
    """A global scale of 1/4 with scales and biases four times as large is the same weight: the same bits, on either
    side of 64 rows."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=36, quant=True, std=0.05, norm_std=0.1)
    plain = run(ming, ctx, syn, T)
    for v in syn.tensors.values():
        if isinstance(v, dict):
            v["s"].mul_(4.0)
            v["b"].mul_(4.0)
    syn.lin = lambda name: ming.linear(*(syn.tensors[name][k] for k in "wsb"), global_scale=0.25)
    syn._build_views()
    scaled = run(ming, ctx, syn, T)
    assert all(np.array_equal(a, b) for a, b in zip(plain[1:], scaled[1:]))


def test_vae_latents_off_alignment(ming, ctx):
    """Latents 2 bytes off a 16-byte boundary give the aligned call's bits."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=29, std=0.05)
    m = syn.model(7)
    buf = torch.empty(7 * 64 + 8, dtype=torch.bfloat16, device="cuda").normal_()
    waves = []
    for lat in (buf[1:1 + 7 * 64], buf[1:1 + 7 * 64].clone()):
        waves.append(torch.empty(7 * 4 * 16, dtype=torch.float32, device="cuda"))
        m.decode(7, lat, waves[-1])
    ctx.sync()
    m.close()
    assert torch.equal(waves[0], waves[1])


@pytest.mark.parametrize("T", [5, 17])
def test_vae_4bit_large_values(ming, ctx, T):
    """SwiGLU rows of about 2^122 (gate and up scaled by 2^61, down by 2^-115): a group's sums of them stay finite where
    the dequantized weights' products do, on either side of 64 rows; the bars are those of check()."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**SMALL), seed=30, quant=True, std=0.05, norm_std=0.1)
    for i in range(syn.spec.n_layers):
        for name, e in (("gate_proj", 61), ("up_proj", 61), ("down_proj", -115)):
            for k in "sb":
                syn.tensors[f"audio.decoder.decoder.layers.{i}.mlp.{name}"][k].mul_(2.0 ** e)
    check(ming, ctx, syn, T)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("T", [9, 23])
def test_vae_infinite_latent(ming, ctx, quant, T):
    """A latent with an infinity makes NaN of exactly the samples that it does in the oracle (a row's norm turns an
    infinite value into NaN), and the others keep their bars."""
    S = syn_mod()
    syn = S.SyntheticVae(ctx, S.VaeSpec(**dict(SMALL, window=4)), seed=31, quant=quant, std=0.05, norm_std=0.1)
    om, spec = oracle_vae(syn), syn.spec
    lat = ming.synth_normal_bf16(32, "vae.inf", T * spec.latent).reshape(T, spec.latent)
    lat[3, 5] = 0x7f80
    lat[4, 11] = 0xff80
    wave = torch.empty(T * spec.patch * spec.hop, dtype=torch.float32, device="cuda")
    m = syn.model(T)
    m.decode(T, torch.from_numpy(lat.view(np.int16)).cuda().view(torch.bfloat16), wave)
    ctx.sync()
    m.close()
    got, ref = wave.cpu().numpy(), oracle.vae_decode(om, lat)
    bad = np.isnan(ref)
    assert bad.any() and not bad.all()
    assert np.array_equal(np.isnan(got), bad)
    assert_close_f32(got[~bad], ref[~bad], "samples beside the infinite latents", 2e-4)
