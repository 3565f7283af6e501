"""AudioVAE decoder (AudioVaeEngine::decode_latents, audiovae.rs:330-372) and the
vae_*.comp entry points on the GPU against the oracle (voxref.AudioVae, vr_vae_*),
through the C ABI. Per-op kernels rel-L2 <= 1e-5; the decoded wave rel-L2 <= 1e-3
(the engine runs the 1x1 and transposed convolutions as f16-weight GEMMs with the
f32 activations split hi/lo, in its own order)."""
import numpy as np
import pytest

import voxref
from conftest import rel_l2
from test_oracle_vae_pins import f16_region
from voxgen_amd import abi, synth
from voxgen_amd.audiovae import AudioVaeEngine
from voxgen_amd.runtime import Model

pytestmark = pytest.mark.gpu


def test_vae_shader_entry_points(ctx):
    rng = np.random.default_rng(11)
    C, L = 16, 300
    arrays = {"dw": rng.normal(0, 0.3, (C, 1, 7)), "dwb": rng.normal(0, 0.1, C),
              "pw": rng.normal(0, 0.2, (8, C, 1)), "pwb": rng.normal(0, 0.1, 8),
              "st": rng.normal(0, 0.3, (C, 12, 6)), "stb": rng.normal(0, 0.1, 12),
              "ct": rng.normal(0, 0.3, (C, 8, 10)), "ctb": rng.normal(0, 0.1, 8),
              "a": rng.uniform(0.5, 1.5, C), "s": rng.normal(1, 0.1, (4, C)), "b": rng.normal(0, 0.1, (4, C))}
    blob, off = f16_region({k: np.asarray(v, np.float16).ravel() for k, v in arrays.items()})
    from voxgen_amd.runtime import TensorDesc
    model = Model(ctx, blob, [TensorDesc("blob", abi.DTYPE_F32, (blob.size // 4,), 0)])
    x = rng.normal(0, 1, (C, L)).astype(np.float32)
    xb = ctx.array(x)
    y = ctx.alloc(C * L * 5 * 4)
    cases = [
        ("conv1d", abi.VaeConvPush(off["dw"], off["dwb"], C, C, L, L, 7, 1, 3, C, 18, 1, 1, 1), C * L),
        ("conv1d", abi.VaeConvPush(off["pw"], off["pwb"], C, 8, L, L, 1, 1, 1, 1, 0, 1, 1, 1), 8 * L),
        ("conv1d", abi.VaeConvPush(off["st"], off["stb"], C, 12, L, L // 3, 6, 3, 1, 1, 3, 1, 1, 1), 12 * (L // 3)),
        ("conv1d", abi.VaeConvPush(off["pw"], off["pwb"], C, 8, L, L, 1, 1, 1, 1, 0, 1, 1, 0), 8 * L),
        ("convt", abi.VaeConvTPush(off["ct"], off["ctb"], C, 8, L, 5 * L, 10, 5, 1, 1, 1, 1), 8 * 5 * L),
    ]
    for kind, push, n in cases:
        print(f"vae op {kind} {n}", flush=True)
        if kind == "conv1d":
            abi.call("vx_vae_conv1d", ctx.handle, model.handle, xb.handle, y.handle, push)
            want = voxref.vae_conv1d(model_blob(blob), x.ravel(), push)
        else:
            abi.call("vx_vae_convtranspose1d", ctx.handle, model.handle, xb.handle, y.handle, push)
            want = voxref.vae_convt1d(model_blob(blob), x.ravel(), push)
        assert rel_l2(y.download(np.float32, n), want) < 1e-5, kind
    push = abi.VaeSnakePush(off["a"], C, L, 1)
    abi.call("vx_vae_snake", ctx.handle, model.handle, xb.handle, y.handle, push)
    assert rel_l2(y.download(np.float32, C * L), voxref.vae_snake(blob, x.ravel(), push)) < 1e-5
    push = abi.VaeScalePush(off["s"], off["b"], C, L, 3, 4, 1, 1)
    z = ctx.array(x)
    abi.call("vx_vae_scale_bias", ctx.handle, model.handle, z.handle, push)
    assert rel_l2(z.download(np.float32, C * L), voxref.vae_scale_bias(blob, x.ravel(), push)) < 1e-6
    abi.call("vx_vae_add", ctx.handle, z.handle, xb.handle, abi.VaeGridPush(C, L))
    abi.call("vx_vae_tanh", ctx.handle, z.handle, C * L)
    want = voxref.vae_tanh(voxref.vae_scale_bias(blob, x.ravel(), push) + x.ravel())
    assert rel_l2(z.download(np.float32, C * L), want) < 1e-6
    small = ctx.alloc(16)   # held in a name: a temporary Buffer frees its handle when .handle is read
    bad = abi.VaeConvPush(off["dw"], off["dwb"], C, C, L, L, 7, 1, 3, C, 18, 1, 1, 1)
    with pytest.raises(abi.VxError) as e:
        abi.call("vx_vae_conv1d", ctx.handle, model.handle, xb.handle, small.handle, bad)
    assert e.value.name == "VX_ERR_BOUNDS"
    model.free()


def model_blob(blob):
    return blob


def engine_case(ctx, dd, frames, seed):
    cfg = synth.audiovae_config(decoder_dim=dd)
    m = synth.build_audiovae(cfg, seed=seed)
    model = Model(ctx, m.data, m.tensors)
    eng = AudioVaeEngine(ctx, model, cfg, strict_geometry=(dd == 2048))
    lat = synth.normal_f32(frames * 64, seed + 1)
    o = voxref.AudioVae(m.data, {t.name: t for t in m.tensors}, cfg)
    return cfg, model, eng, lat, o


@pytest.mark.parametrize("dd,frames", [(256, 8), (2048, 4)])
def test_decode_matches_oracle(ctx, dd, frames):
    print(f"vae decode decoder_dim {dd} frames {frames}", flush=True)
    cfg, model, eng, lat, o = engine_case(ctx, dd, frames, 0x5EED0510 + dd)
    st, wave = eng.decode_latents(lat)
    want = o.decode(lat)
    assert wave.size == frames * 1920 == st.output_samples
    assert rel_l2(wave, want) < 1e-3
    assert st.latent_frames == frames and st.latent_patches == frames // 4 and st.output_sample_rate == 48000
    assert st.checksum == pytest.approx(float(np.sum(wave.astype(np.float64))), abs=1e-6 * wave.size)
    assert st.l2 == pytest.approx(float(np.linalg.norm(wave.astype(np.float64))), rel=1e-9)
    assert st.peak == pytest.approx(float(np.max(np.abs(wave))))
    assert st.scratch_bytes == eng.scratch_bytes() > 0
    lb, wb = ctx.array(lat), ctx.alloc(wave.size * 4)
    eng.decode_latents_gpu(lb, frames, wb)
    # split-K GEMMs accumulate with atomic adds: runs agree to rounding, not bit for bit
    assert rel_l2(wb.download(np.float32, wave.size), wave) < 1e-5
    eng.close()
    model.free()


@pytest.mark.parametrize("frames", [20, 36, 72])
def test_long_decode_tiles(ctx, frames):
    """The residual units and the head take larger tiles from 18, 35 and 69 frames on
    (32, 64/128 and 256 channels). The decoder is causal with under 20 frames of
    history, so a long decode starts like the oracle's decode of its first 4 frames and
    ends like a decode of its last 20 (small tiles but for the 32 channels)."""
    print(f"vae long decode frames {frames}", flush=True)
    cfg, model, eng, lat, o = engine_case(ctx, 2048, frames, 0x5EED0530)
    wave = eng.decode_latents(lat)[1]
    assert rel_l2(wave[:4 * 1920], o.decode(lat[:4 * 64])) < 1e-3
    tail = eng.decode_latents(lat[-20 * 64:])[1]
    assert rel_l2(wave[-1920:], tail[-1920:]) < 1e-5
    eng.close()
    model.free()


@pytest.mark.parametrize("dd,frames", [(512, 12), (1024, 20), (2048, 12), (2048, 44)])
def test_decode_plane_gemms(ctx, dd, frames):
    """Up-convolutions and wide residual units over planes at ragged row counts: small
    tiles (96 rows; 12 rows from the latents), 128 x 128 tiles with a last partial one
    (2112 rows), two K ranges (352 rows of 1024 channels), the one-pass unit of 512
    channels from 2048 rows on, and 16-channel stages behind the planes (512). Whole
    decode up to 20 frames; the first 4 frames of a causal decode beyond."""
    print(f"vae plane gemms decoder_dim {dd} frames {frames}", flush=True)
    cfg, model, eng, lat, o = engine_case(ctx, dd, frames, 0x5EED0550 + dd + frames)
    head = frames if frames <= 20 else 4
    want = o.decode(lat[:head * 64])
    for _ in range(2):
        wave = eng.decode_latents(lat)[1]
        assert rel_l2(wave[:want.size], want) < 1e-5   # two f16 planes: 22 bits of x
    if head < frames:   # the last 20 frames have their whole history in a decode of 40
        tail = eng.decode_latents(lat[-40 * 64:])[1]
        assert rel_l2(wave[-20 * 1920:], tail[-20 * 1920:]) < 1e-5
    eng.close()
    model.free()


def test_decode_large_snake_arguments(ctx):
    """Snake arguments past the reduced-range sine (|a x| >= 32768): with alphas of
    60000 the term sin(a x)^2 / a is below 2e-5, so the wave has to match the oracle
    whatever the sine of so large an argument rounds to."""
    cfg = synth.audiovae_config(decoder_dim=256)
    m = synth.build_audiovae(cfg, seed=0x5EED0540)
    for t in m.tensors:
        if t.name.endswith("alpha"):
            m.data[t.offset:t.offset + t.nbytes].view(np.float16)[::3] = 60000.0
    model = Model(ctx, m.data, m.tensors)
    eng = AudioVaeEngine(ctx, model, cfg, strict_geometry=False)
    lat = 4.0 * synth.normal_f32(8 * 64, 0x5EED0541)
    want = voxref.AudioVae(m.data, {t.name: t for t in m.tensors}, cfg).decode(lat)
    wave = eng.decode_latents(lat)[1]
    assert np.isfinite(wave).all() and rel_l2(wave, want) < 1e-3
    eng.close()
    model.free()


def test_decode_errors(ctx):
    cfg, model, eng, lat, o = engine_case(ctx, 256, 4, 0x5EED0520)
    for bad, code in ((lat[:63], "VX_ERR_SHAPE"), (lat[:128], "VX_ERR_SHAPE"),
                      (np.where(np.arange(lat.size) == 5, np.nan, lat).astype(np.float32), "VX_ERR_INVALID_ARG")):
        with pytest.raises(abi.VxError) as e:
            eng.decode_latents(bad)
        assert e.value.name == code
    with pytest.raises(abi.VxError) as e:
        eng.decode_latents_gpu(ctx.array(lat), 4, ctx.alloc(1024))
    assert e.value.name == "VX_ERR_BOUNDS"
    # A frame count whose activations pass the 32-bit index range is refused by
    # the device-buffer entry as by the host one, before any buffer check or launch.
    patch = cfg["patch_size"]
    with pytest.raises(abi.VxError) as e:
        eng.decode_latents_gpu(ctx.array(lat), (0xFFFFFFFF // patch) * patch, ctx.alloc(1024))
    assert e.value.name == "VX_ERR_UNSUPPORTED"
    with pytest.raises(abi.VxError) as e:
        AudioVaeEngine(ctx, model, cfg, strict_geometry=True)
    assert e.value.name == "VX_ERR_UNSUPPORTED"
    eng.close()
    model.free()


def edited_case(ctx, dd, seed, edits):
    """An engine and oracle over a synthetic decoder some of whose tensors (name ending
    -> (mean, std) of normal values, clipped to the f16 range) are replaced."""
    cfg = synth.audiovae_config(decoder_dim=dd)
    m = synth.build_audiovae(cfg, seed=seed)
    rng = np.random.default_rng(seed)
    for t in m.tensors:
        for end, (mean, std) in edits.items():
            if t.name.endswith(end):
                v = m.data[t.offset:t.offset + t.nbytes].view(np.float16)
                v[:] = np.clip(rng.normal(mean, std, v.size), -65000, 65000).astype(np.float16)
    model = Model(ctx, m.data, m.tensors)
    eng = AudioVaeEngine(ctx, model, cfg, strict_geometry=False)
    return model, eng, voxref.AudioVae(m.data, {t.name: t for t in m.tensors}, cfg)


# The input of a 1x1 convolution, h = snake(depthwise), and of a transposed one, P =
# snake(x scale + bias), far above the f16 range or far below it, with weights that bring
# the result back: (std of the tensors before, after, snake alpha). With alphas of 1 the
# snake's arguments also leave the reduced-range sine.
SCALES = {"large": (3e4, 2e-6, 0.01), "large sine": (3e4, 2e-6, 1.0), "small": (3e-6, 2e4, 1.0)}


@pytest.mark.parametrize("scale", list(SCALES))
@pytest.mark.parametrize("dd,kind,stage", [(192, "unit", 2), (192, "convt", 3), (256, "convt", 5),
                                           (256, "unit", 3), (256, "unit", 4)])
def test_narrow_products_keep_range_and_bits(ctx, dd, kind, stage, scale):
    """Widths whose products are f32 (the 1x1 convolution of 96 channels, the transposed
    ones from 96 and 32) and those whose rows are scaled into the planes (the units of 64
    and 32 channels). Plain f16 planes of such values would overflow, or keep a few bits
    of them."""
    print(f"vae narrow products {dd} {kind} stage {stage} {scale}", flush=True)
    pre, post, al = SCALES[scale]
    if kind == "unit":
        p = "decoder.model.%d.block.{}.block." % stage
        edits = {}
        for r in (2, 3, 4):
            edits |= {p.format(r) + "1": (0.0, pre), p.format(r) + "1.bias": (0.0, pre),
                      p.format(r) + "2.alpha": (al, 0.1 * al), p.format(r) + "3": (0.0, post)}
    else:
        edits = {f"sr_cond_model.{stage}.scale_embed": (0.0, pre), f"sr_cond_model.{stage}.bias_embed": (0.0, pre),
                 f"decoder.model.{stage}.block.0.alpha": (al, 0.1 * al),
                 f"decoder.model.{stage}.block.1": (0.0, post)}
    model, eng, o = edited_case(ctx, dd, 0x5EED0560 + dd, edits)
    lat = synth.normal_f32(8 * 64, 0x5EED0561)
    wave, want = eng.decode_latents(lat)[1], o.decode(lat)
    err = rel_l2(wave, want)
    print(f"rel_l2 {err:.2e} peak {np.abs(want).max():.2f}", flush=True)
    assert np.abs(want).max() > 0.05 and err < 1e-5
    eng.close()
    model.free()


@pytest.mark.parametrize("frames", [48, 132, 252])
def test_decode_is_the_same_bit_for_bit(ctx, frames):
    """Equal decodes give equal bits: no sum depends on which workgroup is first. 132 and
    252 frames are 1056 and 2016 rows of 1024 channels, half the CUs' worth of tiles."""
    print(f"vae bits {frames}", flush=True)
    cfg, model, eng, lat, o = engine_case(ctx, 2048, frames, 0x5EED0570)
    first = eng.decode_latents(lat)[1]
    for _ in range(4):
        assert np.array_equal(eng.decode_latents(lat)[1], first)
    eng.close()
    model.free()
