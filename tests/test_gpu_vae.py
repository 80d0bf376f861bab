"""DC-AE VAE decoder on the GPU (sana_vae_* C ABI) against the oracle and the
reference's own output.

The oracle's decode is bit-exact with the reference's run_vae_decode
(tests/test_oracle_vae.py); here the HIP path (fp16 operands, fp32
accumulation and residuals) is held to a relative L2 of 2e-3 on the decoded
image, the per-forward bar of the DiT.  Decoder shapes go from one level of
each layer type up to the small 4-level decoder and the full Sana 1.0 decoder
(latent 32x32 -> 1024x1024, against the reference's fixture).
"""
import os

import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2, spread_subsample

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
TOL = 2e-3

CONFIGS = {
    "evit1": dict(channels=(128,), attn=(True,)),
    "res1": dict(channels=(64,), attn=(False,)),
    "up2": dict(channels=(64, 128), attn=(False, True)),
    "small": dict(channels=(64, 64, 128, 128), attn=(False, False, True, True)),
}


def build(cfg, full=False):
    import sana_dit
    ora = O.Vae(full=True) if full else O.Vae(cfg=cfg)
    dev = sana_dit.Vae(ora.cfg["channels"], ora.cfg["attn"])
    for name, shape in O.vae_manifest(ora.cfg).items():
        dev.set_weight(name, ora.get(name, shape))
    dev.check_weights()
    return ora, dev


@pytest.mark.parametrize("name,shape", [("evit1", (1, 32, 8, 8)), ("res1", (1, 32, 8, 8)), ("up2", (1, 32, 6, 10)),
                                        ("up2", (2, 32, 4, 4)), ("small", (1, 32, 8, 8))])
def test_decode_vs_oracle(name, shape):
    ora, dev = build(CONFIGS[name])
    try:
        lat = O.randn(shape, 42)
        print(f"{name} {shape}: oracle decode on the host ...", flush=True)
        ref = ora.decode(lat)
        got = dev.decode(lat)
        err = rel_l2(got, ref)
        print(f"{name} {shape}: image rel_l2 {err:.3e}")
        assert got.shape == ref.shape
        assert np.isfinite(got).all()
        assert err < TOL
        again = dev.decode(lat)
        assert np.array_equal(got, again)
    finally:
        dev.close()


# widths around the depthwise 5x5's strips (4 pixels and 2 of border each side)
# and row counts that leave the norms' last group of rows partial
@pytest.mark.parametrize("shape", [(1, 32, 1, 1), (1, 32, 3, 5), (2, 32, 5, 8), (1, 32, 6, 11), (1, 32, 2, 18)])
def test_attention_level_widths_vs_oracle(shape):
    ora, dev = build(CONFIGS["evit1"])
    try:
        lat = O.randn(shape, 13)
        assert rel_l2(dev.decode(lat), ora.decode(lat)) < TOL
    finally:
        dev.close()


def test_small_decode_vs_reference_fixture():
    fx = np.load(os.path.join(GOLDEN, "vae_small.npz"), allow_pickle=False)
    ora, dev = build(CONFIGS["small"])
    try:
        got = dev.decode(fx["latent"])
        err = rel_l2(got, fx["image"])
        print(f"small vs reference image: rel_l2 {err:.3e}")
        assert err < TOL
    finally:
        dev.close()


def test_batch_matches_single():
    ora, dev = build(CONFIGS["up2"])
    try:
        lat = O.randn((2, 32, 4, 6), 7)
        both = dev.decode(lat)
        one = np.concatenate([dev.decode(lat[i:i + 1]) for i in range(2)])
        assert rel_l2(both, one) < 1e-6
    finally:
        dev.close()


# one image's products of 512 channels sum k in four runs at 4 x 4 pixels and in
# two at 40 x 40; the batches take k-groups of 32x64 and 64x64 tiles, then one
# group that folds the runs, on 64x64, 128x64 and 128x128 tiles
@pytest.mark.parametrize("attn", [True, False], ids=["plain", "conv"])
@pytest.mark.parametrize("side,batches", [(4, (2, 80, 130, 260, 520)), (40, (2, 3, 6))])
def test_batches_sum_as_one_image(attn, side, batches):
    ora, dev = build(dict(channels=(128, 512), attn=(False, attn)))
    try:
        lat = O.randn((batches[-1], 32, side, side), 17)
        for b in batches:
            whole = dev.decode(lat[:b])
            assert np.isfinite(whole).all()
            for i in sorted({0, b // 2, b - 1}):
                assert np.array_equal(whole[i:i + 1], dev.decode(lat[i:i + 1])), (b, i)
    finally:
        dev.close()


def test_256_tile_convs_equal_smaller_tiles():
    """The 3x3 convs of 182 x 202 pixels and 256 channels (plain, upsampling,
    conv_in) run on 256x256 tiles, those of the latent's upper part on 128x128
    ones, with the same k order: pixels beyond the convs' reach from
    the cut (1 + 6 latent rows, 1 + 6 + 1 image rows) are bit-identical."""
    ora, dev = build(dict(channels=(256, 256), attn=(False, False)))
    try:
        lat = O.randn((1, 32, 91, 101), 11)
        whole, cut = dev.decode(lat), dev.decode(lat[:, :, :52])
        assert np.isfinite(whole).all()
        assert np.array_equal(whole[:, :, :80], cut[:, :, :80])
        dev2 = build(dict(channels=(256,), attn=(False,)))[1]
        lat = O.randn((1, 32, 182, 202), 12)
        whole, cut = dev2.decode(lat), dev2.decode(lat[:, :, :110])
        assert np.array_equal(whole[:, :, :100], cut[:, :, :100])
        dev2.close()
    finally:
        dev.close()


def test_rejects_bad_input():
    import sana_dit
    with pytest.raises(sana_dit.SanaError):
        sana_dit.Vae((96,), (False,))            # channels not a multiple of 64
    with pytest.raises(sana_dit.SanaError):
        sana_dit.Vae((64, 192), (False, False))  # upsample shortcut ratio 4*64 % 192 != 0
    dev = sana_dit.Vae((64,), (False,))
    try:
        with pytest.raises(sana_dit.SanaError) as e:
            dev.decode(O.randn((1, 32, 4, 4), 1))  # no weights
        assert e.value.code == sana_dit.SANA_ERR_STATE
        with pytest.raises(sana_dit.SanaError) as e:
            dev.set_weight("decoder.conv_in.weight", np.zeros((64, 32, 1, 1), np.float32))
        assert e.value.code == sana_dit.SANA_ERR_SHAPE
    finally:
        dev.close()


def test_full_decoder_vs_reference():
    """Sana 1.0 DC-AE f32c32 decoder, latent 32x32 -> 1024x1024 RGB: the
    fixture keeps a strided subsample of the reference's image, 65536 values
    spread over every row and column, and its L2 norm."""
    path = os.path.join(GOLDEN, "vae_full.npz")
    if not os.path.exists(path):
        pytest.skip("vae_full golden not generated")
    fx = np.load(path, allow_pickle=False)
    import sana_dit
    print("generating the full synthetic decoder on the host ...", flush=True)
    ora = O.Vae(full=True)
    dev = sana_dit.Vae(ora.cfg["channels"], ora.cfg["attn"])
    try:
        for name, shape in O.vae_manifest(ora.cfg).items():
            dev.set_weight(name, ora.get(name, shape))
        lat = O.randn((1, 32, 32, 32), 42)
        got = dev.decode(lat)
        assert got.shape == (1, 3, 1024, 1024)
        stride = int(fx["image__stride"])
        err = rel_l2(got.reshape(-1)[::stride], fx["image__sub"])
        norm_err = abs(np.linalg.norm(got.astype(np.float64)) / float(fx["image__l2"]) - 1.0)
        print(f"full decoder: image subsample rel_l2 {err:.3e}, L2 norm rel diff {norm_err:.3e}")
        assert np.isfinite(got).all()
        assert err < TOL
        assert norm_err < TOL
        sp = spread_subsample(got, fx, "image")
        if sp is not None:
            serr = rel_l2(*sp)
            print(f"full decoder: spread subsample ({sp[1].size} values) rel_l2 {serr:.3e}")
            assert serr < TOL
    finally:
        dev.close()


def test_decoder_input_stage():
    """run_vae_decoder_input: conv_in of the (already scaled) latent, with and
    without the channel-repeat shortcut; needs only the conv_in tensors."""
    import sana_dit
    ora = O.Vae(cfg=CONFIGS["up2"])
    dev = sana_dit.Vae(ora.cfg["channels"], ora.cfg["attn"])
    try:
        for name in ("decoder.conv_in.weight", "decoder.conv_in.bias"):
            dev.set_weight(name, ora.get(name))
        lat = O.randn((2, 32, 5, 7), 3)
        scaled = lat * (np.float32(1.0) / np.float32(0.41407))
        ref = ora.decoder_input(lat)                     # scales, conv_in, + shortcut
        got = dev.decoder_input(scaled)
        assert got.shape == (2, 128, 5, 7)
        assert rel_l2(got, ref) < TOL
        rep = 128 // 32
        short = np.repeat(scaled, rep, axis=1)           # channel oc reads latent channel oc // rep
        assert rel_l2(dev.decoder_input(scaled, in_shortcut=False), ref - short) < TOL
    finally:
        dev.close()
