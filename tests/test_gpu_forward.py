"""Full-model parity of the HIP path against the reference's own CPU outputs.

The golden fixtures (tests/golden/*.npz) hold the outputs of the reference's
src/*.cpp compiled from source (tests/golden/make_golden.py) on the seeded
synthetic Sana-0.6B model of oracle/model_spec.h; the oracle regenerates the
identical weights bit for bit (tests/test_oracle_golden.py pins that), and
they are uploaded here through the C ABI.

Tolerances (relative L2): 2e-3 per forward, 1e-2 on the final latent of the
20-step DPM-Solver++ loop.
"""
import os

import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2, spread_subsample

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
TOL_FORWARD = 2e-3
TOL_LOOP = 1e-2


def golden(name):
    return np.load(os.path.join(GOLDEN, name + ".npz"), allow_pickle=False)


@pytest.fixture(scope="module")
def full_model():
    import sana_dit
    print("generating the seeded 28-block weights on the host ...", flush=True)
    m = O.Model(layers=28, self_heads=36, cross_heads=16)
    d = sana_dit.Dit(layers=28, self_heads=36, cross_heads=16)
    for name, shape in sana_dit.manifest(28).items():
        d.set_weight(name, m.get(name, shape))
    d.check_weights()
    yield m, d
    d.close()


@pytest.mark.parametrize("case,masked", [("cfg2", False), ("cfg2_mask", True)])
def test_forward_1024px_vs_reference(full_model, case, masked):
    m, d = full_model
    fx = golden(case)
    latent = O.randn((1, 32, 32, 32), 42)
    caption = O.randn((2, 300, 2304), 43)
    bias = O.mask_bias(300, 1, 40) if masked else None
    d.set_context(caption, projected=False, bias=bias)
    ctx = d.get_context((2, 300, 1152))
    stride = int(fx["context__stride"])
    ctx_err = rel_l2(ctx.reshape(-1)[::stride], fx["context__sub"])
    got = d.forward(latent, 999.0)
    err = rel_l2(got, fx["noise_pred"])
    guided = got[:1] + np.float32(4.5) * (got[1:] - got[:1])
    gerr = rel_l2(guided, fx["guided"])
    print(f"{case}: context rel_l2 {ctx_err:.2e}, noise_pred rel_l2 {err:.2e}, guided rel_l2 {gerr:.2e}")
    assert ctx_err < 1e-3
    assert err < TOL_FORWARD
    assert gerr < TOL_FORWARD


def test_forward_nonsquare_vs_reference(full_model):
    """A 4x16 latent (64 tokens) against the reference's own forward of it:
    the reference runs each block's depthwise conv on the 8x8 token grid
    (src/transformer.cpp:765-767), and so does the device path."""
    m, d = full_model
    fx = golden("nonsquare")
    latent = O.randn((1, 32, 4, 16), 42)
    d.set_context(O.randn((2, 300, 2304), 43), projected=False)
    got = d.forward(latent, 999.0)
    err = rel_l2(got, fx["noise_pred"])
    print(f"nonsquare 4x16: noise_pred rel_l2 {err:.2e}")
    assert err < TOL_FORWARD


def test_forward_4096px_vs_reference(full_model):
    """4096 px (latent 128x128, 16384 image tokens): the reference's CPU forward
    is too large to store whole, so the fixture keeps, of noise_pred and
    guided, a strided subsample, 65536 values spread over every row and column
    of the grid, and their L2 norms."""
    path = os.path.join(GOLDEN, "cfg5.npz")
    if not os.path.exists(path):
        pytest.skip("cfg5 golden not generated")
    m, d = full_model
    fx = golden("cfg5")
    latent = O.randn((1, 32, 128, 128), 42)
    caption = O.randn((2, 300, 2304), 43)
    d.set_context(caption, projected=False)
    got = d.forward(latent, 999.0)
    guided = got[:1] + np.float32(4.5) * (got[1:] - got[:1])
    res = {}
    for name, arr in (("noise_pred", got), ("guided", guided)):
        stride = int(fx[name + "__stride"])
        res[name] = rel_l2(arr.reshape(-1)[::stride], fx[name + "__sub"])
        norm_err = abs(np.linalg.norm(arr.astype(np.float64)) / float(fx[name + "__l2"]) - 1.0)
        print(f"cfg5 {name}: subsample rel_l2 {res[name]:.2e}, L2 norm rel diff {norm_err:.2e}")
        assert res[name] < TOL_FORWARD
        assert norm_err < TOL_FORWARD
        sp = spread_subsample(arr, fx, name)
        if sp is not None:
            serr = rel_l2(*sp)
            print(f"cfg5 {name}: spread subsample ({sp[1].size} values) rel_l2 {serr:.2e}")
            assert serr < TOL_FORWARD


@pytest.mark.parametrize("masked", [False, True], ids=["nomask", "mask"])
def test_step_device_matches_context_then_forward(full_model, masked):
    """sana_dit_step_device (caption projection, cross K/V and forward in one call,
    the forward's head beside the context GEMMs) gives the noise prediction of
    sana_dit_set_context + sana_dit_forward bit for bit."""
    import torch
    m, d = full_model
    latent = O.randn((1, 32, 32, 32), 42)
    caption = O.randn((2, 300, 2304), 43)
    bias = O.mask_bias(300, 1, 40) if masked else None
    d.set_context(caption, projected=False, bias=bias)
    ref = d.forward(latent, 999.0)
    dev = torch.device("cuda:0")
    d_cap = torch.from_numpy(caption).to(dev)
    d_lat = torch.from_numpy(latent).to(dev)
    d_bias = torch.from_numpy(np.ascontiguousarray(bias, np.float32)).to(dev) if masked else None
    out = torch.empty((2, 32, 32, 32), device=dev)
    for _ in range(2):  # the second call replays the cached block chains
        out.fill_(float("nan"))
        d.step_device(d_cap, 300, d_bias, d_lat, (1, 32, 32, 32), 999.0, out)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.array_equal(got, ref)


def test_block_256_tiles(full_model):
    """One block on 16 x 256 tokens at once (256x256 tiles for the q|k|v split)
    against pairs of them (small tiles): the same sums in the same order."""
    m, d = full_model
    x, ctx, tmod = O.randn((16, 256, 1152), 21), O.randn((16, 300, 1152), 22), 0.1 * O.randn((16, 6 * 1152), 23)
    d.set_context(ctx, projected=True)
    got = d.run_blocks(0, 1, x, tmod)
    for i in range(0, 16, 2):
        d.set_context(ctx[i:i + 2], projected=True)
        ref = d.run_blocks(0, 1, x[i:i + 2], tmod[i:i + 2])
        assert np.array_equal(got[i:i + 2], ref)


def test_forward_deterministic(full_model):
    m, d = full_model
    latent = O.randn((1, 32, 32, 32), 42)
    caption = O.randn((2, 300, 2304), 43)
    d.set_context(caption, projected=False)
    a = d.forward(latent, 999.0)
    b = d.forward(latent, 999.0)
    assert np.array_equal(a, b)


def test_denoise_loop_1024px_vs_reference(full_model):
    path = os.path.join(GOLDEN, "cfg3.npz")
    if not os.path.exists(path):
        pytest.skip("cfg3 golden not generated")
    m, d = full_model
    fx = golden("cfg3")
    latent = O.randn((1, 32, 32, 32), 42)
    caption = O.randn((2, 300, 2304), 43)
    d.set_context(caption, projected=False)
    ts, sg = O.scheduler_timesteps(20)
    fin = d.denoise_loop(latent, ts, sg, 4.5)
    err = rel_l2(fin, fx["final_latent"])
    print(f"cfg3: final latent rel_l2 {err:.2e}")
    assert err < TOL_LOOP


@pytest.fixture(scope="module")
def two_blocks():
    """Two blocks of the full width, as two concurrent chains and as one."""
    import sana_dit
    m = O.Model(layers=2, self_heads=36, cross_heads=16)
    ctxs = []
    for branches in ("1", "0"):
        os.environ["SANA_DIT_CFG_BRANCHES"] = branches
        try:
            d = sana_dit.Dit(layers=2, self_heads=36, cross_heads=16)
        finally:
            del os.environ["SANA_DIT_CFG_BRANCHES"]
        for name, shape in sana_dit.manifest(2).items():
            d.set_weight(name, m.get(name, shape))
        ctxs.append(d)
    yield ctxs
    for d in ctxs:
        d.close()


# few-row products sum k in two or four runs: by k-groups alone, by one group that
# folds them (64x64, 128x64 and 128x128 tiles) in the larger batches
@pytest.mark.parametrize("side,L,batches", [(8, 40, (2, 3, 5, 10)), (12, 77, (2,)), (16, 300, (2, 4, 5, 8)),
                                            (23, 300, (2,)), (32, 300, (2,)), (36, 40, (1,)), (40, 40, (1,))])
def test_batch_equals_single_images(two_blocks, side, L, batches):
    """An image's noise prediction does not depend on its batch, nor on whether
    the batch runs as two chains: bit for bit."""
    n = batches[-1]
    latent, caption = O.randn((n, 32, side, side), 42), O.randn((2 * n, L, 2304), 43)
    bias = np.zeros((2 * n, L), np.float32)
    bias[1::2, L // 2:] = -10000.0

    def run(d, first, count):
        rows = np.r_[first:first + count, n + first:n + first + count]
        d.set_context(caption[rows], projected=False, bias=bias[rows])
        return d.forward(latent[first:first + count], 999.0)

    singles = {i: run(two_blocks[0], i, 1) for i in {0} | {b - 1 for b in batches}}
    assert np.array_equal(run(two_blocks[1], 0, 1), singles[0])
    for b in batches:
        for d in two_blocks:
            whole = run(d, 0, b)
            assert np.isfinite(whole).all()
            for i in (0, b - 1):
                assert np.array_equal(whole[[i, b + i]], singles[i]), (b, i)


SMALL = dict(layers=2, hidden=128, ffn=256, caption=96, latent=8, self_heads=4, cross_heads=2)


@pytest.fixture(scope="module")
def small_model():
    import sana_dit
    m = O.Model(**SMALL)
    d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
        d.set_weight(name, m.get(name, shape))
    d.check_weights()
    yield m, d
    d.close()


def test_small_loop_vs_oracle(small_model):
    m, d = small_model
    latent = O.randn((1, 8, 8, 8), 42)
    caption = O.randn((2, 16, 96), 43)
    ref = m.loop(latent, caption, 6, 4.5)
    d.set_context(caption, projected=False)
    ts, sg = O.scheduler_timesteps(6)
    got = d.denoise_loop(latent, ts, sg, 4.5)
    assert np.isfinite(ref).all(), "oracle loop not finite"
    assert np.isfinite(got).all(), "device loop not finite"
    err = rel_l2(got, ref)
    print(f"small loop rel_l2 {err:.2e}")
    assert err < TOL_LOOP


def test_small_run_blocks_vs_oracle(small_model):
    m, d = small_model
    rng = np.random.default_rng(7)
    x = rng.standard_normal((2, 64, 128)).astype(np.float32)
    ctx = rng.standard_normal((2, 16, 128)).astype(np.float32)
    emb, tmod = m.time(np.array([500.0, 500.0], np.float32))
    ref = x
    for i in range(2):
        ref = m.block(i, ref, ctx, tmod)[2]
    d.set_context(ctx, projected=True)
    got = d.run_blocks(0, 2, x, tmod)
    assert rel_l2(got, ref) < TOL_FORWARD


def test_small_forward_masked_vs_oracle(small_model):
    m, d = small_model
    latent = O.randn((1, 8, 8, 8), 5)
    caption = O.randn((2, 16, 96), 6)
    bias = np.full((2, 16), -10000.0, np.float32)
    bias[0, :3] = 0.0
    bias[1, :11] = 0.0
    ctx = m.project_caption(caption)
    ref = m.forward(latent, ctx, 733.0, bias)
    d.set_context(caption, projected=False, bias=bias)
    got = d.forward(latent, 733.0)
    assert rel_l2(got, ref) < TOL_FORWARD


def test_small_forward_batch2_vs_oracle(small_model):
    """A latent batch of 2 (context batch 4): two chains of two rows, patch embed
    reading latent row b % 2, uncond rows first."""
    m, d = small_model
    latent = O.randn((2, 8, 8, 8), 11)
    caption = O.randn((4, 16, 96), 12)
    ctx = m.project_caption(caption)
    ref = m.forward(latent, ctx, 610.0)
    d.set_context(caption, projected=False)
    got = d.forward(latent, 610.0)
    err = rel_l2(got, ref)
    print(f"small forward, latent batch 2: rel_l2 {err:.2e}")
    assert err < TOL_FORWARD


def test_small_forward_nonsquare_latent(small_model):
    """A 4x16 latent (64 tokens): the reference accepts any H x W whose token
    count is a perfect square and runs each block's depthwise conv on the
    side x side token grid (src/transformer.cpp:18-24, 765-767).  The device
    forward matches the oracle there, equals the 8x8 view of the same data bit
    for bit (patch embedding and final layer see only the flattened index), and
    a 4x8 latent (32 tokens) is refused with the reference's message."""
    import sana_dit
    m, d = small_model
    latent = O.randn((1, 8, 4, 16), 21)
    caption = O.randn((2, 16, 96), 22)
    ref = m.forward(latent, m.project_caption(caption), 420.0)
    d.set_context(caption, projected=False)
    got = d.forward(latent, 420.0)
    assert got.shape == (2, 8, 4, 16)
    err = rel_l2(got, ref)
    print(f"small forward, 4x16 latent: rel_l2 {err:.2e}")
    assert err < TOL_FORWARD
    sq = d.forward(latent.reshape(1, 8, 8, 8), 420.0)
    assert np.array_equal(got.reshape(sq.shape), sq)
    ts, sg = O.scheduler_timesteps(3)
    loop_ns = d.denoise_loop(latent, ts, sg, 4.5)
    loop_sq = d.denoise_loop(latent.reshape(1, 8, 8, 8), ts, sg, 4.5)
    assert np.array_equal(loop_ns.reshape(loop_sq.shape), loop_sq)
    with pytest.raises(sana_dit.SanaError, match="token count must form a square grid"):
        d.forward(O.randn((1, 8, 4, 8), 23), 420.0)


def test_conditioning_dropped_by_its_weights():
    """Uploading a weight the conditioning was computed from (cross-attention
    k / v, caption projection, caption_norm) drops it: the next forward fails
    with SANA_ERR_STATE until sana_dit_set_context runs again; other weights
    keep it."""
    import sana_dit
    m = O.Model(**SMALL)
    d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    try:
        man = sana_dit.manifest(2, 128, 256, 96, 8)
        for name, shape in man.items():
            d.set_weight(name, m.get(name, shape))
        latent = O.randn((1, 8, 8, 8), 51)
        caption = O.randn((2, 16, 96), 52)
        d.set_context(caption, projected=False)
        ref = d.forward(latent, 999.0)
        for name in ("transformer_blocks.0.ff.conv_point.weight", "transformer_blocks.1.attn1.to_q.weight",
                     "scale_shift_table"):
            d.set_weight(name, m.get(name, man[name]))
            assert np.array_equal(d.forward(latent, 999.0), ref), name
        for name in ("transformer_blocks.1.attn2.to_k.weight", "transformer_blocks.0.attn2.to_v.bias",
                     "caption_projection.linear_2.weight", "caption_norm.weight"):
            d.set_weight(name, m.get(name, man[name]))
            with pytest.raises(sana_dit.SanaError) as e:
                d.forward(latent, 999.0)
            assert e.value.code == sana_dit.SANA_ERR_STATE, name
            d.set_context(caption, projected=False)
            assert np.array_equal(d.forward(latent, 999.0), ref), name
    finally:
        d.close()


def test_small_loop_batch2_vs_oracle(small_model):
    """The fused device loop on a latent batch of 2: CFG combines rows b and
    b + 2 of the noise prediction."""
    m, d = small_model
    latent = O.randn((2, 8, 8, 8), 13)
    caption = O.randn((4, 16, 96), 14)
    ref = m.loop(latent, caption, 5, 4.5)
    d.set_context(caption, projected=False)
    ts, sg = O.scheduler_timesteps(5)
    got = d.denoise_loop(latent, ts, sg, 4.5)
    err = rel_l2(got, ref)
    print(f"small loop, latent batch 2: rel_l2 {err:.2e}")
    assert err < TOL_LOOP


def test_small_forward_one_chain_no_graph_vs_oracle(monkeypatch):
    """SANA_DIT_CFG_BRANCHES=0 (the CFG pair as one chain) and
    SANA_DIT_NO_GRAPH=1 (direct launches), both read at context creation."""
    import sana_dit
    monkeypatch.setenv("SANA_DIT_CFG_BRANCHES", "0")
    monkeypatch.setenv("SANA_DIT_NO_GRAPH", "1")
    m = O.Model(**SMALL)
    d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    try:
        for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
            d.set_weight(name, m.get(name, shape))
        latent = O.randn((1, 8, 8, 8), 15)
        caption = O.randn((2, 16, 96), 16)
        ref = m.forward(latent, m.project_caption(caption), 999.0)
        d.set_context(caption, projected=False)
        got = d.forward(latent, 999.0)
        again = d.forward(latent, 999.0)
        err = rel_l2(got, ref)
        print(f"small forward, one chain, no graph: rel_l2 {err:.2e}")
        assert err < TOL_FORWARD
        assert np.array_equal(got, again)
    finally:
        d.close()


def test_small_loop_graph_replays_match_direct_launches(small_model, monkeypatch):
    """The denoise loop on the cached block chains: repeated with a forward and a
    loop of another schedule in between, every result equals the loop launched
    kernel by kernel (SANA_DIT_NO_GRAPH=1, read at context creation)."""
    import sana_dit
    m, d = small_model
    latent = O.randn((1, 8, 8, 8), 21)
    caption = O.randn((2, 16, 96), 22)
    ts6, sg6 = O.scheduler_timesteps(6)
    ts4, sg4 = O.scheduler_timesteps(4)
    d.set_context(caption, projected=False)
    first = d.denoise_loop(latent, ts6, sg6, 4.5)
    d.forward(O.randn((1, 8, 8, 8), 23), 500.0)
    other = d.denoise_loop(latent, ts4, sg4, 4.5)
    replays = [d.denoise_loop(latent, ts6, sg6, 4.5) for _ in range(2)]
    monkeypatch.setenv("SANA_DIT_NO_GRAPH", "1")
    e = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    try:
        for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
            e.set_weight(name, m.get(name, shape))
        e.set_context(caption, projected=False)
        direct6 = e.denoise_loop(latent, ts6, sg6, 4.5)
        direct4 = e.denoise_loop(latent, ts4, sg4, 4.5)
    finally:
        e.close()
    assert np.isfinite(direct6).all() and np.isfinite(direct4).all()
    assert np.array_equal(first, direct6)
    assert np.array_equal(other, direct4)
    for r in replays:
        assert np.array_equal(r, direct6)


def test_small_forward_fewer_tokens_more_chunks(small_model):
    """31 x 31 tokens after 33 x 33: the linear attention splits the fewer
    tokens into more chunks (16 against 9), so the workspace of the larger
    forward must hold them; the result equals a fresh context's."""
    import sana_dit
    m, d = small_model
    caption = O.randn((4, 16, 96), 31)
    lat33, lat31 = O.randn((2, 8, 33, 33), 32), O.randn((2, 8, 31, 31), 33)
    e = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    try:
        for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
            e.set_weight(name, m.get(name, shape))
        e.set_context(caption, projected=False)
        ref = e.forward(lat31, 999.0)
    finally:
        e.close()
    d.set_context(caption, projected=False)
    d.forward(lat33, 999.0)
    assert np.array_equal(d.forward(lat31, 999.0), ref)


@pytest.mark.parametrize("images,masked", [(1, True), (2, False)])
def test_small_step_streams_buffers_and_capture(small_model, images, masked):
    """One step on the context's stream, on a caller's stream with fresh
    buffers (the cached block chains hold none of the caller's), and captured
    into a caller's graph (replayed on new contents with eager steps between):
    all bit-identical."""
    import torch
    m, d = small_model
    dev = torch.device("cuda:0")
    shape = (images, 8, 8, 8)

    def data(seed):
        cap = torch.from_numpy(O.randn((2 * images, 16, 96), seed)).to(dev)
        lat = torch.from_numpy(O.randn(shape, seed + 1)).to(dev)
        bias = torch.zeros((2 * images, 16), device=dev)
        bias[:, 9:] = -10000.0
        return cap, lat, bias if masked else None

    def step(x, stream=None):
        out = torch.empty((2 * images, 8, 8, 8), device=dev)
        torch.cuda.synchronize()
        d.step_device(x[0], 16, x[2], x[1], shape, 999.0, out, stream.cuda_stream if stream else None)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    refs = [step(data(s)) for s in (61, 71, 81)]
    user = torch.cuda.Stream()
    for s, ref in zip((61, 71, 81), refs):
        assert np.array_equal(step(data(s), user), ref)
    x, out = data(61), torch.empty((2 * images, 8, 8, 8), device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=user):
        d.step_device(x[0], 16, x[2], x[1], shape, 999.0, out, user.cuda_stream)
    for s, ref in list(zip((61, 71, 81), refs)) * 2:
        y = data(s)
        x[0].copy_(y[0])
        x[1].copy_(y[1])
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), ref)
        assert np.array_equal(step(data(71)), refs[1])


def test_small_graph_cache_eviction(small_model, monkeypatch):
    """More shapes than the graph cache holds (two chains each), queued on a
    caller's stream without a wait: a graph is dropped only when it has run, and
    every result equals direct launches."""
    import sana_dit
    import torch
    m, _ = small_model
    dev = torch.device("cuda:0")
    cap = torch.from_numpy(O.randn((2, 16, 96), 91)).to(dev)
    lat = torch.from_numpy(O.randn((1, 8, 8, 8), 92)).to(dev)
    shapes = [(L, side, masked) for L in range(16, 0, -1) for side in (8, 7) for masked in (True, False)]
    user = torch.cuda.Stream()

    def run_all():
        d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
        try:
            for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
                d.set_weight(name, m.get(name, shape))
            data = []
            for L, side, masked in shapes:
                bias = torch.zeros((2, L), device=dev)
                bias[:, (L + 1) // 2:] = -10000.0
                data.append((cap[:, :L].contiguous(), bias if masked else None, lat[:, :, :side, :side].contiguous(),
                             torch.empty((2, 8, side, side), device=dev)))
            torch.cuda.synchronize()
            for (L, side, _), (c, b, x, out) in zip(shapes, data):
                d.step_device(c, L, b, x, (1, 8, side, side), 999.0, out, user.cuda_stream)
            torch.cuda.synchronize()
            return [x[3].cpu().numpy() for x in data]
        finally:
            d.close()

    got = run_all()
    monkeypatch.setenv("SANA_DIT_NO_GRAPH", "1")
    for shape, a, b in zip(shapes, got, run_all()):
        assert np.isfinite(a).all() and np.array_equal(a, b), shape


def loop_outputs(d, shape):
    import sana_dit
    prev, last = np.empty(shape, np.float32), np.empty(shape, np.float32)
    sana_dit.check(sana_dit.lib().sana_dit_loop_model_outputs(d.h, sana_dit.ptr(prev), sana_dit.ptr(last)))
    return prev, last


def test_small_capture_leaves_state(small_model):
    """Recording a step (other caption length, masked) and a loop into a caller's
    graphs runs nothing, so forwards and sana_dit_loop_model_outputs answer as
    before; a step recorded after the conditioning was dropped does not bring it
    back."""
    import sana_dit
    import torch
    m, d = small_model
    dev = torch.device("cuda:0")
    latent, caption = O.randn((1, 8, 8, 8), 101), O.randn((2, 16, 96), 102)
    ts6, sg6 = O.scheduler_timesteps(6)
    ts4, sg4 = O.scheduler_timesteps(4)
    d_lat = torch.from_numpy(latent).to(dev)
    cap9 = torch.from_numpy(O.randn((2, 9, 96), 103)).to(dev)
    bias9 = torch.zeros((2, 9), device=dev)
    bias9[:, 4:] = -10000.0
    out, fin = torch.empty((2, 8, 8, 8), device=dev), torch.empty((1, 8, 8, 8), device=dev)
    d.set_context(caption, projected=False)
    loop4 = d.denoise_loop(latent, ts4, sg4, 4.5)
    d.denoise_loop(latent, ts6, sg6, 4.5)
    x0 = loop_outputs(d, latent.shape)
    ref = d.forward(latent, 999.0)
    torch.cuda.synchronize()
    user = torch.cuda.Stream()
    step_graph, loop_graph = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(step_graph, stream=user):
        d.step_device(cap9, 9, bias9, d_lat, (1, 8, 8, 8), 500.0, out, user.cuda_stream)
    assert np.array_equal(d.forward(latent, 999.0), ref)
    with torch.cuda.graph(loop_graph, stream=user):
        d.denoise_loop_device(d_lat, (1, 8, 8, 8), ts4, sg4, 4.5, fin, user.cuda_stream)
    for got, want in zip(loop_outputs(d, latent.shape), x0):
        assert np.array_equal(got, want)
    assert np.array_equal(d.forward(latent, 999.0), ref)
    for _ in range(2):
        fin.fill_(float("nan"))
        loop_graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(fin.cpu().numpy(), loop4)
        d.denoise_loop(latent, ts6, sg6, 4.5)
    d.set_weight("caption_norm.weight", m.get("caption_norm.weight", (128,)))
    with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=user):
        d.step_device(cap9, 9, bias9, d_lat, (1, 8, 8, 8), 500.0, out, user.cuda_stream)
    with pytest.raises(sana_dit.SanaError) as e:
        d.forward(latent, 999.0)
    assert e.value.code == sana_dit.SANA_ERR_STATE


def test_small_growth_after_capture(small_model):
    """A captured step replays correctly after larger eager calls have outgrown
    the buffers it holds (context and workspace), and a capture of a shape that
    was never run is refused with everything as before."""
    import sana_dit
    import torch
    m, _ = small_model
    dev = torch.device("cuda:0")
    d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    user = torch.cuda.Stream()

    def data(images, side, L, seed):
        return (torch.from_numpy(O.randn((2 * images, L, 96), seed)).to(dev),
                torch.from_numpy(O.randn((images, 8, side, side), seed + 1)).to(dev),
                torch.full((2 * images, 8, side, side), float("nan"), device=dev))

    def step(x):
        torch.cuda.synchronize()
        d.step_device(x[0], x[0].shape[1], None, x[1], tuple(x[1].shape), 999.0, x[2], user.cuda_stream)

    def eager(*a):
        x = data(*a)
        step(x)
        torch.cuda.synchronize()
        return x[2].cpu().numpy()

    try:
        for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
            d.set_weight(name, m.get(name, shape))
        ref = eager(1, 8, 16, 111)
        x = data(1, 8, 16, 111)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=user):
            d.step_device(x[0], 16, None, x[1], (1, 8, 8, 8), 999.0, x[2], user.cuda_stream)
        large = data(2, 16, 40, 121)
        torch.cuda.synchronize()
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=user):
            with pytest.raises(sana_dit.SanaError) as e:
                d.step_device(large[0], 40, None, large[1], (2, 8, 16, 16), 999.0, large[2], user.cuda_stream)
        assert e.value.code == sana_dit.SANA_ERR_STATE
        assert np.array_equal(eager(1, 8, 16, 111), ref)
        want = eager(2, 16, 40, 121)
        for _ in range(3):
            x[2].fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(x[2].cpu().numpy(), ref)
            assert np.array_equal(eager(2, 16, 40, 121), want)
        del g
        torch.cuda.synchronize()
    finally:
        d.close()


def test_small_step_after_failed_growth():
    """A step whose workspace does not fit the device fails with
    SANA_ERR_OUT_OF_MEMORY; the context then allocates what the next shape needs
    instead of running on the buffers that were given up."""
    import sana_dit
    import torch
    dev = torch.device("cuda:0")
    m = O.Model(**SMALL)
    d = sana_dit.Dit(layers=2, hidden=128, ffn=256, caption_dim=96, latent_channels=8, self_heads=4, cross_heads=2)
    try:
        for name, shape in sana_dit.manifest(2, 128, 256, 96, 8).items():
            d.set_weight(name, m.get(name, shape))
        cap = torch.from_numpy(O.randn((2, 16, 96), 131)).to(dev)
        lat = torch.from_numpy(O.randn((1, 8, 8, 8), 132)).to(dev)
        out = torch.empty((2, 8, 8, 8), device=dev)

        def step():
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            d.step_device(cap, 16, None, lat, (1, 8, 8, 8), 999.0, out)
            torch.cuda.synchronize()
            return out.cpu().numpy()

        ref = step()
        with pytest.raises(sana_dit.SanaError) as e:  # 1.3 TB for the residual stream alone
            d.step_device(cap, 1, None, lat, (20000, 8, 255, 255), 999.0, out)
        assert e.value.code == sana_dit.SANA_ERR_OUT_OF_MEMORY
        with pytest.raises(sana_dit.SanaError) as e:
            d.forward_device(lat, (1, 8, 8, 8), 999.0, out)
        assert e.value.code == sana_dit.SANA_ERR_STATE
        assert np.array_equal(step(), ref)
    finally:
        d.close()
