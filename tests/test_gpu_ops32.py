"""fp32 op-level kernels (sana_op_*) against 64-bit numpy, at the edges of their
tiles, vector widths and dispatch rules.  Bounds are first-order forward error
bounds in u = 2^-24: a dot product of K terms in any order is off by at most
(K + c) u sum |a b|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
U = 2.0 ** -24


@pytest.fixture(scope="module")
def L():
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible to torch")
    import sana_dit
    return sana_dit


def up(a, offset=0):
    """Device copy whose data starts `offset` floats past a 16-byte boundary."""
    t = torch.zeros(a.size + offset, device="cuda")
    t[offset:] = torch.from_numpy(np.ascontiguousarray(a)).reshape(-1).to("cuda")
    return t[offset:]


def down(t, shape):
    torch.cuda.synchronize()
    return t.cpu().numpy().astype(np.float64).reshape(shape)


# M, N, K, batch, transposed B, row padding of A / B / C, float offset of the bases, bias mode, accumulate
GEMMS = [
    (1, 1, 1, 1, 0, 0, 0, 0, 0), (64, 64, 32, 1, 0, 0, 0, 1, 0), (65, 63, 33, 1, 1, 0, 0, 2, 0),
    (256, 300, 72, 3, 1, 0, 0, 0, 0), (256, 72, 300, 3, 0, 0, 0, 0, 1), (130, 68, 100, 2, 0, 4, 0, 1, 1),
    (130, 68, 100, 2, 1, 4, 0, 2, 0), (100, 70, 36, 1, 0, 1, 0, 1, 0), (100, 70, 36, 1, 1, 0, 1, 1, 0),
    (33, 129, 31, 1, 0, 0, 3, 0, 0), (2048, 1152, 1152, 1, 0, 0, 0, 1, 0), (600, 1152, 64, 1, 1, 0, 0, 1, 0),
    (1000, 64, 33, 7, 0, 3, 2, 2, 1), (5, 4, 0, 1, 0, 4, 0, 1, 0),
    (65, 63, 49, 1, 0, 0, 0, 2, 0), (70, 67, 16, 2, 0, 0, 1, 1, 1), (200, 101, 17, 2, 1, 1, 0, 2, 1),
    (131, 97, 48, 1, 1, 0, 0, 0, 1), (4090, 1151, 300, 1, 0, 1, 0, 1, 1), (4090, 1151, 80, 1, 0, 0, 0, 2, 0),
    (4090, 1152, 40, 1, 0, 0, 0, 1, 0), (4090, 1150, 44, 1, 1, 0, 1, 2, 1), (4090, 1152, 48, 1, 1, 0, 0, 2, 1),
    (1030, 1152, 40, 1, 0, 0, 0, 1, 0), (1030, 1150, 44, 1, 1, 0, 1, 2, 1), (1031, 1154, 33, 1, 0, 2, 0, 1, 0),
]


@pytest.mark.parametrize("M,N,K,batch,bt,pad,off,bias_mode,acc", GEMMS)
def test_gemm_f32(L, M, N, K, batch, bt, pad, off, bias_mode, acc):
    r = np.random.default_rng(M + 3 * N + 7 * K)
    lda, ldb, ldc = K + pad, (K if bt else N) + pad, N + pad
    rows = N if bt else K
    A, B = (r.standard_normal((batch, n, ld), dtype=np.float32) for n, ld in ((M, lda), (rows, ldb)))
    C = r.standard_normal((batch, M, ldc), dtype=np.float32)
    bias = r.standard_normal(M if bias_mode == 2 else N, dtype=np.float32) if bias_mode else None
    dA, dB, dC = up(A, off), up(B, off), up(C, off)
    db = up(bias) if bias_mode else None
    L.check(L.lib().sana_op_gemm_f32(L.ptr(dA) or dC.data_ptr(), lda, M * lda, L.ptr(dB) or dC.data_ptr(), ldb,
                                     rows * ldb, bt, L.ptr(db), bias_mode or 1, dC.data_ptr(), ldc, M * ldc, M, N, K,
                                     batch, acc, None))
    got = down(dC, (batch, M, ldc))
    a = A[:, :, :K].astype(np.float64)
    b = (B[:, :, :K].transpose(0, 2, 1) if bt else B[:, :, :N]).astype(np.float64)
    ref, mag = a @ b, np.abs(a) @ np.abs(b)
    if bias_mode:
        add = (bias[:, None] if bias_mode == 2 else bias[None, :]).astype(np.float64)
        ref, mag = ref + add, mag + np.abs(add)
    if acc:
        ref, mag = ref + C[:, :, :N], mag + np.abs(C[:, :, :N])
    assert (np.abs(got[:, :, :N] - ref) <= (K + 4) * U * mag).all()
    assert np.array_equal(got[:, :, N:], C[:, :, N:].astype(np.float64))  # row padding untouched


def test_gemm_f32_nonfinite(L):
    """An infinity reaches exactly its row, a NaN too."""
    A, B = np.ones((70, 40), np.float32), np.ones((40, 66), np.float32)
    A[3, 39], A[65, 0] = np.inf, np.nan
    dA, dB, dC = up(A), up(B), torch.zeros(70 * 66, device="cuda")
    L.check(L.lib().sana_op_gemm_f32(dA.data_ptr(), 40, 0, dB.data_ptr(), 66, 0, 0, None, 1, dC.data_ptr(), 66, 0, 70,
                                     66, 40, 1, 0, None))
    got = down(dC, (70, 66))
    assert np.isposinf(got[3]).all() and np.isnan(got[65]).all()
    assert (np.delete(got, [3, 65], 0) == 40).all()


@pytest.mark.parametrize("BH,Nq,Nk,D", [(1, 1, 1, 4), (3, 17, 15, 16), (2, 100, 0, 32), (72, 1024, 1024, 32),
                                        (5, 33, 1000, 32), (2, 4096, 777, 72), (32, 529, 529, 72), (2, 40, 300, 80),
                                        (36, 4, 4, 32), (2, 5, 4, 72), (3, 4, 5, 32),
                                        (3, 64, 64, 48), (2, 50, 60, 84), (2, 50, 60, 30), (1, 300, 4096, 64)])
@pytest.mark.parametrize("alias", [False, True])
def test_linear_attention_f32(L, BH, Nq, Nk, D, alias):
    if alias and Nq != Nk:
        pytest.skip("in place only where out has v's shape")
    r = np.random.default_rng(BH + Nq + D)
    q, k, v = (r.standard_normal((BH, n, D), dtype=np.float32) for n in (Nq, Nk, Nk))
    dq, dk, dv = up(q), up(k), up(v)
    keep = torch.zeros(4, device="cuda")
    dk, dv = (dk if Nk else keep), (dv if Nk else keep)
    out = dv if alias else torch.zeros(BH * Nq * D, device="cuda")
    st = torch.zeros(BH * (D + 1) * D, device="cuda")
    L.check(L.lib().sana_op_linear_attention_f32(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), out.data_ptr(), BH, Nq,
                                                 Nk, D, st.data_ptr(), None))
    got = down(out, (BH, Nq, D))
    q, k, v = np.maximum(q, 0).astype(np.float64), np.maximum(k, 0).astype(np.float64), v.astype(np.float64)
    S, ks = np.einsum("btr,btd->brd", v, k), k.sum(1)
    den = np.einsum("btd,bd->bt", q, ks)[:, :, None] + 1e-15
    ref = np.einsum("brd,btd->btr", S, q) / den
    mag = np.einsum("brd,btd->btr", np.einsum("btr,btd->brd", np.abs(v), k), q) / den
    # numerator and denominator each carry a sum over tokens and one over channels
    assert (np.abs(got - ref) <= (2 * (Nk + D) + 8) * U * (mag + np.abs(ref))).all()


@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 64), (6, 65), (7, 128), (9, 129), (33, 300), (4, 512), (5, 513),
                                       (3, 2048), (2, 2049)])
@pytest.mark.parametrize("masked", [False, True])
def test_softmax_f32(L, rows, cols, masked):
    r = np.random.default_rng(rows + cols)
    x = r.standard_normal((rows, cols), dtype=np.float32) * 4
    bias = np.where(r.random((rows, cols)) < 0.3, np.finfo(np.float32).min, 0).astype(np.float32) if masked else None
    d = up(x)
    db = up(bias) if masked else None
    L.check(L.lib().sana_op_softmax_f32(d.data_ptr(), d.data_ptr(), rows, cols, 0.25, L.ptr(db), 1, None))
    got = down(d, (rows, cols))
    s = x.astype(np.float64) * 0.25 + (bias if masked else 0)
    e = np.exp(s - s.max(1, keepdims=True))
    ref = e / e.sum(1, keepdims=True)
    # the exponent's argument is off by at most 3 u max |s|, the sum by cols u, expf by a few u
    fin = np.abs(np.where(s > -1e30, s, 0)).max(1, keepdims=True)
    assert (np.abs(got - ref) <= (cols + 16 + 6 * fin) * U * ref + 1e-37).all()


@pytest.mark.parametrize("B,N,H,D,off", [(2, 7, 3, 8, 0), (1, 5, 16, 72, 0), (2, 3, 5, 6, 0), (3, 4, 2, 4, 1),
                                         (1, 1, 1, 1, 0), (2, 300, 36, 32, 0)])
def test_heads_f32(L, B, N, H, D, off):
    x = np.random.default_rng(B + N).standard_normal((B, N, H, D), dtype=np.float32)
    d, y, z = up(x, off), up(np.zeros(x.size, np.float32), off), up(np.zeros(x.size, np.float32), off)
    L.check(L.lib().sana_op_heads_f32(d.data_ptr(), y.data_ptr(), B, N, H, D, 1, None))
    L.check(L.lib().sana_op_heads_f32(y.data_ptr(), z.data_ptr(), B, N, H, D, 0, None))
    assert np.array_equal(down(y, (B, H, N, D)), x.transpose(0, 2, 1, 3))
    assert np.array_equal(down(z, (B, N, H, D)), x)


def test_gemm_f32_widest_row(L):
    """2^29 columns and more: 32-column tiles would need 2^32 threads in a launch."""
    n = (1 << 29) + 37
    a = torch.full((1,), 1.5, device="cuda")
    b = torch.arange(n, device="cuda", dtype=torch.float32)
    c = torch.full((n,), float("nan"), device="cuda")
    torch.cuda.synchronize()
    L.check(L.lib().sana_op_gemm_f32(a.data_ptr(), 1, 0, b.data_ptr(), n, 0, 0, None, 1, c.data_ptr(), n, 0, 1, n, 1,
                                     1, 0, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(c, b.mul_(1.5))
