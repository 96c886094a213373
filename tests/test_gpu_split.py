"""F32 products on the 16-bit matrix cores (operands in bf16 parts,
csrc/gemm_f32x6.hip) at the sizes where the tiles and taps can go wrong, and
over operands whose values differ widely in size."""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env(orc):
    from __graft_entry__ import ensure_built, load_tsk
    ensure_built()
    tsk = load_tsk()
    tsk.init(0)
    return tsk, orc


# channels in multiples of 32 that are not multiples of the 128-wide tiles
VAE = dict(latent_dim=32, channels=32, c_mults=[1, 2, 3, 3, 4], max_latent=64)


@pytest.fixture(scope="module")
def vae(env):
    tsk, orc = env
    v, ov = tsk.Vae(tsk.vae_config(**VAE)), orc.OracleVae(orc.vae_config(**VAE))
    for k, w in tsk.vae_synthetic_weights(v.tensors(), seed=5, snake_std=0.1).items():
        v.set_tensor(k, w)
        ov.set_tensor(k, w)
    yield v, ov
    v.close()


@pytest.mark.parametrize("T,scale", [(1, 1.0), (3, 1.0), (5, 2.0 ** -12)])
def test_vae_split(vae, T, scale):
    """one output tile and less, odd lengths, and a latent whose values are far
    below 1. Bound: the fp32 decode's 2e-4 (fp32 sums, amplified 50-100 times)"""
    v, ov = vae
    lat = (np.random.default_rng(T).standard_normal((32, T)) * scale).astype(np.float32)
    a, r = v.decode(lat), ov.decode(lat)
    e = rel_l2(a, r)
    print(f"VAE (32-channel groups) T={T} scale {scale:g}: rel-L2 {e:.3e}", flush=True)
    assert a.shape == (2, T * 2048) and e <= 2e-4
    assert np.array_equal(v.decode(lat), a)


def test_vae_split_nan_stays_local(vae):
    """a NaN latent frame reaches its receptive field (about 12 frames) only"""
    v, _ = vae
    lat = np.random.default_rng(9).standard_normal((32, 48)).astype(np.float32)
    ref = v.decode(lat)
    lat[3, 0] = np.nan
    a = v.decode(lat)
    assert np.isnan(a[:, :2048]).all()
    far = slice(20 * 2048, None)
    assert np.isfinite(a[:, far]).all() and rel_l2(a[:, far], ref[:, far]) <= 2e-4


@pytest.fixture(scope="module")
def copier(env):
    """a decoder that repeats its latent: unit kernels (every phase of a transposed convolution reads its own frame),
    zero residual units, SnakeBetas that add nothing (exp(alpha) = 0); 32 output channels"""
    tsk, _ = env
    v = tsk.Vae(tsk.vae_config(latent_dim=32, channels=32, c_mults=[1, 1, 1, 1, 1], out_channels=32, max_latent=8))
    for name, ne in v.tensors():
        w = np.zeros([int(n) for n in reversed(ne) if n > 1], np.float32)
        if name.endswith(".alpha"):
            w[:] = -1000
        elif w.ndim == 3 and w.shape[2] != 7:                          # stride s: taps s / 2 .. 3 s / 2 - 1
            s = w.shape[2] // 2
            w[np.arange(32), np.arange(32), s // 2:3 * s // 2] = 1
        elif name in ("decoder.layers.0.weight", "decoder.layers.7.weight"):
            w[np.arange(32), np.arange(32), 3] = 1
        v.set_tensor(name, w)
    yield v
    v.close()


def test_vae_keeps_every_bit(copier):
    """values that differ by 2^60 within a frame and from frame to frame come through all 36 convolutions as they are:
    no channel and no loud passage costs another one bits"""
    rng = np.random.default_rng(8)
    lat = (rng.standard_normal((32, 8)) * 2.0 ** rng.integers(-30, 30, (32, 8))).astype(np.float32)
    a = copier.decode(lat)
    assert np.array_equal(a, np.repeat(lat, copier.hop, 1))


def test_vae_snake_accuracy(copier):
    """v + sin^2(e^alpha v) e^-beta against 64 bits, arguments up to 2^18: sin^2 to 1.2e-7 (what the fp32 sinf gives)
    and the roundings of the product with e^-beta and of the sum"""
    libm = ctypes.CDLL("libm.so.6")
    libm.expf.restype, libm.expf.argtypes = ctypes.c_float, [ctypes.c_float]
    rng = np.random.default_rng(9)
    try:
        worst = 0.0
        for alpha, beta in [(0.0, 0.0), (0.0, -7.0), (5.0, -7.0), (11.0, -7.0)]:
            ea, eb = np.float32(libm.expf(alpha)), np.float32(libm.expf(-beta))
            copier.set_tensor("decoder.layers.6.alpha", np.full(32, alpha, np.float32))
            copier.set_tensor("decoder.layers.6.beta", np.full(32, beta, np.float32))
            for _ in range(8):
                lat = rng.uniform(-4, 4, (32, 8)).astype(np.float32)
                got = copier.decode(lat)[:, ::copier.hop].astype(np.float64)
                arg = (lat * ea).astype(np.float64)
                ref = lat + np.sin(arg) ** 2 * np.float64(eb)
                err = (np.abs(got - ref) - 2.0 ** -24 * (np.abs(ref) + np.float64(eb))) / np.float64(eb)
                worst = max(worst, float(err.max()))
        print(f"sin^2: max error {worst:.2e}", flush=True)
        assert worst <= 1.2e-7
    finally:
        copier.set_tensor("decoder.layers.6.alpha", np.full(32, -1000, np.float32))


# ---------------------------------------------------------------- F32 nodes
def rows_close(got, w, x, bound):
    """every output row against 64-bit products, relative to |w| |x| of its own row (its sum's condition):
    exact operands, products left out 2^-25, and sums of K terms in fp32"""
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    scale = np.sqrt(((np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T) ** 2).sum(-1))
    err = np.sqrt(((got - ref) ** 2).sum(-1)) / np.maximum(scale, 1e-300)
    print(f"rows: max error / |x||w| {err.max():.2e}", flush=True)
    return err.max() <= bound


@pytest.mark.parametrize("N,K,M", [(9, 32, 4), (63, 480, 132), (65, 1024, 128), (129, 2080, 64), (388, 4096, 96),
                                   (600, 512, 1028)])
def test_mul_mat_split(env, N, K, M):
    """remainders of every tile and of the K halves; rows and weights of very different size keep their own precision"""
    tsk, _ = env
    rng = np.random.default_rng(N + K)
    x = (rng.standard_normal((N, K)) * 2.0 ** rng.integers(-40, 40, (N, 1))).astype(np.float32)
    w = (rng.standard_normal((M, K)) * 2.0 ** rng.integers(-20, 20, (M, 1))).astype(np.float32)
    y = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    scale = 2.0 ** np.floor(np.log2(np.abs(w).max(-1)))           # columns to one size: an error of a small one shows
    assert rows_close(y / scale, w / scale[:, None], x, 2.0 ** -22)


@pytest.mark.parametrize("B,IW,IC,OC,KW,s0,p0,d0", [(2, 65, 160, 36, 3, 1, 1, 1), (3, 31, 96, 128, 7, 2, 3, 2),
                                                    (1, 130, 512, 64, 1, 1, 0, 1), (2, 40, 256, 8, 3, 1, 4, 1)])
def test_conv1d_split(env, B, IW, IC, OC, KW, s0, p0, d0):
    """one output sums input rows of different exponents: steps of 2^30 and more between neighbours, zero rows
    between them, batch items that must not see each other, padding wider than the kernel"""
    tsk, _ = env
    rng = np.random.default_rng(IW + OC)
    e = rng.integers(-35, 35, (B, IW, 1))
    x = (rng.standard_normal((B, IW, IC)) * 2.0 ** e).astype(np.float32)
    x[:, 5:8] = 0
    x[0, 20] *= 2.0 ** -60
    w = (rng.standard_normal((OC, IC, KW)) * 0.05).astype(np.float32)
    y = tsk.conv1d(tsk.to_device(w), tsk.to_device(x), None, s0, p0, d0).numpy().reshape(B, -1, OC)
    xp = np.zeros((B, IW + 2 * p0, IC), np.float32)
    xp[:, p0:p0 + IW] = x
    OW = (IW + 2 * p0 - d0 * (KW - 1) - 1) // s0 + 1
    cols = np.stack([xp[:, k * d0:k * d0 + (OW - 1) * s0 + 1:s0] for k in range(KW)], 2).reshape(B * OW, KW * IC)
    assert rows_close(y.reshape(B * OW, OC), w.transpose(0, 2, 1).reshape(OC, -1), cols, 2.0 ** -22)


def test_split_infinities(env):
    """infinities and NaN give what fp32 products give, and only in the rows and columns that hold them"""
    tsk, _ = env
    rng = np.random.default_rng(2)
    x, w = rng.standard_normal((70, 512)).astype(np.float32), rng.standard_normal((64, 512)).astype(np.float32)
    clean = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    # 1e37: its products (|w| < 6) and their sums stay below fp32's 3.4e38, so that
    # only the infinities make infinities, in fp32 as in 64 bits
    x[3, 7], x[4, 9], w[5, 11], x[6, 0] = np.inf, np.nan, -np.inf, 1e37
    y = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    with np.errstate(all="ignore"):
        ref = (x[:, None, :].astype(np.float64) * w[None]).sum(-1)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    odd = ~np.isfinite(ref)
    assert np.array_equal(y[odd & ~np.isnan(ref)], ref[odd & ~np.isnan(ref)].astype(np.float32))
    same = np.ones_like(odd)
    same[[3, 4, 6]] = False
    same[:, 5] = False
    assert np.array_equal(y[same], clean[same])


@pytest.mark.parametrize("p", [20, 30, 60])
def test_mul_mat_outlier(env, p):
    """one input column 2^p above the rest against zero weights: it may cost the others nothing. Bound: the sums'
    (2^-24 sqrt(K) of the terms at most)"""
    tsk, _ = env
    rng = np.random.default_rng(p)
    x, w = rng.standard_normal((70, 1024)).astype(np.float32), rng.standard_normal((132, 1024)).astype(np.float32)
    x[:, 7] *= 2.0 ** p
    w[:, 7] = 0
    y = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    assert rows_close(y, w, x, 2.0 ** -24)


def test_mul_mat_spread_undone_by_the_weights(env):
    """values of a row spread over 2^60 that the weights undo: every product counts the same"""
    tsk, _ = env
    rng = np.random.default_rng(4)
    e = rng.integers(-30, 31, 1024)
    x = (rng.standard_normal((70, 1024)) * 2.0 ** e).astype(np.float32)
    w = (rng.standard_normal((68, 1024)) * 2.0 ** -e).astype(np.float32)
    y = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    assert rows_close(y, w, x, 2.0 ** -24)


def test_mul_mat_copies_values(env):
    """against a unit matrix every value comes back, all 24 bits of it, whatever the rest of its row is, down to
    fp32's smallest normal numbers"""
    tsk, _ = env
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((100, 512)) * 2.0 ** rng.integers(-120, 100, (100, 512))).astype(np.float32)
    x[np.abs(x) < 2.0 ** -126] = 0
    assert np.array_equal(tsk.mul_mat(tsk.to_device(np.eye(512, dtype=np.float32)), tsk.to_device(x)).numpy(), x)


def test_mul_mat_tiny(env):
    """values so small that parts of them are flushed (2^-112 and less): sums in fp32"""
    tsk, _ = env
    rng = np.random.default_rng(7)
    x = (rng.standard_normal((40, 512)) * 2.0 ** -112).astype(np.float32)
    w = rng.standard_normal((64, 512)).astype(np.float32)
    y = tsk.mul_mat(tsk.to_device(w), tsk.to_device(x)).numpy()
    assert rows_close(y, w, x, 2.0 ** -23)


def test_conv1d_large_rows_beside_small_ones(env):
    """rows just outside an output's taps do not touch it, however much larger they are (2^170 over three rows here),
    and zero rows between them change nothing"""
    tsk, _ = env
    rng = np.random.default_rng(6)
    e = np.array([-100, -100, -50, -50, 120, 120, 0, -100, 0, 45, 45, -60])
    x = (rng.standard_normal((1, 12, 512)) * 2.0 ** e[None, :, None]).astype(np.float32)
    x[0, 8] = 0
    w = (rng.standard_normal((64, 512, 3)) * 0.05).astype(np.float32)
    y = tsk.conv1d(tsk.to_device(w), tsk.to_device(x)).numpy().reshape(12, 64)
    xp = np.concatenate([np.zeros((1, 512), np.float32), x[0], np.zeros((1, 512), np.float32)])
    cols = np.concatenate([xp[k:k + 12] for k in range(3)], 1)
    assert rows_close(y, w.transpose(0, 2, 1).reshape(64, -1), cols, 2.0 ** -23)


def test_f32_nodes_need_no_scratch(env):
    """F32 weights (kernels laid out kw-major): no workspace, and the same bits whatever is bound to the stream and
    when the call is captured"""
    tsk, _ = env
    rng = np.random.default_rng(3)
    x, w = rng.standard_normal((100, 512)).astype(np.float32), rng.standard_normal((64, 512)).astype(np.float32)
    xd, wd, y = tsk.to_device(x), tsk.to_device(w), tsk.empty((100, 64))
    assert tsk.workspace_size(tsk.OP_MUL_MAT, [wd, xd], y) == 0
    kd = tsk.to_device(np.ascontiguousarray(rng.standard_normal((32, 3, 128)).astype(np.float32)))
    kw, xc, yc = tsk.desc(kd, tsk.F32), tsk.to_device(x.reshape(1, 400, 128)), tsk.empty((1, 400, 32))
    kw.ne[0], kw.ne[1], kw.ne[2] = 3, 128, 32
    kw.nb[0], kw.nb[1], kw.nb[2], kw.nb[3] = 4 * 128, 4, 4 * 384, 4 * 384 * 32
    dx, dy = tsk.desc(xc, tsk.F32), tsk.desc(yc, tsk.F32)
    n = ctypes.c_size_t(1)
    srcs = (ctypes.POINTER(type(kw)) * 2)(ctypes.pointer(kw), ctypes.pointer(dx))
    tsk.check(tsk.load().tsk_workspace_size(tsk.OP_CONV1D, srcs, 2, ctypes.byref(dy), ctypes.byref(n)))
    assert n.value == 0
    tsk.mul_mat(wd, xd, out=y)
    tsk.synchronize()
    ref = y.numpy()
    s, buf = tsk.Stream(), tsk.empty((256,), "u8")
    tsk.set_workspace(buf, stream=s)
    tsk.mul_mat(wd, xd, out=y, stream=s)
    s.synchronize()
    assert np.array_equal(y.numpy(), ref)
    tsk.set_workspace(None, stream=s)
    g = tsk.Graph(s, lambda: tsk.mul_mat(wd, xd, out=y, stream=s))
    for _ in range(3):
        g.launch()
        s.synchronize()
        assert np.array_equal(y.numpy(), ref)
    g.destroy()
    s.destroy()
