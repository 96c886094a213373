"""F32 products on the fp16 matrix cores (split operands, csrc/gemm_split.hip)
at the sizes where the tiles, taps and exponents can go wrong."""
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
    below 1 (its exponent follows it). Bound: the fp32 decode's 2e-4 (products
    with an error of 2^-22 per term and fp32 sums, amplified 50-100 times)"""
    v, ov = vae
    lat = (np.random.default_rng(T).standard_normal((32, T)) * scale).astype(np.float32)
    a, r = v.decode(lat), ov.decode(lat)
    e = rel_l2(a, r)
    print(f"VAE (32-channel groups) T={T} scale {scale:g}: rel-L2 {e:.3e}", flush=True)
    assert a.shape == (2, T * 2048) and e <= 2e-4
    assert np.array_equal(v.decode(lat), a)


def test_vae_split_nan_stays_local(vae):
    """a NaN latent frame reaches its receptive field (about 12 frames) only:
    the exponents come from the finite values"""
    v, _ = vae
    lat = np.random.default_rng(9).standard_normal((32, 48)).astype(np.float32)
    ref = v.decode(lat)
    lat[3, 0] = np.nan
    a = v.decode(lat)
    assert np.isnan(a[:, :2048]).all()
    far = slice(20 * 2048, None)
    assert np.isfinite(a[:, far]).all() and rel_l2(a[:, far], ref[:, far]) <= 2e-4
