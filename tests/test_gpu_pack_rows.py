"""GPU test of tdbp_pack_samples at the edges of its loops (one sample, odd
pulses, a load group of 8192 samples and its neighbours), from and into buffers
that start one sample past an aligned address, with pulses on both sides of the
joining threshold, an all-zero pulse, an infinite component and a NaN."""
import numpy as np
import pytest

from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


def _store(v, dtype):
    """Stored values of float32 components, as float32."""
    if dtype == T.CF16:
        with np.errstate(over="ignore"):
            return v.astype(np.float16).astype(np.float32)
    if dtype == T.CBF16:
        u = v.view(np.uint32).astype(np.uint64)
        return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
    return np.clip(np.rint(v), -32767, 32767).astype(np.float32)


def _pack(x, dtype):
    """Stored components and scales: own scales, storage, then the call's."""
    c = np.stack([x.real, x.imag])
    mx = np.fmax.reduce(np.abs(c), axis=(0, 2), initial=0).astype(np.float32)
    own = np.zeros(len(mx), np.float32)
    shift = 14 if dtype == T.CI16 else 13
    ok = (mx > 0) & np.isfinite(mx)
    own[ok] = np.ldexp(np.float32(1), np.frexp(mx[ok])[1] - 1 - shift)
    own[np.isinf(mx)] = 1
    inv = np.where(own > 0, 1 / np.where(own > 0, own, 1), 0).astype(np.float32)[:, None]
    M = own.max()
    low = M / (16 if dtype == T.CI16 else 65536)
    with np.errstate(invalid="ignore"):
        q = _store(np.float32(c * inv), dtype)
    final = np.where((own > 0) & (own < low), own, M) if M else np.ones_like(own)
    for p in np.flatnonzero((own > 0) & (own != final)):
        q[:, p] = _store(np.float32(q[:, p] * (own[p] / final[p])), dtype)
    return q, final


@pytest.mark.parametrize("dtype", [T.CF16, T.CBF16, T.CI16])
@pytest.mark.parametrize("S,shift", [(1, 0), (2, 1), (7, 1), (2047, 0), (8191, 0), (8192, 1),
                                     (8193, 1), (18011, 0)])
def test_words_and_scales(gpu, dtype, S, shift):
    L = 9
    rng = np.random.default_rng(S)
    x = (rng.standard_normal((L, S)) + 1j * rng.standard_normal((L, S))).astype(np.complex64)
    x *= np.float32([1, 2, 0.3, 0, 1e-2, 1e-7, 5, 0.9, 1])[:, None]
    if dtype != T.CI16:   # an integer has no place for either
        x[7, S // 2] = np.nan
        x[8, S - 1] = -np.inf
    if S == 1:
        x[7] = 0.5
    buf = T.DeviceArray.from_host(np.concatenate([np.zeros(shift, np.complex64), x.ravel()]))
    words = T.DeviceArray((shift + L * S + 1,), np.uint32)
    words.zero()
    scale = T.DeviceArray((L,), np.float32)
    T.check(T.lib().tdbp_pack_samples(buf.ptr + 8 * shift, L, S, dtype, words.ptr + 4 * shift,
                                      scale.ptr, None))
    T.sync()
    w = words.download()
    assert w[-1] == 0 and not w[:shift].any()
    w = w[shift:shift + L * S].reshape(L, S)
    half = [(w & 0xFFFF).astype(np.uint16), (w >> 16).astype(np.uint16)]
    got = np.stack([h.view(np.float16).astype(np.float32) if dtype == T.CF16 else
                    (h.astype(np.uint32) << 16).view(np.float32) if dtype == T.CBF16 else
                    h.view(np.int16).astype(np.float32) for h in half])
    q, final = _pack(x, dtype)
    np.testing.assert_array_equal(scale.download(), final)
    np.testing.assert_array_equal(got, q)
