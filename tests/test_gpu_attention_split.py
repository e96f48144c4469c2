"""f32 attention on the bf16 matrix cores (head sizes up to 128), every value as three exact bf16 pieces, against float64."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def exact(q, k, v, scale, causal, z_bias=None, attn_bias=None):
    logits = (q.astype(np.float64) @ k.astype(np.float64).T) * scale
    if z_bias is not None:
        logits = logits + z_bias.astype(np.float64)[None]
    if attn_bias is not None:
        logits = logits + attn_bias.astype(np.float64)
    if causal:
        logits = np.where(np.tril(np.ones(logits.shape, bool)), logits, -np.inf)
    w = np.exp(logits - logits.max(axis=1, keepdims=True))
    return (w / w.sum(axis=1, keepdims=True)) @ v.astype(np.float64)


def run(hip, q, k, v, scale, causal, z_bias=None, attn_bias=None):
    contexts, seq, dim = q.shape
    up = lambda a: None if a is None else hip.DeviceBuffer.from_array(a)
    d_out = hip.DeviceBuffer.from_array(np.full(q.size + 64, 7.5, np.float32))
    keep = [up(a) for a in (q, k, v, z_bias, attn_bias)]
    hip.attention_f32_dev(contexts, seq, dim, scale, causal, *keep, d_out)
    hip.device_synchronize()
    out = d_out.to_array(np.float32, q.size + 64)
    assert (out[q.size:] == 7.5).all(), "wrote past the end of the result"
    return out[:q.size].reshape(q.shape)


# Query tiles of 128 and (from 256 workgroups on) of 256 rows, one key past a stage, short heads, biases on rows of any
# length (a row's last group of four keys reaches into the next row or past the tensor), keys split over workgroups.
@pytest.mark.parametrize("contexts,seq,dim,causal,biased", [
    (1, 1, 64, False, True), (2, 65, 64, True, False), (3, 129, 60, False, True), (2, 191, 36, True, True), (1, 777, 64, False, True),
    (5, 333, 32, False, False), (4, 1001, 64, True, True), (2, 1025, 20, False, True), (128, 513, 64, True, False), (90, 641, 64, False, False),
    (128, 385, 32, True, False), (86, 515, 64, False, True)])
def test_against_float64(hip, contexts, seq, dim, causal, biased):
    rng = np.random.default_rng(seq + dim)
    q, k, v = (rng.normal(size=(contexts, seq, dim)).astype(np.float32) for _ in range(3))
    zb = rng.normal(0, 0.5, (contexts, seq)).astype(np.float32) if biased else None
    ab = rng.normal(0, 0.5, (contexts, seq, seq)).astype(np.float32) if biased else None
    for scale in (1.0 / np.sqrt(dim), -0.3):
        got = run(hip, q, k, v, scale, causal, zb, ab)
        for c in sorted({0, contexts // 2, contexts - 1}):
            want = exact(q[c], k[c], v[c], float(np.float32(scale)), causal, None if zb is None else zb[c], None if ab is None else ab[c])
            # Logits of magnitude L (under 16 here) carry a few roundings of 2^-24·L, which the exponential turns into
            # relative errors of the weights; the weighted sum averages them.  A missing piece costs 2^-17 and more.
            error = got[c] - want
            assert np.sqrt(np.mean(error ** 2)) <= 2.0 ** -20 * np.sqrt(np.mean(want ** 2))
            assert np.abs(error).max() <= 2.0 ** -15


# Heads padded to 96 and 128 values: shared keys in one run (one tile a wavefront, two, wavefronts without any) and in runs, 128-row tiles
# unsplit, in pairs and with their keys cut, 32-key stages cut short; biases up to the longest that are served.
@pytest.mark.parametrize("contexts,seq,causal,biased", [
    (1, 1, False, False), (2, 31, True, False), (3, 33, False, True), (1, 128, True, True), (5, 129, False, False), (2, 255, True, False), (7, 257, False, True),
    (1, 300, True, False), (1, 768, False, True), (1, 769, False, True), (2, 776, True, True), (1, 800, False, True), (1, 832, True, True), (1, 833, True, True), (3, 1001, False, True), (16, 500, True, False), (40, 225, False, False), (70, 289, True, False), (33, 290, True, True)])
@pytest.mark.parametrize("dim", [68, 80, 96, 100, 128])
def test_wide_heads_against_float64(hip, contexts, seq, dim, causal, biased):
    assert hip.attention_f32_launch_plan(contexts, seq, dim, causal, biased, scale=dim ** -0.5)["kernel"] == "split" or (dim > 96 and biased and seq <= 32)
    test_against_float64(hip, contexts, seq, dim, causal, biased)


@pytest.mark.parametrize("contexts,seq", [(2, 150), (2, 400), (80, 260)])  # shared keys in one run and in several, 128-row tiles
@pytest.mark.parametrize("dim", [80, 128])
def test_wide_heads_the_pieces_cannot_carry(hip, contexts, seq, dim):
    rng = np.random.default_rng(dim + seq)
    q, k, v = (rng.normal(size=(contexts, seq, dim)).astype(np.float32) for _ in range(3))
    q[0, 5] *= np.float32(2.0 ** 45)
    k[0, :6] *= np.float32(2.0 ** -45)
    v[1, 40, dim - 1] = np.inf
    got = run(hip, q, k, v, dim ** -0.5, True)
    assert np.abs(got[0] - exact(q[0], k[0], v[0], float(np.float32(dim ** -0.5)), True)).max() <= 2.0 ** -15
    assert not np.isfinite(got[1, 40:, dim - 1]).any() and np.isfinite(got[1, :40]).all() and np.isfinite(got[1, :, :dim - 1]).all()


# keys in as many runs as are no multiple of eight (the merging loads eight at a time): shared keys and 128-row tiles, and on the f32
# matrix cores (a large scale)
@pytest.mark.parametrize("contexts,seq,dim,causal,biased,scale", [
    (1, 700, 80, False, True, None), (1, 700, 128, True, True, None), (1, 890, 64, False, True, None), (2, 400, 96, False, False, None), (3, 1500, 64, True, False, None),
    (4, 1700, 80, False, True, None), (1, 600, 64, False, True, 0.6), (1, 1200, 128, False, False, 0.5)])
def test_infinite_values_in_the_last_run_of_keys(hip, contexts, seq, dim, causal, biased, scale):
    scale = dim ** -0.5 if scale is None else scale
    assert hip.attention_f32_launch_plan(contexts, seq, dim, causal, biased, scale=scale)["key_splits"] % 8 > 0
    rng = np.random.default_rng(seq + dim)
    q, k, v = (rng.normal(size=(contexts, seq, dim)).astype(np.float32) * 0.5 for _ in range(3))
    z, a = (rng.normal(size=shape).astype(np.float32) * 0.5 if biased else None for shape in ((contexts, seq), (contexts, seq, seq)))
    want = run(hip, q, k, v, scale, causal, z, a)
    v[0, seq - 1, dim - 1], v[0, seq - 2, 0] = np.inf, -np.inf
    got = run(hip, q, k, v, scale, causal, z, a)
    assert np.abs(got[0, :, 1:dim - 1] - want[0, :, 1:dim - 1]).max() <= 2.0 ** -14  # either is within 2^-15 of the exact one (above)
    sees = np.arange(seq) if causal else np.full(seq, seq)
    assert (got[0, sees >= seq - 1, dim - 1] == np.inf).all() and np.isfinite(got[0, sees < seq - 1, dim - 1]).all()
    assert (got[0, sees >= seq - 2, 0] == -np.inf).all() and np.isfinite(got[0, sees < seq - 2, 0]).all()
    assert np.isfinite(got[1:]).all()


# shared keys in one run and in several, 128-row tiles; every other pair masked, the last keys of all queries, the keys of a whole run, all keys of
# some queries (zeros, as on the general kernel)
@pytest.mark.parametrize("contexts,seq,causal", [(2, 150, False), (1, 500, True), (1, 700, False), (16, 500, False), (33, 290, True), (4, 1200, False)])
@pytest.mark.parametrize("dim", [64, 80, 128])
@pytest.mark.parametrize("masked", [-np.inf, np.finfo(np.float32).min])
def test_masked_pairs(hip, contexts, seq, dim, causal, masked):
    assert hip.attention_f32_launch_plan(contexts, seq, dim, causal, True, scale=dim ** -0.5)["kernel"] == "split"
    rng = np.random.default_rng(seq + dim)
    q, k, v = (rng.normal(size=(contexts, seq, dim)).astype(np.float32) for _ in range(3))
    zb, ab = (rng.normal(0, 0.5, shape).astype(np.float32) for shape in ((contexts, seq), (contexts, seq, seq)))
    ab[:, 0::2, 1::2] = ab[:, 1::2, 0::2] = masked
    zb[:, seq - 20:] = masked
    if seq > 260:
        zb[:, 128:256] = masked
    nothing = np.zeros(seq, bool)
    if masked == -np.inf:
        nothing[[3, 40, seq - 2]] = True
        ab[:, nothing] = -np.inf
    got = run(hip, q, k, v, dim ** -0.5, causal, zb, ab)
    assert (got[:, nothing] == 0.0).all()
    for c in sorted({0, contexts - 1}):
        with np.errstate(invalid="ignore"):
            want = exact(q[c], k[c], v[c], float(np.float32(dim ** -0.5)), causal, zb[c], ab[c])
        error = (got[c] - want)[~nothing]
        assert np.sqrt(np.mean(error ** 2)) <= 2.0 ** -20 * np.sqrt(np.mean(want[~nothing] ** 2)) and np.abs(error).max() <= 2.0 ** -15


def test_values_the_pieces_cannot_carry(hip):
    rng = np.random.default_rng(9)
    q, k, v = (rng.normal(size=(4, 300, 64)).astype(np.float32) for _ in range(3))
    clean = run(hip, q, k, v, 0.125, True)
    q2, k2, v2 = q.copy(), k.copy(), v.copy()
    k2[0, 290] = -np.inf          # seen by the last rows only: weight 0 or NaN, as in f32 arithmetic
    q2[0, 290:] = np.abs(q2[0, 290:])
    v2[1, 40, 3] = np.inf
    v2[2, :, 7] *= np.float32(2.0 ** -121)
    q2[3, 5] *= np.float32(2.0 ** 45)
    k2[3, :6] *= np.float32(2.0 ** -45)
    got = run(hip, q2, k2, v2, 0.125, True)
    assert np.isfinite(got[0, :290]).all() and (got[0, :256] == clean[0, :256]).all() and np.isfinite(got[0, 290:]).all()
    want = exact(q2[0, 290:291], k2[0, :290], v2[0, :290], 0.125, False)
    assert np.abs(got[0, 290] - want[0]).max() <= 2.0 ** -15
    assert not np.isfinite(got[1, 40:, 3]).any() and np.isfinite(got[1, :40]).all() and np.isfinite(np.delete(got[1], 3, axis=1)).all()
    want = exact(q2[2], k2[2], v2[2], 0.125, True)
    assert (np.abs(got[2, :, 7] - want[:, 7]) <= 2.0 ** -18 * 2.0 ** -119).all()  # its own magnitude, not that of the other columns
    assert np.abs(got[2] - want).max() <= 2.0 ** -15
    want = exact(q2[3], k2[3], v2[3], 0.125, True)
    assert np.abs(got[3] - want).max() <= 2.0 ** -15


@pytest.mark.parametrize("contexts,seq", [(4, 300), (128, 513)])  # 128 and 256 query rows a workgroup
@pytest.mark.parametrize("dim", [32, 64])
def test_small_probabilities_and_values_keep_their_bits(hip, contexts, seq, dim):
    """A key of probability 2^-124 / (seq - 1) holds the only non-zero entry of a column of V; another column is subnormal
    beside large entries of negligible weight."""
    rng = np.random.default_rng(13)
    q, k, v = (np.zeros((contexts, seq, dim), np.float32) for _ in range(3))
    q[..., 0] = 2.0
    k[:, 7, 0] = -86.0  # logit -86, all others 0: every product and sum of them is exact
    v[:, 7, 3] = rng.uniform(1e15, 1e17, contexts)
    v[..., 5] = rng.uniform(1e-39, 1e-38, (contexts, seq))
    v[:, 7, 5] = 1.0
    v[..., 9] = rng.normal(size=(contexts, seq))
    got = run(hip, q, k, v, 0.5, False)
    for c in (0, contexts // 2, contexts - 1):
        want = exact(q[c], k[c], v[c], 0.5, False)
        # the logit in log2 units is rounded at 124 (twice) and log2(e) before it: 3 · 2^-18 · ln 2, and sums of seq terms
        assert np.abs(got[c, :, 3] / want[:, 3] - 1.0).max() <= 1e-5
        # an f32 result of 1e-39 is a multiple of 2^-149; weighted sums of the entries round no more than seq times 2^-24
        assert np.abs(got[c, :, 5] - want[:, 5]).max() <= 2.0 ** -149 + seq * 2.0 ** -24 * 1e-38
        assert np.abs(got[c, :, 9] - want[:, 9]).max() <= 2.0 ** -20


@pytest.mark.parametrize("contexts,seq,dim,causal,biased", [
    (1, 1, 64, False, True), (2, 65, 64, True, False), (3, 129, 60, False, True), (2, 191, 36, True, True), (1, 777, 64, False, True),
    (5, 333, 32, False, False), (4, 1001, 64, True, True), (2, 1025, 20, False, True), (128, 513, 64, True, False), (90, 641, 64, False, False)])
def test_redone_rows_against_float64(hip, contexts, seq, dim, causal, biased):
    """Every query holds a value of 2^41 that meets zeros in K: no logit depends on it, but every workgroup sums in f32."""
    rng = np.random.default_rng(seq + dim)
    q, k, v = (rng.normal(size=(contexts, seq, dim)).astype(np.float32) for _ in range(3))
    q[..., 1] = 2.0 ** 41
    k[..., 1] = 0.0
    zb = rng.normal(0, 0.5, (contexts, seq)).astype(np.float32) if biased else None
    ab = rng.normal(0, 0.5, (contexts, seq, seq)).astype(np.float32) if biased else None
    for scale in (1.0 / np.sqrt(dim), -0.3):
        got = run(hip, q, k, v, scale, causal, zb, ab)
        for c in sorted({0, contexts // 2, contexts - 1}):
            want = exact(q[c], k[c], v[c], float(np.float32(scale)), causal, None if zb is None else zb[c], None if ab is None else ab[c])
            error = got[c] - want  # the bounds of the test above; f32 sums of `dim` and `seq` terms stay within them
            assert np.sqrt(np.mean(error ** 2)) <= 2.0 ** -20 * np.sqrt(np.mean(want ** 2))
            assert np.abs(error).max() <= 2.0 ** -15


def test_redone_rows_take_the_matrix_cores(hip):
    """About five times the ordinary time where every workgroup redoes its rows (a chain of multiply-adds per row: 20 to 45)."""
    n = 128 * 1024 * 64
    data = np.random.default_rng(1).normal(size=n).astype(np.float32)
    wild = data.copy()
    wild[::64] = 2.0 ** 41
    d_q, d_wild, d_out = (hip.DeviceBuffer.from_array(a) for a in (data, wild, data))
    for causal in (False, True):
        def best(d_k):
            times = []
            for _ in range(5):
                start = time.perf_counter()
                hip.attention_f32_dev(128, 1024, 64, 0.125, causal, d_q, d_k, d_q, None, None, d_out)
                hip.device_synchronize()
                times.append(time.perf_counter() - start)
            return min(times)

        assert best(d_wild) <= 15 * best(d_q)


# Keys shared by eight wavefronts of 32-row workgroups: its first and last sequences, wavefronts without keys, a run short of a tile,
# runs of keys put together by a second launch (rows that see none of a run), a grid of exactly one round and the first beyond it.
@pytest.mark.parametrize("contexts,seq,dim,causal,biased", [
    (1, 32, 64, True, False), (1, 33, 64, True, True), (3, 63, 20, False, True), (2, 97, 64, True, False), (1, 255, 64, False, True),
    (4, 256, 32, True, False), (1, 289, 60, True, True), (3, 385, 64, True, False), (1, 1000, 32, True, True), (2, 999, 64, False, True),
    (32, 256, 64, True, False), (33, 256, 64, True, False), (7, 1024, 64, False, False)])
def test_keys_shared_by_the_wavefronts(hip, contexts, seq, dim, causal, biased):
    test_against_float64(hip, contexts, seq, dim, causal, biased)
