"""The split-bf16 forward (attn_fwd_kernel) where it can go wrong: lengths
around its key tiles and query blocks in each launch form (4 or 8 waves, one
block, two at once, two in turn), values that the split cannot carry, operands
of every magnitude, and its error against float64 next to the fp32
instruction's."""

import numpy as np
import pytest

import gpu_helpers as G

pytestmark = pytest.mark.gpu


def _ref(q, k, v, causal, scale=None):
    """float64 O and LSE of (S, D) operands; a score of -inf is a weight of 0."""
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    S, D = q.shape
    with np.errstate(invalid="ignore", over="ignore"):
        s = q @ k.T * np.float64(np.float32(1 / np.sqrt(D) if scale is None else scale))
    if causal:
        s[np.triu(np.ones((S, S), bool), 1)] = -np.inf
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    tot = p.sum(-1, keepdims=True)
    return p @ v / tot, (m + np.log(tot))[:, 0]


def _qkv(H, S, D, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((1, H, S, D), dtype=np.float32) for _ in range(3)]


def _check(q, k, v, causal, heads, log=None):
    o, lse = G.attention_fwd(q, k, v, causal, log=log)
    for h in heads:
        ro, rl = _ref(q[0, h], k[0, h], v[0, h], causal)
        np.testing.assert_allclose(o[0, h], ro, rtol=1e-3, atol=2e-4)
        np.testing.assert_allclose(lse[0, h], rl, rtol=1e-3, atol=2e-4)
    return o, lse


@pytest.mark.parametrize("H,S,D,causal", [
    # 4 waves, one block: one key past a tile, one short of it, one past a block
    (70, 129, 32, False), (70, 191, 32, True), (70, 129, 64, False), (66, 257, 64, False),
    (70, 159, 128, False), (66, 161, 128, True), (65, 255, 128, False), (65, 960, 64, True),
    # 8 waves, one block
    (300, 129, 128, False), (260, 257, 64, False), (300, 385, 32, True), (130, 511, 128, False),
    # two blocks at once: even and odd counts, a last block of one row
    (40, 513, 64, True), (64, 641, 128, True), (30, 385, 32, True), (64, 960, 64, True),
    # two blocks in turn
    (256, 512, 64, True), (256, 400, 128, True),
])
def test_lengths_and_launch_forms(H, S, D, causal):
    q, k, v = _qkv(H, S, D, H + S + D)
    log = []
    _check(q, k, v, causal, (0, H // 2, H - 1), log)
    assert log[0].startswith("attn_fwd_kernel"), log


FORMS = [(70, 200, 64, False), (70, 200, 128, True), (300, 300, 128, True), (40, 640, 64, True)]


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_infinite_keys_get_no_weight(H, S, D, causal):
    """K holding -inf (times positive q) gives scores of -inf: weight 0."""
    q, k, v = _qkv(H, S, D, 1)
    q[..., 0] = np.abs(q[..., 0]) + 0.1
    k[0, 3, 40:50, 0] = -np.inf
    k[0, H - 1, S - 1, 0] = -np.inf
    _check(q, k, v, causal, (0, 3, H - 1))


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_infinite_values(H, S, D, causal):
    """An infinite V element makes its column infinite for the rows that see
    it and changes nothing else."""
    q, k, v = _qkv(H, S, D, 2)
    v[0, 9, 33, 4] = np.inf
    o, _ = G.attention_fwd(q, k, v, causal)
    finite = np.where(np.isinf(v[0, 9]), 0, v[0, 9])
    ro, _ = _ref(q[0, 9], k[0, 9], finite, causal)
    sees = np.arange(S) >= (33 if causal else 0)
    # Masked keys of the same 32-key tile: 0 * inf is NaN, as with the fp32 instruction.
    far = np.arange(S) < 32 if causal else np.zeros(S, bool)
    assert np.isposinf(o[0, 9, sees, 4]).all()
    cols = np.arange(D) != 4
    np.testing.assert_allclose(o[0, 9][:, cols], ro[:, cols], rtol=1e-3, atol=2e-4)
    np.testing.assert_allclose(o[0, 9, far, 4], ro[far, 4], rtol=1e-3, atol=2e-4)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("exponent", [-100, -120])
def test_tiny_values_keep_their_precision(H, S, D, causal, exponent):
    """V below what three bf16 parts can hold without a scale: O to fp32
    precision relative to V's size."""
    q, k, v = _qkv(H, S, D, 3)
    v *= np.float32(2.0 ** exponent)
    o, _ = G.attention_fwd(q, k, v, causal)
    for h in (0, H - 1):
        ro, _ = _ref(q[0, h], k[0, h], v[0, h], causal)
        np.testing.assert_allclose(o[0, h] * 2.0 ** -exponent, ro * 2.0 ** -exponent, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("eq,ek,es", [(-122, 122, 0), (122, -122, 0), (-120, 40, 80), (40, -130, 90), (-60, -60, 120),
                                      (100, -140, 40), (60, 40, -100), (20, 20, -40)])
def test_scores_of_small_and_large_operands(H, S, D, causal, eq, ek, es):
    """Q and K of 2^eq and 2^ek, denormal ones too, which the scale 2^es
    brings back to ordinary scores: O and LSE to fp32 precision."""
    q, k, v = _qkv(H, S, D, 5)
    q, k, scale = np.ldexp(q, eq), np.ldexp(k, ek), np.ldexp(1 / np.sqrt(D), es)
    o, lse = G.attention_fwd(q, k, v, causal, scale)
    for h in (0, H - 1):
        ro, rl = _ref(q[0, h], k[0, h], v[0, h], causal, scale)
        # A score is the sum of D products of a few units: 2^-24 of some D.
        np.testing.assert_allclose(o[0, h], ro, rtol=0, atol=2.0 ** -22 * np.sqrt(D))
        np.testing.assert_allclose(lse[0, h], rl, rtol=0, atol=2.0 ** -22 * np.sqrt(D))


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("exponent", [-112, -120, -125])
def test_tiny_values_beside_large_ones_of_no_weight(H, S, D, causal, exponent):
    """Small V rows keep their precision next to large ones that a query gives
    no weight, or (causal) does not see."""
    q, k, v = _qkv(H, S, D, 6)
    v *= np.float32(2.0 ** exponent)
    q[..., 0], k[..., 0] = 8, 0
    k[:, :, 20:S:7, 0] = -2000                         # weight exp(-1400) at most: 0
    v[:, :, 20:S:7] = 1e6
    o, _ = G.attention_fwd(q, k, v, causal)
    for h in (0, H - 1):
        ro, _ = _ref(q[0, h], k[0, h], v[0, h], causal)
        size, _ = _ref(q[0, h], k[0, h], np.abs(v[0, h]), causal)
        assert (np.abs(o[0, h] - ro) <= 1e-5 * size + 2.0 ** -148).all()


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_tiny_weights_of_large_values(H, S, D, causal):
    """Weights of exp(-86), 2^-124, beside one of 1 whose V is 0."""
    q, k, v = (np.zeros((1, H, S, D), np.float32) for _ in range(3))
    rng = np.random.default_rng(7)
    q[..., 0] = np.sqrt(D)
    k[:, :, 1:, 0] = rng.uniform(-86.4, -85, (1, H, S - 1)).astype(np.float32)
    v[:, :, 1:] = np.ldexp(rng.uniform(-1, 1, (1, H, S - 1, D)).astype(np.float32), 60)
    o, _ = G.attention_fwd(q, k, v, causal)
    for h in (0, H - 1):
        ro, _ = _ref(q[0, h], k[0, h], v[0, h], causal)
        size, _ = _ref(q[0, h], k[0, h], np.abs(v[0, h]), causal)
        # The exponent, about 124 in base 2, has an ulp of 2^-17: 2^-18 ln 2
        # each in the product with the scale and in the sum with the maximum.
        assert (np.abs(o[0, h] - ro) <= 2.0 ** -17 * size).all()


@pytest.mark.parametrize("H,S,D,causal,o_err,lse_err", [
    (80, 2048, 64, True, 4.2e-7, 5.9e-8), (130, 1024, 128, True, 4.0e-7, 5.6e-8), (30, 777, 128, False, 6.8e-7, 5.4e-8),
    (130, 600, 32, False, 5.5e-7, 5.6e-8)])
def test_error_no_larger_than_the_fp32_instructions(H, S, D, causal, o_err, lse_err):
    """Relative 2-norm error against float64 below what the kernel on the
    fp32 matrix instruction measured (its O errors, rounded up)."""
    q, k, v = _qkv(H, S, D, 4)
    o, lse = G.attention_fwd(q, k, v, causal)
    ro, rl = zip(*(_ref(q[0, h], k[0, h], v[0, h], causal) for h in (0, 1)))
    assert np.linalg.norm(o[0, :2] - np.stack(ro)) / np.linalg.norm(ro) <= o_err
    assert np.linalg.norm(lse[0, :2] - np.stack(rl)) / np.linalg.norm(rl) <= lse_err
