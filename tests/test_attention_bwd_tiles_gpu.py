"""The split-bf16 backward (attn_bwd_kernel) where it can go wrong: lengths
around its key and query blocks, the rule that chooses it at D = 64, values
that the split cannot carry, operands of every magnitude, and its error
against float64 next to the fp32 instruction's."""

import numpy as np
import pytest

import gpu_helpers as G
from ember_amd import capi

pytestmark = pytest.mark.gpu


def _ref(q, k, v, do, causal, scale=None):
    """float64 O, LSE, dQ, dK, dV of (S, D) operands."""
    q, k, v, do = (x.astype(np.float64) for x in (q, k, v, do))
    S, D = q.shape
    scale = np.float64(np.float32(1 / np.sqrt(D) if scale is None else scale))
    s = q @ k.T * scale
    if causal:
        s[np.triu(np.ones((S, S), bool), 1)] = -np.inf
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    tot = p.sum(-1, keepdims=True)
    p /= tot
    o = p @ v
    ds = p * (do @ v.T - (do * o).sum(-1, keepdims=True))
    return o, (m + np.log(tot))[:, 0], scale * ds @ k, scale * ds.T @ q, p.T @ do


def _data(H, S, D, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((1, H, S, D), dtype=np.float32) for _ in range(4)]


def _backward(q, k, v, do, causal, heads, scale=None):
    """The kernel's gradients, with O and LSE from the reference at `heads`
    (zero elsewhere: nothing is read across heads), the references and the log."""
    o, lse = np.zeros_like(q), np.zeros(q.shape[:3], np.float32)
    refs = []
    for h in heads:
        r = _ref(q[0, h], k[0, h], v[0, h], do[0, h], causal, scale)
        o[0, h], lse[0, h] = r[0], r[1]
        refs.append(r[2:])
    log = []
    got = G.attention_bwd(q, k, v, o, lse, do, causal, scale, log=log)
    return got, refs, log


def _check(got, refs, heads, unit=1.0, rtol=1e-3, atol=2e-4):
    for h, ref in zip(heads, refs):
        for name, g, r in zip(("dq", "dk", "dv"), got, ref):
            np.testing.assert_allclose(g[0, h] * np.float64(unit), r * unit, rtol=rtol, atol=atol, err_msg=f"{name} head {h}")


@pytest.mark.parametrize("H,S,D,causal", [
    # one past, at and one short of a key block, a query block and both
    (3, 129, 128, False), (3, 159, 128, True), (2, 160, 128, False), (3, 161, 128, True), (2, 255, 128, True),
    (2, 256, 128, False), (2, 257, 128, True), (5, 65, 32, False), (5, 96, 32, True), (3, 127, 32, False),
    (3, 129, 32, True), (2, 385, 32, False), (11, 769, 64, True), (10, 800, 64, False), (13, 513, 64, True),
])
def test_lengths(H, S, D, causal):
    heads = (0, H - 1)
    got, refs, log = _backward(*_data(H, S, D, H + S + D), causal, heads)
    assert log == ["attn_bwd_pre", "attn_bwd_kernel"], log
    _check(got, refs, heads)


@pytest.mark.parametrize("H,S,kernel", [(12, 640, "attn_bwd_w16"), (13, 640, "attn_bwd_kernel"), (40, 512, "attn_bwd_w16"),
                                        (40, 513, "attn_bwd_kernel")])
def test_head_dim_64_rule(H, S, kernel):
    """Walks beyond 512 queries in launches of 64 key blocks or more, in both
    modes, with the same dK and dV."""
    data = _data(H, S, 64, H)
    got, refs, log = _backward(*data, False, (H - 1,))
    assert log[-1] == kernel, log
    _check(got, refs, (H - 1,))
    capi.set_deterministic(True)
    try:
        det, _, log = _backward(*data, False, (H - 1,))
    finally:
        capi.set_deterministic(False)
    assert log[-1] == kernel, log
    assert np.array_equal(det[1], got[1]) and np.array_equal(det[2], got[2])
    assert capi.deterministic_timeouts() == 0


FORMS = [(3, 300, 128, True), (2, 200, 128, False), (4, 200, 32, True), (12, 700, 64, True)]


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_infinite_keys_get_no_weight(H, S, D, causal):
    """K holding -inf (times positive q) has weight 0: dK and dV of the other
    keys, and dQ but for the column that meets 0 * inf, are as without it."""
    q, k, v, do = _data(H, S, D, 1)
    q[..., 0] = np.abs(q[..., 0]) + 0.1
    k[0, H - 1, 40:50, 0] = -np.inf
    far = np.where(np.isinf(k), np.float32(-1e6), k)   # weight exactly 0 in float64 as well
    refs = [_ref(q[0, H - 1], far[0, H - 1], v[0, H - 1], do[0, H - 1], causal)]
    o, lse = np.zeros_like(q), np.zeros(q.shape[:3], np.float32)
    o[0, H - 1], lse[0, H - 1] = refs[0][0], refs[0][1]
    dq, dk, dv = G.attention_bwd(q, k, v, o, lse, do, causal)
    keys = np.ones(S, bool)
    keys[40:50] = False
    np.testing.assert_allclose(dk[0, H - 1][keys], refs[0][3][keys], rtol=1e-3, atol=2e-4)
    np.testing.assert_allclose(dv[0, H - 1], refs[0][4], rtol=1e-3, atol=2e-4)
    np.testing.assert_allclose(dq[0, H - 1][:, 1:], refs[0][2][:, 1:], rtol=1e-3, atol=2e-4)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
@pytest.mark.parametrize("exponent", [-100, -115])
def test_tiny_inputs_keep_their_precision(H, S, D, causal, which, exponent):
    """One input below what three bf16 parts can hold without a scale:
    gradients to fp32 precision relative to their size."""
    f = np.float32(2.0 ** exponent)
    data = dict(zip(("q", "k", "v", "do"), _data(H, S, D, 3)))
    data[which] *= f
    heads = (H - 1,)
    got, refs, _ = _backward(*data.values(), causal, heads)
    for name, g, r in zip(("dq", "dk", "dv"), got, refs[0]):
        size = np.abs(r).max()
        if size < 2.0 ** -120:
            continue                                   # denormal: fp32 itself has no bits left
        np.testing.assert_allclose(g[0, H - 1] / size, r / size, rtol=1e-4, atol=1e-5, err_msg=name)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_zero_first_rows_and_large_values(H, S, D, causal):
    """A first query block of zeros, then rows whose dO is about 2^100: dV
    passes what its scaled sum can hold and is formed again in fp32."""
    q, k, v, do = _data(H, S, D, 5)
    do[0, :, :32] = 0
    q[0, :, :32] = 0
    big = np.float32(2.0 ** 100)
    do *= big
    v /= big
    heads = (0, H - 1)
    got, refs, _ = _backward(q, k, v, do, causal, heads)
    for h, (rq, rk, rv) in zip(heads, refs):
        np.testing.assert_allclose(got[2][0, h] / big, rv / float(big), rtol=1e-3, atol=2e-4)
        np.testing.assert_allclose(got[0][0, h], rq, rtol=1e-3, atol=2e-4)
        np.testing.assert_allclose(got[1][0, h], rk, rtol=1e-3, atol=2e-4)


def _check_sizes(got, refs, heads, rel=1e-5):
    """Each gradient to `rel` of its largest element (denormal: to 2^-148)."""
    for h, ref in zip(heads, refs):
        for name, g, r in zip(("dq", "dk", "dv"), got, ref):
            assert np.abs(g[0, h] - r).max() <= rel * np.abs(r).max() + 2.0 ** -148, f"{name} head {h}"


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("eq,ek,es", [(-122, 122, 0), (122, -122, 0), (-120, 40, 80), (30, -120, 90), (-60, -60, 120),
                                      (60, 40, -100), (20, 20, -40)])
def test_scores_of_small_and_large_operands(H, S, D, causal, eq, ek, es):
    """Q and K of 2^eq and 2^ek, denormal ones too, which the scale 2^es
    brings back to ordinary scores."""
    q, k, v, do = _data(H, S, D, 6)
    heads = (0, H - 1)
    q, k, scale = np.ldexp(q, eq), np.ldexp(k, ek), np.ldexp(1 / np.sqrt(D), es)
    got, refs, _ = _backward(q, k, v, do, causal, heads, scale)
    _check_sizes(got, refs, heads)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("exponent", [-112, -118, -124])
def test_small_gradients_beside_large_ones(H, S, D, causal, exponent):
    """dO rows of 2^exponent among ordinary ones and after a block of zeros:
    their dQ, and dK where the ordinary rows' Q is 0, keep their precision."""
    q, k, v, do = _data(H, S, D, 7)
    large = np.arange(S) % 7 == 3
    do[:, :, :32] = 0
    do[:, :, ~large] *= np.float32(2.0 ** exponent)
    q[:, :, large] = 0
    heads = (0, H - 1)
    got, refs, _ = _backward(q, k, v, do, causal, heads)
    for h, (rq, rk, rv) in zip(heads, refs):
        # 2^-149 per product: dS itself may be denormal.
        assert (np.abs(got[0][0, h] - rq)[~large] <= 1e-5 * np.abs(rq[~large]).max() + S * 2.0 ** -149).all()
        assert (np.abs(got[1][0, h] - rk) <= 1e-5 * np.abs(rk).max() + S * 2.0 ** -149).all()
        np.testing.assert_allclose(got[2][0, h], rv, rtol=1e-3, atol=2e-4)


@pytest.mark.parametrize("H,S,D,causal", FORMS)
def test_tiny_weights_of_large_gradients(H, S, D, causal):
    """Weights of exp(-86), 2^-124, times dO of 2^60 (dV)."""
    q, k, v, do = _data(H, S, D, 8)
    q[:], k[:] = 0, 0
    q[..., 0] = np.sqrt(D)
    k[:, :, 1:, 0] = np.random.default_rng(9).uniform(-86.4, -85, (1, H, S - 1))
    do *= np.float32(2.0 ** 60)
    heads = (0, H - 1)
    got, refs, _ = _backward(q, k, v, do, causal, heads)
    for h, (_, _, rv) in zip(heads, refs):
        p = np.exp(k[0, h, 1:, 0].astype(np.float64))
        size = np.cumsum(np.abs(do[0, h, ::-1]), 0)[::-1][1:] if causal else np.abs(do[0, h]).sum(0)[None]
        # The exponent, about 124 in base 2, has an ulp of 2^-17: 2^-18 ln 2
        # each in the product with the scale and in the difference from lse.
        assert (np.abs(got[2][0, h][1:] - rv[1:]) <= 2.0 ** -17 * p[:, None] * size).all()


@pytest.mark.parametrize("H,S,D,causal", FORMS)
@pytest.mark.parametrize("which,exponent", [("q", 50), ("k", 50), ("v", 113), ("do", 113), ("ds", 26), ("ds", 44)])
def test_large_rows_go_on_with_the_fp32_instruction(H, S, D, causal, which, exponent):
    """One row that the scaled split cannot carry, in the middle of the walk:
    the workgroups that meet it end theirs in fp32, with the same gradients
    on every run in deterministic order."""
    q, k, v, do = _data(H, S, D, 10)
    row, f = S // 2 + 5, np.float32(2.0 ** exponent)
    heads = (0, H - 1)
    if which == "ds":                                  # dS of about f^2, carried at 2^52 and not at 2^88
        v *= f
        do[:, :, row] *= f
    elif which in ("q", "k"):
        x, y = (q, k) if which == "q" else (k, q)
        x[:, :, row, 3], y[..., 3] = f, 0              # finds nothing to multiply but 0
    else:
        x, y = (v, do) if which == "v" else (do, v)
        x[:, :, row, 3] = f
        y[..., 3] /= f
    ref = None
    for det in (False, True, True):
        capi.set_deterministic(det)
        try:
            got, refs, _ = _backward(q, k, v, do, causal, heads)
        finally:
            capi.set_deterministic(False)
        _check_sizes(got, refs, heads)
        if det and ref is not None:
            assert all(np.array_equal(a, b) for a, b in zip(got, ref))
        ref = got if det else None
    assert capi.deterministic_timeouts() == 0


@pytest.mark.parametrize("H,S,D,causal,errs", [
    (8, 1024, 128, True, (5.4e-7, 8.7e-7, 8.1e-7)), (30, 777, 128, False, (6.1e-7, 7.7e-7, 7.6e-7)),
    (16, 1000, 32, True, (3.7e-7, 8.2e-7, 8.3e-7)), (128, 1024, 64, True, (4.7e-7, 8.5e-7, 8.1e-7))])
def test_error_no_larger_than_the_fp32_instructions(H, S, D, causal, errs):
    """Relative 2-norm errors against float64 below what the kernel on the
    fp32 matrix instruction measured (rounded up)."""
    heads = (0, 1)
    data = _data(H, S, D, 4)
    got, refs, _ = _backward(*data, causal, heads)
    for name, g, err, i in zip(("dq", "dk", "dv"), got, errs, range(3)):
        r = np.stack([x[i] for x in refs])
        assert np.linalg.norm(g[0, :2] - r) / np.linalg.norm(r) <= err, name
