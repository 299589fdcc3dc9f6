"""The unfused path's kernels at the edges of their tiles, against the FP64
oracle: sequence lengths around the 32-, 64- and 128-wide tiles and their
remainders, head dims around the 16-, 32-, 64- and 128-column steps (odd ones
take the element-wise loads), one slab (small tiles) and enough slabs for the
large ones, both masks.

Bound: v0 keeps S and P in fp32, so its error is the final rounding to bf16
(half a unit in the last place, at most 2^-8 |O|) plus fp32 sums and
exponentials: at most about (N + D) roundings of 2^-24 of the row's scale and
the exponentials' few units, below 2^-13 of it for N <= 300, D <= 300."""
import numpy as np
import pytest

from gpu_common import HOST_THREADS, run_bits, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fa(fa_lib):
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X")
    return fa_lib


def check_unfused(fa, oracle, B, H, N, D, causal, family="normal_mt19937"):
    q, k, v = oracle.make_inputs(B, H, N, D, family)
    ref = oracle.attention(q, k, v, causal, threads=HOST_THREADS).reshape(-1, D)
    say("unfused", B, H, N, D, causal, family)
    got = run_bits(fa, "v0_unfused", q, k, v, causal)
    out = oracle.bf16_to_f32(got).astype(np.float64).reshape(-1, D)
    scale = np.abs(ref).max(axis=1, keepdims=True)
    bound = 2.0 ** -8 * np.abs(ref) + 2.0 ** -13 * scale
    assert np.all(np.abs(out - ref) <= bound), (B, H, N, D, causal, family, float((np.abs(out - ref) - bound).max()))


@pytest.mark.parametrize("head_dim", [1, 5, 8, 24, 33, 64, 72, 96, 128, 136, 200, 256, 264])
def test_edges(fa, oracle_mod, head_dim):
    for n in (1, 31, 33, 64, 65, 129):
        for causal in (False, True):
            check_unfused(fa, oracle_mod, 1, 2, n, head_dim, causal)


@pytest.mark.parametrize("B,H,N,D", [(4, 16, 250, 72), (2, 32, 256, 64), (1, 29, 300, 33), (16, 16, 128, 96)])
def test_many_slabs(fa, oracle_mod, B, H, N, D):
    for causal in (False, True):
        check_unfused(fa, oracle_mod, B, H, N, D, causal)


@pytest.mark.parametrize("H,N,D", [(2, 300, 200), (1, 545, 264), (3, 257, 400)])
def test_column_tiles_of_many_query_blocks(fa, oracle_mod, H, N, D):
    """Two to four tiles of columns with more than eight blocks of 32 queries:
    the second round of eight, whole and partial, and a third."""
    for causal in (False, True):
        check_unfused(fa, oracle_mod, 1, H, N, D, causal)


@pytest.mark.parametrize("H,N,D", [(32, 500, 72), (64, 300, 33), (300, 257, 40), (128, 256, 64), (171, 256, 64), (513, 65, 8), (24, 448, 200)])
def test_two_large_tiles_per_cu(fa, oracle_mod, H, N, D):
    """The large tiles of scores: two or more for every CU dense and causal, dense
    only (the causal launch has 384 of 128 x 128), just above two, and the lower
    limit beyond head_dim 128 (384 dense, 240 causal)."""
    for causal in (False, True):
        check_unfused(fa, oracle_mod, 1, H, N, D, causal)


@pytest.mark.parametrize("cols", [1, 2, 5, 255, 257, 511, 513, 1023, 1024, 1025, 2047, 2049, 4097, 8191, 8193, 16385, 32767,
                                  32769])
def test_softmax_lengths_and_addresses(fa, cols):
    """Rows of every register variant's first and last lengths, at each of the
    four positions that a row of floats can have against 16 bytes, one to six
    rows. Bound: (x - max) * log2(e) carries two roundings of up to 2^-24 of an
    exponent of at most 60, 5e-6 of the weight; the sum and the final product add
    less than 2^-20; weights below fp32's normal range may be flushed."""
    import torch

    rng = np.random.default_rng(cols)
    for offset in range(4):
        rows = 1 + (offset + cols) % 6
        x = rng.normal(0, 4, size=(rows, cols)).astype(np.float32)
        t = torch.full((rows * cols + 8,), 7.0, dtype=torch.float32, device="cuda")
        t[offset:offset + rows * cols] = torch.from_numpy(x.reshape(-1)).cuda()
        say("softmax", rows, cols, offset)
        assert fa.launch_softmax_rows_inplace(t.data_ptr() + 4 * offset, rows, cols)
        torch.cuda.synchronize()
        got = t.cpu().numpy().astype(np.float64)
        assert np.all(got[:offset] == 7.0) and np.all(got[offset + rows * cols:] == 7.0)
        xd = x.astype(np.float64)
        e = np.exp(xd - xd.max(axis=1, keepdims=True))
        want = e / e.sum(axis=1, keepdims=True)
        np.testing.assert_allclose(got[offset:offset + rows * cols].reshape(rows, cols), want, rtol=1e-5, atol=2e-38)


@pytest.mark.parametrize("N,D", [(70, 8), (200, 64), (129, 130)])
def test_causal_masked_weights(fa, oracle_mod, N, D):
    """Scores above the diagonal are neither written nor read, and their
    weights are one value per row. A row whose scores are all -infinity gives
    its weight to the masked keys in equal parts (their score is the lowest
    finite float; the last row, without masked keys, comes out 0), and a NaN in
    V reaches every row: both as if the whole matrix were there."""
    rng = np.random.default_rng(N)
    shape = (1, 2, N, D)
    q, k = np.zeros(shape), rng.normal(size=shape)
    q[..., 0] = 1.0
    v = rng.uniform(-1, 1, shape)
    k[0, 1, :, 0] = -np.inf
    bits = [oracle_mod.bf16_bits(x) for x in (q, k, v)]
    say("masked weights", N, D)
    out = oracle_mod.bf16_to_f32(run_bits(fa, "v0_unfused", *bits, True)).astype(np.float64)
    vf = oracle_mod.bf16_to_f32(bits[2]).astype(np.float64)
    for row in range(N):
        want = vf[0, 1, row + 1:].mean(axis=0) if row < N - 1 else np.zeros(D)
        assert np.all(np.abs(out[0, 1, row] - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -14), row
    ref = oracle_mod.attention(*(x[:, :1].copy() for x in bits), True, threads=HOST_THREADS).reshape(N, D)
    assert np.all(np.abs(out[0, 0] - ref) <= 2.0 ** -8 * np.abs(ref) + 2.0 ** -13)
    bits[2][0, 0, N - 1, D - 1] = 0x7FC0
    out = oracle_mod.bf16_to_f32(run_bits(fa, "v0_unfused", *bits, True))
    assert np.isnan(out[0, 0, :, D - 1]).all() and np.isfinite(out[0, 0, :, :D - 1]).all() and np.isfinite(out[0, 1]).all()


@pytest.mark.parametrize("H,N,D", [(2, 1, 8), (2, 70, 33), (2, 200, 64), (1, 545, 264), (70, 250, 64)])
def test_workspace_of_nans(fa, oracle_mod, H, N, D):
    """Whatever the score workspace holds is not read: with NaN everywhere in it
    (causal launches leave the scores above the diagonal as they are) the output
    is that of a zeroed one, bit for bit."""
    import torch

    from gpu_common import from_dev, nan_like, to_dev

    q, k, v = (to_dev(x) for x in oracle_mod.make_inputs(1, H, N, D, "normal_mt19937"))
    shape = fa.AttentionShape(1, H, N, D)
    for causal in (False, True):
        say("workspace of NaNs", H, N, D, causal)
        out = []
        for fill in (0.0, float("nan")):
            ws = torch.full((fa.unfused_workspace_bytes(shape) // 4,), fill, dtype=torch.float32, device="cuda")
            o = nan_like(q)
            assert fa.launch_attention_unfused(q, k, v, o, ws, shape, causal)
            out.append(from_dev(o))
        assert np.array_equal(out[0], out[1]) and np.isfinite(oracle_mod.bf16_to_f32(out[1])).all()


def test_causal_rows_beyond_the_registers(fa, oracle_mod):
    """More than 32768 keys: the softmax that walks a row in memory, causal, on a
    workspace of NaNs, checked on rows around the register limit and at both ends
    (the bound of the file: N roundings of 2^-24 of either sign add up to about
    sqrt(N) 2^-24 = 2^-16.5 of the row's scale, under 2^-13)."""
    import torch

    from gpu_common import from_dev, nan_like, to_dev

    N, D = 32801, 8
    qb, kb, vb = oracle_mod.make_inputs(1, 1, N, D, "normal_mt19937")
    q, k, v = (to_dev(x) for x in (qb, kb, vb))
    shape = fa.AttentionShape(1, 1, N, D)
    say("causal rows beyond the registers", N, D)
    ws = torch.full((fa.unfused_workspace_bytes(shape) // 4,), float("nan"), dtype=torch.float32, device="cuda")
    o = nan_like(q)
    assert fa.launch_attention_unfused(q, k, v, o, ws, shape, True)
    out = oracle_mod.bf16_to_f32(from_dev(o)).astype(np.float64).reshape(N, D)
    assert np.isfinite(out).all()
    qf, kf, vf = (oracle_mod.bf16_to_f32(x).astype(np.float64).reshape(N, D) for x in (qb, kb, vb))
    for row in (0, 1, 31, 32, 255, 256, 1000, 16383, 32767, 32768, 32799, 32800):
        x = kf[:row + 1] @ qf[row] / np.sqrt(D)
        w = np.exp(x - x.max())
        want = w @ vf[:row + 1] / w.sum()
        bound = 2.0 ** -8 * np.abs(want) + 2.0 ** -13 * np.abs(vf[:row + 1]).max()
        assert np.all(np.abs(out[row] - want) <= bound), (row, out[row], want)


@pytest.mark.parametrize("N,D", [(1, 8), (1, 33), (4, 64), (64, 96), (70, 200), (300, 130)])
@pytest.mark.parametrize("equal_scores", [True, False])
def test_infinite_v(fa, oracle_mod, N, D, equal_scores):
    """An infinity in V gives an infinity wherever its weight is positive, also
    where the weight needs fewer than 24 bits (seq_len 1, causal row 0, equal
    scores over a power of two), and NaN where two of opposite sign meet or the
    weight is 0 (causal rows before its key): the products of the whole matrix."""
    rng = np.random.default_rng(N * 1000 + D)
    q, k, v = (rng.normal(size=(1, 2, N, D)) for _ in range(3))
    if equal_scores:
        q[:] = 0.0
    v[0, 0, N // 2, 0] = np.inf
    v[0, 0, 0, D - 1] = -np.inf
    v[0, 1, N - 1, 3] = -np.inf
    v[0, 1, 0, 3] = np.inf
    v[0, 1, 0, 5] = np.nan
    bits = [oracle_mod.bf16_bits(x) for x in (q, k, v)]
    qf, kf, vf = (oracle_mod.bf16_to_f32(b).astype(np.float64)[0] for b in bits)
    for causal in (False, True):
        s = np.einsum("hqd,hkd->hqk", qf, kf) / np.sqrt(D)
        if causal:
            s = np.where(np.arange(N)[None, :] > np.arange(N)[:, None], -np.inf, s)
        w = np.exp(s - s.max(axis=-1, keepdims=True))
        w /= w.sum(axis=-1, keepdims=True)
        with np.errstate(invalid="ignore"):
            want = np.stack([(w[h][:, :, None] * vf[h][None]).sum(axis=1) for h in range(2)])
        say("infinite V", N, D, equal_scores, causal)
        out = oracle_mod.bf16_to_f32(run_bits(fa, "v0_unfused", *bits, causal)).astype(np.float64)[0]
        special = ~np.isfinite(want)
        assert np.array_equal(out[special], want[special], equal_nan=True), (N, D, equal_scores, causal)
        scale = np.where(special, 0.0, np.abs(want)).max(axis=2, keepdims=True)
        with np.errstate(invalid="ignore"):
            wrong = ~(np.abs(out - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -13 * scale)
        assert not wrong[~special].any(), (N, D, equal_scores, causal)


@pytest.mark.parametrize("D", [8, 33, 64])
def test_subnormal_v(fa, oracle_mod, D):
    """The matrix cores keep bf16's subnormal values: with one key O is V."""
    v = np.arange(1, D + 1, dtype=np.uint16).reshape(1, 1, 1, D)
    v[..., ::2] |= 0x8000
    ones = np.full_like(v, 0x3F80)
    for causal in (False, True):
        say("subnormal V", D, causal)
        assert np.array_equal(run_bits(fa, "v0_unfused", ones, ones, v, causal), v)
