"""The audio decoder through the C ABI against the oracle: each convolution
kernel (with and without the fused Snake, residual accumulation, every tile
shape, ragged channel counts and signal edges), the whole decoder at a tiny
and at the released configuration within the reference's own decode bounds
(codec_test.cpp:60-62: RMS within 1e-4, samples within 1e-3), determinism,
the device entry point, errors, and a checkpoint written with the
reference's tensor names."""
import math
import os

import numpy as np
import pytest

import omnivoice_amd as ov
import oracle

pytestmark = pytest.mark.gpu

TINY = dict(codebooks=3, codebook_size=16, codebook_dim=8, hidden=24, latent=12,
            channels=32, ratios=[2, 3, 4])


def _gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not _gpu_available():
        pytest.skip("no GPU")


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def close(got, want, rtol=1e-4):
    scale = max(float(np.abs(want).max()), 1e-3)
    err = float(np.abs(got - want).max())
    assert err <= rtol * scale, (err, scale)


@pytest.mark.parametrize("cin,cout,length,kernel,dilation,snake,accumulate", [
    (16, 32, 300, 7, 1, False, False),    # 32 x 128 tiles
    (48, 64, 150, 7, 3, True, False),     # 64 x 64 tiles
    (32, 96, 97, 7, 9, True, True),       # ragged output channels and positions
    (21, 40, 64, 1, 1, True, True),       # ragged input channels, one tap
    (256, 1024, 25, 7, 1, False, False),  # the decoder's input convolution shape
    (64, 64, 5, 7, 9, True, False),       # signal shorter than the taps' spread
    (128, 128, 40000, 7, 1, True, True),  # long signals: hundreds of tiles
    (64, 64, 40000, 7, 3, True, False),
    (48, 96, 40000, 1, 1, True, True),    # long, one tap, ragged channels
])
def test_conv1d_matches_oracle(cin, cout, length, kernel, dilation, snake, accumulate):
    rng = np.random.default_rng(cin + cout + length)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, kernel)) / math.sqrt(cin * kernel)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    alpha = np.exp(0.3 * rng.standard_normal(cin)).astype(np.float32) if snake else None
    y0 = rng.standard_normal((cout, length)).astype(np.float32)
    y = dev(y0)
    ov.op_conv1d(dev(x), w, b, y, alpha=dev(alpha) if snake else None, dilation=dilation,
                 accumulate=accumulate)
    xin = oracle.snake(x, alpha) if snake else x
    want = oracle.conv1d(xin, w, b, dilation) + (y0 if accumulate else 0)
    close(y.cpu().numpy(), want)


@pytest.mark.parametrize("cin,cout,length,kernel,dilation", [
    (1, 1, 1, 7, 10), (31, 32, 255, 7, 9), (32, 31, 257, 7, 10), (33, 33, 129, 7, 1),
    (64, 64, 127, 1, 1), (65, 65, 64, 1, 1), (63, 129, 65, 7, 3), (130, 200, 63, 1, 1),
    (97, 128, 16500, 7, 9), (40, 130, 16400, 1, 1), (17, 16, 300, 2, 1)])
def test_conv1d_tile_edges(cin, cout, length, kernel, dilation):
    """Edges of the tiles, chunks and windows against 64 bits. Bound: every operand is kept to
    2^-24 and what is left out of a product is below 2^-23 of it; each 16-deep product rounds
    its two sums once, five of six of them small: K / 8 + 8 roundings of 2^-24 of sum |w x|."""
    rng = np.random.default_rng(cin + cout + length)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, kernel)) / math.sqrt(cin * kernel)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    y = dev(np.zeros((cout, length)))
    ov.op_conv1d(dev(x), w, b, y, dilation=dilation)
    pad = (kernel - 1) * dilation // 2
    xp = np.pad(x.astype(np.float64), ((0, 0), (pad, kernel * dilation)))
    want, size = b.astype(np.float64)[:, None], np.abs(b)[:, None].astype(np.float64)
    for k in range(kernel):
        at = xp[:, k * dilation:k * dilation + length]
        want = want + w[:, :, k].astype(np.float64) @ at
        size = size + np.abs(w[:, :, k]).astype(np.float64) @ np.abs(at)
    assert (np.abs(y.cpu().numpy() - want) <= (cin * kernel / 8 + 8) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("cin,cout,length,stride", [
    (32, 31, 1, 1), (33, 33, 63, 2), (31, 64, 65, 3), (64, 96, 64, 4), (65, 40, 129, 5),
    (40, 32, 33, 6), (16, 65, 100, 7), (128, 20, 66, 8)])
def test_conv_transpose1d_tile_edges(cin, cout, length, stride):
    """Every stride at the edges of the tiles against 64 bits, with the bound of the test above
    (two taps reach each output)."""
    rng = np.random.default_rng(cin + cout + length)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    w = (rng.standard_normal((cin, cout, 2 * stride)) / math.sqrt(2 * cin)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    y = dev(np.zeros((cout, length * stride)))
    ov.op_conv_transpose1d(dev(x), w, b, y, stride)

    def run(x, w, b):
        full = np.zeros((cout, (length + 2) * stride))
        for k in range(2 * stride):
            full[:, k:k + (length - 1) * stride + 1:stride] += w[:, :, k].T @ x
        pad = (stride + 1) // 2
        return full[:, pad:pad + length * stride] + b[:, None]
    x, w, b = (v.astype(np.float64) for v in (x, w, b))
    size = run(np.abs(x), np.abs(w), np.abs(b))
    bound = (2 * cin / 8 + 8) * 2.0 ** -24 * size
    assert (np.abs(y.cpu().numpy() - run(x, w, b)) <= bound).all()


def precise(got, want, terms, more=0.0):
    """The root mean square of the error against 64 bits, for sums of `terms` random products.
    Each 16-deep product rounds the running sum once (to 2^-24 of it), the second accumulator,
    the final addition and the bias a few times more, independently: sqrt(terms / 16 + 4)
    roundings, and `more` for what comes with them. A partial product left out, hi lo the least
    of them, is an error of 2^-18.7 of the sum, the bound under 2^-20 up to 3700 terms."""
    err = np.sqrt(np.mean((got - want) ** 2)) / np.sqrt(np.mean(want ** 2))
    bound = (math.sqrt(terms / 16 + 4) + more) * 2.0 ** -24
    assert err <= bound, (err / 2.0 ** -24, bound / 2.0 ** -24)


def conv_exact(x, w, b, dilation=1, stride=1, padding=0, groups=1, positions=None):
    """Conv1d in 64 bits, x [in][L], w [out][in / groups][k], the first `positions` outputs."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    kernel, per = w.shape[2], w.shape[1]
    n = (x.shape[1] + 2 * padding - (kernel - 1) * dilation - 1) // stride + 1
    n = n if positions is None else positions
    x = np.pad(x, ((0, 0), (padding, padding)))
    y = np.zeros((w.shape[0], n))
    out = w.shape[0] // groups
    for g in range(groups):
        for k in range(kernel):
            at = x[g * per:(g + 1) * per, k * dilation:k * dilation + (n - 1) * stride + 1:stride]
            y[g * out:(g + 1) * out] += w[g * out:(g + 1) * out, :, k] @ at
    return y + b.astype(np.float64)[:, None]


@pytest.mark.parametrize("cin,cout,length,kernel,dilation,stride,padding,groups,elu,split", [
    (1, 65, 1003, 10, 1, 5, 0, 1, False, 0),       # the first feature convolution
    (40, 130, 611, 3, 1, 2, 0, 1, False, 1 << 20), # a strided window, split
    (96, 96, 50, 3, 1, 1, 1, 1, True, 1 << 20),    # k3 of an activated input, split
    (96, 96, 50, 3, 1, 1, 1, 1, True, 0),
    (64, 40, 333, 16, 1, 8, 4, 1, False, 0),       # a downsampling layer
    (96, 96, 70, 32, 1, 1, 16, 4, False, 1 << 20), # grouped, an even kernel's first outputs
    (300, 130, 33, 1, 1, 1, 0, 1, False, 1 << 20), # one tap, split
    (300, 70, 30, 7, 3, 1, 9, 1, False, 1 << 20),  # seven taps, split, 128 x 32 tiles
    (520, 300, 190, 7, 1, 1, 3, 1, False, 1 << 20),
    (40, 24, 70, 7, 1, 1, 3, 1, False, 1 << 20),   # narrow layers, split
    (70, 64, 90, 7, 9, 1, 27, 1, False, 1 << 20),
    (33, 129, 8193, 7, 1, 1, 3, 1, False, 0),      # 128 x 64 tiles
    (32, 129, 8201, 7, 9, 1, 27, 1, False, 0),     # the same, of one chunk
    (17, 200, 8193, 7, 1, 1, 3, 1, False, 1 << 20),
    (40, 300, 8129, 1, 1, 1, 0, 1, False, 0),      # one tap: past three narrow tiles a CU
    (40, 300, 8065, 1, 1, 1, 0, 1, False, 0),      # and not
    (40, 300, 8129, 3, 1, 2, 1, 1, False, 0),
])
def test_strided_and_split_conv1d_precision(cin, cout, length, kernel, dilation, stride, padding,
                                            groups, elu, split):
    rng = np.random.default_rng(cin + cout + length)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    per = cin // groups
    w = (rng.standard_normal((cout, per, kernel)) / math.sqrt(per * kernel)).astype(np.float32)
    b = (0.1 * rng.standard_normal(cout)).astype(np.float32)
    positions = (length + 2 * padding - (kernel - 1) * dilation - 1) // stride + 1
    if kernel % 2 == 0 and padding == kernel // 2:
        positions = length
    xin = np.where(x > 0, x, np.expm1(x.astype(np.float64))) if elu else x
    want = conv_exact(xin, w, b, dilation, stride, padding, groups, positions)
    y = dev(np.zeros((cout, positions)))
    ov.op_conv1d_strided(dev(x), w, b, y, dilation, stride, padding, groups, elu, split)
    # each input of an ELU carries its rounding too
    precise(y.cpu().numpy(), want, per * kernel, more=1.0 if elu else 0.0)


@pytest.mark.parametrize("cin,kernel,stride", [(40, 4, 2), (33, 3, 1), (9, 16, 8)])
def test_strided_conv1d_of_a_snake(cin, kernel, stride):
    """Each channel of a strided window by its own alpha."""
    rng = np.random.default_rng(kernel)
    x = rng.standard_normal((cin, 203)).astype(np.float32)
    w = (rng.standard_normal((70, cin, kernel)) / math.sqrt(cin * kernel)).astype(np.float32)
    b = rng.standard_normal(70).astype(np.float32)
    alpha = np.exp(rng.standard_normal(cin)).astype(np.float32)
    want = conv_exact(oracle.snake(x, alpha), w, b, 1, stride, 1)
    y = dev(np.zeros(want.shape))
    ov.op_conv1d_strided(dev(x), w, b, y, stride=stride, padding=1, alpha=dev(alpha))
    precise(y.cpu().numpy(), want, cin * kernel, more=4.0)  # the Snake's roundings on both sides


def _huge(rng, shape, share=0.03):
    """Random values, some of them next to the largest float32 (past bf16's largest)."""
    x = rng.standard_normal(shape).astype(np.float32)
    top = np.float32(np.finfo(np.float32).max)
    at = rng.random(shape) < share
    x[at] = (rng.choice([-1, 1], at.sum()) * top * rng.uniform(0.999, 1.0, at.sum()))
    return x


def _finite_and_close(got, want, size):
    """Sums formed in double from the operands: one rounding, and those of the bias and what is
    added after it. Ordinary sums, of under 600 terms here, by the tile edges' bound."""
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert (np.abs(got - want) <= 80 * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("cin,cout,length,kernel,stride,groups,split", [
    (32, 32, 140, 7, 1, 1, 0), (40, 33, 90, 1, 1, 1, 0), (40, 70, 300, 7, 1, 1, 0),
    (300, 130, 40, 1, 1, 1, 1 << 20), (40, 130, 211, 3, 2, 1, 0), (64, 64, 60, 8, 4, 4, 1 << 20)])
def test_conv1d_of_the_largest_values(cin, cout, length, kernel, stride, groups, split):
    """Finite inputs and weights that round to bf16's infinity give finite sums."""
    rng = np.random.default_rng(cin + cout + kernel)
    per, padding = cin // groups, (kernel - 1) // 2
    tiny = 2.0 ** -12
    b = rng.standard_normal(cout).astype(np.float32)
    for big_weights in (False, True):
        x = _huge(rng, (cin, length))
        w = (tiny * rng.standard_normal((cout, per, kernel))).astype(np.float32)
        if big_weights:
            x, w = (tiny * rng.standard_normal(x.shape)).astype(np.float32), _huge(rng, w.shape)
        want = conv_exact(x, w, b, 1, stride, padding, groups)
        size = conv_exact(np.abs(x), np.abs(w), np.abs(b), 1, stride, padding, groups)
        y = dev(np.zeros(want.shape))
        ov.op_conv1d_strided(dev(x), w, b, y, 1, stride, padding, groups, False, split)
        _finite_and_close(y.cpu().numpy(), want, size)


@pytest.mark.parametrize("cin,cout,length,kernel,stride,split", [
    (40, 33, 300, 1, 1, 0), (300, 130, 40, 1, 1, 1 << 20), (300, 70, 30, 7, 1, 1 << 20),
    (40, 130, 211, 3, 2, 0), (70, 20, 90, 8, 4, 1 << 20)])
def test_strided_and_split_conv1d_keep_infinities(cin, cout, length, kernel, stride, split):
    """Infinite and NaN inputs give what 64 bits give, in the outputs that they reach only."""
    rng = np.random.default_rng(cin + kernel)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    x[3, 9], x[17, 20], x[20, 20], x[5, 27] = np.inf, np.inf, -np.inf, np.nan
    w = rng.standard_normal((cout, cin, kernel)).astype(np.float32)
    b = np.zeros(cout, np.float32)
    with np.errstate(invalid="ignore"):
        want = conv_exact(x, w, b, 1, stride, (kernel - 1) // 2)
    y = dev(np.zeros(want.shape))
    ov.op_conv1d_strided(dev(x), w, b, y, 1, stride, (kernel - 1) // 2, split_floats=split)
    got, finite = y.cpu().numpy(), np.isfinite(want)
    assert (np.isfinite(got) == finite).all()
    np.testing.assert_array_equal(got[~finite], want[~finite].astype(np.float32))
    np.testing.assert_allclose(got[finite], want[finite], rtol=1e-4, atol=1e-4)


def test_conv1d_of_the_smallest_values():
    """Inputs around 2^-118, whose low parts are below bf16's least value 2^-133, against 64
    bits: each is kept to half of that, beside the tile edges' bound."""
    rng = np.random.default_rng(7)
    x = (2.0 ** -118 * rng.standard_normal((40, 300))).astype(np.float32)
    w = (2.0 ** 20 * rng.standard_normal((33, 40, 7))).astype(np.float32)
    b = np.zeros(33, np.float32)
    y = dev(np.zeros((33, 300)))
    ov.op_conv1d(dev(x), w, b, y)
    size = conv_exact(np.abs(x), np.abs(w), b, padding=3)
    kept = np.abs(w).astype(np.float64).sum((1, 2))[:, None] * 2.0 ** -134
    err = np.abs(y.cpu().numpy() - conv_exact(x, w, b, padding=3))
    assert (err <= (40 * 7 / 8 + 8) * 2.0 ** -24 * size + kept).all()


@pytest.mark.parametrize("cin,cout,length,stride", [(40, 33, 50, 3), (33, 40, 70, 8)])
def test_conv_transpose1d_of_the_largest_values(cin, cout, length, stride):
    rng = np.random.default_rng(stride)
    x, tiny = _huge(rng, (cin, length)), 2.0 ** -12
    w = (tiny * rng.standard_normal((cin, cout, 2 * stride))).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    y = dev(np.zeros((cout, length * stride)))
    ov.op_conv_transpose1d(dev(x), w, b, y, stride)

    def run(x, w, b):
        full = np.zeros((cout, (length + 2) * stride))
        for k in range(2 * stride):
            full[:, k:k + (length - 1) * stride + 1:stride] += w[:, :, k].T @ x
        pad = (stride + 1) // 2
        return full[:, pad:pad + length * stride] + b[:, None]
    x, w, b = (v.astype(np.float64) for v in (x, w, b))
    _finite_and_close(y.cpu().numpy(), run(x, w, b), run(np.abs(x), np.abs(w), np.abs(b)))


@pytest.mark.parametrize("channels,length", [(20, 150), (48, 140), (100, 66), (65, 16321)])
def test_residual_unit_of_the_largest_values(channels, length):
    """Inputs, and results of the first convolution, that round to bf16's infinity. Alphas of
    one: the Snake adds at most one, of nothing to such values."""
    rng = np.random.default_rng(channels)
    x = _huge(rng, (channels, length), share=20.0 / (channels * length))
    w1 = np.zeros((channels, channels, 7), np.float32)
    w1[:, :, 3] = np.eye(channels)
    w2 = (2.0 ** -12 * rng.standard_normal((channels, channels))).astype(np.float32)
    zero = np.zeros(channels, np.float32)
    y0 = rng.standard_normal((channels, length)).astype(np.float32)
    v = x.astype(np.float64)
    v = v + np.where(np.abs(v) < 1e6, np.sin(v) ** 2, 0.0)
    size = conv_exact(np.abs(v), np.abs(w2)[:, :, None], zero) + np.abs(y0)
    y = dev(y0)
    ov.op_residual_unit(dev(x), w1, zero, dev(np.ones(channels)), w2, zero, y)
    _finite_and_close(y.cpu().numpy(), conv_exact(v, w2[:, :, None], zero) + y0, size)


@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("channels,length,dilation", [
    (5, 131, 9), (32, 257, 1), (48, 300, 3), (64, 129, 1), (100, 65, 9), (128, 70, 3),
    # the wider tiles, which take over where the narrow ones number twice the CUs
    (40, 32641, 3), (64, 32700, 9), (65, 16321, 1), (96, 16400, 9), (128, 16385, 3)])
def test_residual_unit_precision(channels, length, dilation, second):
    """Either product of a fused unit against 64 bits, the other one an exact scaling by powers
    of two. The Snake, of a small alpha, adds a few roundings and turns the sum by under 1 %."""
    rng = np.random.default_rng(channels + length)
    x, y0 = (rng.standard_normal((channels, length)).astype(np.float32) for _ in range(2))
    alpha = (0.002 * np.exp(0.3 * rng.standard_normal(channels))).astype(np.float32)
    b1, b2 = (0.1 * rng.standard_normal((2, channels))).astype(np.float32)
    scaling = np.diag(2.0 ** rng.integers(-2, 3, channels)).astype(np.float32)
    if second:
        w1 = np.zeros((channels, channels, 7), np.float32)
        w1[:, :, 3] = scaling
        w2 = rng.standard_normal((channels, channels)) / math.sqrt(channels)
    else:
        w1 = rng.standard_normal((channels, channels, 7)) / math.sqrt(7 * channels)
        w2 = scaling
    w1, w2 = w1.astype(np.float32), w2.astype(np.float32)
    v = conv_exact(x, w1, b1, dilation, padding=3 * dilation)
    a = alpha.astype(np.float64)[:, None]
    v = v + np.sin(a * v) ** 2 / (a + 1e-9)
    want = conv_exact(v, w2[:, :, None], b2) + y0
    y = dev(y0)
    ov.op_residual_unit(dev(x), w1, b1, dev(alpha), w2, b2, y, dilation)
    precise(y.cpu().numpy(), want, channels * (1 if second else 7), more=2.0)


@pytest.mark.parametrize("channels,frames", [(32, 5), (64, 11), (128, 23), (192, 43), (256, 3)])
def test_fused_residual_units_match_oracle(channels, frames):
    """Decoders whose blocks' units run fused (16 to 128 channels, ragged ones too; the narrower
    tiles, at signals this short), next to 256 channels that do not."""
    cfg = dict(TINY, channels=channels * 2, ratios=[5, 2])
    codes = np.random.default_rng(frames).integers(0, 16, size=(3, frames)).astype(np.int32)
    close(ov.Codec.synthetic(cfg, 31).decode(codes), oracle.Codec(cfg, 31).decode(codes),
          rtol=2e-4)


def test_conv1d_keeps_infinities():
    """An infinite input makes its outputs infinite, not NaN; NaN stays where it reaches."""
    x = np.ones((32, 200), dtype=np.float32)
    x[3, 50], x[5, 120] = np.inf, np.nan
    w = np.full((32, 32, 7), 0.5, dtype=np.float32)
    y = dev(np.zeros((32, 200)))
    ov.op_conv1d(dev(x), w, np.zeros(32, np.float32), y)
    got = y.cpu().numpy()
    assert np.isposinf(got[:, 47:54]).all() and np.isnan(got[:, 117:124]).all()
    rest = np.delete(got, [*range(47, 54), *range(117, 124)], axis=1)
    assert np.isfinite(rest).all()


@pytest.mark.parametrize("cin,cout,length,stride,snake", [
    (64, 32, 40, 8, True), (32, 16, 33, 5, True), (128, 64, 70, 4, False),
    (16, 8, 9, 2, True), (48, 24, 31, 3, True), (1024, 512, 25, 8, True),
    (256, 128, 10000, 4, True)])  # long signal over four phases
def test_conv_transpose1d_matches_oracle(cin, cout, length, stride, snake):
    rng = np.random.default_rng(cin * stride + length)
    x = rng.standard_normal((cin, length)).astype(np.float32)
    w = (rng.standard_normal((cin, cout, 2 * stride)) / math.sqrt(2 * cin)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    alpha = np.exp(0.3 * rng.standard_normal(cin)).astype(np.float32) if snake else None
    y = dev(np.zeros((cout, length * stride)))
    ov.op_conv_transpose1d(dev(x), w, b, y, stride, alpha=dev(alpha) if snake else None)
    xin = oracle.snake(x, alpha) if snake else x
    close(y.cpu().numpy(), oracle.conv_transpose1d(xin, w, b, stride))


def test_synthetic_values_match_oracle():
    for tensor, scale, exp in [(1000, 0.35, False), (1205, 0.25, False), (1200, 0.1, True)]:
        np.testing.assert_array_equal(
            ov.codec_synthetic_values(1234, tensor, 17, 5000, scale, exp),
            oracle.codec_values(1234, tensor, 5000, scale, exp, first=17))


@pytest.mark.parametrize("frames", [1, 7, 40])
def test_tiny_decode_matches_oracle(frames):
    codec = ov.Codec.synthetic(TINY, 77)
    codes = np.random.default_rng(frames).integers(0, 16, size=(3, frames)).astype(np.int32)
    got = codec.decode(codes)
    want = oracle.Codec(TINY, 77).decode(codes)
    assert got.shape == want.shape == (frames * 24,)
    close(got, want, rtol=2e-4)


def test_decode_matches_transformers_fixture():
    """The GPU decoder against transformers' DAC decoder (HiggsAudioV2's
    output padding, no tanh) on the same synthetic weights
    (tests/golden/codec_tiny.json)."""
    import json
    from conftest import GOLDEN
    with open(os.path.join(GOLDEN, "codec_tiny.json")) as f:
        golden = json.load(f)
    codec = ov.Codec.synthetic(golden["config"], golden["seed"])
    got = codec.decode(np.array(golden["codes"], dtype=np.int32))
    close(got, np.array(golden["audio"]), rtol=2e-4)


@pytest.fixture(scope="module")
def released():
    cfg = ov.codec_released_config()
    return cfg, ov.Codec.synthetic(cfg, 1234), oracle.Codec(oracle.codec_released_config(), 1234)


@pytest.mark.parametrize("frames", [3, 25])
def test_released_decode_within_reference_bounds(released, frames):
    cfg, codec, model = released
    codes = np.random.default_rng(frames).integers(0, 1024, size=(8, frames)).astype(np.int32)
    got = codec.decode(codes)
    want = model.decode(codes)
    assert got.shape == want.shape == (frames * 960,)
    rms_got = float(np.sqrt(np.mean(got.astype(np.float64) ** 2)))
    rms_want = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    worst = float(np.abs(got - want).max())
    print(f"rms {rms_got:.6f} vs {rms_want:.6f}, max |d sample| {worst:.2e}")
    assert abs(rms_got - rms_want) < 1e-4
    assert worst < 1e-3


def test_decode_deterministic_and_device_entry(released):
    import torch
    cfg, codec, _ = released
    codes = np.random.default_rng(5).integers(0, 1024, size=(8, 50)).astype(np.int32)
    a = codec.decode(codes)
    b = codec.decode(codes)
    np.testing.assert_array_equal(a, b)
    codes_dev = torch.from_numpy(codes).cuda()
    audio = torch.empty(codec.samples(50), dtype=torch.float32, device="cuda")
    codec.decode_device(codes_dev, audio)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(audio.cpu().numpy(), a)
    # a shorter decode after a longer one reuses the grown buffers
    short = codec.decode(codes[:, :4])
    np.testing.assert_array_equal(short, codec.decode(codes[:, :4].copy()))


def test_decode_errors_carry_reference_prefix(released):
    _, codec, _ = released
    bad = np.zeros((8, 3), dtype=np.int32)
    bad[2, 1] = 1024
    with pytest.raises(ov.GeneratorError, match="^OmniVoice decode: code outside the codebook"):
        codec.decode(bad)
    with pytest.raises(ov.GeneratorError, match="^OmniVoice decode: no frames"):
        codec.decode(np.zeros((8, 0), dtype=np.int32))


def _checkpoint_tensors(cfg, seed):
    """The synthetic decoder written under the reference's tensor names and
    shapes (codec.cpp:112-181)."""
    v = lambda tid, shape, scale, exp=False: ov.codec_synthetic_values(
        seed, tid, 0, int(np.prod(shape)), scale, exp).reshape(shape)
    C, E, D, H, Lat = (cfg[k] for k in ("codebooks", "codebook_size", "codebook_dim",
                                        "hidden", "latent"))
    t = {}
    for c in range(C):
        p = f"quantizer.quantizers.{c}"
        t[p + ".codebook.embed"] = v(1000 + 4 * c, (E, D), 0.35)
        t[p + ".project_out.weight"] = v(1001 + 4 * c, (H, D), D ** -0.5)
        t[p + ".project_out.bias"] = v(1002 + 4 * c, (H,), 0.01)
    t["fc2.weight"] = v(1100, (Lat, H), H ** -0.5)
    t["fc2.bias"] = v(1101, (Lat,), 0.01)
    ch = cfg["channels"]
    t["acoustic_decoder.conv1.weight"] = v(1102, (ch, Lat, 7), (7 * Lat) ** -0.5)
    t["acoustic_decoder.conv1.bias"] = v(1103, (ch,), 0.01)
    for i, s in enumerate(cfg["ratios"]):
        p, base, out = f"acoustic_decoder.block.{i}", 1200 + 32 * i, ch // 2
        t[p + ".snake1.alpha"] = v(base, (1, ch, 1), 0.1, True)
        t[p + ".conv_t1.weight"] = v(base + 1, (ch, out, 2 * s), (2 * ch) ** -0.5)
        t[p + ".conv_t1.bias"] = v(base + 2, (out,), 0.01)
        for u in range(3):
            q, uid = f"{p}.res_unit{u + 1}", base + 4 + 6 * u
            t[q + ".snake1.alpha"] = v(uid, (1, out, 1), 0.1, True)
            t[q + ".conv1.weight"] = v(uid + 1, (out, out, 7), (7 * out) ** -0.5)
            t[q + ".conv1.bias"] = v(uid + 2, (out,), 0.01)
            t[q + ".snake2.alpha"] = v(uid + 3, (1, out, 1), 0.1, True)
            t[q + ".conv2.weight"] = v(uid + 4, (out, out, 1), 0.3 * out ** -0.5)
            t[q + ".conv2.bias"] = v(uid + 5, (out,), 0.01)
        ch = out
    t["acoustic_decoder.snake1.alpha"] = v(1400, (1, ch, 1), 0.1, True)
    t["acoustic_decoder.conv2.weight"] = v(1401, (1, ch, 7), 0.1 * (7 * ch) ** -0.5)
    t["acoustic_decoder.conv2.bias"] = v(1402, (1,), 0.01)
    return t


def test_checkpoint_matches_synthetic_decoder(tmp_path):
    from safetensors.numpy import save_file
    os.makedirs(tmp_path / "audio_tokenizer")
    save_file(_checkpoint_tensors(TINY, 99), str(tmp_path / "audio_tokenizer" /
                                                 "model.safetensors"))
    codes = np.random.default_rng(3).integers(0, 16, size=(3, 11)).astype(np.int32)
    from_file = ov.Codec.load(TINY, str(tmp_path)).decode(codes)
    np.testing.assert_array_equal(from_file, ov.Codec.synthetic(TINY, 99).decode(codes))
    # a tensor of the wrong shape is named
    t = _checkpoint_tensors(TINY, 99)
    t["fc2.bias"] = np.zeros(5, dtype=np.float32)
    save_file(t, str(tmp_path / "audio_tokenizer" / "model.safetensors"))
    with pytest.raises(ov.GeneratorError, match="^OmniVoice audio tokenizer: .*fc2.bias"):
        ov.Codec.load(TINY, str(tmp_path))
