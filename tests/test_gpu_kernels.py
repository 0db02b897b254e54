"""Operator parity on the MI355X: every HIP kernel, called through the C ABI,
against the CPU oracle on the same seeded inputs. Bit-exact throughout."""
import numpy as np
import pytest

from tsac_hip.synthetic import bf16_bits, bf16_float, random_linear

pytestmark = pytest.mark.gpu

EDGE_BITS = np.array([0, 0x8000, 0x0001, 0x8001, 0x3F00, 0xBF00, 0x3FC0, 0xBFC0, 0x42FE, 0xC300,
                      0x2F80, 0xAF80], np.uint16)  # tests/metal_optimized.cpp:152-153


@pytest.fixture(scope="module")
def torch():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    return torch


@pytest.fixture(scope="module")
def native():
    from tsac_hip import native

    native.library()
    return native


def dev(torch, array):
    a = np.ascontiguousarray(array)
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(a.copy()).cuda()


def host(tensor, dtype=np.uint16):
    return tensor.cpu().numpy().view(dtype)


def empty(torch, shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda")


# ---------------------------------------------------------------- qlinear

def _activations(rng, m, k, pattern=False):
    if pattern:  # tests/metal_optimized.cpp:105-108
        i = np.arange(m * k)
        return bf16_bits(((i * 73 + i // 17) % 257 - 128).astype(np.float32) * np.float32(0.03125)).reshape(m, k)
    return bf16_bits(rng.standard_normal((m, k)).astype(np.float32))


@pytest.mark.parametrize("n", [1024, 4096])
@pytest.mark.parametrize("m", [1, 3, 64, 1024, 4096])
def test_qlinear_config_shapes_match_oracle(torch, native, oracle, n, m):
    """K=1024 qlinear, GEMV, small-M and GEMM paths, against the oracle (rows sampled for large M)."""
    rng = np.random.default_rng(n * 7 + m)
    values, scales, bias = random_linear(rng, 1024, n, bias_std=0.1, row_scales=True)
    x = _activations(rng, m, 1024)
    linear = native.DeviceLinear(values, scales, bias)
    dx = dev(torch, x)
    outputs = {}
    paths = [native.PATH_GEMM] + ([native.PATH_GEMV] if m <= 8 else []) + ([native.PATH_SMALL] if m <= 1024 else [])
    for path in paths:
        y = empty(torch, (m, n), torch.int16)
        linear.apply(dx, y, path)
        outputs[path] = host(y)
    if m > 8:  # the GEMV path in blocks of 8 columns covers every row too
        y = empty(torch, (m, n), torch.int16)
        for r in range(0, m, 8):
            linear.apply(dx[r:r + 8], y[r:r + 8], native.PATH_GEMV)
        outputs[native.PATH_GEMV] = host(y)
    assert np.array_equal(outputs[native.PATH_GEMM], outputs[native.PATH_GEMV])
    if m <= 1024:
        assert np.array_equal(outputs[native.PATH_GEMM], outputs[native.PATH_SMALL])
    rows = np.arange(m) if m <= 64 else np.unique(np.r_[0, 1, 127, 128, m - 1, rng.integers(0, m, 40)])
    expected = oracle.qlinear(values, scales, bias, x[rows])
    assert np.array_equal(outputs[native.PATH_GEMM][rows], expected)


@pytest.mark.parametrize("k,n", [(512, 1536), (512, 512), (512, 2048), (2048, 512), (1024, 512), (512, 1024),
                                 (256, 256), (4096, 1024)])
@pytest.mark.parametrize("columns", [1, 2, 3, 6, 8, 14, 33, 64, 96])
def test_qlinear_reference_projection_shapes(torch, native, oracle, k, n, columns):
    """Projection shapes of the reference model at the column counts of
    tests/metal_optimized.cpp:96-146, with the integer-pattern activations."""
    rng = np.random.default_rng(k + n + columns)
    values, scales, bias = random_linear(rng, k, n, bias_std=0.1)
    x = _activations(rng, columns, k, pattern=True)
    linear = native.DeviceLinear(values, scales, bias)
    y = empty(torch, (columns, n), torch.int16)
    linear.apply(dev(torch, x), y, native.PATH_GEMM)
    expected = oracle.qlinear(values, scales, bias, x)
    assert np.array_equal(host(y), expected)
    if columns <= 8:
        linear.apply(dev(torch, x), y, native.PATH_GEMV)
        assert np.array_equal(host(y), expected)
    if columns <= 64 and k <= 2048:
        y.zero_()
        linear.apply(dev(torch, x), y, native.PATH_SMALL)
        assert np.array_equal(host(y), expected)


def test_qlinear_edge_bits_and_zero_blocks(torch, native, oracle):
    """BF16 edge patterns with whole zero blocks (tests/metal_optimized.cpp:148-203)."""
    rng = np.random.default_rng(1)
    values, scales, bias = random_linear(rng, 1024, 512)
    for columns in (3, 1, 3, 2, 6, 3, 40):
        i = np.arange(columns * 1024)
        x = np.where((i // 256) % 3 == 0, 0, EDGE_BITS[i % EDGE_BITS.size]).astype(np.uint16).reshape(columns, 1024)
        expected = oracle.qlinear(values, scales, bias, x)
        linear = native.DeviceLinear(values, scales, bias)
        for path in (native.PATH_GEMM, native.PATH_SMALL) + ((native.PATH_GEMV,) if columns <= 8 else ()):
            y = empty(torch, (columns, 512), torch.int16)
            linear.apply(dev(torch, x), y, path)
            assert np.array_equal(host(y), expected)


def test_qlinear_rejects_nonfinite(torch, native):
    rng = np.random.default_rng(2)
    linear = native.DeviceLinear(*random_linear(rng, 512, 512))
    for bad in (0x7F80, 0x7FC1):
        x = np.zeros((3, 512), np.uint16)
        x[0, 0] = bad
        y = empty(torch, (3, 512), torch.int16)
        with pytest.raises(native.HipError, match="finite"):
            linear.apply(dev(torch, x), y)


def test_qlinear_fused_residual(torch, native, oracle):
    rng = np.random.default_rng(3)
    values, scales, bias = random_linear(rng, 2048, 512)
    # 77 and 300 rows at N = 512 take the small-M kernel automatically (few GEMM tiles).
    for m, path in ((3, native.PATH_AUTO), (77, native.PATH_AUTO), (40, native.PATH_SMALL), (64, native.PATH_AUTO),
                    (300, native.PATH_AUTO), (300, native.PATH_GEMM)):
        x = _activations(rng, m, 2048)
        skip = bf16_bits(((np.arange(m * 512) % 31) - 15).astype(np.float32) / 32).reshape(m, 512)
        q = empty(torch, (m, 2048), torch.int8)
        s = empty(torch, (m, 8), torch.float32)
        native.bf8l(dev(torch, x), m, 2048, q, s)
        linear = native.DeviceLinear(values, scales, bias)
        y = dev(torch, skip)
        linear.apply_quantized(q, s, m, y, residual=y, path=path)
        plain = oracle.qlinear(values, scales, bias, x)
        expected = np.array([[oracle.add_bf16(int(a), int(b)) for a, b in zip(r1, r2)]
                             for r1, r2 in zip(skip, plain)], np.uint16)
        assert np.array_equal(host(y), expected)


def _tile_offsets(m, k):
    """Byte offset of (row, k) in the MFMA operand-tile layout of bf8l_tiles."""
    r = np.arange(m)[:, None]
    c = np.arange(k)[None, :]
    return ((r // 32) * (k // 32) + c // 32) * 1024 + ((r % 32) + 32 * ((c // 16) % 2)) * 16 + c % 16


@pytest.mark.parametrize("m,k,n", [(9, 256, 64), (130, 512, 192), (77, 2048, 512), (300, 512, 1536),
                                   (129, 4096, 1024), (1000, 1024, 320)])
def test_gemm_tiles_and_rows_layouts_agree(torch, native, oracle, m, k, n):
    """The GEMM on operand tiles (encode path), on row-major activations, and
    the GEMV in blocks of eight columns agree bit for bit with the oracle, with
    and without a residual, at row and column counts that leave partial tiles."""
    rng = np.random.default_rng(m * 31 + k + n)
    values, scales, bias = random_linear(rng, k, n, bias_std=0.1)
    x = _activations(rng, m, k)
    linear = native.DeviceLinear(values, scales, bias)
    padded = native.tile_rows(m)
    assert padded % 128 == 0 and padded >= m
    q_rows = empty(torch, (m, k), torch.int8)
    s_rows = empty(torch, (m, k // 256), torch.float32)
    native.bf8l(dev(torch, x), m, k, q_rows, s_rows)
    q_tiles = empty(torch, (padded * k,), torch.int8)
    s_tiles = empty(torch, (k // 256, padded), torch.float32)
    native.bf8l_tiles(dev(torch, x), m, k, q_tiles, s_tiles)
    # The tile layout holds the same bytes and scales as the rows.
    assert np.array_equal(host(q_tiles, np.int8)[_tile_offsets(m, k)], host(q_rows, np.int8))
    assert np.array_equal(host(s_tiles, np.float32)[:, :m].T, host(s_rows, np.float32))
    expected = oracle.qlinear(values, scales, bias, x)
    skip = bf16_bits(rng.standard_normal((m, n)).astype(np.float32))
    with_skip = np.array([[oracle.add_bf16(int(a), int(b)) for a, b in zip(r1, r2)]
                          for r1, r2 in zip(skip, expected)], np.uint16)
    for residual, want in ((False, expected), (True, with_skip)):
        results = []
        for q, s, path in ((q_tiles, s_tiles, native.PATH_GEMM_TILES), (q_rows, s_rows, native.PATH_GEMM)):
            y = dev(torch, skip) if residual else empty(torch, (m, n), torch.int16)
            linear.apply_quantized(q, s, m, y, residual=y if residual else None, path=path)
            results.append(host(y))
        y = dev(torch, skip) if residual else empty(torch, (m, n), torch.int16)
        for r in range(0, m, 8):
            linear.apply_quantized(q_rows[r:r + 8], s_rows[r:r + 8], min(8, m - r), y[r:r + 8],
                                   residual=y[r:r + 8] if residual else None, path=native.PATH_GEMV)
        results.append(host(y))
        for got in results:
            assert np.array_equal(got, want)


@pytest.mark.parametrize("k,n,with_residual", [(512, 1536, False), (2048, 512, True)])
def test_gemm_many_tiles_per_workgroup(torch, native, k, n, with_residual):
    """At the encode's 2580 x 12 rows every persistent workgroup walks several
    tiles (LDS reuse across tiles, output staging between them); the GEMM on
    operand tiles must equal the GEMV in blocks of eight columns, on two runs."""
    rng = np.random.default_rng(k + n)
    m = 30960
    linear = native.DeviceLinear(*random_linear(rng, k, n, bias_std=0.1))
    x = dev(torch, _activations(rng, m, k))
    skip = dev(torch, bf16_bits(rng.standard_normal((m, n)).astype(np.float32)))
    padded = native.tile_rows(m)
    q_tiles = empty(torch, (padded * k,), torch.int8)
    s_tiles = empty(torch, (k // 256 * padded,), torch.float32)
    native.bf8l_tiles(x, m, k, q_tiles, s_tiles)
    q_rows = empty(torch, (m, k), torch.int8)
    s_rows = empty(torch, (m, k // 256), torch.float32)
    native.bf8l(x, m, k, q_rows, s_rows)
    want = skip.clone()
    for r in range(0, m, 8):
        native_rows = min(8, m - r)
        linear.apply_quantized(q_rows[r:r + 8], s_rows[r:r + 8], native_rows, want[r:r + 8],
                               residual=want[r:r + 8] if with_residual else None, path=native.PATH_GEMV)
    want = host(want)
    for _ in range(2):
        y = skip.clone()
        linear.apply_quantized(q_tiles, s_tiles, m, y, residual=y if with_residual else None,
                               path=native.PATH_GEMM_TILES)
        assert np.array_equal(host(y), want)


def test_gemm_output_beyond_32bit_byte_range(torch, native, oracle):
    """Outputs are addressed through 32-bit buffer ranges, so an output matrix
    past 2^31 bytes takes several launches of row chunks (K=256, N=8192: 130,944
    rows per launch); rows on both sides of the chunk boundary, in both
    activation layouts and with a residual, must match the oracle."""
    rng = np.random.default_rng(31)
    k, n = 256, 8192
    m = 131072 + 300
    assert m * n * 2 > 2 ** 31
    values, scales, bias = random_linear(rng, k, n, bias_std=0.1)
    linear = native.DeviceLinear(values, scales, bias)
    x = _activations(rng, m, k)
    dx = dev(torch, x)
    rows = np.unique(np.r_[0, 1, 130943, 130944, 130945, 131071, 131072, m - 1, rng.integers(0, m, 24)])
    expected = oracle.qlinear(values, scales, bias, x[rows])
    index = torch.from_numpy(rows).cuda()
    padded = native.tile_rows(m)
    q_tiles = empty(torch, (padded * k,), torch.int8)
    s_tiles = empty(torch, (k // 256 * padded,), torch.float32)
    native.bf8l_tiles(dx, m, k, q_tiles, s_tiles)
    q_rows = empty(torch, (m, k), torch.int8)
    s_rows = empty(torch, (m, k // 256), torch.float32)
    native.bf8l(dx, m, k, q_rows, s_rows)
    y = empty(torch, (m, n), torch.int16)
    for q, s, path in ((q_tiles, s_tiles, native.PATH_GEMM_TILES), (q_rows, s_rows, native.PATH_GEMM)):
        y.zero_()
        linear.apply_quantized(q, s, m, y, path=path)
        assert np.array_equal(host(y.index_select(0, index)), expected)
    skip = bf16_bits(rng.standard_normal((rows.size, n)).astype(np.float32))
    y.zero_()
    y.index_copy_(0, index, dev(torch, skip))
    linear.apply_quantized(q_tiles, s_tiles, m, y, residual=y, path=native.PATH_GEMM_TILES)
    with_skip = np.array([[oracle.add_bf16(int(a), int(b)) for a, b in zip(r1, r2)]
                          for r1, r2 in zip(skip, expected)], np.uint16)
    assert np.array_equal(host(y.index_select(0, index)), with_skip)
    del y, q_tiles, q_rows
    torch.cuda.empty_cache()


def test_gemm_repeatable(torch, native):
    """Two launches of the persistent GEMM give identical bytes."""
    rng = np.random.default_rng(8)
    m, k, n = 4000, 512, 1536
    linear = native.DeviceLinear(*random_linear(rng, k, n))
    x = dev(torch, _activations(rng, m, k))
    outputs = []
    for _ in range(2):
        y = empty(torch, (m, n), torch.int16)
        linear.apply(x, y, native.PATH_GEMM)
        outputs.append(host(y))
    assert np.array_equal(outputs[0], outputs[1])


def test_bf8l_matches_oracle(torch, native, oracle):
    rng = np.random.default_rng(4)
    for k in (256, 512, 1024, 2048, 4096):
        x = bf16_bits((rng.standard_normal((5, k)) * 10.0 ** rng.uniform(-30, 30, (5, 1))).astype(np.float32))
        q = empty(torch, (5, k), torch.int8)
        s = empty(torch, (5, k // 256), torch.float32)
        native.bf8l(dev(torch, x), 5, k, q, s)
        for r in range(5):
            eq, es = oracle.bf8l(bf16_float(x[r]))
            assert np.array_equal(host(q, np.int8)[r], eq)
            assert np.array_equal(host(s, np.float32)[r], bf16_float(es))


# ---------------------------------------------------------------- elementwise

def test_gelu_exhaustive(torch, native, oracle):
    x = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    out = empty(torch, 65536, torch.int16)
    native.gelu(dev(torch, x), out)
    assert np.array_equal(host(out), oracle.gelu_batch(x))


def test_layer_norm_matches_oracle(torch, native, oracle):
    rng = np.random.default_rng(5)
    for width in (256, 512, 1024, 2048):
        rows = 9
        x = bf16_bits((rng.standard_normal((rows, width)) * 10.0 ** rng.uniform(-3, 3, (rows, 1))).astype(np.float32))
        x[0] = np.resize(EDGE_BITS, width)
        g = bf16_bits((1 + 0.1 * rng.standard_normal(width)).astype(np.float32))
        b = bf16_bits((0.1 * rng.standard_normal(width)).astype(np.float32))
        out = empty(torch, (rows, width), torch.int16)
        native.layer_norm(dev(torch, x), rows, width, dev(torch, g), dev(torch, b), out)
        expected = np.stack([oracle.layer_norm(r, g, b) for r in x])
        assert np.array_equal(host(out), expected)


def _tiny_rows(rng, width):
    """Rows around the magnitudes where FTZ sums start to differ from plain sums:
    values at and just below 2^-56, squares that are subnormal, sums that cancel
    to subnormals, BF16 subnormals, signed zeros and the largest finite values."""
    rows = []
    for exponent in (-56, -57, -63, -64, -70, -100, -126, -130):
        rows.append(bf16_bits((rng.standard_normal(width) * 2.0 ** exponent).astype(np.float32)))
    mixed = bf16_bits(rng.standard_normal(width).astype(np.float32))
    mixed[::3] = bf16_bits((rng.standard_normal(mixed[::3].size) * 1e-30).astype(np.float32))
    rows.append(mixed)
    boundary = np.where(rng.random(width) < 0.5, 0x2380, 0x237F).astype(np.uint16)
    boundary |= (rng.random(width) < 0.5).astype(np.uint16) << 15
    rows.append(boundary)
    cancel = bf16_bits((rng.standard_normal(width) * 2.0 ** -120).astype(np.float32))
    cancel[1::2] = cancel[0::2] ^ 0x8000  # pairs sum to signed zeros
    cancel[-1] = 0x0003
    rows.append(cancel)
    rows.append(np.resize(np.array([0x0001, 0x8001, 0x007F, 0x807F, 0x0000, 0x8000], np.uint16), width))
    rows.append(np.resize(np.array([0x7F7F, 0xFF7F, 0x0080, 0x8080], np.uint16), width))
    return np.stack(rows)


def test_layer_norm_small_magnitudes(torch, native, oracle):
    rng = np.random.default_rng(15)
    for width in (256, 512, 2048):
        x = _tiny_rows(rng, width)
        rows = x.shape[0]
        g = bf16_bits((1 + 0.1 * rng.standard_normal(width)).astype(np.float32))
        b = bf16_bits((0.1 * rng.standard_normal(width)).astype(np.float32))
        out = empty(torch, (rows, width), torch.int16)
        native.layer_norm(dev(torch, x), rows, width, dev(torch, g), dev(torch, b), out)
        expected = np.stack([oracle.layer_norm(r, g, b) for r in x])
        assert np.array_equal(host(out), expected)


def test_bf8l_small_magnitudes(torch, native, oracle):
    rng = np.random.default_rng(16)
    for k in (256, 512, 2048):
        x = _tiny_rows(rng, k)
        rows = x.shape[0]
        q = empty(torch, (rows, k), torch.int8)
        s = empty(torch, (rows, k // 256), torch.float32)
        native.bf8l(dev(torch, x), rows, k, q, s)
        for r in range(rows):
            eq, es = oracle.bf8l(bf16_float(x[r]))
            assert np.array_equal(host(q, np.int8)[r], eq), r
            assert np.array_equal(host(s, np.float32)[r], bf16_float(es)), r


def test_softmax_matches_oracle(torch, native, oracle):
    rng = np.random.default_rng(6)
    for amplitude in (0.0, 1 / 32, 1.0, 40.0, 300.0):  # tests/metal_range.cpp:144
        x = bf16_bits((rng.standard_normal((7, 1024)) * amplitude).astype(np.float32))
        out = empty(torch, (7, 1024), torch.int16)
        native.softmax(dev(torch, x), 7, 1024, out)
        assert np.array_equal(host(out), np.stack([oracle.softmax(r) for r in x]))
    bad = np.zeros((1, 1024), np.uint16)
    bad[0, 5] = 0x7F80
    with pytest.raises(native.HipError):
        native.softmax(dev(torch, bad), 1, 1024, out)


def test_rotary_and_add_match_oracle(torch, native, oracle):
    rng = np.random.default_rng(7)
    v = bf16_bits(rng.standard_normal(4096).astype(np.float32) * 4)
    c = bf16_bits(rng.uniform(-1, 1, 4096).astype(np.float32))
    out = empty(torch, 4096, torch.int16)
    native.rotary(dev(torch, v), dev(torch, c), out)
    assert np.array_equal(host(out), oracle.rotary(v, c))
    a = bf16_bits(rng.standard_normal((6, 512)).astype(np.float32))
    b = bf16_bits(rng.standard_normal((3, 512)).astype(np.float32))
    out = empty(torch, (6, 512), torch.int16)
    native.add(dev(torch, a), dev(torch, b), 6, 512, 3, out)
    expected = np.array([[oracle.add_bf16(int(x), int(y)) for x, y in zip(a[r], b[r % 3])] for r in range(6)],
                        np.uint16)
    assert np.array_equal(host(out), expected)


# ---------------------------------------------------------------- attention

def _pattern_attention(heads, hw, frames):
    width = heads * hw
    i = np.arange(width)
    q = bf16_bits((((i * 37 + 19) % 257) - 128).astype(np.float32) / np.float32(128))
    i = np.arange(frames * width)
    k = bf16_bits((((i * 73 + i // 17) % 257) - 128).astype(np.float32) / np.float32(64))
    v = bf16_bits((((i * 31 + i // 7) % 127) - 63).astype(np.float32) / np.float32(32))
    return q, k, v


@pytest.mark.parametrize("heads,hw", [(4, 128), (16, 64), (1, 128), (2, 64)])
def test_attention_decode_matches_oracle(torch, native, oracle, heads, hw):
    """One query over T cached keys (tests/attention.cpp frame sweep + the long histories)."""
    rng = np.random.default_rng(heads * hw)
    scale = np.float32(1 / np.sqrt(hw))
    for frames in (1, 3, 4, 8, 9, 15, 16, 17, 33, 63, 64, 65, 127, 128, 129, 257, 1024, 1290):
        for pattern in (True, False):
            if pattern:
                q, k, v = _pattern_attention(heads, hw, frames)
            else:
                w = heads * hw
                q = bf16_bits(rng.standard_normal(w).astype(np.float32) * 2)
                k = bf16_bits(rng.standard_normal(frames * w).astype(np.float32) * 2)
                v = bf16_bits(rng.standard_normal(frames * w).astype(np.float32))
            for prefill in (False, True):
                out = empty(torch, heads * hw, torch.int16)
                native.attention(dev(torch, q), dev(torch, k), dev(torch, v), 0, 1, frames, heads, hw, scale,
                                 prefill, out)
                assert np.array_equal(host(out), oracle.attention(q, k, v, heads, hw, scale, prefill)), \
                    (frames, pattern, prefill)


@pytest.mark.parametrize("heads,hw", [(1, 128), (2, 64)])
def test_attention_decode_long_histories(torch, native, oracle, heads, hw):
    """Histories past 64 blocks (the merge's running-maximum scan carried from
    one chunk of 64 blocks to the next), the longest one workgroup's LDS holds
    (256 blocks), one block more (partials in scratch and a merge launch), and
    a block whose scores are all NaN (the merge's plain sequential loop)."""
    rng = np.random.default_rng(21 + hw)
    scale = np.float32(1 / np.sqrt(hw))
    w = heads * hw
    cases = [(frames, False) for frames in (4097, 8191, 16384, 16385)] + [(5000, True)]
    for frames, poisoned in cases:
        q = bf16_bits(rng.standard_normal(w).astype(np.float32) * 2)
        k = bf16_bits(rng.standard_normal(frames * w).astype(np.float32) * 2)
        v = bf16_bits(rng.standard_normal(frames * w).astype(np.float32))
        if poisoned:
            q[3] = 0  # 0 * inf = NaN in every score of block 70
            k.reshape(frames, w)[70 * 64:71 * 64, 3] = 0x7F80
        out = empty(torch, w, torch.int16)
        native.attention(dev(torch, q), dev(torch, k), dev(torch, v), 0, 1, frames, heads, hw, scale, False, out)
        assert np.array_equal(host(out), oracle.attention(q, k, v, heads, hw, scale, False)), (frames, poisoned)


def test_attention_decode_batched_sequences(torch, native, oracle):
    """Three lanes with their own caches, as the decode step runs them."""
    rng = np.random.default_rng(11)
    heads, hw, frames, lanes, extent = 4, 128, 200, 3, 256
    w = heads * hw
    q = bf16_bits(rng.standard_normal((lanes, w)).astype(np.float32))
    k = bf16_bits(rng.standard_normal((lanes, extent, w)).astype(np.float32))
    v = bf16_bits(rng.standard_normal((lanes, extent, w)).astype(np.float32))
    out = empty(torch, (lanes, w), torch.int16)
    scale = np.float32(0.0883883461356163)
    native.attention(dev(torch, q), dev(torch, k), dev(torch, v), extent * w, lanes, frames, heads, hw, scale,
                     False, out)
    for lane in range(lanes):
        expected = oracle.attention(q[lane], k[lane, :frames], v[lane, :frames], heads, hw, scale, False)
        assert np.array_equal(host(out)[lane], expected)


def test_attention_decode_split_scratch_and_capture(torch, native, oracle):
    """Histories split over several workgroups per (sequence, head), in shapes
    that grow, shrink and grow the per-stream scratch in turn (its arrival
    counters must be zero again after every launch), then one such call
    captured in a graph and replayed with eager calls on the same stream
    between the replays."""
    rng = np.random.default_rng(31)

    def case(sequences, heads, hw, frames):
        w = heads * hw
        q = bf16_bits(rng.standard_normal((sequences, w)).astype(np.float32) * 2)
        k = bf16_bits(rng.standard_normal((sequences, frames, w)).astype(np.float32) * 2)
        v = bf16_bits(rng.standard_normal((sequences, frames, w)).astype(np.float32))
        scale = np.float32(1 / np.sqrt(hw))
        expected = np.stack([oracle.attention(q[s], k[s], v[s], heads, hw, scale, False) for s in range(sequences)])
        args = (dev(torch, q), dev(torch, k), dev(torch, v), frames * w, sequences, frames, heads, hw, scale, False)
        return args, expected

    shapes = [(1, 2, 64, 1290), (3, 16, 64, 2580), (1, 2, 64, 700), (2, 4, 128, 5000), (3, 16, 64, 2580),
              (2, 1, 128, 257)]
    cases = [case(*shape) for shape in shapes]
    for shape, (args, expected) in zip(shapes, cases):
        out = empty(torch, expected.shape, torch.int16)
        native.attention(*args, out)
        assert np.array_equal(host(out), expected), shape
    (args, expected), (other, other_expected) = cases[1], cases[3]
    out = empty(torch, expected.shape, torch.int16)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        native.attention(*args, out)
    for replay in range(3):
        out.zero_()
        other_out = empty(torch, other_expected.shape, torch.int16)
        native.attention(*other, other_out)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(out), expected), replay
        assert np.array_equal(host(other_out), other_expected), replay


@pytest.mark.parametrize("heads,hw,rotary", [(4, 128, True), (4, 128, False), (16, 64, True)])
def test_attention_causal_matches_oracle(torch, native, oracle, heads, hw, rotary):
    """Every query of several causal sequences (one with a replay prefix) against
    the oracle's single-query attention over keys 0..t."""
    rng = np.random.default_rng(heads + hw + rotary)
    w = heads * hw
    lengths = [1, 12, 70, 300, 129]
    replays = [0, 0, 0, 256, 5]
    starts = np.cumsum([0] + lengths[:-1]).astype(np.int32)
    rows = sum(lengths)
    qkv = bf16_bits(rng.standard_normal((rows, 3 * w)).astype(np.float32))
    context = max(lengths)
    rotations = bf16_bits(rng.uniform(-1, 1, (context, hw)).astype(np.float32)) if rotary else None
    scale = np.float32(1 / np.sqrt(hw))
    out = empty(torch, (rows, w), torch.int16)
    native.attention_causal(dev(torch, qkv), heads, hw, dev(torch, starts), dev(torch, np.array(lengths, np.int32)),
                            dev(torch, np.array(replays, np.int32)), len(lengths), max(lengths),
                            dev(torch, rotations) if rotary else None, scale, out)
    got = host(out)
    for s, (start, length, replay) in enumerate(zip(starts, lengths, replays)):
        seq = qkv[start:start + length]
        q, k, v = seq[:, :w].copy(), seq[:, w:2 * w].copy(), seq[:, 2 * w:].copy()
        if rotary:
            for t in range(length):
                for h in range(heads):
                    q[t, h * hw:(h + 1) * hw] = oracle.rotary(q[t, h * hw:(h + 1) * hw], rotations[t])
                    k[t, h * hw:(h + 1) * hw] = oracle.rotary(k[t, h * hw:(h + 1) * hw], rotations[t])
        for t in range(length):
            expected = oracle.attention(q[t], k[:t + 1], v[:t + 1], heads, hw, scale, t < replay)
            assert np.array_equal(got[start + t], expected), (s, t)


def test_calibration_probes(torch, native):
    """The calibration kernels run, report their operation count, and reject
    sizes they cannot stream."""
    data = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    native.probe_read(data)
    assert native.probe_mfma(8, 3) == 8 * 4 * 4 * 3 * 65536
    torch.cuda.synchronize()
    with pytest.raises(native.HipError, match="multiple of 64 KiB"):
        native.probe_read(data[:1000])


@pytest.mark.parametrize("heads,hw", [(16, 64), (4, 128)])
@pytest.mark.parametrize("lengths,kind", [([65, 31, 33, 64, 1] * 8, "normal"), ([330], "normal"), ([129, 96], "spread"),
                                          ([100], "dead infinity"), ([70], "zeros"), ([65], "tiny"), ([12] * 9, "normal"),
                                          ([1, 16, 15, 2, 7], "spread"), ([9, 16], "zeros"), ([16], "tiny"),
                                          ([12, 16, 1, 7, 2], "rotated"), ([65, 31, 8], "rotated")])
def test_attention_causal_branches(torch, native, oracle, heads, hw, lengths, kind):
    """The causal kernels' own choices: sequences of at most 16 rows and longer ones, edges
    of the query and 64-key tiles, scores more than 87 below the maximum (where weights
    and their sums meet subnormals), and the last block's dead keys, whose values may be
    infinite, and whose terms must not turn a zero sum's sign; replay counts of none,
    some, all and more than all of a sequence's rows."""
    rng = np.random.default_rng(sum(lengths) + hw)
    w, rows = heads * hw, sum(lengths)
    replays = [(0, n // 2, n, n + 9, 1)[i % 5] for i, n in enumerate(lengths)]
    if len(lengths) == 1:
        replays = [lengths[0] // 2]
    qkv = rng.standard_normal((rows, 3 * w)).astype(np.float32)
    if kind == "spread":
        qkv[:, :w] *= 60
    elif kind == "dead infinity":
        qkv[90, 2 * w:] = np.inf
    elif kind == "zeros":
        qkv[:, 2 * w:2 * w + hw] = 0
        qkv[::3, 2 * w + hw:] *= -0.0
    elif kind == "tiny":
        qkv[:, :w] *= 60
        qkv[:, 2 * w:] *= 1e-38
    qkv = bf16_bits(qkv)
    starts = np.cumsum([0] + lengths[:-1]).astype(np.int32)
    scale = np.float32(1 / np.sqrt(hw))
    out = empty(torch, (rows, w), torch.int16)
    rotations = bf16_bits(rng.uniform(-1, 1, (max(lengths), hw)).astype(np.float32)) if kind == "rotated" else None
    native.attention_causal(dev(torch, qkv), heads, hw, dev(torch, starts), dev(torch, np.array(lengths, np.int32)),
                            dev(torch, np.array(replays, np.int32)), len(lengths), max(lengths),
                            dev(torch, rotations) if kind == "rotated" else None, scale, out)
    got = host(out)
    for start, length, replay in list(zip(starts, lengths, replays))[:5]:
        seq = qkv[start:start + length]
        q, k, v = seq[:, :w].copy(), seq[:, w:2 * w].copy(), seq[:, 2 * w:].copy()
        if kind == "rotated":
            for part in (q, k):
                for t in range(length):
                    for h in range(0, w, hw):
                        part[t, h:h + hw] = oracle.rotary(part[t, h:h + hw], rotations[t])
        for t in range(length):
            expected = oracle.attention(q[t], k[:t + 1], v[:t + 1], heads, hw, scale, t < replay)
            finite = np.isfinite(bf16_float(expected))
            assert np.array_equal(got[start + t][finite], expected[finite]), (length, t)
            assert not np.isfinite(bf16_float(got[start + t][~finite])).any()


@pytest.mark.parametrize("heads,hw", [(8, 64), (4, 128)])
@pytest.mark.parametrize("lengths,pairs", [([64, 33, 17, 8], 32), ([64, 33, 17, 49], 1280), ([330], 8), ([129, 96], 16),
                                           ([65, 128], 1024), ([129, 70, 100], 480), ([129, 70, 100], 96),
                                           ([330, 257], 32)])
@pytest.mark.parametrize("kind", ["normal", "spread", "zeros", "dead infinity"])
def test_attention_causal_workgroups(torch, native, oracle, heads, hw, lengths, pairs, kind):
    """Every choice of waves and queries a workgroup, by the count of (sequence, head)
    pairs: the same sequences again and again equal the first ones, which equal the
    oracle; rotated in the kernel, they equal a launch of one set. Some sequences have
    replayed rows, which round the values of queries below 64."""
    rng = np.random.default_rng(sum(lengths) + hw)
    w, rows, sets = heads * hw, sum(lengths), max(1, pairs // (heads * len(lengths)))
    replays = [(40, 0, length + 1, 5)[i % 4] for i, length in enumerate(lengths)]
    qkv = rng.standard_normal((rows, 3 * w)).astype(np.float32)
    if kind == "spread":
        qkv[:, :w] *= 60
    elif kind == "zeros":
        qkv[:, 2 * w:2 * w + hw] = 0
        qkv[::3, 2 * w + hw:] *= -0.0
    elif kind == "dead infinity":
        qkv[lengths[0] - 2, 2 * w:] = np.inf
    qkv = bf16_bits(qkv)
    angles = rng.standard_normal((max(lengths), hw // 2))
    rotations = bf16_bits(np.stack([np.cos(angles), np.sin(angles)], axis=-1).reshape(-1, hw).astype(np.float32))
    scale = np.float32(1 / np.sqrt(hw))

    def run(n, rotated):
        many = np.array(lengths * n, np.int32)
        starts = np.cumsum(np.concatenate([[0], many[:-1]])).astype(np.int32)
        out = empty(torch, (rows * n, w), torch.int16)
        native.attention_causal(dev(torch, np.tile(qkv, (n, 1))), heads, hw, dev(torch, starts), dev(torch, many),
                                dev(torch, np.array(replays * n, np.int32)), len(many), max(lengths),
                                dev(torch, rotations) if rotated else None, scale, out)
        return host(out).reshape(n, rows, w)

    assert np.array_equal(run(sets, True), np.tile(run(1, True), (sets, 1, 1)))
    got = run(sets, False)
    assert np.array_equal(got, np.tile(got[:1], (sets, 1, 1)))
    start = 0
    for length, replay in zip(lengths, replays):
        seq = qkv[start:start + length]
        q, k, v = seq[:, :w].copy(), seq[:, w:2 * w].copy(), seq[:, 2 * w:].copy()
        for t in range(length):
            expected = oracle.attention(q[t], k[:t + 1], v[:t + 1], heads, hw, scale, t < replay)
            finite = np.isfinite(bf16_float(expected))
            assert np.array_equal(got[0, start + t][finite], expected[finite]), (length, t)
            assert not np.isfinite(bf16_float(got[0, start + t][~finite])).any()
        start += length


@pytest.mark.parametrize("heads,hw,lengths,sequences", [(8, 64, [256, 250, 193], 480), (8, 64, [384, 330], 536), (8, 64, [200, 70, 64, 1], 800),
                                                        (8, 64, [65, 64, 30], 900), (4, 128, [96, 65, 7], 1200)])
def test_attention_causal_of_full_devices(torch, native, oracle, heads, hw, lengths, sequences):
    """Launches that fill the device with workgroups of one wave (of 32 queries for the first
    set on 256 compute units, two waves for the second, of 16 for the others): the
    sequences lie over the rows of the first few, which equal the oracle."""
    rng = np.random.default_rng(sum(lengths))
    w, rows, n = heads * hw, sum(lengths), len(lengths)
    qkv = bf16_bits(rng.standard_normal((rows, 3 * w)).astype(np.float32))
    qkv[5, 2 * w:] = bf16_bits(np.zeros(w, np.float32))
    starts = np.resize(np.cumsum([0] + lengths[:-1]), sequences).astype(np.int32)
    replays = [(40, 0, length + 1, 5)[i % 4] for i, length in enumerate(lengths)]
    rotations = bf16_bits(rng.uniform(-1, 1, (max(lengths), hw)).astype(np.float32))
    scale = np.float32(1 / np.sqrt(hw))
    for rotated in (True, False):
        out = empty(torch, (rows, w), torch.int16)
        native.attention_causal(dev(torch, qkv), heads, hw, dev(torch, starts),
                                dev(torch, np.resize(lengths, sequences).astype(np.int32)),
                                dev(torch, np.resize(replays, sequences).astype(np.int32)), sequences, max(lengths),
                                dev(torch, rotations) if rotated else None, scale, out)
        got = host(out)
        for start, length, replay in zip(starts[:n], lengths, replays):
            seq = qkv[start:start + length]
            q, k, v = seq[:, :w].copy(), seq[:, w:2 * w].copy(), seq[:, 2 * w:].copy()
            if rotated:
                for part in (q, k):
                    for t in range(length):
                        for h in range(0, w, hw):
                            part[t, h:h + hw] = oracle.rotary(part[t, h:h + hw], rotations[t])
            for t in range(length):
                expected = oracle.attention(q[t], k[:t + 1], v[:t + 1], heads, hw, scale, t < replay)
                assert np.array_equal(got[start + t], expected), (rotated, length, t)


@pytest.mark.parametrize("sequences,length", [(4_300_000, 1), (300_000, 20)])
def test_attention_causal_of_very_many_sequences(torch, native, sequences, length):
    """More (sequence, head) pairs than one launch takes. The sequences lie over the same
    few rows, so that each of them gives what a call of one of each gives."""
    heads, hw, starts = 16, 64, 61
    rng = np.random.default_rng(length)
    w = heads * hw
    qkv = dev(torch, bf16_bits(rng.standard_normal((starts * length, 3 * w)).astype(np.float32)))
    scale = np.float32(1 / np.sqrt(hw))

    def run(n):
        start = (torch.arange(n, device="cuda") % starts * length).to(torch.int32)
        lengths, replay = torch.full_like(start, length), torch.zeros_like(start)
        if n > starts:
            # the last of them alone, where an earlier slice does not reach
            start[-1], qkv_last = starts * length, torch.cat([qkv, qkv[:length]])
        else:
            qkv_last = qkv
        out = torch.zeros((qkv_last.shape[0], w), dtype=torch.int16, device="cuda")
        native.attention_causal(qkv_last, heads, hw, start, lengths, replay, n, length, None, scale, out)
        return host(out)

    few, many = run(starts), run(sequences)
    assert np.array_equal(many[:starts * length], few)
    assert np.array_equal(many[starts * length:], few[:length])


def test_attention_causal_with_a_loose_bound(torch, native):
    """max_length bounds the lengths; tiles past a sequence's end do nothing, however many."""
    heads, hw, lengths = 2, 64, [130, 17, 64, 1]
    rng = np.random.default_rng(3)
    w, rows = heads * hw, sum(lengths)
    qkv = dev(torch, bf16_bits(rng.standard_normal((rows, 3 * w)).astype(np.float32)))
    starts = dev(torch, np.cumsum([0] + lengths[:-1]).astype(np.int32))
    args = (heads, hw, starts, dev(torch, np.array(lengths, np.int32)), dev(torch, np.zeros(4, np.int32)), 4)
    tight = empty(torch, (rows, w), torch.int16)
    native.attention_causal(qkv, *args, 130, None, np.float32(0.125), tight)
    for bound in (2_200_000, 4_194_240):
        loose = empty(torch, (rows, w), torch.int16)
        native.attention_causal(qkv, *args, bound, None, np.float32(0.125), loose)
        assert np.array_equal(host(loose), host(tight)), bound


@pytest.mark.parametrize("k", [256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("columns", range(1, 9))
def test_qlinear_quantises_in_the_gemv(torch, native, oracle, k, columns):
    """Up to 8 rows the projection quantises inside the GEMV; where the output overlaps
    the input it takes two launches, and an output over the input must still be made
    from the input as it was. A nonfinite input fails, and the next call does not."""
    rng = np.random.default_rng(k + columns)
    values, scales, bias = random_linear(rng, k, k)
    linear = native.DeviceLinear(values, scales, bias)
    x = _activations(rng, columns, k)
    x[0, :256] = 0
    expected = oracle.qlinear(values, scales, bias, x)
    dx, y = dev(torch, x), empty(torch, (columns, k), torch.int16)
    linear.apply(dx, y)
    assert np.array_equal(host(y), expected)
    bad = x.copy()
    bad[columns - 1, k - 1] = 0x7F80
    with pytest.raises(native.HipError, match="finite"):
        linear.apply(dev(torch, bad), y)
    linear.apply(dx, dx)
    assert np.array_equal(host(dx), expected)


@pytest.mark.parametrize("count", [1, 7, 8, 9, 2047, 2048, 2055, 65536 + 3])
def test_gelu_vectors_and_remainders(torch, native, oracle, count):
    x = np.random.default_rng(count).integers(0, 65536, count).astype(np.uint16)
    out = empty(torch, (count + 8,), torch.int16)
    out.fill_(77)
    native.gelu(dev(torch, x), out[:count])
    assert np.array_equal(host(out)[:count], oracle.gelu_batch(x))
    assert (host(out)[count:] == 77).all()


@pytest.mark.parametrize("rows,width,period", [(1, 8, 1), (5, 24, 3), (7, 20, 2), (4, 512, 4), (3, 512, 100), (9, 1, 2),
                                               (257, 1024, 12)])
def test_add_vectors_and_periods(torch, native, rows, width, period):
    """Rows of whole vectors or not, the second operand's rows repeating or not."""
    rng = np.random.default_rng(rows * width)
    a = bf16_bits(rng.standard_normal((rows, width)).astype(np.float32))
    b = bf16_bits(rng.standard_normal((period, width)).astype(np.float32))
    out = empty(torch, (rows, width), torch.int16)
    native.add(dev(torch, a), dev(torch, b), rows, width, period, out)
    assert np.array_equal(host(out), bf16_bits(bf16_float(a) + bf16_float(b[np.arange(rows) % period])))


@pytest.mark.parametrize("width", [256, 512, 1024, 2048])
def test_layer_norm_of_many_rows(torch, native, oracle, width):
    """A row per wave from 2,048 rows on (on 256 compute units): the same rows give the
    bits of a call of few rows, which spreads them."""
    rng = np.random.default_rng(width)
    rows = 2049
    x = bf16_bits(rng.standard_normal((rows, width)).astype(np.float32))
    x[::7] = bf16_bits((rng.standard_normal((len(x[::7]), width)) * 1e-19).astype(np.float32))
    gain, bias = (dev(torch, bf16_bits(rng.standard_normal(width).astype(np.float32))) for _ in range(2))
    many, few = (empty(torch, (rows, width), torch.int16) for _ in range(2))
    native.layer_norm(dev(torch, x), rows, width, gain, bias, many)
    for r in range(0, rows, 683):
        native.layer_norm(dev(torch, x[r:r + 683]), min(683, rows - r), width, gain, bias, few[r:r + 683])
    assert np.array_equal(host(many), host(few))
    # at addresses that are multiples of two only, and in place
    shifted = [torch.empty(t.numel() + 1, dtype=torch.int16, device="cuda")[1:].copy_(t.flatten())
               for t in (dev(torch, x), gain, bias)]
    native.layer_norm(shifted[0], rows, width, shifted[1], shifted[2], shifted[0])
    assert np.array_equal(host(shifted[0]).reshape(rows, width), host(few))


@pytest.mark.parametrize("k", [256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("rows", [1, 5, 33, 130])
def test_quantised_tiles_of_wide_rows(torch, native, oracle, k, rows):
    """Rows of 2048 and 4096 values in operand tiles, 8 rows a wave, against the row-major call."""
    rng = np.random.default_rng(k + rows)
    x = dev(torch, bf16_bits(rng.standard_normal((rows, k)).astype(np.float32)))
    padded = native.tile_rows(rows)
    q, s = empty(torch, (rows, k), torch.int8), empty(torch, (rows, k // 256), torch.float32)
    tq, ts = empty(torch, (padded * k,), torch.int8), empty(torch, (k // 256, padded), torch.float32)
    native.bf8l(x, rows, k, q, s)
    native.bf8l_tiles(x, rows, k, tq, ts)
    m, j = np.arange(rows)[:, None], np.arange(k)[None, :]
    at = ((m // 32) * (k // 32) + j // 32) * 1024 + ((m % 32) + 32 * ((j // 16) % 2)) * 16 + j % 16
    assert np.array_equal(tq.cpu().numpy()[at], q.cpu().numpy())
    assert np.array_equal(ts.cpu().numpy()[:, :rows].T, s.cpu().numpy())


def test_qlinear_calls_overlap_on_threads(torch, native):
    """Calls of different sizes on threads and streams of their own share the kept buffers:
    each gives what it gives alone."""
    import threading

    rng = np.random.default_rng(5)
    linear = native.DeviceLinear(*random_linear(rng, 1024, 1024))
    rows = (5, 40, 700, 5000, 30000)
    inputs = [dev(torch, bf16_bits(rng.standard_normal((m, 1024)).astype(np.float32))) for m in rows]
    outputs = [[empty(torch, (m, 1024), torch.int16) for _ in range(8)] for m in rows]
    alone = [empty(torch, (m, 1024), torch.int16) for m in rows]
    for x, y in zip(inputs, alone):
        linear.apply(x, y)
    torch.cuda.synchronize()
    failures = []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            for y in outputs[i]:
                linear.apply(inputs[i], y, stream=stream)
        except Exception as e:  # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(rows))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
    for i, m in enumerate(rows):
        assert all(bool((y == alone[i]).all()) for y in outputs[i]), m


def test_qlinear_buffer_grows_beside_a_capture(torch, native):
    """One thread's call allocates its buffer while another thread's stream is captured in
    the thread-local mode (the global one forbids the call's wait for its stream);
    neither disturbs the other, and the graph replays like its eager calls."""
    import threading

    rng = np.random.default_rng(6)
    linear = native.DeviceLinear(*random_linear(rng, 1024, 256))
    x = dev(torch, bf16_bits(rng.standard_normal((150000, 1024)).astype(np.float32)))
    y, alone = empty(torch, (150000, 256), torch.int16), empty(torch, (150000, 256), torch.int16)
    small, wanted, captured = dev(torch, np.arange(65536, dtype=np.uint16)), *(empty(torch, (65536,), torch.int16)
                                                                               for _ in range(2))
    native.gelu(small, wanted)
    stream, capturing = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    failures = []

    def work():
        try:
            linear.apply(x, y, stream=stream)
        except Exception as e:  # noqa: BLE001
            failures.append(e)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=capturing, capture_error_mode="thread_local"):
        native.gelu(small, captured)
        thread = threading.Thread(target=work)
        thread.start()
        thread.join()
    assert not failures, failures
    linear.apply(x, alone)
    assert bool((y == alone).all())
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert bool((captured == wanted).all())
