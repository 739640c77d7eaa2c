"""Parity of the HIP library with the CPU oracle, through the C ABI.

Known-answer and cross-path checks follow the reference's device probe
(tests/cpp/muse_glimmer_cuda_kernel_probe.cpp:650-1904).  The bar, from the
build's contract: dequantized weights bit-exact; float outputs within
max|y - ref| / max|ref| <= 2e-3 of the CPU engine's double-accumulate matmul;
argmax indices exact.
"""
import ctypes
import struct

import numpy as np
import pytest

from neuralfn_amd import kquant, tile_ops

pytestmark = pytest.mark.gpu

TOLERANCE = 2e-3  # max relative error allowed against the CPU oracle
K_ENCODINGS = [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K]
ALL_PACKED = K_ENCODINGS + [kquant.Q8_0]


def torch_():
    import torch
    return torch


def to_device(array, device):
    return torch_().from_numpy(np.ascontiguousarray(array)).to(device)


def normalised_error(actual, expected):
    scale = np.max(np.abs(expected))
    return float(np.max(np.abs(actual.astype(np.float64) - expected.astype(np.float64))) / scale)


def assert_bits_equal(a, b, label=""):
    a = a.detach().cpu().numpy() if hasattr(a, "detach") else a
    b = b.detach().cpu().numpy() if hasattr(b, "detach") else b
    assert a.shape == b.shape, label
    mismatch = np.flatnonzero(a.reshape(-1).view(np.uint32) != b.reshape(-1).view(np.uint32))
    assert mismatch.size == 0, f"{label}: {mismatch.size} values differ, first at {mismatch[:4]}"


def random_packed(encoding, out_dim, in_dim, seed):
    rng = np.random.default_rng(seed)
    elements, nbytes = kquant.BLOCKS[encoding]
    blocks = rng.integers(0, 256, (out_dim * in_dim // elements, nbytes), dtype=np.uint8)
    offsets = {kquant.Q4_K: (0, 2), kquant.Q5_K: (0, 2), kquant.Q6_K: (208,), kquant.Q8_0: (0,)}
    for offset in offsets[encoding]:
        blocks[:, offset + 1] = (blocks[:, offset + 1] & 0x83) | 0x24
    return blocks.reshape(-1)


def probe_packed(encoding, out_dim, in_dim, seed):
    """make_packed of the reference probe (:1290-1327): patterned bytes, fixed d/dmin."""
    _, nbytes = kquant.BLOCKS[encoding]
    total = kquant.packed_nbytes(encoding, out_dim, in_dim)
    index = np.arange(total, dtype=np.uint64)
    packed = ((index * np.uint64(seed * 2 + 17) + np.uint64(seed)) & np.uint64(0xFF)).astype(np.uint8)
    blocks = packed.reshape(out_dim, in_dim // 256, nbytes)
    rows = np.arange(out_dim)[:, None]
    if encoding in (kquant.Q4_K, kquant.Q5_K):
        blocks[:, :, 0], blocks[:, :, 1], blocks[:, :, 2], blocks[:, :, 3] = 0x00, 0x28, 0x00, 0x24
        for scale in range(12):
            blocks[:, :, 4 + scale] = (1 + (scale + rows + seed) % 4).astype(np.uint8)
    else:
        for scale in range(16):
            blocks[:, :, 192 + scale] = (((scale + rows + seed) % 11 - 5) & 0xFF).astype(np.uint8)
        blocks[:, :, 208], blocks[:, :, 209] = 0x00, 0x28
    return packed


# ---------------------------------------------------------------- dequantize

@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_dequantize_bit_exact(cuda, oracle, encoding):
    out_dim, in_dim = 37, 1024
    if encoding in (kquant.F32, kquant.BF16):
        packed = kquant.quantize(encoding, kquant.synthetic_weights(3, out_dim, in_dim))
    else:
        packed = random_packed(encoding, out_dim, in_dim, 21 + encoding)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    actual = tile_ops.dequantize(weight).cpu().numpy()
    expected = oracle.dequantize(encoding, packed, out_dim, in_dim)
    assert_bits_equal(actual, expected, kquant.NAMES[encoding])


@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_dequantize_bit_exact_quantized_weights(cuda, oracle, encoding):
    out_dim, in_dim = 64, 6656
    packed = kquant.quantize(encoding, kquant.synthetic_weights(17, out_dim, in_dim))
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    assert_bits_equal(tile_ops.dequantize(weight), oracle.dequantize(encoding, packed, out_dim, in_dim))


def test_q4_k_known_answer_through_the_abi(cuda, oracle):
    # probe :650-746
    block = bytes([0x00, 0x3C, 0x00, 0x38]) + bytes(range(1, 9)) + bytes(4) + bytes([0x21] * 128)
    packed = np.frombuffer(block, np.uint8).copy()
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, packed, 1, 256)
    values = tile_ops.dequantize(weight).cpu().numpy()[0]
    assert np.all(values[:32] == -1.5) and np.all(values[32:64] == 1.0)
    assert np.all(values[64:96] == -0.5) and np.all(values[96:128] == 4.0)
    x = ((np.arange(256) % 17 - 8) / 19.0).astype(np.float32)[None, :]
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    expected = float(np.dot(values.astype(np.float64), x[0].astype(np.float64)))
    assert abs(y[0, 0] - expected) <= 2e-4


# ------------------------------------------------------- generic float linear

@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_generic_linear_rows5_with_bias(cuda, oracle, encoding):
    # probe :748-897: rows 5, out 5, in 512, patterned bytes, bias, tol 5e-3 absolute
    rows, out_dim, in_dim = 5, 5, 512
    if encoding in (kquant.F32, kquant.BF16):
        packed = kquant.quantize(encoding, kquant.synthetic_weights(4, out_dim, in_dim, 1.0))
    else:
        packed = kquant.patterned_bytes(encoding, out_dim, in_dim)
    r, c = np.arange(rows)[:, None], np.arange(in_dim)[None, :]
    x = (((r * 37 + c * 13) % 257 - 128) / 257.0).astype(np.float32)
    bias = ((np.arange(out_dim) - 2) / 7.0).astype(np.float32)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda), to_device(bias, cuda)).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x, bias=bias)
    assert np.max(np.abs(y - expected)) <= 5e-3
    assert normalised_error(y, expected) <= 1e-5


@pytest.mark.parametrize("rows", [1, 2, 3, 7, 16, 23])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_generic_linear_against_oracle(cuda, oracle, encoding, rows):
    out_dim, in_dim = 257, 1024
    packed = kquant.quantize(encoding, kquant.synthetic_weights(31 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(77 + rows, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= TOLERANCE


@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_generic_linear_many_rows_decodes_every_weight_exactly(cuda, oracle, encoding):
    """More than 16 rows of the generic linear run on the float matrix cores.  One-hot input
    rows make every output a single product with 1.0, so the result is the decoded weight
    matrix itself and has to equal the dequantize entry point's bit for bit (all eight
    sub-blocks of a K-quant block, both halves of every nibble, rows past the last tile)."""
    out_dim, in_dim = 203, 768
    if encoding in (kquant.F32, kquant.BF16):
        packed = kquant.quantize(encoding, kquant.synthetic_weights(9, out_dim, in_dim, 1.0))
    else:
        packed = kquant.quantize(encoding, kquant.synthetic_weights(9 + encoding, out_dim, in_dim))
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    decoded = tile_ops.dequantize(weight).cpu().numpy()
    assert np.array_equal(decoded, oracle.dequantize(encoding, packed, out_dim, in_dim))
    x = np.eye(in_dim, dtype=np.float32)
    bias = ((np.arange(out_dim) % 7 - 3) * 0.25).astype(np.float32)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    assert np.array_equal(y, decoded.T)
    y = tile_ops.linear(weight, to_device(x[:300] * 2.0, cuda), to_device(bias, cuda)).cpu().numpy()
    assert np.array_equal(y, decoded.T[:300] * 2.0 + bias[None, :])


@pytest.mark.parametrize("rows", [17, 128, 129, 300])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_generic_linear_many_rows_against_oracle(cuda, oracle, encoding, rows):
    out_dim, in_dim = 321, 2048
    packed = kquant.quantize(encoding, kquant.synthetic_weights(41 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(78 + rows, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= 1e-5


@pytest.mark.parametrize("rows,out_dim,in_dim", [
    (1, 1, 256), (2, 67, 4352), (3, 130, 512),    # one pass over the weights, rows in LDS
    (1, 3, 16384), (3, 40, 16384),                # ... of rows that fill LDS, or do not fit it
    (4, 33, 288), (31, 65, 768), (47, 129, 288),  # 32 x 32 tiles; an odd last step of 32 columns
    (60, 5000, 256), (100, 6600, 320), (200, 6600, 512),  # 32 x 64, 32 x 128 and 64 x 128 tiles (F32: up to 64 x 64)
])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_forms_at_their_edges(cuda, oracle, encoding, rows, out_dim, in_dim):
    """Every form of the exact linear against the oracle's double sums, a row six orders of
    magnitude larger than the others among them.  Bound: a float sum of K terms is off by at
    most K 2^-24 of the sum of magnitudes; with random signs by about sqrt(K) of that, and the
    largest output of a row is some four standard deviations: 1e-5 covers K = 16,384."""
    if in_dim % kquant.BLOCKS[encoding][0]:
        in_dim += 256 - in_dim % 256  # whole blocks
    packed = kquant.quantize(encoding, kquant.synthetic_weights(5 + rows, out_dim, in_dim))
    x = kquant.synthetic_activations(6 + rows, rows, in_dim) + np.float32(0.3)
    x[rows - 1] *= np.float32(1e6)
    bias = np.linspace(-1, 1, out_dim, dtype=np.float32)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda), to_device(bias, cuda)).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x, bias=bias)
    for row in {0, rows // 2, rows - 1}:
        assert normalised_error(y[row], expected[row]) <= 1e-5, row
    assert normalised_error(y[: rows - 1], expected[: rows - 1]) <= 1e-5 if rows > 1 else True


@pytest.mark.parametrize("rows", [7, 8, 9, 16, 17, 39])  # the last and the first of those cut by 8, 16 and 32 rows
@pytest.mark.parametrize("out_dim", [33, 3000, 8300])  # 32 x 32 (few, many) and, by two, 32 x 64 tiles (F32: 64 x 32)
@pytest.mark.parametrize("encoding,in_dim", [
    (encoding, in_dim) for encoding in ALL_PACKED + [kquant.F32, kquant.BF16]
    for in_dim in ((512, 3584) if kquant.BLOCKS[encoding][0] == 256 else (544,))])
def test_exact_linear_cuts_the_rows_that_are_there(cuda, oracle, encoding, in_dim, out_dim, rows):
    """The forms of a few tiles: walks over K that go through LDS and short ones that do not, rows of an
    odd number of 32 columns where the format has them.  Bound: as above."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(9, out_dim, in_dim))
    x = kquant.synthetic_activations(10 + rows, rows, in_dim) + np.float32(0.3)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    assert normalised_error(y, oracle.linear(encoding, packed, out_dim, in_dim, x)) <= 1e-5


@pytest.mark.parametrize("rows", [100, 200])  # 32 x 128 and 64 x 128 tiles
@pytest.mark.parametrize("out_dim", [6529, 6592, 6593])  # one, 64 and 65 rows in the last tile's pair of waves
@pytest.mark.parametrize("encoding,in_dim", [
    (encoding, 64 * units) for encoding in ALL_PACKED + [kquant.BF16]
    for units in ((4, 20) if kquant.BLOCKS[encoding][0] == 256 else (1, 3, 5))])  # K groups of none, one, two and five units
def test_exact_linear_tiles_of_128_columns(cuda, oracle, encoding, in_dim, out_dim, rows):
    """The form whose waves turn their weights in LDS and wait in pairs.  Bound: as above."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(7 + rows, out_dim, in_dim))
    x = kquant.synthetic_activations(8 + rows, rows, in_dim) + np.float32(0.3)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    assert normalised_error(y, oracle.linear(encoding, packed, out_dim, in_dim, x)) <= 1e-5


@pytest.mark.parametrize("out_dim,in_dim", [(67, 512), (6656, 768), (9000, 256), (33, 2048)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_rows_carry_the_same_bits_within_a_form(cuda, encoding, out_dim, in_dim):
    """What the header says of a row's bits: the same whichever other rows come with it, among one
    to three rows and among four to 32."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(5, out_dim, in_dim))
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(6, 32, in_dim), cuda)
    three, many = tile_ops.linear(weight, x[:3]), tile_ops.linear(weight, x)
    for rows in (1, 2):
        assert_bits_equal(tile_ops.linear(weight, x[3 - rows:3]), three[3 - rows:], f"{rows} rows")
    for rows in (4, 5, 16, 17, 31):
        assert_bits_equal(tile_ops.linear(weight, x[32 - rows:]), many[32 - rows:], f"{rows} rows")
    assert normalised_error(three.cpu().numpy(), many[:3].cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("rows,out_dim", [(257, 7232), (333, 6656), (509, 5056)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.BF16])
def test_exact_linear_of_many_rows_rounds_as_that_of_64(cuda, encoding, rows, out_dim):
    """Shapes where 32 x 64 tiles and those of 128 columns cost alike: they stay with the former (Q4_K, Q5_K),
    whose sums are cut among eight waves and not four, and carry the bits of a call of 64 rows, which
    takes 32 x 64 tiles at these widths.  (The other formats: within the bound of every form.)"""
    in_dim = 4096
    packed = random_packed(encoding, out_dim, in_dim, 66) if encoding != kquant.BF16 else kquant.quantize(
        encoding, kquant.synthetic_weights(66, out_dim, in_dim))
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(67, rows, in_dim), cuda)
    many, few = tile_ops.linear(weight, x), tile_ops.linear(weight, x[:64])
    if encoding in (kquant.Q4_K, kquant.Q5_K):
        assert_bits_equal(many[:64].contiguous(), few, f"64 of {rows} rows")
    assert normalised_error(many[:64].cpu().numpy(), few.cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("in_dim", [2 ** 23, 2 ** 23 + 256])
@pytest.mark.parametrize("encoding", [kquant.Q8_0, kquant.BF16])
def test_exact_linear_on_both_sides_of_its_longest_rows(cuda, encoding, in_dim):
    """Past 2^23 columns the kernel for any width takes the call.  Bound: its lanes add 2^17 products
    one after another, which with random signs is off by about sqrt(2^17) 2^-24 = 2e-5 of the result;
    1e-4 leaves five standard deviations."""
    torch = torch_()
    out_dim, rows = 3, 5
    packed = kquant.quantize(encoding, kquant.synthetic_weights(64, out_dim, in_dim))
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(65, rows, in_dim), cuda)
    y = tile_ops.linear(weight, x).double()
    expected = torch.stack([(x.double() * row.double()).sum(dim=1) for row in tile_ops.dequantize(weight)], dim=1)
    assert float((y - expected).abs().max() / expected.abs().max()) <= 1e-4


@pytest.mark.parametrize("rows,out_dim,in_dim", [(3, 67, 512), (5, 67, 512), (60, 5000, 256), (100, 6600, 256), (200, 6600, 256)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_of_infinities_nan_and_large_activations(cuda, oracle, encoding, rows, out_dim, in_dim):
    """Activations that are infinite, NaN or whose products with the codes (but not with the
    weights) leave the float range: what the products with the decoded weights give."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(5 + rows, out_dim, in_dim))
    x = kquant.synthetic_activations(6 + rows, rows, in_dim)
    x[0, 37] = np.inf
    x[1, 200] = np.nan
    x[2] *= np.float32(3e37) / np.abs(x[2]).max()
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    w = oracle.dequantize(encoding, packed, out_dim, in_dim).reshape(out_dim, in_dim).astype(np.float64)
    with np.errstate(invalid="ignore"):
        expected = x.astype(np.float64) @ w.T
    assert np.array_equal(np.isnan(y), np.isnan(expected))
    infinite = np.isinf(expected)
    assert infinite[0].any() and np.array_equal(np.isinf(y), infinite) and np.array_equal(y[infinite], expected[infinite])
    for row in {2, rows - 1}:
        assert normalised_error(y[row], expected[row]) <= 1e-5, row


@pytest.mark.parametrize("rows,out_dim,in_dim", [(2, 67, 512), (3, 67, 512), (5, 67, 512), (60, 5000, 256), (100, 6600, 256), (200, 6600, 256)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_of_weights_that_are_not_finite(cuda, oracle, encoding, rows, out_dim, in_dim):
    """Infinite block scales and minimums, infinite and NaN float weights, and rows of zeros among
    the activations: what the products with the decoded weights give."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(5 + rows, out_dim, in_dim)).copy()
    row_bytes = kquant.row_stride_bytes(encoding, in_dim)
    infinity, nan = (b"\x00\x7c", b"\x00\x7e")  # halves
    if encoding == kquant.F32:
        infinity, nan = (np.float32(v).tobytes() for v in (np.inf, np.nan))
    elif encoding == kquant.BF16:
        infinity, nan = (np.float32(v).tobytes()[2:] for v in (np.inf, np.nan))
    scale = {kquant.Q6_K: 208}.get(encoding, 0)
    minimum = {kquant.Q4_K: 2, kquant.Q5_K: 2}.get(encoding, scale)
    for row, offset, value in ((1, scale, infinity), (2, minimum, infinity), (out_dim - 1, scale, nan)):
        at = row * row_bytes + offset
        packed[at:at + len(value)] = np.frombuffer(value, dtype=np.uint8)
    x = kquant.synthetic_activations(6 + rows, rows, in_dim)
    x[rows - 2] = 0.0
    if encoding in (kquant.Q6_K, kquant.Q8_0):  # a block of positive codes, times infinity, times positive activations
        at, nbytes = 3 * row_bytes, kquant.BLOCKS[encoding][1]
        packed[at:at + nbytes] = 0x7f if encoding == kquant.Q8_0 else 0xff
        if encoding == kquant.Q6_K:
            packed[at + 192:at + 208] = 1
        packed[at + scale:at + scale + 2] = np.frombuffer(infinity, dtype=np.uint8)
        x[rows - 1] = np.abs(x[rows - 1]) + np.float32(0.25)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy()
    w = oracle.dequantize(encoding, packed, out_dim, in_dim).reshape(out_dim, in_dim).astype(np.float64)
    with np.errstate(invalid="ignore"):
        expected = x.astype(np.float64) @ w.T
    assert (~np.isfinite(expected)).sum(axis=0)[[1, 2, out_dim - 1]].min() > 0
    assert np.array_equal(np.isnan(y), np.isnan(expected))
    infinite = np.isinf(expected)
    assert np.array_equal(np.isinf(y), infinite) and np.array_equal(y[infinite], expected[infinite])
    if encoding in (kquant.Q6_K, kquant.Q8_0):
        assert expected[rows - 1, 3] == np.inf
    finite = np.isfinite(expected)
    assert normalised_error(y[finite], expected[finite]) <= 1e-5


@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_small_tiles_of_special_operands(cuda, oracle, encoding):
    """The matrix-core kernel's 32 x 32 tiles (five and 17 rows into more outputs than the vector kernel takes
    them for) with operands that are not finite, large or tiny."""
    for rows, out_dim, in_dim in ((5, 6700, 512), (17, 2100, 256)):
        test_exact_linear_of_infinities_nan_and_large_activations(cuda, oracle, encoding, rows, out_dim, in_dim)
        test_exact_linear_of_weights_that_are_not_finite(cuda, oracle, encoding, rows, out_dim, in_dim)
        test_exact_linear_of_tiny_operands(cuda, oracle, encoding, rows, out_dim, in_dim, -36)


@pytest.mark.parametrize("in_dim,out_dim", [(256, 368), (256, 369), (512, 736), (512, 737), *((1024, n) for n in (90, 94, 368, 369)),
                                            *((1280, n) for n in (368, 369, 736, 737)), (2304, 368), (2304, 369),
                                            *((3328, n) for n in (736, 737, 1104, 1105)), (4352, 737), (5376, 736)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_carries_the_same_bits_from_four_to_32_rows(cuda, encoding, in_dim, out_dim):
    """Which kernel and which form of it runs from four to 32 rows hangs on the weight alone (outputs and widths on
    both sides of every line)."""
    weight = tile_ops.PackedWeight.from_numpy(
        encoding, kquant.quantize(encoding, kquant.synthetic_weights(60, out_dim, in_dim)), out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(61, 32, in_dim), cuda)
    all_rows = tile_ops.linear(weight, x)
    for rows in (4, 5, 9, 12, 17, 24):
        assert_bits_equal(tile_ops.linear(weight, x[:rows].contiguous()), all_rows[:rows].contiguous(), f"{rows} rows")


@pytest.mark.parametrize("rows,out_dim,in_dim", [(4, 300, 2048), (5, 33, 1280), (7, 368, 1536), (12, 352, 8192), (17, 2, 1088), (97, 65, 4096)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_of_row_groups(cuda, oracle, encoding, rows, out_dim, in_dim):
    """More than three rows into few outputs on the vector kernel, two or three of them a workgroup: row for
    row the bits of the call of three rows (F32 and bf16, whose waves may share a row or not: its bound), a
    last group of one or two, nothing written past the end."""
    if encoding not in (kquant.F32, kquant.BF16, kquant.Q8_0):
        in_dim = -(-in_dim // 256) * 256
    packed = kquant.quantize(encoding, kquant.synthetic_weights(50, out_dim, in_dim))
    x = kquant.synthetic_activations(51, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    bias = torch_().linspace(-1.0, 1.0, out_dim, device=cuda)
    device_x = to_device(x, cuda)
    y = tile_ops.linear(weight, device_x, bias)
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x) + bias.cpu().numpy()
    assert normalised_error(y.cpu().numpy(), expected) <= 1e-5
    if encoding in ALL_PACKED:
        for first in range(0, rows, 3):
            part = tile_ops.linear(weight, device_x[first:first + 3].contiguous(), bias)
            assert_bits_equal(y[first:first + 3].contiguous(), part, f"rows {first} on")


@pytest.mark.parametrize("in_dim", [4096, 4352, 8192])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_exact_linear_of_few_outputs_rounds_no_more_than_of_many(cuda, encoding, in_dim):
    """Few outputs run on the vector kernel and many on the matrix-core one (eight rows of 320 and of 8,192): against
    float64 the former are no further off, over 2,560 values each, whose root mean squares are known to 1.4 percent
    (1 / sqrt(2 x 2,560)): three times that for their ratio is 6 percent."""
    packed = torch_().from_numpy(kquant.quantize(encoding, kquant.synthetic_weights(62, 256, in_dim)).reshape(256, -1)).to(cuda)
    chosen = torch_().from_numpy(np.random.default_rng(64).integers(0, 256, 8192)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, 8192, in_dim, packed.index_select(0, chosen).reshape(-1))
    few = tile_ops.PackedWeight(encoding, 320, in_dim, packed.index_select(0, chosen[:320]).reshape(-1))
    x = to_device(kquant.synthetic_activations(63, 8, in_dim), cuda)
    exact = x.double() @ tile_ops.dequantize(few).reshape(320, in_dim).double().T.contiguous()
    error = [((y.double() - exact).norm() / exact.norm()).item()
             for y in (tile_ops.linear(few, x), tile_ops.linear(weight, x)[:, :320])]
    assert error[0] <= 1.06 * error[1], error


@pytest.mark.parametrize("exponent", [-33, -35, -36, -37])
@pytest.mark.parametrize("rows,out_dim,in_dim", [(3, 67, 512), (5, 67, 512), (60, 5000, 256), (100, 6600, 256), (200, 6600, 256)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_of_tiny_operands(cuda, oracle, encoding, rows, out_dim, in_dim, exponent):
    """Activations, and float weights, down to the smallest normal floats: a bf16 term of one of
    them would be below 2^-133, the smallest bf16 number.  Products and sums are normal floats, so
    that the bound is that of the edges' test, plus half a unit of the smallest float."""
    tiny = np.float32(10.0) ** np.float32(exponent)
    x = kquant.synthetic_activations(6 + rows, rows, in_dim) + np.float32(0.3)
    w = kquant.synthetic_weights(5 + rows, out_dim, in_dim, 1.0)
    packed = kquant.quantize(encoding, w)
    decoded = oracle.dequantize(encoding, packed, out_dim, in_dim).reshape(out_dim, in_dim).astype(np.float64)

    def check(packed, decoded, x):
        weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
        y = tile_ops.linear(weight, to_device(x, cuda)).cpu().numpy().astype(np.float64)
        expected = x.astype(np.float64) @ decoded.T
        for row in range(rows):
            assert np.max(np.abs(y[row] - expected[row])) <= 1e-5 * np.max(np.abs(expected[row])) + 2.0 ** -150, row

    check(packed, decoded, x * tiny)
    mixed = x * tiny
    mixed[:, in_dim // 2:] *= np.float32(1e6)  # tiny next to ordinary ones
    check(packed, decoded, mixed)
    if encoding in (kquant.F32, kquant.BF16):
        packed = kquant.quantize(encoding, w * tiny)
        check(packed, oracle.dequantize(encoding, packed, out_dim, in_dim).reshape(out_dim, in_dim).astype(np.float64), x)


# ------------------------------------------------------------ public Q8_1 path

def crafted_q8_input(rows, in_dim):
    """probe :899-920: every 32-block has scale exactly 1/32."""
    x = np.zeros((rows, in_dim), np.float32)
    for row in range(rows):
        for block in range(in_dim // 32):
            for lane in range(32):
                code = 0
                if lane == 0:
                    code = -127
                elif lane == 1:
                    code = 127
                elif lane == 2:
                    code = 64 - 2 * (row % 5)
                elif lane >= 4:
                    magnitude = 1 + (block * 11 + (lane // 2) * 7 + row * 3) % 96
                    code = magnitude if lane % 2 == 0 else -magnitude
                x[row, block * 32 + lane] = code * 0.03125
    return x


@pytest.mark.parametrize("encoding", K_ENCODINGS)
def test_q8_1_quantize_and_linear(cuda, oracle, encoding):
    rows, out_dim, in_dim = 5, 7, 512
    _, nbytes = kquant.BLOCKS[encoding]
    packed = kquant.patterned_bytes(encoding, out_dim, in_dim, multiplier=41, offset=23)
    x = crafted_q8_input(rows, in_dim)
    bias = ((np.arange(out_dim) - 3) / 9.0).astype(np.float32)
    codes, scales, sums = tile_ops.quantize_q8_1(to_device(x, cuda))
    o_codes, o_scales, o_sums = oracle.quantize_q8_1(x)
    assert np.array_equal(codes.cpu().numpy(), o_codes)
    assert np.max(np.abs(scales.cpu().numpy() - o_scales)) <= 1e-7
    assert np.max(np.abs(sums.cpu().numpy() - o_sums)) <= 2e-5
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.linear_q8_1(weight, codes, scales, sums, to_device(bias, cuda)).cpu().numpy()
    expected = oracle.linear_q8_1(encoding, packed, out_dim, in_dim, o_codes, o_scales, bias)
    assert np.max(np.abs(y - expected)) <= 8e-3  # probe :1019-1022


def test_q8_1_quantize_random_matches_oracle(cuda, oracle):
    x = kquant.synthetic_activations(5, 4, 6656)
    x[1, 64:96] = 0.0
    codes, scales, sums = tile_ops.quantize_q8_1(to_device(x, cuda))
    o_codes, o_scales, o_sums = oracle.quantize_q8_1(x)
    assert np.array_equal(codes.cpu().numpy(), o_codes)
    assert np.array_equal(scales.cpu().numpy(), o_scales)
    assert np.max(np.abs(sums.cpu().numpy() - o_sums)) <= 2e-5


def test_q8_1_multi_decode_bit_exact_with_single(cuda):
    # probe :1026-1202
    in_dim = 512
    specs = [(kquant.Q4_K, 5, 3), (kquant.Q5_K, 7, 5), (kquant.Q6_K, 3, 7), (kquant.Q4_K, 9, 11)]
    weights = [tile_ops.PackedWeight.from_numpy(e, probe_packed(e, n, in_dim, s), n, in_dim)
               for e, n, s in specs]
    x = (((np.arange(in_dim) * 19 + 7) % 251 - 125) / 47.0).astype(np.float32)[None, :]
    codes, scales, sums = tile_ops.quantize_q8_1(to_device(x, cuda))
    singles = [tile_ops.linear_q8_1(w, codes, scales, sums) for w in weights]
    fused = tile_ops.linear_q8_1_multi_decode(weights, codes, scales, sums)
    for index, (a, b) in enumerate(zip(singles, fused)):
        assert_bits_equal(a, b, f"projection {index}")
    fused2 = tile_ops.linear_q8_1_multi_decode(weights[:2], codes, scales, sums)
    assert_bits_equal(singles[0], fused2[0])
    assert_bits_equal(singles[1], fused2[1])


# ----------------------------------------------- small-batch K-quant entry points

@pytest.fixture(scope="module")
def mixed(cuda):
    """probe :1278-1390: rows 5, K 512, Q4_K x129, Q5_K x17, Q6_K x33."""
    in_dim, rows = 512, 5
    specs = [(kquant.Q4_K, 129, 3), (kquant.Q5_K, 17, 5), (kquant.Q6_K, 33, 7)]
    packed = [probe_packed(e, n, in_dim, s) for e, n, s in specs]
    weights = [tile_ops.PackedWeight.from_numpy(e, p, n, in_dim)
               for (e, n, _), p in zip(specs, packed)]
    r, c = np.arange(rows)[:, None], np.arange(in_dim)[None, :]
    x = (((c * 19 + r * 23 + 7) % 251 - 125) / 47.0).astype(np.float32)
    gate = (((np.arange(rows * in_dim) * 13 + 11) % 101 - 50) / 17.0).astype(np.float32)
    return dict(specs=specs, packed=packed, weights=weights, x=x, gate=gate.reshape(rows, in_dim),
                rows=rows, in_dim=in_dim)


def test_small_batch_against_both_oracles(cuda, oracle, mixed):
    rows, in_dim = mixed["rows"], mixed["in_dim"]
    x = to_device(mixed["x"], cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    outputs = tile_ops.multi_linear(mixed["weights"], x, workspace)
    o_codes, o_scales, _ = oracle.quantize_q8_1(mixed["x"])
    for (encoding, out_dim, _), packed, y in zip(mixed["specs"], mixed["packed"], outputs):
        y = y.cpu().numpy()
        exact = oracle.linear(encoding, packed, out_dim, in_dim, mixed["x"])
        assert normalised_error(y, exact) <= TOLERANCE
        # The reference checks this entry point against its int8-activation
        # path (probe :1444-1458).  This library keeps 16 bits of every
        # activation here, so it has to sit closer to the float oracle than
        # that int8 result does, not within the int8 path's own tolerance.
        q8 = oracle.linear_q8_1(encoding, packed, out_dim, in_dim, o_codes, o_scales)
        assert normalised_error(y, exact) <= normalised_error(q8, exact)


def test_one_row_paths_agree_bit_for_bit(cuda, oracle, mixed):
    in_dim = mixed["in_dim"]
    x = to_device(mixed["x"][:1], cuda)
    workspace = tile_ops.small_batch_workspace(1, in_dim)
    grouped = tile_ops.multi_linear(mixed["weights"], x, workspace)
    direct = tile_ops.mmvq_linear(mixed["weights"][0], x, workspace)
    assert_bits_equal(grouped[0], direct, "dedicated vs grouped one-row")  # probe :1520-1529
    for (encoding, out_dim, _), packed, y in zip(mixed["specs"], mixed["packed"], grouped):
        exact = oracle.linear(encoding, packed, out_dim, in_dim, mixed["x"][:1])
        assert normalised_error(y.cpu().numpy(), exact) <= TOLERANCE


@pytest.mark.parametrize("prologue", ["plain", "gated", "swiglu"])
def test_verifier_rows_equal_row_by_row(cuda, mixed, prologue):
    # probe :1588-1640: batched verifier == the one-row call per row, bit for bit
    rows, in_dim = mixed["rows"], mixed["in_dim"]
    x = to_device(mixed["x"], cuda)
    second = to_device(mixed["gate"], cuda) if prologue != "plain" else None
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    one = tile_ops.small_batch_workspace(1, in_dim)
    batched = tile_ops.multi_linear(mixed["weights"], x, workspace, second, "mmvq", prologue)
    for row in range(rows):
        single = tile_ops.multi_linear(
            mixed["weights"], x[row:row + 1], one,
            second[row:row + 1] if second is not None else None, "mmq", prologue)
        for b, s in zip(batched, single):
            assert_bits_equal(b[row:row + 1], s, f"{prologue} row {row}")


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("prologue", ["gated", "swiglu"])
def test_fused_prologue_equals_materialised(cuda, oracle, mixed, prologue, rows):
    # probe :1659-1692, 1764-1833
    in_dim = mixed["in_dim"]
    x = to_device(mixed["x"][:rows], cuda)
    g = to_device(mixed["gate"][:rows], cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    if prologue == "gated":
        materialised = tile_ops.sigmoid_gate(x, g)
        host = oracle.sigmoid_gate(mixed["x"][:rows], mixed["gate"][:rows])
    else:
        materialised = tile_ops.swiglu(x, g)  # x is the gate operand, g is `up`
        host = oracle.swiglu(mixed["x"][:rows], mixed["gate"][:rows])
    np.testing.assert_allclose(materialised.cpu().numpy(), host, rtol=2e-6, atol=1e-7)
    baseline = tile_ops.multi_linear(mixed["weights"], materialised, workspace)
    fused = tile_ops.multi_linear(mixed["weights"], x, workspace, g, "mmq", prologue)
    for b, f in zip(baseline, fused):
        assert_bits_equal(b, f, prologue)


@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K])
@pytest.mark.parametrize("in_dim,out_dim", [(256, 1), (2304, 70), (4096, 1037), (6656, 16384), (8192, 513)])
def test_gate_up_swiglu_equals_the_two_calls(cuda, oracle, encoding, in_dim, out_dim):
    """nfn_mi355_k_quant_mmvq_gate_up_swiglu_float32_v1 = the grouped one-row call on [gate, up]
    followed by the element-wise SwiGLU, bit for bit; a projection fed from its output equals the
    SwiGLU-prologue call on the two separate results."""
    gate = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, out_dim, in_dim, 91), out_dim, in_dim)
    up = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, out_dim, in_dim, 92), out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(93, 1, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(1, max(in_dim, (out_dim + 255) // 256 * 256))
    separate = tile_ops.multi_linear([gate, up], x, workspace)
    expected = tile_ops.swiglu(separate[0], separate[1])
    fused = tile_ops.gate_up_swiglu(gate, up, x)
    assert_bits_equal(fused, expected, "gate/up with SwiGLU")
    if out_dim % 256 == 0:
        down = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, 40, out_dim, 94), 40, out_dim)
        (by_prologue,) = tile_ops.multi_linear([down], separate[0], workspace, separate[1], "mmq", "swiglu")
        (plain,) = tile_ops.multi_linear([down], fused, workspace)
        assert_bits_equal(plain, by_prologue, "the projection behind")
    exact_gate = oracle.linear(encoding, gate.data.cpu().numpy(), out_dim, in_dim, x.cpu().numpy())
    exact_up = oracle.linear(encoding, up.data.cpu().numpy(), out_dim, in_dim, x.cpu().numpy())
    exact = oracle.swiglu(exact_gate, exact_up)
    assert normalised_error(fused.cpu().numpy(), exact) <= 2 * TOLERANCE


@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
@pytest.mark.parametrize("rows,in_dim,out_dim", [(5, 256, 1), (16, 2304, 70), (8, 6656, 1037), (16, 6656, 16384),
                                                 (11, 16384, 513)])
def test_gate_up_swiglu_rows_equals_the_two_calls(cuda, oracle, encoding, rows, in_dim, out_dim):
    """nfn_mi355_k_quant_mmq_gate_up_swiglu_float32_v1 = the grouped small-batch call on [gate, up]
    followed by the element-wise SwiGLU, bit for bit; a projection fed from its output equals the
    SwiGLU-prologue call on the two separate results."""
    gate = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, out_dim, in_dim, 191), out_dim, in_dim)
    up = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, out_dim, in_dim, 192), out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(193, rows, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(rows, max(in_dim, (out_dim + 255) // 256 * 256))
    separate = tile_ops.multi_linear([gate, up], x, workspace)
    expected = tile_ops.swiglu(separate[0], separate[1])
    assert tile_ops.gate_up_swiglu_rows_supported(gate, up, rows)
    fused = tile_ops.gate_up_swiglu_rows(gate, up, x, rows, workspace)
    assert_bits_equal(fused, expected, "gate/up with SwiGLU")
    if out_dim % 256 == 0:
        down = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, 40, out_dim, 194), 40, out_dim)
        (by_prologue,) = tile_ops.multi_linear([down], separate[0], workspace, separate[1], "mmq", "swiglu")
        (plain,) = tile_ops.multi_linear([down], fused, workspace)
        assert_bits_equal(plain, by_prologue, "the projection behind")
    if out_dim <= 2048:
        exact_gate = oracle.linear(encoding, gate.data.cpu().numpy(), out_dim, in_dim, x.cpu().numpy())
        exact_up = oracle.linear(encoding, up.data.cpu().numpy(), out_dim, in_dim, x.cpu().numpy())
        exact = oracle.swiglu(exact_gate, exact_up)
        assert normalised_error(fused.cpu().numpy(), exact) <= 2 * TOLERANCE


def test_gate_up_swiglu_rows_from_the_norm_handoff(cuda):
    """With a null input the call multiplies from the fp16 rows the dual norm left in the workspace:
    the same bits as the call on the normalized rows."""
    torch = torch_()
    rows, width, out_dim = 16, 6656, 640
    rng = np.random.default_rng(7)
    pending = to_device(rng.standard_normal((rows, width)).astype(np.float32), cuda)
    residual = to_device(rng.standard_normal((rows, width)).astype(np.float32), cuda)
    _, first = norm_weight(1.0 + 0.1 * rng.standard_normal(width), kquant.F32, cuda)
    _, second = norm_weight(1.0 + 0.1 * rng.standard_normal(width), kquant.BF16, cuda)
    gate = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, out_dim, width, 195), out_dim, width)
    up = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, out_dim, width, 196), out_dim, width)
    workspace = tile_ops.small_batch_workspace(rows, width)
    _, normalized, _ = tile_ops.dual_rms_add_capture(pending, residual, first, False, second, False, 1e-6, 1e-6,
                                                      handoff_workspace=workspace)
    handed = tile_ops.gate_up_swiglu_rows(gate, up, None, rows, workspace)
    ordinary = tile_ops.gate_up_swiglu_rows(gate, up, normalized, rows, workspace)
    assert_bits_equal(handed, ordinary, "from the handoff")


def test_gate_up_swiglu_rows_fails_closed(cuda):
    lib = tile_ops.load()
    in_dim, out_dim, rows = 512, 24, 8
    make = lambda e, n, k, seed: tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, k, seed), n, k)
    gate, up = make(kquant.Q4_K, out_dim, in_dim, 1), make(kquant.Q4_K, out_dim, in_dim, 2)
    x = to_device(kquant.synthetic_activations(3, 16, in_dim), cuda)
    out = torch_().empty((16, out_dim), dtype=torch_().float32, device=cuda)
    workspace = tile_ops.small_batch_workspace(16, in_dim)
    call = lib.nfn_mi355_k_quant_mmq_gate_up_swiglu_float32_v1
    ref = lambda w: ctypes.byref(w.descriptor(0))
    arguments = lambda g, u, r=rows, n=workspace.numel(): (ref(g), ref(u), x.data_ptr(), out.data_ptr(), r,
                                                           workspace.data_ptr(), n, None)
    assert call(*arguments(gate, up)) == 0
    assert call(*arguments(gate, make(kquant.Q5_K, out_dim, in_dim, 4))) == 1
    assert call(*arguments(gate, make(kquant.Q4_K, out_dim + 1, in_dim, 5))) == 1
    assert call(*arguments(gate, make(kquant.Q4_K, out_dim, 256, 6))) == 1
    assert call(*arguments(gate, up, 4)) == 1
    assert call(*arguments(gate, up, 17)) == 1
    assert call(*arguments(gate, up, rows, 64)) == 1
    assert call(None, ref(up), x.data_ptr(), out.data_ptr(), rows, workspace.data_ptr(), workspace.numel(), None) == 1
    assert call(ref(gate), ref(up), x.data_ptr(), None, rows, workspace.data_ptr(), workspace.numel(), None) == 1
    assert call(ref(gate), ref(up), x.data_ptr(), out.data_ptr(), rows, None, workspace.numel(), None) == 1
    torch_().cuda.synchronize()


def test_gate_up_swiglu_fails_closed(cuda):
    lib = tile_ops.load()
    in_dim, out_dim = 512, 24
    make = lambda e, n, k, seed: tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, k, seed), n, k)
    gate, up = make(kquant.Q4_K, out_dim, in_dim, 1), make(kquant.Q4_K, out_dim, in_dim, 2)
    x = to_device(kquant.synthetic_activations(3, 1, 16384), cuda)
    out = torch_().empty((1, out_dim), dtype=torch_().float32, device=cuda)
    call = lib.nfn_mi355_k_quant_mmvq_gate_up_swiglu_float32_v1
    ref = lambda w: ctypes.byref(w.descriptor(0))
    assert call(ref(gate), ref(up), x.data_ptr(), out.data_ptr(), None) == 0
    assert call(ref(gate), ref(make(kquant.Q5_K, out_dim, in_dim, 4)), x.data_ptr(), out.data_ptr(), None) == 1
    assert call(ref(gate), ref(make(kquant.Q4_K, out_dim + 1, in_dim, 5)), x.data_ptr(), out.data_ptr(), None) == 1
    assert call(ref(gate), ref(make(kquant.Q4_K, out_dim, 256, 6)), x.data_ptr(), out.data_ptr(), None) == 1
    six = make(kquant.Q6_K, out_dim, in_dim, 7)
    assert call(ref(six), ref(six), x.data_ptr(), out.data_ptr(), None) == 1
    wide = make(kquant.Q4_K, 8, 8448, 8)
    assert call(ref(wide), ref(wide), x.data_ptr(), out.data_ptr(), None) == 1
    assert call(None, ref(up), x.data_ptr(), out.data_ptr(), None) == 1
    assert call(ref(gate), ref(up), None, out.data_ptr(), None) == 1
    assert call(ref(gate), ref(up), x.data_ptr(), None, None) == 1
    torch_().cuda.synchronize()


def test_elementwise_prologues_over_the_float_range(cuda, oracle):
    """The sigmoid of the two element-wise operators (and of the fused prologues, which share
    it) is built from the hardware's exp2 and reciprocal: 2e-6 of the oracle over twenty
    decades of either sign, the saturated ends, zeros, infinities and NaN."""
    rng = np.random.default_rng(5)
    magnitudes = 10.0 ** rng.uniform(-20, 3, 4096)
    gate = (magnitudes * rng.choice([-1.0, 1.0], 4096)).astype(np.float32)
    special = np.array([0.0, -0.0, 86.9, -86.9, 87.0, -87.0, 88.4, -88.4, 88.8, -88.8, 104.0,
                        -104.0, 1e30, -1e30, np.inf, -np.inf, np.nan, 1e-40, -1e-40],
                       np.float32)
    gate = np.concatenate([gate, special, np.linspace(-30, 30, 4096).astype(np.float32)])
    other = rng.uniform(-3, 3, gate.size).astype(np.float32)
    for name in ("sigmoid_gate", "swiglu"):
        first, second = (other, gate) if name == "sigmoid_gate" else (gate, other)
        got = getattr(tile_ops, name)(to_device(first[None, :], cuda),
                                      to_device(second[None, :], cuda)).cpu().numpy()[0]
        with np.errstate(all="ignore"):
            want = getattr(oracle, name)(first[None, :], second[None, :])[0]
        assert np.array_equal(np.isnan(got), np.isnan(want)), name
        finite = ~np.isnan(want)
        np.testing.assert_allclose(got[finite], want[finite], rtol=2e-6, atol=1e-35, err_msg=name)


def test_small_batch_fails_closed_on_device(cuda, mixed):
    # probe :1834-1866 with real device buffers
    rows, in_dim = mixed["rows"], mixed["in_dim"]
    lib = tile_ops.load()
    x = to_device(mixed["x"], cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    weight = mixed["weights"][0]
    out = torch_().full((rows, weight.output_dim), 123.0, device=cuda)

    def call(descriptor, test_rows, ws_bytes):
        array = (ctypes.POINTER(tile_ops.PackedWeightDescriptor) * 1)(ctypes.pointer(descriptor))
        outs = (ctypes.c_void_p * 1)(out.data_ptr())
        return lib.nfn_native_tile_k_quant_mmq_multi_linear_float32_v1(
            array, x.data_ptr(), outs, 1, test_rows, workspace.data_ptr(), ws_bytes, None)

    good = weight.descriptor()
    for field, value in (("data_nbytes", good.data_nbytes - 1), ("encoding", 0xFFFF),
                         ("row_stride_bytes", good.row_stride_bytes - 1)):
        bad = weight.descriptor()
        setattr(bad, field, value)
        assert call(bad, rows, workspace.numel()) == tile_ops.INVALID
    need = lib.nfn_native_tile_k_quant_mmq_workspace_bytes_v1(rows, in_dim)
    assert call(good, rows, need - 1) == tile_ops.INVALID
    assert call(good, 17, workspace.numel()) == tile_ops.INVALID
    torch_().cuda.synchronize()
    assert bool((out == 123.0).all()), "a rejected call wrote to its output"
    assert call(good, rows, need) == 0


@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_small_batch_quantized_weights(cuda, oracle, encoding, rows):
    out_dim, in_dim = 272, 1024
    packed = kquant.quantize(encoding, kquant.synthetic_weights(50 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(60 + rows, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    y = tile_ops.multi_linear([weight], to_device(x, cuda), workspace)[0].cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= TOLERANCE


@pytest.mark.parametrize("rows", [5, 9, 16])
@pytest.mark.parametrize("in_dim", [256, 2304, 8192, 8448, 19968])
def test_small_batch_half_kernel_shapes(cuda, oracle, in_dim, rows):
    """Five rows and more run on the fp16 matrix cores behind a conversion launch.  Row lengths:
    one block (seven of the eight waves of a workgroup have no K range), nine blocks (ranges
    of one and two blocks), the longest row that is one chunk of K (activation fragments loaded
    once), the first length past it (two chunks, the second of one block for some waves) and
    three chunks.  Projections of 40, 8 and 19 rows: partial 16-row tiles and
    tiles of different projections and formats in one call.  Activations of very different
    magnitude per row: every row carries its own power-of-two scale."""
    specs = [(kquant.Q4_K, 40), (kquant.Q5_K, 8), (kquant.Q6_K, 19), (kquant.Q8_0, 24)]
    packed = [random_packed(e, n, in_dim, 90 + i) for i, (e, n) in enumerate(specs)]
    weights = [tile_ops.PackedWeight.from_numpy(e, p, n, in_dim) for (e, n), p in zip(specs, packed)]
    x = kquant.synthetic_activations(91 + rows, rows, in_dim)
    x *= (10.0 ** np.linspace(-6, 5, rows)).astype(np.float32)[:, None]
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    outputs = tile_ops.multi_linear(weights, to_device(x, cuda), workspace)
    again = tile_ops.multi_linear(weights, to_device(x, cuda), workspace)
    for (encoding, out_dim), p, y, z in zip(specs, packed, outputs, again):
        expected = oracle.linear(encoding, p, out_dim, in_dim, x)
        for row in range(rows):  # per row: the rows differ by eleven orders of magnitude
            assert normalised_error(y[row:row + 1].cpu().numpy(), expected[row:row + 1]) <= TOLERANCE
        assert_bits_equal(y, z, "the same call twice")
    # a single projection alone gives the bits it gives inside the group
    alone = tile_ops.multi_linear(weights[2:3], to_device(x, cuda), workspace)[0]
    assert_bits_equal(alone, outputs[2], "single projection = its place in the group")


@pytest.mark.parametrize("in_dim", [512, 8448])
def test_small_batch_half_kernel_many_tiles(cuda, oracle, in_dim):
    """More 16-row tiles than twice the compute units: workgroups take three tiles, in a group of
    two and a group of one, and with two chunks of K they load their activation fragments
    again for every (group, chunk)."""
    rows = 7
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    specs = [(kquant.Q4_K, 16 * 2 * units + 200), (kquant.Q6_K, 16 * units - 200 + 5)]
    packed = [random_packed(e, n, in_dim, 95 + i) for i, (e, n) in enumerate(specs)]
    weights = [tile_ops.PackedWeight.from_numpy(e, p, n, in_dim) for (e, n), p in zip(specs, packed)]
    x = kquant.synthetic_activations(96, rows, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    for group in (weights[:1], weights):  # 2 x units + 13 tiles of one format, then both formats
        outputs = tile_ops.multi_linear(group, to_device(x, cuda), workspace)
        for (encoding, out_dim), p, y in zip(specs, packed, outputs):
            expected = oracle.linear(encoding, p, out_dim, in_dim, x)
            assert normalised_error(y.cpu().numpy(), expected) <= TOLERANCE


@pytest.mark.parametrize("in_dim", [2048, 3840, 4096, 4352])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_small_batch_half_kernel_short_rows(cuda, oracle, encoding, in_dim):
    """Rows of up to 4,096 columns (two blocks a wave) keep two tiles of weights in flight: one tile a
    workgroup, three (a group of two and a group of one), shares of one and of two blocks, and the
    first length past the line.  A tile's rows are the same bits wherever the tile lies."""
    rows = 9
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    packed = random_packed(encoding, 16 * 2 * units + 24, in_dim, 97).reshape(16 * 2 * units + 24, -1)
    x = kquant.synthetic_activations(98, rows, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    outputs = []
    for out_dim in (24, 16 * 2 * units + 24):
        weight = tile_ops.PackedWeight.from_numpy(encoding, packed[:out_dim].reshape(-1), out_dim, in_dim)
        outputs.append(tile_ops.multi_linear([weight], to_device(x, cuda), workspace)[0].cpu())
    checked = np.r_[0:24, 16 * units - 8:16 * units + 40, 16 * 2 * units - 16:16 * 2 * units + 24]
    expected = oracle.linear(encoding, packed[checked].reshape(-1), len(checked), in_dim, x)
    assert normalised_error(outputs[1].numpy()[:, checked], expected) <= TOLERANCE
    assert_bits_equal(outputs[0], outputs[1][:, :24].contiguous(), "one tile = its place among many")


@pytest.mark.parametrize("family,rows", [("mmq", 5), ("mmq", 16), ("mmvq", 7), ("mmvq", 16)])
@pytest.mark.parametrize("encoding,in_dim", [(kquant.Q4_K, 512), (kquant.Q5_K, 768), (kquant.Q6_K, 768), (kquant.Q8_0, 512),
                                             (kquant.Q8_0, 6144)])
def test_small_batch_tiles_of_fewer_rows(cuda, oracle, encoding, in_dim, family, rows):
    """Tiles of as few rows as keep every workgroup at its number of tiles: the fewest rows there are, one tile a
    workgroup with and without a remainder, two, three, and so many that tiles stay whole; alone and beside another
    projection.  A row has the bits it has in a launch of its own."""
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    most = 7 * 32 * units + 9
    packed = random_packed(encoding, most, in_dim, 31).reshape(most, -1)
    x = kquant.synthetic_activations(32, rows, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)

    def run(*spans):
        weights = [tile_ops.PackedWeight.from_numpy(encoding, packed[a:b].reshape(-1), b - a, in_dim) for a, b in spans]
        return [y.cpu() for y in tile_ops.multi_linear(weights, to_device(x, cuda), workspace, family=family)]

    (own,) = run((0, 40))
    expected = oracle.linear(encoding, packed[:40].reshape(-1), 40, in_dim, x)
    assert normalised_error(own.numpy(), expected) <= TOLERANCE
    sizes = [4 * units - 3, 4 * units + 1, 13 * units, 16 * units + 5, 26 * units, 26 * units + 1, 2 * 32 * units + 7, most]
    for out_dim in sizes if in_dim < 6144 else sizes[:5]:
        (y,) = run((0, out_dim))
        assert_bits_equal(y[:, :40].contiguous(), own, f"first rows of {out_dim}")
        (last,) = run((out_dim - 40, out_dim))
        assert_bits_equal(y[:, -40:].contiguous(), last, f"last rows of {out_dim}")
        middle = out_dim // 2
        (between,) = run((middle - 20, middle + 20))
        assert_bits_equal(y[:, middle - 20:middle + 20].contiguous(), between, f"middle rows of {out_dim}")
    first, second = run((0, 13 * units + 2), (40, 40 + 9 * units))
    assert_bits_equal(first[:, :40].contiguous(), own, "beside another projection")
    (alone,) = run((40, 80))
    assert_bits_equal(second[:, :40].contiguous(), alone, "the other projection")


@pytest.mark.parametrize("rows", [5, 16])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_gate_up_swiglu_rows_tiles_of_fewer_rows(cuda, encoding, rows):
    """The pair form's tiles likewise."""
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    in_dim, most = 512, 16 * units + 9
    packed = [random_packed(encoding, most, in_dim, seed).reshape(most, -1) for seed in (41, 42)]
    x = to_device(kquant.synthetic_activations(43, rows, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)

    def run(begin, end):
        gate, up = (tile_ops.PackedWeight.from_numpy(encoding, p[begin:end].reshape(-1), end - begin, in_dim) for p in packed)
        return tile_ops.gate_up_swiglu_rows(gate, up, x, rows, workspace).cpu()

    for out_dim in (4 * units + 1, 13 * units, most):
        y = run(0, out_dim)
        assert_bits_equal(y[:, :40].contiguous(), run(0, 40), f"first rows of {out_dim}")
        assert_bits_equal(y[:, -40:].contiguous(), run(out_dim - 40, out_dim), f"last rows of {out_dim}")


@pytest.mark.parametrize("in_dim", [4096, 8192, 8448, 16384])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K])
def test_decode_dot_kernel_row_lengths(cuda, oracle, encoding, in_dim):
    """The one-token kernel keeps a lane's activation operands in registers for rows of one or two
    64-unit slices (up to 8,192 columns) and reads them from LDS for longer rows; the verifier
    rows must equal it bit for bit at every length, grouped projections the single one."""
    out_dims = (40, 8, 19)  # a wave's rows cross the boundaries between the projections
    packed = [random_packed(encoding, n, in_dim, 80 + i) for i, n in enumerate(out_dims)]
    weights = [tile_ops.PackedWeight.from_numpy(encoding, p, n, in_dim) for p, n in zip(packed, out_dims)]
    x = kquant.synthetic_activations(81, 4, in_dim)
    workspace = tile_ops.small_batch_workspace(4, in_dim)
    one = tile_ops.multi_linear(weights, to_device(x[:1], cuda), workspace)
    for y, p, n in zip(one, packed, out_dims):
        expected = oracle.linear(encoding, p, n, in_dim, x[:1])
        assert normalised_error(y.cpu().numpy(), expected) <= TOLERANCE
    single = tile_ops.mmvq_linear(weights[1], to_device(x[:1], cuda), workspace)
    assert_bits_equal(single, one[1], "single projection = its place in the group")
    for rows in (2, 4):
        batch = tile_ops.multi_linear(weights, to_device(x[:rows], cuda), workspace, family="mmvq")
        for row in range(rows):
            alone = tile_ops.multi_linear(weights, to_device(x[row:row + 1], cuda), workspace)
            for whole, part in zip(batch, alone):
                assert_bits_equal(whole[row:row + 1].contiguous(), part, f"verifier row {row} of {rows}")


@pytest.mark.parametrize("in_dim", [256, 2304, 4096, 6656, 8448, 16384])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_verifier_matrix_core_rows_equal_the_one_row_kernel(cuda, oracle, encoding, in_dim):
    """From four rows on the verifier family's projections run on the int8 matrix cores, one
    pass over the weights: every row must still carry the one-row kernel's bits (for Q6_K both
    of its one-row kernels: rows of fewer than 16 blocks and the streaming one).
    Row lengths: one block (15 empty classes), 9 blocks, exactly one 16-block slice, 26 blocks
    (classes of one and two blocks), 33 and 64 blocks; output widths off the 32-row tile."""
    out_dims = (40, 8, 70)
    packed = [random_packed(encoding, n, in_dim, 90 + i) for i, n in enumerate(out_dims)]
    weights = [tile_ops.PackedWeight.from_numpy(encoding, p, n, in_dim) for p, n in zip(packed, out_dims)]
    x = kquant.synthetic_activations(91, 16, in_dim)
    x *= (10.0 ** np.arange(-3, 5).repeat(2))[:, None].astype(np.float32)  # rows of very different size
    one = tile_ops.small_batch_workspace(1, in_dim)
    alone = [tile_ops.multi_linear(weights, to_device(x[row:row + 1], cuda), one) for row in range(16)]
    for y, p, n in zip(alone[3], packed, out_dims):
        assert normalised_error(y.cpu().numpy(), oracle.linear(encoding, p, n, in_dim, x[3:4])) <= TOLERANCE
    for rows in (4, 5, 8, 9, 13, 16):
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        batch = tile_ops.multi_linear(weights, to_device(x[:rows], cuda), workspace, family="mmvq")
        for row in range(rows):
            for whole, part in zip(batch, alone[row]):
                assert_bits_equal(whole[row:row + 1].contiguous(), part, f"row {row} of {rows}")


@pytest.mark.parametrize("in_dim,out_dim", [(256, 40), (2304, 33), (6656, 70), (4096, 12289), (12544, 31), (512, 24577), (12544, 4100), (4352, 12289)])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_two_and_three_rows_equal_the_one_row_kernel_on_either_kernel(cuda, oracle, encoding, in_dim, out_dim):
    """Two and three rows of the one-row arithmetic run on the matrix cores where that is faster and the
    workspace has room for the operands: the same bits with it, with the records alone, and from the
    records that the call leaves.  Behind the prologues the same rows as alone."""
    packed = random_packed(encoding, 64, in_dim, 90).reshape(64, -1)
    chosen = torch_().from_numpy(np.random.default_rng(91).integers(0, 64, out_dim)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim,
                                   torch_().from_numpy(packed).to(cuda).index_select(0, chosen).reshape(-1))
    x = to_device(kquant.synthetic_activations(92, 3, in_dim) * np.array([[1.0], [1.0e3], [1.0e-3]], dtype=np.float32), cuda)
    second = to_device(kquant.synthetic_activations(93, 3, in_dim), cuda)
    one = tile_ops.small_batch_workspace(1, in_dim)
    for prologue in ("plain", "gated", "swiglu"):
        with_second = {} if prologue == "plain" else {"prologue": prologue}
        alone = [tile_ops.multi_linear([weight], x[r:r + 1].contiguous(), one, **with_second,
                                       **({"second": second[r:r + 1].contiguous()} if with_second else {}))[0] for r in range(3)]
        for rows, family in ((2, "mmq"), (2, "mmvq"), (3, "mmvq")):
            room = tile_ops.small_batch_workspace(rows, in_dim)
            for workspace in (room, room[:(rows * in_dim // 32 * 72 + 255) // 256 * 256]):
                batch = tile_ops.multi_linear([weight], x[:rows], workspace, family=family, **with_second,
                                              **({"second": second[:rows]} if with_second else {}))[0]
                for row in range(rows):
                    assert_bits_equal(batch[row:row + 1].contiguous(), alone[row], f"{prologue} {family} row {row} of {rows}")
            if family == "mmvq":
                assert_bits_equal(tile_ops.multi_linear_prequantized([weight], rows, workspace, family=family)[0], batch, "records")


@pytest.mark.parametrize("rows,prologue", [(3, "plain"), (4, "plain"), (3, "swiglu"), (4, "gated")])
@pytest.mark.parametrize("in_dim", [256, 8192, 8448, 12544])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q8_0])
def test_small_batches_of_three_and_four_rows(cuda, oracle, encoding, in_dim, rows, prologue):
    """Three and four rows of the other family: the same bits alone and beside a projection of another format,
    the prologue fused or materialised; Q8_0 in the one-row arithmetic, the rest to rounding."""
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, in_dim, 94 + n), n, in_dim)
               for e, n in ((encoding, 77), (kquant.Q6_K, 20))]
    x, second = (to_device(kquant.synthetic_activations(seed, rows, in_dim), cuda) for seed in (95, 96))
    arguments = {} if prologue == "plain" else {"prologue": prologue, "second": second}
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    exact = tile_ops.multi_linear(weights, x, workspace, family="mmvq", **arguments)
    alone = tile_ops.multi_linear(weights[:1], x, workspace, **arguments)[0]
    both = tile_ops.multi_linear(weights, x, workspace, **arguments)
    assert_bits_equal(both[0], alone, "beside another format")
    if encoding == kquant.Q8_0:
        assert_bits_equal(alone, exact[0], "the verifier's rows")
    for got, expected in zip(both, exact):
        assert normalised_error(got.cpu().numpy(), expected.cpu().numpy()) <= TOLERANCE
    if prologue != "plain":
        applied = tile_ops.sigmoid_gate(x, second) if prologue == "gated" else tile_ops.swiglu(x, second)
        assert_bits_equal(tile_ops.multi_linear(weights[:1], applied, workspace)[0], alone, "materialised")


@pytest.mark.parametrize("prologue", ["plain", "gated", "swiglu"])
@pytest.mark.parametrize("encoding,rows,out_dim,in_dim", [
    *((encoding, 2, out_dim, in_dim) for encoding in ALL_PACKED for out_dim, in_dim in ((77, 12544), (12289, 512))),
    *((encoding, rows, 77, 8448) for encoding in (kquant.Q4_K, kquant.Q5_K, kquant.Q8_0) for rows in (3, 4)),
    (kquant.Q8_0, 3, 12289, 512), (kquant.Q8_0, 4, 77, 4096),
])
def test_small_batches_leave_the_records_of_a_verifier_call(cuda, encoding, rows, out_dim, in_dim, prologue):
    """The other family at two rows, and at three and four where it quantizes inside its kernels, writes nothing
    into its workspace: records that a verifier call left there serve the prequantized call behind it."""
    packed = torch_().from_numpy(random_packed(encoding, 64, in_dim, 86).reshape(64, -1)).to(cuda)
    chosen = torch_().from_numpy(np.random.default_rng(87).integers(0, 64, out_dim)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, packed.index_select(0, chosen).reshape(-1))
    x, other, second = (to_device(kquant.synthetic_activations(seed, rows, in_dim), cuda) for seed in (88, 89, 85))
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    expected = tile_ops.multi_linear([weight], x, workspace, family="mmvq")[0]
    before = workspace.clone()
    tile_ops.multi_linear([weight], other, workspace, **({} if prologue == "plain" else {"prologue": prologue, "second": second}))
    assert bool((workspace == before).all())
    after = tile_ops.multi_linear_prequantized([weight], rows, workspace, family="mmvq")[0]
    assert_bits_equal(after, expected, "from the records")


@pytest.mark.parametrize("rows", [3, 4])
@pytest.mark.parametrize("in_dim", [8192, 8448])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K])
def test_lm_head_of_three_and_four_rows_is_the_maximum_of_the_calls_logits(cuda, encoding, in_dim, rows):
    """The fused choice and its value are those of the small-batch call's logits, bit for bit, on both sides
    of the widths at which their kernels change."""
    out_dim = 4133
    packed = torch_().from_numpy(random_packed(encoding, 64, in_dim, 81).reshape(64, -1)).to(cuda)
    chosen = torch_().from_numpy(np.random.default_rng(82).integers(0, 64, out_dim)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, packed.index_select(0, chosen).reshape(-1))
    x = to_device(kquant.synthetic_activations(83, rows, in_dim), cuda)
    logits = tile_ops.multi_linear([weight], x, tile_ops.small_batch_workspace(rows, in_dim))[0]
    indices, values = tile_ops.lm_head_argmax(weight, x)
    best = logits.max(dim=1)
    assert_bits_equal(values.reshape(-1), best.values, "the largest logit")
    for row in range(rows):
        assert indices[row].item() == int((logits[row] == best.values[row]).nonzero()[0].item())


@pytest.mark.parametrize("in_dim", [4096, 4352, 6656])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_verifier_matrix_core_rows_of_many_tiles_a_workgroup(cuda, encoding, in_dim):
    """Up to eight tokens a wave's share of a row's blocks moves on from tile to tile (rows of 16,
    17 and 26 blocks: even shares, one wave with a block more, two) and comes round after four
    tiles: five and six tiles a workgroup, the last one part of a tile, against the one-row call."""
    torch = torch_()
    units = torch.cuda.get_device_properties(0).multi_processor_count
    out_dim = 32 * (5 * units + units // 3) + 9
    rows_of = torch.from_numpy(random_packed(encoding, 512, in_dim, 77).reshape(512, -1)).to(cuda)
    chosen = torch.randint(0, 512, (out_dim,), generator=torch.Generator().manual_seed(78)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, rows_of.index_select(0, chosen).reshape(-1))
    x = to_device(kquant.synthetic_activations(79, 8, in_dim), cuda)
    one = tile_ops.small_batch_workspace(1, in_dim)
    alone = [tile_ops.mmvq_linear(weight, x[row:row + 1], one) for row in range(8)]
    for rows in (4, 7, 8):
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        batch = tile_ops.multi_linear([weight], x[:rows], workspace, family="mmvq")[0]
        for row in range(rows):
            assert_bits_equal(batch[row:row + 1].contiguous(), alone[row], f"row {row} of {rows}")


@pytest.mark.parametrize("in_dim,out_dim", [(256, 42000), (1024, 50000), (6656, 8704), (6656, 13000)])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_verifier_matrix_core_rows_whose_waves_wait_by_counts(cuda, encoding, in_dim, out_dim):
    """Waves without a block of their own over six tiles, halves of tiles shared by two workgroups (one
    and two a workgroup), tokens that leave some waves nothing to add, against the one-row call."""
    weight = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, out_dim, in_dim, 81), out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(82, 8, in_dim), cuda)
    one = tile_ops.small_batch_workspace(1, in_dim)
    alone = [tile_ops.mmvq_linear(weight, x[row:row + 1], one) for row in range(8)]
    for rows in (4, 5, 7, 8):
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        batch = tile_ops.multi_linear([weight], x[:rows], workspace, family="mmvq")[0]
        for row in range(rows):
            assert_bits_equal(batch[row:row + 1].contiguous(), alone[row], f"row {row} of {rows}")


@pytest.mark.parametrize("in_dim,over", [(2048, 64), (4096, 8), (4352, 33), (6656, 64)])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_verifier_matrix_core_rows_by_halves(cuda, encoding, in_dim, over):
    """A few tiles more than compute units, up to eight tokens: halves of tiles (rows of eight blocks: the
    right ones empty), walks of an even and an odd number of steps, the last tile part of one, with the
    quantizer's fill of the outputs and with one of its own, against the one-row call."""
    torch = torch_()
    out_dim = 32 * (torch.cuda.get_device_properties(0).multi_processor_count + over) - 5
    rows_of = torch.from_numpy(random_packed(encoding, 512, in_dim, 83).reshape(512, -1)).to(cuda)
    chosen = torch.randint(0, 512, (out_dim,), generator=torch.Generator().manual_seed(84)).to(cuda)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, rows_of.index_select(0, chosen).reshape(-1))
    x = to_device(kquant.synthetic_activations(85, 8, in_dim), cuda)
    one = tile_ops.small_batch_workspace(1, in_dim)
    alone = [tile_ops.mmvq_linear(weight, x[row:row + 1], one) for row in range(8)]
    for rows in (4, 5, 8):
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        batch = tile_ops.multi_linear([weight], x[:rows], workspace, family="mmvq")[0]
        for row in range(rows):
            assert_bits_equal(batch[row:row + 1].contiguous(), alone[row], f"row {row} of {rows}")
        again = tile_ops.multi_linear_prequantized([weight], rows, workspace)[0]
        assert_bits_equal(again, batch, f"{rows} rows prequantized")


@pytest.mark.parametrize("in_dim,out_dim", [(6656, 3000), (6656, 4608), (13312, 2100), (4096, 2500)])
def test_q6k_rows_carry_the_same_bits_wherever_their_wave_starts(cuda, oracle, in_dim, out_dim):
    """The Q6_K streaming kernel hands a wave a contiguous range of rows, and how many depends on
    the launch (output width, tokens per pass, waves per workgroup, the other projections of the
    call); a row of 26 or 52 blocks then starts inside a 16-block pass.  Its bits must not depend
    on where: verifier rows at 2, 4 and 16 tokens equal the one-row call, and a projection alone
    equals the same projection inside a group."""
    encoding = kquant.Q6_K
    packed = random_packed(encoding, out_dim, in_dim, 61)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    other = tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, 256, in_dim, 62), 256, in_dim)
    x = kquant.synthetic_activations(63, 16, in_dim)
    one = tile_ops.small_batch_workspace(1, in_dim)
    alone = [tile_ops.mmvq_linear(weight, to_device(x[row:row + 1], cuda), one) for row in range(16)]
    picked = np.arange(0, out_dim, 37)
    expected = oracle.linear(encoding, packed.reshape(out_dim, -1)[picked].reshape(-1), picked.size, in_dim, x[:1])
    assert normalised_error(alone[0].cpu().numpy()[:, picked], expected) <= TOLERANCE
    grouped = tile_ops.multi_linear([other, weight], to_device(x[:1], cuda), one, family="mmvq")
    assert_bits_equal(grouped[1], alone[0], "a projection alone = its place in a group")
    for rows in (2, 4, 16):
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        batch = tile_ops.multi_linear([weight], to_device(x[:rows], cuda), workspace, family="mmvq")[0]
        for row in range(rows):
            assert_bits_equal(batch[row:row + 1].contiguous(), alone[row], f"row {row} of {rows}")


@pytest.mark.parametrize("prologue", ["gated", "swiglu"])
def test_verifier_matrix_core_rows_with_prologues_and_mixed_formats(cuda, prologue):
    """Fused prologues go through the quantizer launch; the Q6_K and Q8_0 projections of the same
    call read the records it wrote."""
    in_dim, rows = 1280, 11
    specs = [(kquant.Q4_K, 33), (kquant.Q6_K, 40), (kquant.Q5_K, 64), (kquant.Q8_0, 24)]
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, in_dim, 95 + i), n, in_dim)
               for i, (e, n) in enumerate(specs)]
    x = to_device(kquant.synthetic_activations(96, rows, in_dim), cuda)
    g = to_device(kquant.synthetic_activations(97, rows, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    one = tile_ops.small_batch_workspace(1, in_dim)
    batch = tile_ops.multi_linear(weights, x, workspace, g, "mmvq", prologue)
    again = tile_ops.multi_linear_prequantized(weights, rows, workspace)
    for row in range(rows):
        alone = tile_ops.multi_linear(weights, x[row:row + 1], one, g[row:row + 1], "mmvq", prologue)
        for whole, reused, part, (encoding, _) in zip(batch, again, alone, specs):
            assert_bits_equal(whole[row:row + 1].contiguous(), part, f"{kquant.NAMES[encoding]} row {row}")
            assert_bits_equal(reused[row:row + 1].contiguous(), part, f"prequantized {kquant.NAMES[encoding]} row {row}")


@pytest.mark.parametrize("magnitude", [1e-4, 1.0, 1e3])
@pytest.mark.parametrize("encoding", ALL_PACKED)
@pytest.mark.parametrize("rows", [5, 16])
def test_small_batch_keeps_the_bound_for_weights_of_other_magnitudes(cuda, oracle, encoding, rows, magnitude):
    """The 5..16-row kernels of the mmq family hold weights as fp16 on their way into the matrix
    instruction: the block factors d * sc of tensors far smaller (or larger) than the N(0, 0.02)
    of the other tests must not leave that format's range."""
    in_dim, out_dim = 1536, 72
    weights = kquant.synthetic_weights(500 + encoding, out_dim, in_dim) * np.float32(magnitude / 0.02)
    packed = kquant.quantize(encoding, weights)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    x = kquant.synthetic_activations(501, rows, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    (y,) = tile_ops.multi_linear([weight], to_device(x, cuda), workspace)
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y.cpu().numpy(), expected) <= TOLERANCE
    indices, maxima = tile_ops.lm_head_argmax(weight, to_device(x, cuda))
    for row in range(rows):
        assert abs(float(maxima[row]) - expected[row].max()) <= TOLERANCE * np.max(np.abs(expected[row]))


# ------------------------------------------------------------------- argmax

def test_argmax_rows_tie_rule_at_vocabulary_width(cuda):
    # probe :1869-1904
    rows, width = 3, 202048
    values = np.full((rows, width), -9.0, np.float32)
    values[0, 17] = 10.0
    values[0, 123] = 10.0
    values[1, width - 1] = 5.5
    values[2, 0] = -1.0
    indices, maxima = tile_ops.argmax_rows(to_device(values, cuda))
    assert indices.cpu().tolist() == [17, width - 1, 0]
    assert maxima.cpu().tolist() == [10.0, 5.5, -1.0]


def test_argmax_rows_random_and_nan(cuda, oracle):
    rng = np.random.default_rng(1)
    values = rng.standard_normal((4, 50001)).astype(np.float32)
    values[1, 100] = np.nan
    values[2, :] = np.nan
    values[3, 7] = values[3].max()
    indices, maxima = tile_ops.argmax_rows(to_device(values, cuda))
    indices = indices.cpu().tolist()
    assert indices[0] == oracle.argmax(values[0])
    assert indices[1] == int(np.nanargmax(values[1]))
    assert indices[2] == 0 and maxima.cpu()[2].item() == -np.inf
    assert indices[3] == min(7, int(np.argmax(values[3])))


@pytest.mark.parametrize("rows", [1, 3, 5, 8, 16])
@pytest.mark.parametrize("encoding", [kquant.Q6_K, kquant.Q4_K, kquant.Q5_K, kquant.Q8_0])
def test_lm_head_fused_argmax_against_oracle(cuda, oracle, encoding, rows):
    out_dim, in_dim = 4099, 1024
    packed = kquant.quantize(encoding, kquant.synthetic_weights(80 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(90 + rows, rows, in_dim, rms_normalize=True)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    indices, maxima = tile_ops.lm_head_argmax(weight, to_device(x, cuda))
    logits = oracle.linear(encoding, packed, out_dim, in_dim, x)
    scale = np.max(np.abs(logits))
    for row in range(rows):
        ordered = np.sort(logits[row])[::-1]
        assert abs(maxima.cpu()[row].item() - ordered[0]) <= TOLERANCE * scale
        if ordered[0] - ordered[1] > 2 * TOLERANCE * scale:  # argmax exact on non-tied rows
            assert indices.cpu()[row].item() == oracle.argmax(logits[row])
        else:
            assert logits[row, indices.cpu()[row].item()] >= ordered[0] - 2 * TOLERANCE * scale


@pytest.mark.parametrize("out_dim", [33, 4096, 4097, 8192, 9001, 12288, 12289, 24576, 24577])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q8_0])
def test_lm_head_one_row_leaves_what_lies_behind_its_workspace(cuda, encoding, out_dim):
    """Small vocabularies are spread over more workgroups, each of which leaves a candidate: with the query's
    workspace and with less nothing behind it is written, and the choice is that of the logits."""
    in_dim, lib = 256, tile_ops.load()
    packed = torch_().from_numpy(random_packed(encoding, 64, in_dim, 97).reshape(64, -1)).to(cuda)
    chosen = torch_().from_numpy(np.random.default_rng(98).integers(0, 63, out_dim)).to(cuda)
    chosen[out_dim - 1] = 63
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, packed.index_select(0, chosen).reshape(-1))
    x = to_device(kquant.synthetic_activations(99, 1, in_dim), cuda)
    logits = tile_ops.linear(weight, x)[0].cpu().numpy()
    asked = lib.nfn_mi355_lm_head_argmax_workspace_bytes_v1(1, out_dim)
    assert asked >= (out_dim + 31) // 32 * 16
    for nbytes in (asked, asked - 16, asked - 256):
        workspace = torch_().full((asked + 65536,), 0x5a, dtype=torch_().uint8, device=cuda)
        indices, maxima = (torch_().zeros(1, dtype=d, device=cuda) for d in (torch_().int64, torch_().float32))
        descriptor = weight.descriptor()
        status = lib.nfn_mi355_lm_head_argmax_v1(ctypes.byref(descriptor), x.data_ptr(), indices.data_ptr(),
                                                 maxima.data_ptr(), 1, workspace.data_ptr(), nbytes, None)
        torch_().cuda.synchronize()
        assert bool((workspace[nbytes:] == 0x5a).all())
        if nbytes == asked:
            assert status == 0
        if status == 0:
            best = logits.max()
            assert abs(maxima.item() - best) <= 1e-5 * np.abs(logits).max()
            assert logits[indices.item()] >= best - 2e-5 * np.abs(logits).max()


@pytest.mark.parametrize("rows", [1, 2, 5, 16])
def test_lm_head_fused_argmax_tie_goes_to_lowest_index(cuda, rows):
    # Identical vocabulary rows, two in one 32-row tile and one far away: the
    # lowest index must win for every token (all tokens carry the same input).
    out_dim, in_dim = 3000, 512
    w = kquant.synthetic_weights(5, out_dim, in_dim)
    x = np.repeat(kquant.synthetic_activations(6, 1, in_dim), rows, axis=0)
    best = w[100] * 0 + np.sign(x[0]) * 0.05
    w[100] = best
    w[110] = best
    w[2900] = best
    packed = kquant.quantize(kquant.Q6_K, w)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q6_K, packed, out_dim, in_dim)
    indices, _ = tile_ops.lm_head_argmax(weight, to_device(x, cuda))
    assert indices.cpu().tolist() == [100] * rows


def test_lm_head_fused_argmax_fails_closed(cuda):
    """Row counts and forms the call does not take, refused before any launch (the weights
    behind these descriptors do not exist)."""
    lib = tile_ops.load()
    torch = torch_()
    out_dim = 4096
    x = torch.zeros((16, 32768), dtype=torch.float32, device=cuda)
    indices = torch.full((16,), -7, dtype=torch.int64, device=cuda)
    maxima = torch.zeros(16, dtype=torch.float32, device=cuda)
    nbytes = lib.nfn_mi355_lm_head_argmax_workspace_bytes_v1(16, out_dim)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=cuda)

    def call(encoding, in_dim, rows, size=nbytes):
        descriptor = tile_ops.make_descriptor(encoding, 0x1000, out_dim, in_dim)
        return lib.nfn_mi355_lm_head_argmax_v1(ctypes.byref(descriptor), x.data_ptr(), indices.data_ptr(),
                                               maxima.data_ptr(), rows, workspace.data_ptr(), size, None)

    assert call(kquant.Q6_K, 1024, 17) == 1           # beyond a block of 16
    assert call(kquant.Q6_K, 1024, 0) == 1
    assert call(kquant.F32, 1024, 9) == 1             # 9..16 rows: packed formats only
    assert call(kquant.Q4_K, 32768, 9) == 1           # ... of at most 16,384 columns
    assert call(kquant.Q6_K, 1024, 16, 4096) == 1     # workspace too small
    torch.cuda.synchronize()
    assert int(indices[0]) == -7


@pytest.mark.parametrize("shape", [(130, 256), (515, 6656)])
def test_q8_0_one_token_and_verifier(cuda, oracle, shape):
    out_dim, in_dim = shape
    packed = random_packed(kquant.Q8_0, out_dim, in_dim, 61)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q8_0, packed, out_dim, in_dim)
    x = kquant.synthetic_activations(62, 5, in_dim)
    workspace = tile_ops.small_batch_workspace(5, in_dim)
    expected = oracle.linear(kquant.Q8_0, packed, out_dim, in_dim, x)
    batched = tile_ops.multi_linear([weight], to_device(x, cuda), workspace, family="mmvq")[0]
    assert normalised_error(batched.cpu().numpy(), expected) <= TOLERANCE
    for row in range(5):
        single = tile_ops.mmvq_linear(weight, to_device(x[row:row + 1], cuda), workspace)
        assert_bits_equal(single, batched[row:row + 1], f"row {row}")
    one = tile_ops.multi_linear([weight], to_device(x[:1], cuda), workspace, family="mmq")[0]
    assert_bits_equal(one, batched[:1], "mmq at one row")


# ------------------------------------------------ Q6_K rows of 16 blocks and more (streaming kernel)

@pytest.mark.parametrize("shape", [(777, 4096), (1301, 6656), (64, 8192), (33, 4352)])
def test_q6_k_long_rows_one_token_and_verifier(cuda, oracle, shape):
    # row counts that leave partial passes and waves without rows; K of exactly
    # 16 blocks, of 26 (rows straddle passes) and of 32
    out_dim, in_dim = shape
    packed = random_packed(kquant.Q6_K, out_dim, in_dim, 51)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q6_K, packed, out_dim, in_dim)
    x = kquant.synthetic_activations(52, 3, in_dim)
    workspace = tile_ops.small_batch_workspace(3, in_dim)
    expected = oracle.linear(kquant.Q6_K, packed, out_dim, in_dim, x)
    batched = tile_ops.multi_linear([weight], to_device(x, cuda), workspace, family="mmvq")[0]
    assert normalised_error(batched.cpu().numpy(), expected) <= TOLERANCE
    for row in range(3):
        single = tile_ops.mmvq_linear(weight, to_device(x[row:row + 1], cuda), workspace)
        assert_bits_equal(single, batched[row:row + 1], f"row {row}")
    one = tile_ops.multi_linear([weight], to_device(x[:1], cuda), workspace, family="mmq")[0]
    assert_bits_equal(one, batched[:1], "mmq at one row")


@pytest.mark.parametrize("out_dims", [(1301, 257, 63, 910), (1, 4097, 2), (513, 1)])
@pytest.mark.parametrize("in_dim", [4352, 6656])
def test_q6_k_long_rows_grouped_projections_end_in_partial_waves(cuda, oracle, in_dim, out_dims):
    """Where each projection's waves begin and how many rows its last one lacks reach the streaming kernel packed: every
    projection of a call has the bits of its own call, for one token and for two and three of the verifier."""
    x = kquant.synthetic_activations(66, 3, in_dim)
    packed = [random_packed(kquant.Q6_K, out_dim, in_dim, 67 + out_dim) for out_dim in out_dims]
    weights = [tile_ops.PackedWeight.from_numpy(kquant.Q6_K, p, out_dim, in_dim) for p, out_dim in zip(packed, out_dims)]
    workspace = tile_ops.small_batch_workspace(3, in_dim)
    for rows, family in ((1, "mmq"), (1, "mmvq"), (2, "mmvq"), (3, "mmvq")):
        together = tile_ops.multi_linear(weights, to_device(x[:rows], cuda), workspace, family=family)
        for weight, y in zip(weights, together):
            alone = tile_ops.multi_linear([weight], to_device(x[:rows], cuda), workspace, family=family)[0]
            assert_bits_equal(y, alone, f"{weight.output_dim} outputs, {rows} rows")
    for p, out_dim, y in zip(packed, out_dims, together):
        assert normalised_error(y.cpu().numpy(), oracle.linear(kquant.Q6_K, p, out_dim, in_dim, x)) <= TOLERANCE


@pytest.mark.parametrize("per_unit,in_dim,prologue", [(8.0, 12288, "plain"), (11.99, 12544, "swiglu"),
                                                      (17.3, 16384, "plain"), (23.9, 12288, "gated")])
def test_q6_k_long_rows_with_fewer_waves_a_workgroup(cuda, oracle, per_unit, in_dim, prologue):
    """One token over rows of 48 blocks and more: output widths that would leave compute units
    without a sixteen-wave workgroup run with 8 to 12 waves (one row a wave, then two, the last
    workgroups short of rows); two rows of the verifier family take another form and give the
    same bits."""
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    out_dim = int(per_unit * units)
    packed = random_packed(kquant.Q6_K, 256, in_dim, 57).reshape(256, -1)
    chosen = np.random.default_rng(58).integers(0, 256, out_dim)
    weight = tile_ops.PackedWeight(kquant.Q6_K, out_dim, in_dim, torch_().from_numpy(packed).to(cuda).index_select(
        0, torch_().from_numpy(chosen).to(cuda)).reshape(-1))
    x = kquant.synthetic_activations(59, 2, in_dim)
    options = {} if prologue == "plain" else {"second": to_device(x, cuda), "prologue": prologue}
    workspace = tile_ops.small_batch_workspace(2, in_dim)
    batch = tile_ops.multi_linear([weight], to_device(x, cuda), workspace, family="mmvq", **options)[0]
    for row in range(2):
        here = {k: v[row:row + 1] if k == "second" else v for k, v in options.items()}
        single = tile_ops.multi_linear([weight], to_device(x[row:row + 1], cuda), workspace, **here)[0]
        assert_bits_equal(single, batch[row:row + 1].contiguous(), f"row {row}")
    if prologue == "plain":
        expected = oracle.linear(kquant.Q6_K, packed.reshape(-1), 256, in_dim, x)[:, chosen]
        assert normalised_error(batch.cpu().numpy(), expected) <= TOLERANCE


def test_q6_k_long_rows_tensor_two_bytes_off_a_word(cuda, oracle):
    """The streaming kernel reads word-aligned pieces when the tensor starts on a four-byte
    boundary; a tensor that does not is read the plain way and gives the same bits."""
    out_dim, in_dim = 33, 4352
    packed = random_packed(kquant.Q6_K, out_dim, in_dim, 53)
    aligned = tile_ops.PackedWeight.from_numpy(kquant.Q6_K, packed, out_dim, in_dim)
    holder = torch_().empty(packed.size + 2, dtype=torch_().uint8, device=cuda)
    holder[2:].copy_(torch_().from_numpy(packed.reshape(-1)))
    shifted = tile_ops.PackedWeight(kquant.Q6_K, out_dim, in_dim, holder[2:])
    assert shifted.data.data_ptr() % 4 == 2
    x = kquant.synthetic_activations(54, 1, in_dim)
    workspace = tile_ops.small_batch_workspace(1, in_dim)
    a = tile_ops.mmvq_linear(aligned, to_device(x, cuda), workspace)
    b = tile_ops.mmvq_linear(shifted, to_device(x, cuda), workspace)
    assert normalised_error(a.cpu().numpy(), oracle.linear(kquant.Q6_K, packed, out_dim, in_dim, x)) <= TOLERANCE
    assert_bits_equal(a, b, "aligned and shifted tensor")


@pytest.mark.parametrize("encoding,in_dim", [(kquant.Q6_K, 4352), (kquant.Q6_K, 6656), (kquant.Q6_K, 768),
                                             (kquant.Q8_0, 4352), (kquant.Q8_0, 1280)])
def test_verifier_matrix_core_rows_tensor_two_bytes_off_a_word(cuda, encoding, in_dim):
    """The matrix-core rows kernel fetches Q6_K blocks from the word at or before their first
    byte (rows of an odd number of blocks alternate between the two cases, and so does a tensor
    that starts two bytes past a word) and Q8_0 rows as they lie: a shifted tensor gives the
    bits of the aligned one, which the other tests tie to the one-row call."""
    out_dim = 75
    packed = random_packed(encoding, out_dim, in_dim, 55)
    aligned = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    holder = torch_().empty(packed.size + 2, dtype=torch_().uint8, device=cuda)
    holder[2:].copy_(torch_().from_numpy(packed.reshape(-1)))
    shifted = tile_ops.PackedWeight(encoding, out_dim, in_dim, holder[2:])
    assert shifted.data.data_ptr() % 4 == 2
    for rows in (4, 16):
        x = to_device(kquant.synthetic_activations(56, rows, in_dim), cuda)
        workspace = tile_ops.small_batch_workspace(rows, in_dim)
        a = tile_ops.multi_linear([aligned], x, workspace, family="mmvq")[0]
        b = tile_ops.multi_linear([shifted], x, workspace, family="mmvq")[0]
        assert_bits_equal(a, b, f"aligned and shifted tensor, {rows} rows")
        single = tile_ops.mmvq_linear(shifted, x[rows - 1:rows], workspace)
        assert_bits_equal(single, a[rows - 1:rows].contiguous(), "the one-row call on the shifted tensor")


def shifted_copy(array, offset, device):
    """The values of `array` in a tensor that starts `offset` bytes into an allocation and ends with it."""
    flat = torch_().from_numpy(np.ascontiguousarray(array)).reshape(-1).view(torch_().uint8)
    holder = torch_().empty(flat.numel() + offset, dtype=torch_().uint8, device=device)
    holder[offset:].copy_(flat)
    return holder[offset:]


def shifted_floats(array, device):
    flat = torch_().empty(array.size + 1, dtype=torch_().float32, device=device)[1:]
    flat.copy_(torch_().from_numpy(np.ascontiguousarray(array)).reshape(-1))
    assert flat.data_ptr() % 16 == 4
    return flat.reshape(array.shape)


@pytest.mark.parametrize("rows,out_dim,in_dim", [(1, 75, 768), (3, 1030, 512), (5, 75, 768), (60, 5000, 256),
                                                 (100, 6600, 256), (200, 6600, 256)])
@pytest.mark.parametrize("encoding", ALL_PACKED + [kquant.F32, kquant.BF16])
def test_exact_linear_on_tensors_off_a_word(cuda, encoding, rows, out_dim, in_dim):
    """Every form: weights two bytes (floats four) and activations four bytes off the boundary that
    their loads would like, at the end of their allocations: the bits of the aligned call."""
    packed = kquant.quantize(encoding, kquant.synthetic_weights(57, out_dim, in_dim))
    x, bias = kquant.synthetic_activations(58, rows, in_dim), kquant.synthetic_activations(59, 1, out_dim)[0]
    aligned = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    data = shifted_copy(packed, 4 if encoding == kquant.F32 else 2, cuda)
    shifted = tile_ops.PackedWeight(encoding, out_dim, in_dim, data)
    assert shifted.data.data_ptr() % 16 in (2, 4)
    expected = tile_ops.linear(aligned, to_device(x, cuda), to_device(bias, cuda))
    assert_bits_equal(tile_ops.linear(shifted, shifted_floats(x, cuda), shifted_floats(bias, cuda)), expected)


@pytest.mark.parametrize("rows", [1, 3, 4, 16, 17, 21, 40])
@pytest.mark.parametrize("in_dim", [256, 512, 768, 1280, 2304])
@pytest.mark.parametrize("encoding", [kquant.Q6_K, kquant.Q8_0])
def test_exact_linear_of_blocks_past_a_word(cuda, oracle, encoding, in_dim, rows):
    """Blocks that start two bytes past a word are read from the word before them: rows of odd and even
    numbers of blocks, tensors that start at a word and two bytes past it, the first and the last block of
    a tensor.  Bound as for the forms' edges above."""
    out_dim = 35 if rows < 40 else 5000  # (32 x 64 tiles)
    packed = random_packed(encoding, out_dim, in_dim, 64)
    x = kquant.synthetic_activations(65, rows, in_dim)
    aligned = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    shifted = tile_ops.PackedWeight(encoding, out_dim, in_dim, shifted_copy(packed, 2, cuda))
    y = tile_ops.linear(aligned, to_device(x, cuda))
    assert_bits_equal(tile_ops.linear(shifted, to_device(x, cuda)), y)
    checked = np.r_[0:35] if out_dim == 35 else np.r_[0:33, 4960:5000]
    expected = oracle.linear(encoding, packed.reshape(out_dim, -1)[checked].reshape(-1), len(checked), in_dim, x)
    assert normalised_error(y.cpu().numpy()[:, checked], expected) <= 1e-5


@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_lm_head_one_row_on_tensors_off_a_word(cuda, encoding):
    out_dim, in_dim = 4099, 1280
    packed = random_packed(encoding, out_dim, in_dim, 60)
    x = kquant.synthetic_activations(61, 1, in_dim)
    aligned = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    shifted = tile_ops.PackedWeight(encoding, out_dim, in_dim, shifted_copy(packed, 2, cuda))
    indices, maxima = tile_ops.lm_head_argmax(aligned, to_device(x, cuda))
    again, again_maxima = tile_ops.lm_head_argmax(shifted, shifted_floats(x, cuda))
    assert torch_().equal(indices, again)
    assert_bits_equal(maxima, again_maxima)


@pytest.mark.parametrize("rows,out_dim,in_dim", [(17, 129, 1536), (96, 130, 3072), (300, 1030, 1280), (700, 6656, 512)])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_on_tensors_off_a_word(cuda, encoding, rows, out_dim, in_dim):
    """Up to 32 rows, K shares of 128-row tiles, and 256-row tiles; the output four bytes off as well."""
    packed = random_packed(encoding, out_dim, in_dim, 62)
    x = kquant.synthetic_activations(63, rows, in_dim)
    aligned = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    shifted = tile_ops.PackedWeight(encoding, out_dim, in_dim, shifted_copy(packed, 2, cuda))
    out = shifted_floats(np.zeros((rows, out_dim), dtype=np.float32), cuda)
    expected = tile_ops.gemm(aligned, to_device(x, cuda))
    assert_bits_equal(tile_ops.gemm(shifted, shifted_floats(x, cuda), out=out), expected)


@pytest.mark.parametrize("in_dim", [256, 1024, 6656, 6912])
@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_fp16_rows_last_row_of_a_tensor_and_shifted_tensors(cuda, encoding, in_dim):
    """The fp16 small-batch kernel brings Q6_K and Q8_0 blocks into LDS in 16-byte pieces from
    wherever a row starts; the piece behind a tensor's very last block would reach past the
    tensor and is fetched another way.  The last row of a tensor gives the bits the same row
    gives inside a taller tensor (where its blocks go the ordinary way), for a last tile of
    one row and of several, and a tensor that starts one, two or three bytes past a word gives
    the bits of the aligned one.  (The other tests tie these bits to the oracle.)"""
    torch = torch_()
    tall_dim = 53
    packed = random_packed(encoding, tall_dim, in_dim, 57)
    tall = tile_ops.PackedWeight.from_numpy(encoding, packed, tall_dim, in_dim)
    rows = 16
    x = to_device(kquant.synthetic_activations(58, rows, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    expected = tile_ops.multi_linear([tall], x, workspace)[0]
    row_bytes = packed.size // tall_dim
    for out_dim in (1, 16, 17, 37, 48):
        short = tile_ops.PackedWeight.from_numpy(encoding, packed.reshape(-1)[:out_dim * row_bytes].copy(),
                                                 out_dim, in_dim)
        got = tile_ops.multi_linear([short], x, workspace)[0]
        assert_bits_equal(got, expected[:, :out_dim].contiguous(), f"a tensor of {out_dim} rows")
    for shift in (1, 2, 3):
        if shift != 2 and encoding != kquant.Q8_0 and encoding != kquant.Q6_K:
            continue
        holder = torch.empty(packed.size + shift, dtype=torch.uint8, device=cuda)
        holder[shift:].copy_(torch.from_numpy(packed.reshape(-1)))
        shifted = tile_ops.PackedWeight(encoding, tall_dim, in_dim, holder[shift:])
        assert shifted.data.data_ptr() % 4 == shift
        got = tile_ops.multi_linear([shifted], x, workspace)[0]
        assert_bits_equal(got, expected, f"a tensor {shift} bytes past a word")
    # the fused argmax over the short tensors' last tile
    short = tile_ops.PackedWeight.from_numpy(encoding, packed.reshape(-1)[:37 * row_bytes].copy(), 37, in_dim)
    indices, maxima = tile_ops.lm_head_argmax(short, x)
    assert torch.equal(maxima.cpu(), expected[:, :37].max(dim=1).values.cpu())


@pytest.mark.parametrize("rows", [1, 3, 8, 16])
def test_q6_k_long_rows_lm_head(cuda, oracle, rows):
    out_dim, in_dim = 5003, 6656
    packed = kquant.quantize(kquant.Q6_K, kquant.synthetic_weights(83, out_dim, in_dim))
    x = kquant.synthetic_activations(93 + rows, rows, in_dim, rms_normalize=True)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q6_K, packed, out_dim, in_dim)
    indices, maxima = tile_ops.lm_head_argmax(weight, to_device(x, cuda))
    logits = oracle.linear(kquant.Q6_K, packed, out_dim, in_dim, x)
    scale = np.max(np.abs(logits))
    for row in range(rows):
        ordered = np.sort(logits[row])[::-1]
        assert abs(maxima.cpu()[row].item() - ordered[0]) <= TOLERANCE * scale
        if ordered[0] - ordered[1] > 2 * TOLERANCE * scale:
            assert indices.cpu()[row].item() == oracle.argmax(logits[row])
    # the fused result equals argmax over the unfused logits of the same kernel
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    family = "mmvq" if rows == 1 else "mmq"  # one row: dot kernel; more: matrix cores (fp16 from three rows of Q6_K)
    unfused = tile_ops.multi_linear([weight], to_device(x, cuda), workspace, family=family)[0]
    assert torch_().equal(unfused.max(dim=1).values.cpu(), maxima.cpu())


@pytest.mark.parametrize("rows", [1, 4, 16])
def test_lm_head_full_vocabulary_planted_maxima(cuda, oracle, rows):
    # The benchmark's lm_head (Q6_K, 6656 -> 202048, 1.1 GB) with random bytes
    # and planted rows: every token's winner is known, one of them twice (the
    # lower index must win), one at the last vocabulary row.
    torch = torch_()
    out_dim, in_dim = 202048, 6656
    generator = torch.Generator(device=cuda).manual_seed(11)
    blocks = torch.randint(0, 256, (out_dim * in_dim // 256, 210), generator=generator,
                           device=cuda, dtype=torch.uint8)
    blocks[:, 209] = (blocks[:, 209] & 0x03) | 0x14          # d in [2^-10, 2^-9)
    packed = blocks.reshape(out_dim, -1)
    x = kquant.synthetic_activations(95, rows, in_dim, rms_normalize=True)
    planted = {0: [17, 150000], 1: [202047], 2: [101010], 3: [4096]}
    planted.update({token: [7919 * token + 13] for token in range(4, 16)})
    planted[9] = [202032, 31]  # the first row of the last 16-row tile, and an earlier row
    expected_index, expected_value = [], []
    for token in range(rows):
        strong = (np.sign(x[token]) * 8.0).astype(np.float32).reshape(1, in_dim)
        row_bytes = kquant.quantize(kquant.Q6_K, strong)
        for index in planted[token]:
            packed[index] = to_device(row_bytes, cuda)
        expected_index.append(min(planted[token]))
        expected_value.append(oracle.linear(kquant.Q6_K, row_bytes, 1, in_dim, x[token:token + 1])[0, 0])
    weight = tile_ops.PackedWeight(kquant.Q6_K, out_dim, in_dim, packed.reshape(-1))
    indices, maxima = tile_ops.lm_head_argmax(weight, to_device(x, cuda))
    assert indices.cpu().tolist() == expected_index
    for token in range(rows):
        # a planted row of one token also scores against the other tokens, but never
        # as high as that token's own planted row
        assert abs(maxima.cpu()[token].item() - expected_value[token]) <= TOLERANCE * abs(expected_value[token])


# ---------------------------- dual RMS normalisation and the prequantized handoff

def norm_weight(values, encoding, device):
    """A [1, width] norm weight as a packed-weight descriptor (F32 or BF16 row)."""
    values = np.ascontiguousarray(values, dtype=np.float32)
    if encoding == kquant.BF16:
        values = (values.view(np.uint32) & 0xffff0000).view(np.float32)  # exactly representable
        raw = (values.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8)
    else:
        raw = values.view(np.uint8)
    return values, tile_ops.PackedWeight(encoding, 1, values.size, to_device(raw.copy(), device))


def probe_rms_input(rows, width):
    index = np.arange(rows * width)
    return (((index % 37) - 18) / 11.0).astype(np.float32).reshape(rows, width)  # probe :222-225


@pytest.mark.parametrize("weights", ["none", "f32", "bf16_centered"])
def test_dual_rms_add_capture_against_oracle(cuda, oracle, weights):
    rows, width = 3, 6656
    x = probe_rms_input(rows, width)
    residual = np.random.default_rng(31).standard_normal((rows, width)).astype(np.float32)
    first = second = None
    first_values = second_values = None
    centered = weights == "bf16_centered"
    if weights != "none":
        encoding = kquant.F32 if weights == "f32" else kquant.BF16
        rng = np.random.default_rng(32)
        first_values, first = norm_weight(rng.standard_normal(width) * 0.2, encoding, cuda)
        second_values, second = norm_weight(rng.standard_normal(width) * 0.2 + 1.0, encoding, cuda)
    hidden, normalized, captured = tile_ops.dual_rms_add_capture(
        to_device(x, cuda), to_device(residual, cuda), first, centered, second, False, 1e-8, 1e-5)
    expected_hidden, expected_normalized = oracle.dual_rms_add_capture(
        x, residual, first_values, centered, second_values, False, 1e-8, 1e-5)
    assert_bits_equal(hidden, expected_hidden, "hidden")
    assert_bits_equal(normalized, expected_normalized, "normalized")
    assert_bits_equal(captured, hidden, "residual capture")
    # the CPU engine's double form, at the reference probe's tolerance (:243-256)
    for row in range(rows):
        reference_hidden = oracle.rms_norm(x[row], first_values, centered, 1e-8) + residual[row]
        assert np.max(np.abs(hidden.cpu().numpy()[row] - reference_hidden)) <= 2e-5
        reference_normalized = oracle.rms_norm(reference_hidden, second_values, False, 1e-5)
        assert np.max(np.abs(normalized.cpu().numpy()[row] - reference_normalized)) <= 2e-5


@pytest.mark.parametrize("width", [6656, 12288 + 32])
@pytest.mark.parametrize("weights", ["none", "f32_centered", "bf16"])
def test_rms_norm_family_against_oracle(cuda, oracle, weights, width):
    # the single normalisation and its fused forms (probe :243-330): plain, with the
    # input kept as the residual, with the Q8_1 form of the output, with a residual added
    rows = 3
    rng = np.random.default_rng(35)
    x = probe_rms_input(rows, width) if width == 6656 else \
        rng.standard_normal((rows, width)).astype(np.float32)
    residual = rng.standard_normal((rows, width)).astype(np.float32)
    values = weight = None
    centered = weights == "f32_centered"
    if weights != "none":
        encoding = kquant.F32 if centered else kquant.BF16
        values, weight = norm_weight(rng.standard_normal(width) * 0.3, encoding, cuda)
    device_x = to_device(x, cuda)
    expected = oracle.rms_norm_strict(x, values, centered, 1e-6)
    plain = tile_ops.rms_norm(device_x, weight, centered, 1e-6)
    assert_bits_equal(plain["output"], expected, "plain")
    for row in range(rows):  # the CPU engine's double form at the probe's tolerance
        assert np.max(np.abs(expected[row] - oracle.rms_norm(x[row], values, centered, 1e-6))) <= 2e-5
    captured = tile_ops.rms_norm(device_x, weight, centered, 1e-6, capture=True)
    assert_bits_equal(captured["output"], expected, "capture output")
    assert_bits_equal(captured["captured"], x, "captured residual")
    added = tile_ops.rms_norm(device_x, weight, centered, 1e-6, residual=to_device(residual, cuda))
    assert_bits_equal(added["output"], oracle.rms_norm_strict(x, values, centered, 1e-6, residual),
                      "add residual")
    fused = tile_ops.rms_norm(device_x, weight, centered, 1e-6, q8=True)
    assert_bits_equal(fused["output"], expected, "q8 output")
    assert_bits_equal(fused["captured"], x, "q8 captured residual")
    codes, scales, sums = tile_ops.quantize_q8_1(plain["output"])
    assert torch_().equal(fused["codes"], codes)
    assert_bits_equal(fused["scales"], scales.reshape(rows, -1), "q8 scales")
    assert_bits_equal(fused["sums"], sums.reshape(rows, -1), "q8 sums")


def test_cooperative_dual_rms_equals_the_ordinary_entry_point(cuda):
    rows, width = 4, 6656
    x = to_device(probe_rms_input(rows, width), cuda)
    residual = to_device(np.random.default_rng(36).standard_normal((rows, width)).astype(np.float32),
                         cuda)
    _, first = norm_weight(np.random.default_rng(37).standard_normal(width), kquant.F32, cuda)
    _, half = norm_weight(np.random.default_rng(38).standard_normal(width), kquant.BF16, cuda)
    ordinary = tile_ops.dual_rms_add_capture(x, residual, first, True, None, False, 1e-8, 1e-5)
    outputs = [torch_().empty_like(x) for _ in range(3)]
    stream = tile_ops._stream_handle()
    cooperative = tile_ops.load().nfn_native_tile_glimmer_dual_rms_add_capture_cooperative_batch_float32_v1
    descriptor = first.descriptor(stream)
    assert cooperative(x.data_ptr(), ctypes.byref(descriptor), residual.data_ptr(),
                       outputs[0].data_ptr(), None, outputs[1].data_ptr(), outputs[2].data_ptr(),
                       rows, width, 1e-8, True, 1e-5, False, stream) == 0
    for a, b in zip(ordinary, outputs):
        assert_bits_equal(a, b)
    bf16 = half.descriptor(stream)
    assert cooperative(x.data_ptr(), ctypes.byref(bf16), residual.data_ptr(), outputs[0].data_ptr(),
                       None, outputs[1].data_ptr(), outputs[2].data_ptr(), rows, width, 1e-8, True,
                       1e-5, False, stream) == 1  # F32 norm weights only


def test_dual_rms_add_capture_wide_rows(cuda, oracle):
    # wider than the register-resident kernel takes: the kernel that walks memory in batches
    rows, width = 2, 12288 + 32
    rng = np.random.default_rng(34)
    x = rng.standard_normal((rows, width)).astype(np.float32)
    residual = rng.standard_normal((rows, width)).astype(np.float32)
    first_values, first = norm_weight(rng.standard_normal(width) * 0.3, kquant.F32, cuda)
    hidden, normalized, captured = tile_ops.dual_rms_add_capture(
        to_device(x, cuda), to_device(residual, cuda), first, True, None, False, 1e-6, 1e-6)
    expected_hidden, expected_normalized = oracle.dual_rms_add_capture(
        x, residual, first_values, True, None, False, 1e-6, 1e-6)
    assert_bits_equal(hidden, expected_hidden, "hidden")
    assert_bits_equal(normalized, expected_normalized, "normalized")
    assert_bits_equal(captured, hidden, "residual capture")


def test_dual_rms_handoff_equals_ordinary_path(cuda, oracle):
    # probe :1694-1762: the handoff's three outputs and the projection fed from
    # its records equal the ordinary dual RMS followed by the ordinary one-row call.
    width = 6656
    x = probe_rms_input(1, width)
    residual = np.random.default_rng(33).standard_normal((1, width)).astype(np.float32)
    specs = [(kquant.Q4_K, 129), (kquant.Q5_K, 33), (kquant.Q6_K, 70), (kquant.Q8_0, 17)]
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, width, 40 + i), n, width)
               for i, (e, n) in enumerate(specs)]
    workspace = tile_ops.small_batch_workspace(1, width)
    ordinary = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda),
                                             first_eps=1e-8, second_eps=1e-5)
    ordinary_out = tile_ops.multi_linear(weights, ordinary[1], workspace)
    workspace.zero_()
    handoff = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda),
                                            first_eps=1e-8, second_eps=1e-5,
                                            handoff_workspace=workspace)
    handoff_out = tile_ops.multi_linear_prequantized(weights, 1, workspace)
    for a, b, label in zip(ordinary, handoff, ("hidden", "normalized", "capture")):
        assert_bits_equal(a, b, label)
    for a, b, (encoding, _) in zip(ordinary_out, handoff_out, specs):
        assert_bits_equal(a, b, kquant.NAMES[encoding])
    # and the values are right, not just equal
    normalized = ordinary[1].cpu().numpy()
    for (encoding, out_dim), weight, y in zip(specs, weights, ordinary_out):
        exact = oracle.linear(encoding, weight.data.cpu().numpy(), out_dim, width, normalized)
        assert normalised_error(y.cpu().numpy(), exact) <= TOLERANCE


@pytest.mark.parametrize("rows", [1, 5, 16])
def test_prequantized_reuses_the_records_of_a_verifier_call(cuda, rows):
    # The engine's verifier quantizes once for Q and feeds K, V and the gate from the
    # same workspace (resident_glimmer_cuda.cpp:3649-3666).
    in_dim = 1024
    x = to_device(kquant.synthetic_activations(51, rows, in_dim), cuda)
    specs = [(kquant.Q4_K, 64), (kquant.Q6_K, 40), (kquant.Q5_K, 24), (kquant.Q8_0, 48)]
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, in_dim, 60 + i), n, in_dim)
               for i, (e, n) in enumerate(specs)]
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    direct = tile_ops.multi_linear(weights[1:], x, workspace, family="mmvq")
    workspace.zero_()
    tile_ops.multi_linear(weights[:1], x, workspace, family="mmvq")
    reused = tile_ops.multi_linear_prequantized(weights[1:], rows, workspace)
    for a, b, (encoding, _) in zip(direct, reused, specs[1:]):
        assert_bits_equal(a, b, kquant.NAMES[encoding])


@pytest.mark.parametrize("rows,width", [(5, 6656), (16, 6656), (9, 256), (16, 8192)])
def test_dual_rms_block_handoff_equals_ordinary_path(cuda, oracle, rows, width):
    """The 5..16-row form of the handoff: the norm kernel leaves the fp16 rows that the
    small-batch call would have converted its input to, and the projections fed from them
    equal the ordinary dual RMS followed by the ordinary call, bit for bit; rows several
    orders of magnitude apart keep their own scales."""
    rng = np.random.default_rng(70 + rows)
    x = probe_rms_input(rows, width) * (10.0 ** rng.integers(-3, 4, (rows, 1))).astype(np.float32)
    residual = (rng.standard_normal((rows, width)) *
                10.0 ** rng.integers(-2, 3, (rows, 1))).astype(np.float32)
    scale = tile_ops.PackedWeight.from_numpy(
        kquant.F32, kquant.quantize(kquant.F32, rng.uniform(0.5, 1.5, (1, width)).astype(np.float32)),
        1, width)
    specs = [(kquant.Q4_K, 129), (kquant.Q5_K, 33), (kquant.Q6_K, 70), (kquant.Q8_0, 17)]
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, width, 40 + i), n, width)
               for i, (e, n) in enumerate(specs)]
    workspace = tile_ops.small_batch_workspace(rows, width)
    arguments = dict(first_weight=scale, second_weight=scale, first_eps=1e-8, second_eps=1e-5)
    ordinary = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda), **arguments)
    ordinary_out = tile_ops.multi_linear(weights, ordinary[1], workspace)
    workspace.zero_()
    handoff = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda),
                                            handoff_workspace=workspace, **arguments)
    handoff_out = tile_ops.multi_linear_prequantized(weights, rows, workspace, family="mmq")
    again = tile_ops.multi_linear_prequantized(weights[1:3], rows, workspace, family="mmq")
    for a, b, label in zip(ordinary, handoff, ("hidden", "normalized", "capture")):
        assert_bits_equal(a, b, label)
    for a, b, (encoding, _) in zip(ordinary_out, handoff_out, specs):
        assert_bits_equal(a, b, kquant.NAMES[encoding])
    for a, b in zip(ordinary_out[1:3], again):
        assert_bits_equal(a, b, "a second consumer of the same rows")
    normalized = ordinary[1].cpu().numpy()
    for (encoding, out_dim), weight, y in zip(specs, weights, ordinary_out):
        exact = oracle.linear(encoding, weight.data.cpu().numpy(), out_dim, width, normalized)
        for row in range(rows):
            assert normalised_error(y.cpu().numpy()[row], exact[row]) <= TOLERANCE


@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K])
@pytest.mark.parametrize("width", [256, 4096, 6656, 8192])
@pytest.mark.parametrize("weights", ["none", "f32", "bf16_centered"])
def test_dual_rms_inside_the_projection_launch_equals_the_two_calls(cuda, oracle, encoding, width, weights):
    """nfn_mi355_dual_rms_mmvq_multi_linear_float32_v1: the three rows of the norm kernel and
    the projections of the normalized row, bit for bit what the dual RMS call followed by the
    grouped one-row call gives."""
    rng = np.random.default_rng(width + encoding)
    x = (rng.standard_normal((1, width)) * 3.0).astype(np.float32)
    residual = rng.standard_normal((1, width)).astype(np.float32)
    first = second = None
    centered = weights == "bf16_centered"
    if weights != "none":
        kind = kquant.F32 if weights == "f32" else kquant.BF16
        make = lambda seed: tile_ops.PackedWeight.from_numpy(
            kind, kquant.quantize(kind, np.random.default_rng(seed).uniform(-0.3, 0.3, (1, width)).astype(np.float32)
                                  + (0.0 if centered else 1.0)), 1, width)
        first, second = make(1), make(2)
    specs = [129, 33, 70, 300] if width <= 4096 else [4096, 256, 256, 4096]
    projections = [tile_ops.PackedWeight.from_numpy(encoding, random_packed(encoding, n, width, 50 + i), n, width)
                   for i, n in enumerate(specs)]
    workspace = tile_ops.small_batch_workspace(1, width)
    arguments = dict(first_weight=first, first_centered=centered, second_weight=second,
                     second_centered=centered, first_eps=1e-8, second_eps=1e-5)
    ordinary = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda), **arguments)
    ordinary_out = tile_ops.multi_linear(projections, ordinary[1], workspace)
    fused = tile_ops.dual_rms_multi_linear(to_device(x, cuda), to_device(residual, cuda), projections,
                                           **arguments)
    for a, b, label in zip(ordinary, fused[:3], ("hidden", "normalized", "capture")):
        assert_bits_equal(a, b, label)
    for a, b, n in zip(ordinary_out, fused[3], specs):
        assert_bits_equal(a, b, f"projection of {n} rows")


@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q5_K])
@pytest.mark.parametrize("width,outputs", [(256, 30001), (4096, 20000), (8192, 12803)])
def test_dual_rms_inside_a_projection_launch_of_many_rows(cuda, encoding, width, outputs):
    """One normalising workgroup a compute unit, however many rows it then has: the bits of the two calls."""
    packed = torch_().from_numpy(random_packed(encoding, 64, width, 55).reshape(64, -1)).to(cuda)
    chosen = torch_().from_numpy(np.random.default_rng(56).integers(0, 64, outputs)).to(cuda)
    weights = [tile_ops.PackedWeight(encoding, n, width, packed.index_select(0, chosen[:n]).reshape(-1)) for n in (outputs, 33)]
    x, residual = (to_device(kquant.synthetic_activations(seed, 1, width), cuda) for seed in (57, 58))
    ordinary = tile_ops.dual_rms_add_capture(x, residual)
    fused = tile_ops.dual_rms_multi_linear(x, residual, weights)
    for a, b in zip((*ordinary, *tile_ops.multi_linear(weights, ordinary[1], tile_ops.small_batch_workspace(1, width))),
                    (*fused[:3], *fused[3])):
        assert_bits_equal(a, b, f"{outputs} rows")


def test_dual_rms_inside_the_projection_launch_fails_closed(cuda):
    lib = tile_ops.load()
    width = 512
    x = to_device(probe_rms_input(1, width), cuda)
    rows = [torch_().empty_like(x) for _ in range(3)]
    make = lambda e, n, k, seed: tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, k, seed), n, k)
    good, five, six = make(kquant.Q4_K, 24, width, 1), make(kquant.Q5_K, 24, width, 2), make(kquant.Q6_K, 24, width, 3)
    out = [torch_().empty((1, 24), dtype=torch_().float32, device=cuda) for _ in range(2)]
    call = lib.nfn_mi355_dual_rms_mmvq_multi_linear_float32_v1
    head = [x.data_ptr(), None, x.data_ptr(), rows[0].data_ptr(), None, rows[1].data_ptr(), rows[2].data_ptr()]
    tail = [1e-8, False, 1e-5, False]
    def run(weights, width_argument=width, count=None, head_arguments=head, tail_arguments=tail):
        descriptors = tile_ops._descriptor_array([w.descriptor(0) for w in weights])
        pointers = tile_ops._pointer_array(out[:len(weights)])
        return call(*head_arguments, width_argument, *tail_arguments, descriptors, pointers,
                    len(weights) if count is None else count, None)
    assert run([good, good]) == 0
    assert run([good, five]) == 1          # two encodings: two launches, not this call
    assert run([six]) == 1                 # no dot kernel of this form
    assert run([good], count=0) == 1
    assert run([good], width_argument=256) == 1   # the projections' input width differs
    assert run([good], tail_arguments=[0.0, False, 1e-5, False]) == 1
    assert run([good], head_arguments=[None] + head[1:]) == 1
    # Every workgroup reads the two input rows while the first one stores the three result
    # rows: in-place calls (the engine's residual_output == residual_input) are refused, as are
    # results or projection outputs laid over a row that is read.
    residual_in = to_device(probe_rms_input(1, width), cuda)
    in_place = [x.data_ptr(), None, residual_in.data_ptr(), rows[0].data_ptr(), None,
                rows[1].data_ptr(), residual_in.data_ptr()]
    assert run([good], head_arguments=in_place) == 1
    over_input = [x.data_ptr(), None, residual_in.data_ptr(), x.data_ptr(), None,
                  rows[1].data_ptr(), rows[2].data_ptr()]
    assert run([good], head_arguments=over_input) == 1
    partly = [x.data_ptr(), None, residual_in.data_ptr(), rows[0].data_ptr(), None,
              x.data_ptr() + 4 * (width - 1), rows[2].data_ptr()]
    assert run([good], head_arguments=partly) == 1
    kept = out[0]
    out[0] = residual_in[:, :24]  # a projection's output over the residual row
    assert run([good]) == 0  # (x is both inputs here: not touched)
    assert run([good], head_arguments=[x.data_ptr(), None, residual_in.data_ptr()] + head[3:]) == 1
    out[0] = kept
    wide = make(kquant.Q4_K, 8, 8448, 4)
    wide_x = to_device(probe_rms_input(1, 8448), cuda)
    wide_rows = [torch_().empty_like(wide_x) for _ in range(3)]
    wide_head = [wide_x.data_ptr(), None, wide_x.data_ptr(), wide_rows[0].data_ptr(), None,
                 wide_rows[1].data_ptr(), wide_rows[2].data_ptr()]
    assert run([wide], width_argument=8448, head_arguments=wide_head) == 1
    torch_().cuda.synchronize()


@pytest.mark.parametrize("rows,width", [(4, 256), (5, 6656), (9, 2304), (16, 6656), (16, 8192)])
def test_dual_rms_block_handoff_of_the_exact_family_equals_ordinary_path(cuda, rows, width):
    """nfn_mi355_dual_rms_add_capture_mmvq_rows_float32_v1: the norm kernel leaves the rows'
    activation records and their matrix-operand copy, and the reference's prequantized consumer
    fed from them gives the bits of the dual RMS followed by the verifier call (and so of the
    one-row call on every row); rows several orders of magnitude apart keep their own scales."""
    rng = np.random.default_rng(170 + rows)
    x = probe_rms_input(rows, width) * (10.0 ** rng.integers(-3, 4, (rows, 1))).astype(np.float32)
    residual = (rng.standard_normal((rows, width)) *
                10.0 ** rng.integers(-2, 3, (rows, 1))).astype(np.float32)
    scale = tile_ops.PackedWeight.from_numpy(
        kquant.F32, kquant.quantize(kquant.F32, rng.uniform(0.5, 1.5, (1, width)).astype(np.float32)),
        1, width)
    specs = [(kquant.Q4_K, 129), (kquant.Q5_K, 33), (kquant.Q6_K, 70), (kquant.Q8_0, 17)]
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, width, 140 + i), n, width)
               for i, (e, n) in enumerate(specs)]
    workspace = tile_ops.small_batch_workspace(rows, width)
    arguments = dict(first_weight=scale, second_weight=scale, first_eps=1e-8, second_eps=1e-5)
    ordinary = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda), **arguments)
    ordinary_out = tile_ops.multi_linear(weights, ordinary[1], workspace, family="mmvq")
    workspace.zero_()
    handoff = tile_ops.dual_rms_add_capture(to_device(x, cuda), to_device(residual, cuda),
                                            handoff_workspace=workspace, handoff_family="mmvq",
                                            **arguments)
    handoff_out = tile_ops.multi_linear_prequantized(weights, rows, workspace, family="mmvq")
    again = tile_ops.multi_linear_prequantized(weights[1:3], rows, workspace, family="mmvq")
    for a, b, label in zip(ordinary, handoff, ("hidden", "normalized", "capture")):
        assert_bits_equal(a, b, label)
    for a, b, (encoding, _) in zip(ordinary_out, handoff_out, specs):
        assert_bits_equal(a, b, kquant.NAMES[encoding])
    for a, b in zip(ordinary_out[1:3], again):
        assert_bits_equal(a, b, "a second consumer of the same rows")
    one = tile_ops.small_batch_workspace(1, width)
    alone = tile_ops.multi_linear(weights, ordinary[1][rows - 1:rows].contiguous(), one, family="mmvq")
    for a, b in zip(handoff_out, alone):
        assert_bits_equal(a[rows - 1:rows].contiguous(), b, "the one-row call on the last row")


def test_block_handoff_of_the_exact_family_fails_closed(cuda):
    width = 512
    lib = tile_ops.load()
    x = to_device(probe_rms_input(16, width), cuda)
    outputs = [torch_().empty_like(x) for _ in range(3)]
    workspace = tile_ops.small_batch_workspace(16, width)
    head = [x.data_ptr(), None, x.data_ptr(), outputs[0].data_ptr(), None, outputs[1].data_ptr(),
            outputs[2].data_ptr()]
    tail = [1e-8, False, 1e-5, False]
    handoff = lib.nfn_mi355_dual_rms_add_capture_mmvq_rows_float32_v1
    required = lib.nfn_native_tile_k_quant_mmq_workspace_bytes_v1(8, width)
    assert handoff(*head, 8, width, *tail, workspace.data_ptr(), required, None) == 0
    assert handoff(*head, 4, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 0
    assert handoff(*head, 3, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 17, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 8, width, *tail, workspace.data_ptr(), required - 1, None) == 1
    assert handoff(*head, 8, width, *tail, None, required, None) == 1
    assert handoff(*head, 8, 384, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 8, 8448, *tail, workspace.data_ptr(), 1 << 30, None) == 1
    assert handoff(*head, 8, width, 0.0, False, 1e-5, False, workspace.data_ptr(), required, None) == 1
    torch_().cuda.synchronize()


def test_block_handoff_fails_closed(cuda):
    width = 512
    lib = tile_ops.load()
    x = to_device(probe_rms_input(16, width), cuda)
    outputs = [torch_().empty_like(x) for _ in range(3)]
    workspace = tile_ops.small_batch_workspace(16, width)
    head = [x.data_ptr(), None, x.data_ptr(), outputs[0].data_ptr(), None, outputs[1].data_ptr(),
            outputs[2].data_ptr()]
    tail = [1e-8, False, 1e-5, False]
    handoff = lib.nfn_mi355_dual_rms_add_capture_mmq_f16_float32_v1
    required = lib.nfn_native_tile_k_quant_mmq_workspace_bytes_v1(8, width)
    assert handoff(*head, 8, width, *tail, workspace.data_ptr(), required, None) == 0
    assert handoff(*head, 4, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 17, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 8, width, *tail, workspace.data_ptr(), required - 1, None) == 1
    assert handoff(*head, 8, width, *tail, None, required, None) == 1
    assert handoff(*head, 8, 384, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 8, 8448, *tail, workspace.data_ptr(), 1 << 30, None) == 1
    assert handoff(*head, 8, width, 0.0, False, 1e-5, False, workspace.data_ptr(), required, None) == 1
    torch_().cuda.synchronize()
    out = torch_().empty((16, 8), dtype=torch_().float32, device=cuda)
    packed = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, 8, width, 1),
                                              8, width)
    plain = tile_ops.PackedWeight.from_numpy(
        kquant.F32, kquant.quantize(kquant.F32, kquant.synthetic_weights(2, 8, width, 1.0)), 8, width)
    prequantized = lib.nfn_mi355_k_quant_mmq_multi_linear_prequantized_float32_v1
    pointers = tile_ops._pointer_array([out])
    good = tile_ops._descriptor_array([packed.descriptor(0)])
    assert prequantized(good, pointers, 1, 8, workspace.data_ptr(), required, None) == 0
    assert prequantized(good, pointers, 1, 4, workspace.data_ptr(), workspace.numel(), None) == 1
    assert prequantized(good, pointers, 1, 17, workspace.data_ptr(), workspace.numel(), None) == 1
    assert prequantized(good, pointers, 1, 8, workspace.data_ptr(), required - 1, None) == 1
    assert prequantized(good, pointers, 0, 8, workspace.data_ptr(), required, None) == 1
    assert prequantized(good, pointers, 1, 8, None, required, None) == 1
    # a projection that the fp16 kernel does not take has no use for the rows in the workspace
    other = tile_ops._descriptor_array([plain.descriptor(0)])
    assert prequantized(other, pointers, 1, 8, workspace.data_ptr(), required, None) == 1
    torch_().cuda.synchronize()


def test_handoff_and_prequantized_fail_closed(cuda):
    width = 512
    lib = tile_ops.load()
    x = to_device(probe_rms_input(2, width), cuda)
    outputs = [torch_().empty_like(x) for _ in range(3)]
    workspace = tile_ops.small_batch_workspace(2, width)
    head = [x.data_ptr(), None, x.data_ptr(), outputs[0].data_ptr(), None, outputs[1].data_ptr(),
            outputs[2].data_ptr()]
    tail = [1e-8, False, 1e-5, False]
    handoff = lib.nfn_native_tile_glimmer_dual_rms_add_capture_mmvq_q8_float32_v1
    required = lib.nfn_native_tile_k_quant_mmq_workspace_bytes_v1(1, width)
    assert handoff(*head, 1, width, *tail, workspace.data_ptr(), required, None) == 0
    assert handoff(*head, 2, width, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    assert handoff(*head, 1, width, *tail, workspace.data_ptr(), required - 1, None) == 1
    assert handoff(*head, 1, width, *tail, None, required, None) == 1
    assert handoff(*head, 1, 480, *tail, workspace.data_ptr(), workspace.numel(), None) == 1
    plain = lib.nfn_native_tile_glimmer_dual_rms_add_capture_float32_v1
    assert plain(*head, 2, width, *tail, None) == 0
    assert plain(*head, 2, width, 0.0, False, 1e-5, False, None) == 1
    assert plain(*head, 2, 65537, *tail, None) == 1
    assert plain(*head, 0, width, *tail, None) == 1
    torch_().cuda.synchronize()
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, random_packed(kquant.Q4_K, 8, width, 1),
                                              8, width)
    out = torch_().empty((16, 8), dtype=torch_().float32, device=cuda)
    prequantized = lib.nfn_native_tile_k_quant_mmvq_multi_linear_prequantized_float32_v1
    descriptor = weight.descriptor(0)
    descriptors = tile_ops._descriptor_array([descriptor])
    pointers = tile_ops._pointer_array([out])
    big = tile_ops.small_batch_workspace(16, width)
    assert prequantized(descriptors, pointers, 1, 17, big.data_ptr(), big.numel(), None) == 1
    assert prequantized(descriptors, pointers, 1, 2, big.data_ptr(), required, None) == 1
    assert prequantized(descriptors, pointers, 0, 1, big.data_ptr(), big.numel(), None) == 1
    assert prequantized(descriptors, pointers, 1, 1, None, big.numel(), None) == 1


# ------------------------------------------------ the benchmark's geometries

def config_layer(seed, encoding=kquant.Q4_K):
    shapes = {"q": (4096, 6656), "k": (256, 6656), "v": (256, 6656), "o": (6656, 4096)}
    return {name: (shape, kquant.quantize(encoding, kquant.synthetic_weights(seed + i, *shape)))
            for i, (name, shape) in enumerate(shapes.items())}


@pytest.mark.parametrize("rows", [1, 4, 8])
def test_config1_attention_projections(cuda, oracle, rows):
    layer = config_layer(1000)
    x = kquant.synthetic_activations(2000 + rows, rows, 6656)
    attn = kquant.synthetic_activations(3000 + rows, rows, 4096)
    weights = {n: tile_ops.PackedWeight.from_numpy(kquant.Q4_K, p, *s) for n, (s, p) in layer.items()}
    workspace = tile_ops.small_batch_workspace(16, 6656)
    q, k, v = tile_ops.multi_linear([weights["q"], weights["k"], weights["v"]],
                                    to_device(x, cuda), workspace)
    (o,) = tile_ops.multi_linear([weights["o"]], to_device(attn, cuda), workspace)
    for name, y, source in (("q", q, x), ("k", k, x), ("v", v, x), ("o", o, attn)):
        (out_dim, in_dim), packed = layer[name]
        expected = oracle.linear(kquant.Q4_K, packed, out_dim, in_dim, source)
        assert normalised_error(y.cpu().numpy(), expected) <= TOLERANCE, name
    if rows == 1:  # config 0 is the Q projection at M=1 through the decode GEMV
        direct = tile_ops.mmvq_linear(weights["q"], to_device(x, cuda), workspace)
        assert_bits_equal(direct, q, "config 0")


def test_config4_mixed_formats_dispatch(cuda, oracle):
    # per-tensor formats drawn by seed, V/O/down at least Q5_K; decode (M=1)
    rng = np.random.default_rng(4)
    low = [kquant.Q4_K, kquant.Q5_K, kquant.Q6_K, kquant.Q8_0]
    high = [kquant.Q5_K, kquant.Q6_K, kquant.Q8_0]
    in_dim = 1024
    names = {"q": (512, low), "k": (256, low), "v": (256, high), "gate": (768, low)}
    x = kquant.synthetic_activations(41, 1, in_dim)
    weights, packed_all = [], []
    for index, (name, (out_dim, choices)) in enumerate(names.items()):
        encoding = int(rng.choice(choices))
        packed = kquant.quantize(encoding, kquant.synthetic_weights(400 + index, out_dim, in_dim))
        packed_all.append((encoding, out_dim, packed))
        weights.append(tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim))
    workspace = tile_ops.small_batch_workspace(1, in_dim)
    outputs = tile_ops.multi_linear(weights, to_device(x, cuda), workspace)
    for (encoding, out_dim, packed), y in zip(packed_all, outputs):
        expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
        assert normalised_error(y.cpu().numpy(), expected) <= TOLERANCE


@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_against_oracle(cuda, oracle, encoding):
    # 160 rows: one full and one ragged 256-row tile is not covered here but by
    # the ragged test below; 384 columns = three 128-column tiles
    rows, out_dim, in_dim = 160, 384, 1024
    packed = kquant.quantize(encoding, kquant.synthetic_weights(70 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(71, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= TOLERANCE


@pytest.mark.parametrize("in_dim", [256, 768])
@pytest.mark.parametrize("encoding", K_ENCODINGS)
def test_prefill_gemm_ragged_tiles_and_odd_block_count(cuda, oracle, encoding, in_dim):
    # 300 rows (full tiles and a ragged one), 200 columns (ragged), K of one or
    # three blocks (odd: the kernel's two-block loop runs its first block ahead)
    rows, out_dim = 300, 200
    packed = random_packed(encoding, out_dim, in_dim, 41)
    x = kquant.synthetic_activations(72, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= TOLERANCE


@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_tall_tiles(cuda, oracle, encoding):
    # 512 rows x 16384 columns = 2 x 128 tiles: enough workgroups for the
    # 256-row tile variant (smaller problems run the 128-row one); K of two
    # blocks (even count).  The oracle checks a spread of rows.
    rows, out_dim, in_dim = 512, 16384, 512
    assert tile_ops.gemm_tile_rows(encoding, rows, in_dim, [out_dim]) == 256
    packed = random_packed(encoding, out_dim, in_dim, 43)
    x = kquant.synthetic_activations(74, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    picked = np.array([0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 300, 383, 384, 447, 448, 511])
    expected = oracle.linear(encoding, packed, out_dim, in_dim, np.ascontiguousarray(x[picked]))
    assert normalised_error(y[picked], expected) <= TOLERANCE


@pytest.mark.parametrize("rows,tiles,in_dim", [(1624, 0.25, 256), (1000, 0.5, 512), (1712, 0.25, 768), (1537, 0.25, 1280)])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_eight_waves_a_tile(cuda, oracle, encoding, rows, tiles, in_dim):
    """Tiles of 512 rows, one on every compute unit: a last tile of 88, 488, 176 and one row (waves
    past the rows that the fp16 copy is padded to), a last column tile of 125, one to five blocks of
    K.  The oracle checks rows at the edges of waves and tiles."""
    units = torch_().cuda.get_device_properties(0).multi_processor_count
    out_dim = int(tiles * units) * 128 - 3
    assert tile_ops.gemm_tile_rows(encoding, rows, in_dim, [out_dim]) == 512
    packed = random_packed(encoding, 256, in_dim, 46).reshape(256, -1)
    chosen = np.random.default_rng(47).integers(0, 256, out_dim)
    weight = tile_ops.PackedWeight(encoding, out_dim, in_dim, torch_().from_numpy(packed).to(cuda).index_select(
        0, torch_().from_numpy(chosen).to(cuda)).reshape(-1))
    x = kquant.synthetic_activations(76, rows, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda)).cpu().numpy()
    picked = np.array(sorted({r for edge in range(0, rows + 1, 64) for r in (edge - 1, edge, edge + 31, edge + 32)
                              if 0 <= r < rows} | {rows - 1}))
    expected = oracle.linear(encoding, packed.reshape(-1), 256, in_dim, np.ascontiguousarray(x[picked]))[:, chosen]
    for row, want in zip(picked, expected):
        assert normalised_error(y[row], want) <= TOLERANCE, row


def test_prefill_gemm_plans():
    # Host logic only.  A problem of many tiles but not one per compute unit: shares of at
    # least twelve 256-value blocks, 256-row tiles while two shares or more fit.
    wide = 33 * 128
    assert tile_ops.gemm_plan(kquant.Q4_K, 96, 4096, wide) == (128, 1)    # sixteen blocks: one share
    assert tile_ops.gemm_plan(kquant.Q4_K, 96, 6144, wide) == (128, 2)
    assert tile_ops.gemm_plan(kquant.Q4_K, 96, 9216, wide) == (128, 3)
    assert tile_ops.gemm_plan(kquant.Q4_K, 200, 9216, wide) == (256, 3)
    assert tile_ops.gemm_plan(kquant.Q4_K, 200, 12544, wide) == (256, 4)
    assert tile_ops.gemm_plan(kquant.Q4_K, 2048, 6656, 16384) == (256, 1)
    # A K too short for shares: 256-row tiles from half a workgroup a unit on.
    assert tile_ops.gemm_plan(kquant.Q4_K, 512, 4096, 6656) == (128, 1)
    assert tile_ops.gemm_plan(kquant.Q4_K, 700, 4096, 6656) == (256, 1)
    # A narrow projection (the K and V projections of the workload): small tiles, short shares.
    assert tile_ops.gemm_plan(kquant.Q4_K, 1024, 6656, 256) == (128, 4)
    assert tile_ops.gemm_plan(kquant.Q6_K, 2048, 6656, 256) == (128, 4)


def test_prefill_gemm_tile_rows(cuda):
    # Host logic only.  Low tiles where high ones would leave units idle, by the widths of the whole launch.
    for encoding in ALL_PACKED:
        assert tile_ops.gemm_tile_rows(encoding, 32, 6656, [4096]) == 32
        assert tile_ops.gemm_tile_rows(encoding, 128, 6656, [4096]) == 128
        assert tile_ops.gemm_tile_rows(encoding, 4096, 6656, [16384, 16384]) == 512
    assert tile_ops.gemm_tile_rows(kquant.Q4_K, 160, 6656, [16384, 16384]) == 256
    assert tile_ops.gemm_tile_rows(kquant.Q4_K, 160, 4096, [6656]) == 128
    call, widths, out = tile_ops.load().nfn_mi355_k_quant_gemm_tile_rows_v1, (ctypes.c_int64 * 2)(128, 0), ctypes.c_int(7)
    for encoding, count, in_dim in ((kquant.Q4_K, 2, 256), (kquant.Q4_K, 0, 256), (kquant.Q4_K, 5, 256),
                                    (kquant.Q4_K, 1, 128), (kquant.BF16, 1, 256)):
        assert call(encoding, 64, in_dim, ctypes.addressof(widths), count, tile_ops.GEMM_F16, ctypes.addressof(out)) == 1
    assert call(kquant.Q4_K, 64, 256, None, 1, tile_ops.GEMM_F16, ctypes.addressof(out)) == 1 and out.value == 7


def test_prefill_gemm_workspace_of_a_longer_chunk(cuda):
    """The workspace of a long chunk serves the short ones behind it, which split K further, and a
    call takes any workspace that holds what its own plan needs: the fp16 rows in whole 256-row
    tiles, eight bytes a row, an output per share, 256 bytes."""
    in_dim, out_dim = 6656, 16384
    query = tile_ops.load().nfn_mi355_k_quant_gemm_workspace_bytes_v1
    packed = random_packed(kquant.Q4_K, out_dim, in_dim, 5)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, packed, out_dim, in_dim)
    large = torch_().empty(query(512, in_dim, out_dim, tile_ops.GEMM_F16), dtype=torch_().uint8, device=cuda)
    for rows in (512, 256, 128, 17):
        x = to_device(kquant.synthetic_activations(rows, rows, in_dim), cuda)
        y = tile_ops.gemm(weight, x, workspace=large)
        _, shares = tile_ops.gemm_plan(kquant.Q4_K, rows, in_dim, out_dim)
        padded = (rows + 255) // 256 * 256
        needed = (padded * (in_dim * 2 + 8) + 255) // 256 * 256 + (shares * rows * out_dim * 4 if shares > 1 else 0) + 256
        assert needed <= large.numel()
        assert_bits_equal(tile_ops.gemm(weight, x, workspace=large[:needed]), y, str(rows))
        with pytest.raises(tile_ops.TileOpsError):
            tile_ops.gemm(weight, x, workspace=large[:needed - 1])


def gemm_query(rows, in_dim, *out_dims):
    lib = tile_ops.load()
    if len(out_dims) == 1:
        return lib.nfn_mi355_k_quant_gemm_workspace_bytes_v1(rows, in_dim, out_dims[0], tile_ops.GEMM_F16)
    widths = (ctypes.c_int64 * len(out_dims))(*out_dims)
    return lib.nfn_mi355_k_quant_gemm_multi_workspace_bytes_v1(rows, in_dim, ctypes.addressof(widths), len(out_dims),
                                                               tile_ops.GEMM_F16)


def gemm_weight(cuda, encoding, out_dim, in_dim, seed):
    """(weight, its 256 different rows, which of them each output has)"""
    packed = random_packed(encoding, 256, in_dim, seed)
    chosen = np.random.default_rng(seed + 2).integers(0, 256, out_dim)
    device_rows = torch_().from_numpy(packed.reshape(256, -1)).to(cuda)
    return tile_ops.PackedWeight(encoding, out_dim, in_dim, device_rows.index_select(
        0, torch_().from_numpy(chosen).to(cuda)).reshape(-1)), packed, chosen


@pytest.mark.parametrize("rows,in_dim,out_dim,taken", [(33, 4096, 5373, 4), (128, 2304, 2049, 4), (35, 11776, 5376, 6),
                                                       (36, 1536, 2073, 3), (33, 11520, 2080, 8)])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_cut_beyond_the_plan(cuda, oracle, encoding, rows, in_dim, out_dim, taken):
    """Few tiles and a K that the plan leaves whole or in long shares: with the workspace of the query the
    call cuts further (three to eight shares, some of unequal lengths, a last column tile of one), with the
    plan's it does not; both keep the bound, and a projection beside another the single call's bits."""
    _, shares = tile_ops.gemm_plan(encoding, rows, in_dim, out_dim)
    least = (256 * (in_dim * 2 + 8) + 255) // 256 * 256 + (shares * rows * out_dim * 4 if shares > 1 else 0) + 256
    asked = gemm_query(rows, in_dim, out_dim)
    assert [tile_ops.gemm_launch(encoding, rows, in_dim, [out_dim], n)[0][1] for n in (asked, least)] == [taken, shares]
    assert shares < taken
    weight, packed, chosen = gemm_weight(cuda, encoding, out_dim, in_dim, 46)
    x = kquant.synthetic_activations(77, rows, in_dim)
    expected = oracle.linear(encoding, packed, 256, in_dim, x)[:, chosen]
    device_x = to_device(x, cuda)
    results = []
    for nbytes in (asked, least):
        workspace = torch_().full((nbytes + 4096,), 0x5a, dtype=torch_().uint8, device=cuda)
        results.append(tile_ops.gemm(weight, device_x, workspace=workspace[:nbytes]))
        assert normalised_error(results[-1].cpu().numpy(), expected) <= TOLERANCE
        assert bool((workspace[nbytes:] == 0x5a).all())
    assert not torch_().equal(*results), "the sums of more shares round differently"
    with pytest.raises(tile_ops.TileOpsError):
        tile_ops.gemm(weight, device_x, workspace=workspace[:least - 1])
    for y in tile_ops.gemm_multi([weight, weight], device_x):
        assert_bits_equal(y, tile_ops.gemm(weight, device_x), kquant.NAMES[encoding])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_cut_beyond_the_plan_beside_others(cuda, encoding, mixed):
    """Projections that the call cuts into three, six and four shares beside one that keeps the plan's two, of one
    encoding and of two: with the grouped query's workspace in one launch an encoding, with what the largest one
    needs in several, each time with the single calls' bits and nothing written behind the workspace."""
    rows, in_dim, out_dims = 40, 4096, (4353, 256, 2300, 5000)
    other = kquant.Q6_K if encoding != kquant.Q6_K else kquant.Q4_K
    encodings = [encoding, encoding, other if mixed else encoding, encoding]
    weights = [gemm_weight(cuda, e, n, in_dim, 49 + i)[0] for i, (e, n) in enumerate(zip(encodings, out_dims))]
    x = to_device(kquant.synthetic_activations(78, rows, in_dim), cuda)
    alone = [tile_ops.gemm(w, x) for w in weights]
    together = gemm_query(rows, in_dim, *out_dims)
    activations = (256 * (in_dim * 2 + 8) + 255) // 256 * 256
    one = activations + 5 * rows * 2300 * 4 + 256  # (the six shares of one projection, and no other beside it)
    for nbytes in (together, one):
        launched = tile_ops.gemm_launch(encoding, rows, in_dim, out_dims, nbytes)
        assert [shares for _, shares in launched] == [3, 2, 6, 4 if nbytes == together else 1]
        workspace = torch_().full((nbytes + 4096,), 0x5a, dtype=torch_().uint8, device=cuda)
        outputs = tile_ops.gemm_multi(weights, x, workspace=workspace[:nbytes])
        for i, (y, single) in enumerate(zip(outputs, alone)):
            if launched[i][1] == tile_ops.gemm_launch(encodings[i], rows, in_dim, [out_dims[i]],
                                                      gemm_query(rows, in_dim, out_dims[i]))[0][1]:
                assert_bits_equal(y, single, f"projection {i}")
            else:
                assert_bits_equal(y, tile_ops.gemm(weights[i], x, workspace=workspace[:nbytes]), f"projection {i}")
        assert bool((workspace[nbytes:] == 0x5a).all())


@pytest.mark.parametrize("rows,in_dim,out_dims", [(333, 6656, [4096, 256, 256, 4096]), (1000, 4096, [6656]), (2048, 16384, [6656]),
                                                  (1100, 11520, [2080, 4097]), (700, 1536, [16384, 130, 2073]), (40, 512, [64])])
def test_prefill_gemm_workspace_lets_every_shorter_call_take_its_shares(rows, in_dim, out_dims):
    """Host logic only.  The query looks at few row counts, the largest first, and at none that cannot need more; with
    its workspace a call of any count takes the shares and tiles that it would with all the room there is."""
    nbytes = gemm_query(rows, in_dim, *out_dims)
    for encoding in (kquant.Q4_K, kquant.Q6_K):
        for count in sorted({*range(1, rows, 23), *range(128, rows, 128), 32, 33, rows}):
            assert (tile_ops.gemm_launch(encoding, count, in_dim, out_dims, nbytes) ==
                    tile_ops.gemm_launch(encoding, count, in_dim, out_dims, 1 << 60)), count


def test_prefill_gemm_launch_says_what_runs():
    """Host logic only.  The height and the shares that the queries report are those of a call with the workspace at
    hand: 257 rows of 8,704 -> 2,999 are cut in two by the plan (tiles of 128 rows), in four with room for it (256)."""
    rows, in_dim, out_dim = 257, 8704, 2999
    plan_bytes = (512 * (in_dim * 2 + 8) + 255) // 256 * 256 + 2 * rows * out_dim * 4 + 256
    assert tile_ops.gemm_plan(kquant.Q4_K, rows, in_dim, out_dim) == (256, 2)
    assert tile_ops.gemm_tile_rows(kquant.Q4_K, rows, in_dim, [out_dim]) == 256
    assert tile_ops.gemm_launch(kquant.Q4_K, rows, in_dim, [out_dim], gemm_query(rows, in_dim, out_dim)) == [(256, 4)]
    assert tile_ops.gemm_launch(kquant.Q4_K, rows, in_dim, [out_dim], plan_bytes) == [(128, 2)]
    for rows in (17, 40, 333, 2000):
        for out_dims in ([4096], [4353, 256, 2300, 5000], [16384, 16384]):
            for encoding in ALL_PACKED:
                launched = tile_ops.gemm_launch(encoding, rows, 4096, out_dims, gemm_query(rows, 4096, *out_dims))
                assert {height for height, _ in launched} == {tile_ops.gemm_tile_rows(encoding, rows, 4096, out_dims)}
                for n, (_, shares) in zip(out_dims, launched):
                    single = tile_ops.gemm_launch(encoding, rows, 4096, [n], gemm_query(rows, 4096, n))
                    assert single[0][1] == shares >= tile_ops.gemm_plan(encoding, rows, 4096, n)[1]
    least = (256 * (4096 * 2 + 8) + 255) // 256 * 256 + 256
    assert tile_ops.gemm_launch(kquant.Q4_K, 200, 4096, [16384], least)[0][1] == 1
    for arguments in ((kquant.Q4_K, 200, 4096, [16384], least - 1), (kquant.Q4_K, 200, 4096, [], least),
                      (kquant.Q4_K, 0, 4096, [64], least), (kquant.Q4_K, 200, 4100, [64], least),
                      (kquant.BF16, 200, 4096, [64], least), (kquant.Q4_K, 200, 4096, [0], least)):
        with pytest.raises(tile_ops.TileOpsError):
            tile_ops.gemm_launch(*arguments)


@pytest.mark.parametrize("rows,in_dim,plan", [
    (96, 1536, (128, 1)),    # six blocks: one share
    (96, 3072, (128, 2)),    # twelve blocks -> two shares of six
    (96, 4608, (128, 3)),    # eighteen -> three
    (200, 6656, (128, 4)),   # 26 blocks -> four shares of unequal length (7, 7, 6, 6)
    (200, 12544, (128, 4)),  # 49 blocks -> (13, 12, 12, 12)
])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_split_k(cuda, oracle, encoding, rows, in_dim, plan):
    # few tiles and a long K: the launch splits K into shares (of at least six 256-value
    # blocks for a narrow projection, at most four) and a second launch sums them in share order
    out_dim = 130
    assert tile_ops.gemm_plan(encoding, rows, in_dim, out_dim) == plan
    packed = kquant.quantize(encoding, kquant.synthetic_weights(70 + encoding, out_dim, in_dim))
    x = kquant.synthetic_activations(71, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda)).cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    assert normalised_error(y, expected) <= TOLERANCE
    again = tile_ops.gemm(weight, to_device(x, cuda)).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))  # fixed summation order


@pytest.mark.parametrize("rows,out_dim,in_dim,plan", [
    (1, 1, 256, (32, 1)), (17, 129, 1536, (32, 2)), (32, 31, 4608, (32, 6)),   # rows of one fragment, K shares
    (20, 97, 6656, (32, 8)), (31, 128, 2560, (32, 3)),                         # shares of unequal length
    (17, 40000, 512, (32, 1)), (33, 129, 1536, (128, 1)),                      # enough tiles without shares; past the kernel's rows
])
@pytest.mark.parametrize("encoding", ALL_PACKED)
def test_prefill_gemm_few_rows(cuda, oracle, encoding, rows, out_dim, in_dim, plan):
    # up to 32 rows: the kernel that cuts the columns among a workgroup's waves
    assert tile_ops.gemm_plan(encoding, rows, in_dim, out_dim) == plan
    packed = random_packed(encoding, out_dim, in_dim, 90 + rows)
    x = kquant.synthetic_activations(91, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda)).cpu().numpy()
    assert normalised_error(y, oracle.linear(encoding, packed, out_dim, in_dim, x)) <= TOLERANCE
    again = tile_ops.gemm(weight, to_device(x, cuda)).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))  # fixed summation order


def test_prefill_gemm_multi_equals_single_calls(cuda, oracle):
    """nfn_mi355_k_quant_gemm_multi_float32_v1: one conversion of the input, the single call's bits."""
    rows, in_dim = 300, 1024
    specs = [(kquant.Q4_K, 384), (kquant.Q6_K, 130), (kquant.Q8_0, 17), (kquant.Q5_K, 256)]
    weights = [tile_ops.PackedWeight.from_numpy(
        e, kquant.quantize(e, kquant.synthetic_weights(70 + i, n, in_dim)), n, in_dim)
        for i, (e, n) in enumerate(specs)]
    x = to_device(kquant.synthetic_activations(71, rows, in_dim), cuda)
    grouped = tile_ops.gemm_multi(weights, x)
    for weight, y in zip(weights, grouped):
        assert_bits_equal(y, tile_ops.gemm(weight, x), kquant.NAMES[weight.encoding])
    lib = tile_ops.load()
    descriptors = [w.descriptor(0) for w in weights]
    outputs = [torch_().empty((rows, w.output_dim), dtype=torch_().float32, device=cuda) for w in weights]
    workspace = torch_().empty(1 << 24, dtype=torch_().uint8, device=cuda)

    def call(count=4, rows=rows, nbytes=workspace.numel(), mode=tile_ops.GEMM_F16, descs=descriptors):
        return lib.nfn_mi355_k_quant_gemm_multi_float32_v1(
            tile_ops._descriptor_array(descs), x.data_ptr(), tile_ops._pointer_array(outputs), count,
            rows, workspace.data_ptr(), nbytes, mode, None)

    assert call() == 0
    assert call(count=0) == 1 and call(count=5) == 1 and call(rows=0) == 1
    assert call(nbytes=1024) == 1 and call(mode=tile_ops.GEMM_INT8) == 1
    other = tile_ops.PackedWeight.from_numpy(
        kquant.Q4_K, kquant.quantize(kquant.Q4_K, kquant.synthetic_weights(72, 64, 512)), 64, 512)
    assert call(descs=descriptors[:3] + [other.descriptor(0)]) == 1  # another input width
    torch_().cuda.synchronize()


@pytest.mark.parametrize("rows", [17, 200, 300, 640])
@pytest.mark.parametrize("specs", [
    [(kquant.Q4_K, 4096), (kquant.Q4_K, 256), (kquant.Q4_K, 130), (kquant.Q4_K, 4000)],  # one launch
    [(kquant.Q6_K, 1000), (kquant.Q8_0, 300), (kquant.Q6_K, 17), (kquant.Q8_0, 2048)],   # two, interleaved
    [(kquant.Q5_K, 5000), (kquant.Q5_K, 129)],
])
def test_prefill_gemm_multi_launches_equal_single_calls(cuda, specs, rows):
    """Projections of one encoding in one launch, each with its own K shares: the single call's bits,
    with the workspace for one launch and with the smallest allowed (more launches); nothing is
    written behind either."""
    in_dim = 6656
    weights = [tile_ops.PackedWeight.from_numpy(e, random_packed(e, n, in_dim, 80 + i), n, in_dim)
               for i, (e, n) in enumerate(specs)]
    x = to_device(kquant.synthetic_activations(81, rows, in_dim), cuda)
    expected = [tile_ops.gemm(weight, x) for weight in weights]
    lib = tile_ops.load()
    widths = np.array([n for _, n in specs], dtype=np.int64)
    together = lib.nfn_mi355_k_quant_gemm_multi_workspace_bytes_v1(
        rows, in_dim, widths.ctypes.data, len(specs), tile_ops.GEMM_F16)
    least = max(lib.nfn_mi355_k_quant_gemm_workspace_bytes_v1(rows, in_dim, n, tile_ops.GEMM_F16) for _, n in specs)
    assert together >= least
    for nbytes in (together, least):
        workspace = torch_().full((nbytes + 4096,), 0x5a, dtype=torch_().uint8, device=cuda)
        for weight, y, single in zip(weights, tile_ops.gemm_multi(weights, x, workspace=workspace[:nbytes]), expected):
            assert_bits_equal(y, single, kquant.NAMES[weight.encoding])
        assert bool((workspace[nbytes:] == 0x5a).all())
    assert lib.nfn_mi355_k_quant_gemm_multi_workspace_bytes_v1(rows, in_dim, widths.ctypes.data, 5, tile_ops.GEMM_F16) == 0


@pytest.mark.parametrize("encoding", [kquant.Q4_K, kquant.Q6_K])
def test_fp16_rows_activation_range(cuda, oracle, encoding):
    """The fp16 small-batch kernel scales every eighth of K of a row by its own power of two:
    rows far outside the fp16 range, a zero row, a row whose eighths differ by twelve orders of
    magnitude and a row with an eighth of zeros keep the bound."""
    rows, out_dim, in_dim = 8, 96, 2048
    packed = kquant.quantize(encoding, kquant.synthetic_weights(78, out_dim, in_dim))
    x = kquant.synthetic_activations(74, rows, in_dim)
    x *= np.array([1.0, 1.0e6, 1.0e-6, 3.0e20, 2.0e-22, 0.0, 1.0, 1.0], dtype=np.float32)[:, None]
    x[6, :256] *= 1.0e6
    x[6, 1280:1536] *= 1.0e-6
    x[7, 512:768] = 0.0
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    y = tile_ops.multi_linear([weight], to_device(x, cuda), workspace)[0].cpu().numpy()
    expected = oracle.linear(encoding, packed, out_dim, in_dim, x)
    for row in range(rows):
        if row == 5:
            assert np.all(y[row] == 0.0)
        else:
            assert normalised_error(y[row:row + 1], expected[row:row + 1]) <= TOLERANCE


def test_prefill_gemm_activation_range(cuda, oracle):
    # rows scaled far outside the fp16 range, and a zero row: the per-row power
    # of two keeps every row at the same relative accuracy
    rows, out_dim, in_dim = 6, 128, 512
    packed = kquant.quantize(kquant.Q4_K, kquant.synthetic_weights(77, out_dim, in_dim))
    x = kquant.synthetic_activations(73, rows, in_dim)
    x *= np.array([1.0, 1.0e6, 1.0e-6, 3.0e20, 2.0e-22, 0.0], dtype=np.float32)[:, None]
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    expected = oracle.linear(kquant.Q4_K, packed, out_dim, in_dim, x)
    for row in range(rows - 1):
        assert normalised_error(y[row:row + 1], expected[row:row + 1]) <= TOLERANCE
    assert np.all(y[rows - 1] == 0.0)


def test_prefill_gemm_reserved_mode_is_refused(cuda):
    lib = tile_ops.load()
    assert lib.nfn_mi355_k_quant_gemm_workspace_bytes_v1(64, 512, 128, tile_ops.GEMM_INT8) == 0
    assert lib.nfn_mi355_k_quant_gemm_workspace_bytes_v1(64, 512, 128, tile_ops.GEMM_F16) > 0


def test_prefill_gemm_full_size_row_subset(cuda, oracle):
    # the benchmark's prefill shape (M=512, 6656 -> 16384): check a slice of output columns.
    rows, out_dim, in_dim = 512, 16384, 6656
    torch = torch_()
    generator = torch.Generator(device="cpu").manual_seed(5)
    packed = random_packed(kquant.Q4_K, 256, in_dim, 91)
    full = np.tile(packed.reshape(256, -1), (out_dim // 256, 1)).reshape(-1)
    x = kquant.synthetic_activations(92, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, full, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    expected = oracle.linear(kquant.Q4_K, packed, 256, in_dim, x)
    assert normalised_error(y[:, :256], expected) <= TOLERANCE
    # every 256-column stripe repeats the same weights
    assert np.array_equal(y[:, :256], y[:, out_dim - 256:])


def gemm_subset_check(cuda, oracle, encoding, rows, out_dim, in_dim, seed, plan):
    """A full-size GEMM with distinct random weights in every column, compared with the oracle on a
    spread of rows (tile edges, both halves of every 256-row tile kind) and of column stripes
    (first, last and interior 128-column tiles, edges of each)."""
    assert tile_ops.gemm_plan(encoding, rows, in_dim, out_dim) == plan
    packed = random_packed(encoding, out_dim, in_dim, seed)
    x = kquant.synthetic_activations(seed + 1, rows, in_dim)
    weight = tile_ops.PackedWeight.from_numpy(encoding, packed, out_dim, in_dim)
    y = tile_ops.gemm(weight, to_device(x, cuda), tile_ops.GEMM_F16).cpu().numpy()
    rng = np.random.default_rng(seed + 2)
    picked_rows = np.unique(np.concatenate([
        np.array([0, 1, 31, 32, 127, 128, 255, rows - 256, rows - 129, rows - 128, rows - 33, rows - 1]),
        rng.integers(0, rows, 12)]))
    starts = [0, 120, out_dim // 2 - 8, out_dim - 136, out_dim - 16]
    picked_columns = np.unique(np.concatenate([np.arange(start, start + 16) for start in starts] +
                                              [rng.integers(0, out_dim, 48)]))
    row_bytes = packed.size // out_dim
    stripe = np.ascontiguousarray(packed.reshape(out_dim, row_bytes)[picked_columns]).reshape(-1)
    expected = oracle.linear(encoding, stripe, picked_columns.size, in_dim,
                             np.ascontiguousarray(x[picked_rows]))
    assert normalised_error(y[np.ix_(picked_rows, picked_columns)], expected) <= TOLERANCE
    return y


@pytest.mark.parametrize("rows", [512, 2048])
def test_prefill_gemm_config3_gate_up_shape(cuda, oracle, rows):
    # SwiGLU FFN prefill, gate / up projection: 6,656 -> 16,384 at both row counts
    gemm_subset_check(cuda, oracle, kquant.Q4_K, rows, 16384, 6656, 300 + rows, (256, 1))


@pytest.mark.parametrize("rows,plan", [(512, (256, 4)), (2048, (256, 1))])
def test_prefill_gemm_config3_down_shape(cuda, oracle, rows, plan):
    # the down projection 16,384 -> 6,656 (64 blocks of K): 512 rows give 104 tall tiles for 256
    # compute units, so K is split into four shares; 2,048 rows run unsplit
    y = gemm_subset_check(cuda, oracle, kquant.Q4_K, rows, 6656, 16384, 400 + rows, plan)
    assert np.all(np.isfinite(y))


@pytest.mark.parametrize("encoding", [kquant.Q5_K, kquant.Q6_K, kquant.Q8_0])
def test_prefill_gemm_config4_prefill_shapes(cuda, oracle, encoding):
    # the mixed-format profile's prefill half: 1,024 rows, FFN down in the formats it may draw
    gemm_subset_check(cuda, oracle, encoding, 1024, 6656, 16384, 500 + encoding, (256, 2))


def test_decode_gemv_is_deterministic(cuda):
    # the same call must return the same bits every time (fixed reduction order)
    out_dim, in_dim = 520, 6656
    packed = random_packed(kquant.Q4_K, out_dim, in_dim, 5)
    weight = tile_ops.PackedWeight.from_numpy(kquant.Q4_K, packed, out_dim, in_dim)
    x = to_device(kquant.synthetic_activations(8, 1, in_dim), cuda)
    workspace = tile_ops.small_batch_workspace(1, in_dim)
    first = tile_ops.mmvq_linear(weight, x, workspace).cpu().numpy()
    for _ in range(20):
        assert_bits_equal(tile_ops.mmvq_linear(weight, x, workspace), first)


@pytest.mark.gpu
@pytest.mark.parametrize("prologue", ["plain", "swiglu"])
@pytest.mark.parametrize("rows", [5, 8])
def test_many_tile_launches_at_five_to_eight_rows_equal_narrow_ones(cuda, prologue, rows):
    """With two or more 32-row tiles per compute unit the 5..8-row launches quantize the
    activations once (a quantizer launch and the workspace) instead of once per tile in the
    kernel: same records, so the same bits as a launch over a slice of the rows."""
    in_dim, out_dim, narrow = 512, 16640, 96  # 2 x 520 tiles; the slice is three tiles
    packed = [random_packed(kquant.Q4_K, out_dim, in_dim, 70 + index) for index in range(2)]
    wide = [tile_ops.PackedWeight.from_numpy(kquant.Q4_K, p, out_dim, in_dim) for p in packed]
    row_bytes = packed[0].size // out_dim
    first, last = out_dim - narrow, out_dim
    sliced = [tile_ops.PackedWeight.from_numpy(kquant.Q4_K, p.reshape(-1)[first * row_bytes:].copy(),
                                               narrow, in_dim) for p in packed]
    x = to_device(kquant.synthetic_activations(71, rows, in_dim), cuda)
    second = to_device(kquant.synthetic_activations(72, rows, in_dim), cuda) if prologue != "plain" else None
    workspace = tile_ops.small_batch_workspace(rows, in_dim)
    many = tile_ops.multi_linear(wide, x, workspace, second, "mmq", prologue)
    few = tile_ops.multi_linear(sliced, x, workspace, second, "mmq", prologue)
    for whole, part in zip(many, few):
        assert_bits_equal(whole[:, first:last].contiguous(), part, "many tiles vs few")
