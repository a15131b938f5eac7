"""GPU parity of the streaming 16-bit softmax at the places where its parts can go wrong: the range in which row sums take the
short division, and the edges of the walker's 64-value chunks and 512-column steps.  Bit-exact against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from ratchet_amd import Device

    d = Device(0)
    yield d
    d.close()


def _to(oracle, a, bf):
    a = np.asarray(a, np.float32)
    return oracle.cast(a, np.uint16, dst_bf16=True) if bf else a.astype(np.float16)


def _same(got, want, bf):
    g, w = got.view(np.uint16), want.view(np.uint16)
    lim = 0x7f80 if bf else 0x7c00
    return bool((((g == w) | (((g & 0x7fff) > lim) & ((w & 0x7fff) > lim)))).all())


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("cols", [8, 64, 72, 504, 512, 520, 1024, 1096, 2176, 4096])
def test_row_sums_on_both_sides_of_the_short_division(dev, oracle, cols, kind):
    """rows shifted so that their sums run from subnormal (f16) or below 2^-100 (bf16), through the range of the short
    division, to infinity; with results that are subnormal themselves"""
    bf = kind == "bf16"
    rng = np.random.default_rng(cols)
    top = 88.0 if bf else 11.0
    low = -92.0 if bf else -17.0
    rows = 256
    x = rng.standard_normal((1, rows, cols)).astype(np.float32)
    x[0] += np.linspace(low, top - np.log(cols), rows)[:, None].astype(np.float32)
    x[0, ::7] = np.where(rng.random((len(x[0, ::7]), cols)) < 0.9, x[0, ::7] - (40.0 if bf else 8.0), x[0, ::7])
    x[0, 3], x[0, 5], x[0, 9, : cols // 2] = top + 3, -np.inf, -np.inf
    xb = _to(oracle, x, bf)
    want = oracle.softmax(xb, bf16=bf)
    assert _same(dev.softmax(dev.upload(xb, bf16=bf)).to_numpy(), want, bf)


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("cols", [193, 505, 513, 1001, 1023, 1535, 1537, 2047, 2561, 3073, 3583, 3585, 4095])
def test_ragged_rows_under_a_mask_shared_by_heads(dev, oracle, cols, kind):
    """rows that are not whole vectors, whose last vector overlaps the one before it, under an [S, T] mask of three heads: the
    variant that takes a mask row for two heads (an even number of 512-column steps), with a head left over, and the other one"""
    bf = kind == "bf16"
    rng = np.random.default_rng(cols)
    x = _to(oracle, 2 * rng.standard_normal((1, 3, 250, cols)), bf)
    m = np.triu(np.full((250, cols), -np.inf, np.float32), k=1 + max(cols - 250, 0))
    m[100:140] = rng.standard_normal((40, cols))
    m = _to(oracle, m, bf)
    full = np.ascontiguousarray(np.broadcast_to(m, x.shape))
    want = oracle.softmax(oracle.binary("add", x, full, bf16=bf), bf16=bf)
    dx, dm = dev.upload(x, bf16=bf), dev.upload(m, bf16=bf)
    assert _same(dev.softmax_masked(dx, dm).to_numpy(), want, bf)
    dev.softmax_masked(dx, dm, out=dx)
    assert _same(dx.to_numpy(), want, bf)


@pytest.mark.parametrize("heads,rows,cols", [(1, 3840, 6152), (1, 3841, 6152), (1, 4500, 6656),      # under a mask: one round in registers; two, so parked in y
                                             (2, 1920, 6152), (2, 1930, 6152), (1, 3900, 4104)])                    # two rows to a wave, as without a mask; registers
@pytest.mark.parametrize("masked", [False, True])
def test_rows_of_4097_to_8192_columns_around_a_round(dev, oracle, heads, rows, cols, masked):
    """both sides of the choice between registers and parking in y; also in place"""
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((1, heads, rows, cols), np.float32).astype(np.float16)
    m = np.triu(np.full((rows, cols), -np.inf, np.float16), k=1 + cols - rows)
    want = oracle.softmax(oracle.binary("add", x, np.ascontiguousarray(np.broadcast_to(m, x.shape))) if masked else x)
    dx = dev.upload(x)
    for out in (None, dx):
        got = dev.softmax_masked(dx, dev.upload(m), out=out) if masked else dev.softmax(dx, out=out)
        assert _same(got.to_numpy(), want, False)


def _hard_rows(rng, cols, bf):
    """rows whose sums run through subnormals, ties and many powers of two, stop growing, pass infinity, meet NaN or are all masked"""
    rows = [rng.standard_normal(cols) * s + m for s, m in ((1, 0), (2, 0), (4, -3), (0.3, 5), (1, -14), (1, -16), (0.01, 0), (8, -8), (1, 6))]
    rows += [np.full(cols, v) for v in (0.0, -1.0, 3.0, -7.0, -9.7, 8.0, 12.0, -np.inf)]
    rows += [rng.standard_normal(cols) * s + m for s, m in (((1, -85), (2, -90), (1, 85), (3, 80)) if bf else ((3, 4),))]
    rows += [np.sort(rng.standard_normal(cols) * 3), -np.sort(rng.standard_normal(cols) * 3), np.linspace(-17, 5, cols)]
    for k in (1, 8, 31, 33, cols // 2, cols - 1):
        rows += [np.where(np.arange(cols) < k, rng.standard_normal(cols), -np.inf), np.where(np.arange(cols) < k, -np.inf, rng.standard_normal(cols))]
    for at, v in ((0, 11.2), (cols - 1, np.inf), (5, np.inf), (cols // 2, np.nan), (cols - 1, np.nan)):
        rows.append(np.where(np.arange(cols) == at, v, rng.standard_normal(cols)))
    rows.append(np.where(np.arange(cols) % max(cols - 1, 1) == 0, np.where(np.arange(cols) == 0, np.inf, np.nan), 1.0))
    return np.stack(rows)


@pytest.mark.parametrize("kind,heads,rows,cols", [
    ("f16", 2, 33, 2056), ("f16", 2, 33, 3072), ("f16", 2, 40, 3080), ("f16", 4, 40, 4096), ("f16", 2, 33, 4104), ("f16", 2, 33, 5128), ("f16", 6, 35, 6144),
    ("f16", 2, 33, 7176), ("f16", 2, 33, 8184), ("f16", 2, 33, 8192),
    ("f16", 4, 3850, 257), ("f16", 4, 3850, 511), ("f16", 4, 3850, 513), ("f16", 4, 3841, 1001), ("f16", 4, 3850, 1537), ("f16", 4, 3850, 2047),
    ("bf16", 4, 33, 1032), ("bf16", 4, 33, 1536), ("bf16", 4, 33, 2048), ("bf16", 2, 33, 2057), ("bf16", 2, 33, 2056), ("bf16", 2, 33, 4095), ("bf16", 2, 33, 4096),
    ("bf16", 2, 33, 4104), ("bf16", 2, 33, 7168), ("bf16", 2, 33, 8192), ("bf16", 4, 10241, 264), ("bf16", 4, 10241, 520), ("bf16", 4, 3850, 1023)])
def test_several_rows_to_a_wave(dev, oracle, kind, heads, rows, cols):
    """softmax16_row_kernel at the edges of its chunks, of both its lane counts and of rows a wave; plain (an odd number of rows
    among them), under a mask and in place"""
    bf = kind == "bf16"
    rng = np.random.default_rng(cols)
    hard = _hard_rows(rng, cols, bf)
    n = heads * rows
    x = hard[rng.integers(0, len(hard), n)] if n > 2 * len(hard) else np.concatenate([hard, rng.standard_normal((max(n - len(hard), 0), cols))])[:n]
    x = _to(oracle, x, bf).reshape(1, heads, rows, cols)
    m = np.where(rng.random((rows, cols)) < 0.1, -np.inf, 0.5 * rng.standard_normal((rows, cols)))
    m[0] = -np.inf
    m = _to(oracle, m, bf)
    dx, dm = dev.upload(x, bf16=bf), dev.upload(m, bf16=bf)
    want = oracle.softmax(oracle.binary("add", x, np.ascontiguousarray(np.broadcast_to(m, x.shape)), bf16=bf), bf16=bf)
    assert _same(dev.softmax_masked(dx, dm).to_numpy(), want, bf)
    odd = np.ascontiguousarray(x.reshape(1, n, cols)[:, : n - 1])
    assert _same(dev.softmax(dev.upload(odd, bf16=bf)).to_numpy(), oracle.softmax(odd, bf16=bf), bf)
    dev.softmax(dx, out=dx)
    assert _same(dx.to_numpy(), oracle.softmax(x, bf16=bf), bf)


def _plain_masked_in_place(dev, oracle, kind, heads, rows, cols, seed):
    """the oracle's bits without a mask, under one of `rows` rows that the heads share, and both in place; rows of _hard_rows among N(0, 1)"""
    bf = kind == "bf16"
    rng = np.random.default_rng(seed)
    hard = _hard_rows(rng, cols, bf)
    x = rng.standard_normal((heads * rows, cols), np.float32)
    at = rng.permutation(heads * rows)[: 4 * len(hard)]
    x[at] = hard[np.arange(len(at)) % len(hard)]
    x = _to(oracle, x, bf).reshape(1, heads, rows, cols)
    m = np.where(rng.random((rows, cols)) < 0.1, -np.inf, 0.5 * rng.standard_normal((rows, cols), np.float32))
    m = _to(oracle, m, bf)
    dm = dev.upload(m, bf16=bf)
    for mask in (None, m):
        want = oracle.softmax(x if mask is None else oracle.binary("add", x, np.ascontiguousarray(np.broadcast_to(m, x.shape)), bf16=bf), bf16=bf)
        dx = dev.upload(x, bf16=bf)
        assert _same((dev.softmax(dx) if mask is None else dev.softmax_masked(dx, dm)).to_numpy(), want, bf), (mask is None, "another buffer")
        dev.softmax(dx, out=dx) if mask is None else dev.softmax_masked(dx, dm, out=dx)
        assert _same(dx.to_numpy(), want, bf), (mask is None, "in place")


@pytest.mark.parametrize("kind,heads,rows,cols", [
    ("f16", 4, 4101, 1001), ("f16", 4, 4101, 1033), ("f16", 4, 4101, 2047), ("bf16", 4, 5951, 1001), ("bf16", 4, 4301, 1033), ("bf16", 4, 4101, 2047),       # four rows a wave: 16384 in a trip, not whole vectors
    ("bf16", 4, 4301, 1032), ("bf16", 4, 4101, 2048), ("bf16", 2, 4101, 2057), ("bf16", 2, 4101, 3080),                          # two: 8192
    ("f16", 2, 3100, 4104), ("f16", 2, 2100, 7176), ("bf16", 2, 3100, 5128), ("bf16", 2, 2100, 8192)])                           # 6144 and 4096
def test_several_rows_to_a_wave_in_several_trips(dev, oracle, kind, heads, rows, cols):
    """on 256 CUs more rows than the waves of softmax16_row_kernel hold at one time: they store one set of rows while the next one loads"""
    _plain_masked_in_place(dev, oracle, kind, heads, rows, cols, rows + cols)


@pytest.mark.parametrize("kind,heads,rows,cols", [
    ("bf16", 4, 2100, 1024), ("bf16", 4, 2047, 1536), ("bf16", 4, 2048, 1536), ("bf16", 4, 1920, 2048), ("bf16", 4, 1800, 2304), ("bf16", 4, 3840, 2304), ("bf16", 4, 2500, 2304),
    ("bf16", 4, 4100, 511), ("bf16", 4, 4100, 513), ("bf16", 2, 300, 4095), ("bf16", 2, 300, 4097),
    ("f16", 4, 4100, 511), ("f16", 4, 4100, 513), ("f16", 4, 5700, 1001), ("f16", 2, 4096, 2056), ("f16", 2, 4097, 2056), ("f16", 2, 3840, 7176), ("f16", 2, 4200, 7176),
    ("f16", 2, 5760, 4104), ("f16", 2, 4900, 4104), ("f16", 2, 5760, 5120), ("f16", 2, 5760, 6008), ("f16", 2, 5760, 6144), ("f16", 2, 32, 3080), ("f16", 2, 33, 3080)])
def test_both_sides_of_several_rows_to_a_wave(dev, oracle, kind, heads, rows, cols):
    """the same bits on either side of the lines at which softmax16_row_kernel takes over (on 256 CUs)"""
    _plain_masked_in_place(dev, oracle, kind, heads, rows, cols, rows + cols)


@pytest.mark.parametrize("rows,cols", [(1030, 8192), (1640, 5120), (1367, 6144), (2051, 4104), (1403, 6008), (181, 5120), (175, 6000)])
def test_f16_rows_of_4097_to_8192_columns_under_a_mask_of_three_heads(dev, oracle, rows, cols):
    """softmax16_stream_kernel with fifteen rows a block in registers, which has the masks that an odd number of rows share: masks large enough for the
    table of tile classes (with uniform and with mixed tiles) and smaller ones, rows that fill the kernel's steps and rows that do not, a single row of
    mask (under an odd number of rows), one head; also in place"""
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((1, 3, rows, cols), np.float32)
    x[0, :, ::50] = _hard_rows(rng, cols, False)[rng.integers(0, 20, (3, len(x[0, 0, ::50])))]
    x = x.astype(np.float16)
    m = np.where(np.arange(cols)[None, :] > np.arange(rows)[:, None] * (cols // rows), -np.inf, 0.0).astype(np.float16)
    m[:, 512:1024], m[::7, 2048:2560] = -0.5, (0.3 * rng.standard_normal((len(m[::7]), 512))).astype(np.float16)
    for heads, mask in ((3, m), (1, m), (3 if rows % 2 else 1, m[rows // 2:rows // 2 + 1])):
        part = np.ascontiguousarray(x[:, :heads, :rows - (rows + 1) % 2] if len(mask) == 1 else x[:, :heads])
        want = oracle.softmax(oracle.binary("add", part, np.ascontiguousarray(np.broadcast_to(mask, part.shape))))
        dx, dm = dev.upload(part), dev.upload(mask)
        assert _same(dev.softmax_masked(dx, dm).to_numpy(), want, False), (heads, mask.shape)
        dev.softmax_masked(dx, dm, out=dx)
        assert _same(dx.to_numpy(), want, False), (heads, mask.shape, "in place")


def test_f16_rows_of_8192_columns_beyond_2_gib(dev, oracle):
    """several rows to a wave have 32-bit offsets: a tensor of 2 GiB and more goes in chunks to the kernel that keeps fifteen rows a block in registers"""
    rng = np.random.default_rng(5)
    rows, cols, reps = 131072 + 90, 8192, 130
    block = rng.standard_normal((1009, cols), np.float32).astype(np.float16)
    x = np.tile(block, (reps, 1))[:rows]
    got = dev.softmax(dev.upload(x)).to_numpy()
    want = oracle.softmax(block)
    for k in range(0, rows, 1009):
        n = min(1009, rows - k)
        assert np.array_equal(got[k:k + n].view(np.uint16), want[:n].view(np.uint16)), k
