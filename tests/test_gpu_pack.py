"""GPU parity of the packed chunk-embedding codec (src/packops.rs:172-438) against the CPU
oracle, through the C ABI.

Every step is exact arithmetic in the reference's order (column sums, Haar butterflies,
max-abs scaling, rounding, integer rANS64), so the GPU's bytes must equal the oracle's bytes
and the GPU's decoded floats must equal the oracle's decoded floats bit for bit.  Cases cover
the window split at 1024 rows, odd column lengths (mirror-edge Haar), empty and one-row
matrices, a batch of mixed sizes, NaN input (the reference panics: an error here), and
malformed buffers (truncated, leftover bytes, corrupt stream).
"""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def codec():
    from witchcraft_amd import codec as c
    return c


def _emb(rows, cols, seed, smooth=True):
    rng = np.random.default_rng(seed)
    if smooth:
        base = rng.normal(0, 1, cols)
        x = base + np.cumsum(rng.normal(0, 0.15, (rows, cols)), axis=0) + rng.normal(0, 0.3, (rows, cols))
    else:
        x = rng.normal(0, 1, (rows, cols))
    n = np.linalg.norm(x, axis=1, keepdims=True)
    return (x / np.where(n == 0, 1, n)).astype(np.float32)


SHAPES = [(1, 128), (2, 128), (7, 128), (64, 128), (333, 128), (1024, 128), (1025, 128), (2500, 128),
          (40, 5), (17, 255), (300, 1), (3, 64)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_packed_bytes_equal_oracle(codec, rows, cols):
    x = _emb(rows, cols, rows * 31 + cols, smooth=rows % 2 == 0)
    got = codec.embeddings_to_packed(x)
    want = orc.embeddings_to_packed(x)
    assert len(got) == len(want)
    assert got == want


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_unpacked_floats_equal_oracle(codec, rows, cols):
    x = _emb(rows, cols, rows * 17 + cols)
    buf = orc.embeddings_to_packed(x)
    got = codec.embeddings_from_packed(buf, cols)
    want = orc.embeddings_from_packed(buf, cols)
    assert got.shape == (rows, cols)
    assert got.view(np.uint32).tolist() == want.view(np.uint32).tolist()


def test_batch_of_mixed_matrices(codec):
    mats = [_emb(r, 128, r) for r in (0, 5, 1024, 1, 2049, 333, 0, 77)]
    packed = codec.embeddings_to_packed_batch(mats)
    assert packed == [orc.embeddings_to_packed(m) for m in mats]
    back = codec.embeddings_from_packed_batch(packed, 128)
    for m, b, buf in zip(mats, back, packed):
        assert b.shape == m.shape
        if m.shape[0]:
            assert b.view(np.uint32).tolist() == orc.embeddings_from_packed(buf, 128).view(np.uint32).tolist()
            assert float((m * b).sum(1).min()) > 0.99


def test_scale_extremes(codec):
    """Large low-frequency coefficients (symbols far above 8192) and tiny windows."""
    x = np.ones((900, 128), np.float32)
    x[:, 0] = 50.0  # huge DC term, many large symbols
    x[::7, 3] = -3.0
    assert codec.embeddings_to_packed(x) == orc.embeddings_to_packed(x)
    z = np.zeros((3, 128), np.float32)
    assert codec.embeddings_to_packed(z) == orc.embeddings_to_packed(z)


def test_nan_input_is_an_error(codec):
    x = _emb(10, 128, 1)
    x[4, 9] = np.nan
    with pytest.raises(RuntimeError):
        codec.embeddings_to_packed(x)


def test_malformed_buffers_are_errors(codec):
    x = _emb(50, 128, 3)
    buf = orc.embeddings_to_packed(x)
    for bad in (buf + b"\0", buf[:-3], buf[:10]):
        with pytest.raises(RuntimeError):
            codec.embeddings_from_packed(bad, 128)
    # flip bytes inside the stream: either decodes to something or reports corruption, never faults
    b = bytearray(buf)
    b[-20] ^= 0xFF
    try:
        codec.embeddings_from_packed(bytes(b), 128)
    except RuntimeError:
        pass


def _or_refused(fn, *args):
    try:
        return fn(*args)
    except (RuntimeError, ValueError):
        return "refused"


@pytest.mark.parametrize("rows,cols", [(1, 1), (21, 3), (64, 1), (13, 5), (127, 1), (127, 8), (341, 3), (512, 2),
                                       (205, 5), (344, 3), (1024, 2), (73, 57)])
@pytest.mark.parametrize("kind", ["smooth", "two", "flat"])
def test_coder_lengths_and_histograms(codec, rows, cols, kind):
    """Value counts around the coder's steps (8 and 64 symbols, 1024 staged positions) on histograms
    from one dominant symbol to hundreds of rare ones; what the oracle refuses is refused."""
    rng = np.random.default_rng(rows)
    if kind == "two":  # a constant with one step: few nonzero coefficients
        x = np.full((rows, cols), 0.5, np.float32)
        x[rows // 2:] = 0.51
    elif kind == "flat":
        x = rng.uniform(-0.4, 0.4, (rows, cols)).astype(np.float32)
    else:
        x = _emb(rows, cols, rows) * rng.uniform(0.1, 0.9, (rows, 1)).astype(np.float32)
    buf = _or_refused(orc.embeddings_to_packed, x)
    assert _or_refused(codec.embeddings_to_packed, x) == buf
    if buf != "refused":
        got, want = codec.embeddings_from_packed(buf, cols), orc.embeddings_from_packed(buf, cols)
        assert got.view(np.uint32).tolist() == want.view(np.uint32).tolist()


@pytest.mark.parametrize("rows,cols,big", [(31, 128, 2.0), (32, 128, 8.0), (33, 128, 40.0), (65, 64, 150.0),
                                           (96, 32, 300.0), (512, 128, 900.0), (9, 250, 2500.0)])
def test_symbols_across_the_counters(codec, rows, cols, big):
    """Rows around the column sums' blocks of 32, and values past 1 (scaled by the largest one below 1)
    whose symbols fall on both sides of the per-lane counters (64), of the first histogram pass (8,192)
    and of the 16 bits a symbol is stored in: the oracle's bytes."""
    rng = np.random.default_rng(rows)
    x = _emb(rows, cols, rows)
    at = rng.integers(0, x.size, 12)
    x.reshape(-1)[at] = np.linspace(1.0, big, at.size).astype(np.float32) * rng.choice([-1, 1], at.size)
    buf = _or_refused(orc.embeddings_to_packed, x)
    assert buf != "refused"
    assert codec.embeddings_to_packed(x) == buf


@pytest.mark.parametrize("delta", [-1, -3, 1])
def test_histogram_totals_other_than_the_slots(codec, delta):
    """A frequency changed in the stored histogram: slots left uncovered decode as the oracle
    decodes them (or both refuse); a total above 4096 is refused."""
    b = bytearray(orc.embeddings_to_packed(_emb(40, 128, 9)))
    at = 4 + 128 + 2 + 2  # first symbol's frequency
    f = int.from_bytes(b[at:at + 2], "little") + delta
    b[at:at + 2] = f.to_bytes(2, "little")
    got, want = (_or_refused(fn, bytes(b), 128) for fn in (codec.embeddings_from_packed, orc.embeddings_from_packed))
    if isinstance(want, str):
        assert isinstance(got, str)
    else:
        assert got.view(np.uint32).tolist() == want.view(np.uint32).tolist()
    assert delta < 0 or isinstance(got, str)


def test_window_of_one_symbol_decodes_like_any_other(codec):
    """The slot table of a window with one symbol (4,096 slots of one run) is formed by all threads: five
    rows of one value take no longer to decode than five of many (0.95 times as long; 1.85 times when
    one thread wrote the run)."""
    import time
    rng = np.random.default_rng(4)
    flat, many = np.full((5, 128), 0.5, np.float32), rng.uniform(-0.3, 0.3, (5, 128)).astype(np.float32)
    best = []
    for x in (flat, many):
        bufs = codec.embeddings_to_packed_batch([x])
        times = []
        for _ in range(60):
            t0 = time.perf_counter()
            codec.embeddings_from_packed_batch(bufs, 128)
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    assert best[0] < 1.4 * best[1], best
