"""GPU parity of untranspose (transpose_i / transpose_o on the device) and of
decode-to-materialize (any encoding -> plain values, stored or row order)
against the oracle's permutations and the values that were encoded."""
import numpy as np
import pytest

import fastlanesgpu_amd as fls
import fls_testlib as T

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(2027)


@pytest.mark.parametrize("n_vec", [1, 3, 257])
def test_transpose_matches_oracle(n_vec):
    x = RNG.integers(0, 2**32, n_vec * 1024, dtype=np.uint64).astype(np.uint32)
    fwd = T.from_dev(fls.transpose_vectors(T.to_dev(x), n_vec))
    inv = T.from_dev(fls.transpose_vectors(T.to_dev(x), n_vec, inverse=True))
    for v in range(n_vec):
        s = slice(1024 * v, 1024 * (v + 1))
        np.testing.assert_array_equal(fwd[s], T.o_perm("orc_transpose_i_u32", x[s]))
        np.testing.assert_array_equal(inv[s], T.o_perm("orc_transpose_o_u32", x[s]))
    back = T.from_dev(fls.transpose_vectors(T.to_dev(fwd), n_vec, inverse=True))
    np.testing.assert_array_equal(back, x)


def column_values(n, seed):
    """Sorted runs with noise: every encoding has something to work with."""
    r = np.random.default_rng(seed)
    base = np.sort(r.integers(0, 5_000_000, n)).astype(np.uint32)
    runs = np.repeat(r.integers(0, 1 << 20, n // 37 + 1), 37)[:n].astype(np.uint32)
    return np.where(r.random(n) < 0.5, base, runs).astype(np.uint32)


KINDS = ["bitpack", "bitpack_t", "delta", "rle", "for", "exhaustive"]


def encode(x, kind):
    if kind == "bitpack":
        return fls.bitpack_column(x).to_device()
    return T.encode_any(x, kind)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1, 1000, 1024, 5_000 + 7, 300_000 + 11])
def test_decode_rows_is_the_encoded_column(kind, n):
    x = column_values(n, n)
    col = encode(x, kind)
    got = T.from_dev(fls.decode_column(col, n, fls.ORDER_ROWS))
    assert got.size == n
    np.testing.assert_array_equal(got, x)


@pytest.mark.parametrize("kind", ["bitpack_t", "delta", "rle"])
@pytest.mark.parametrize("n", [5_000 + 7, 4 * 1024 + 1, 4 * 1024 + 130])
def test_decode_rows_into_an_unaligned_output(kind, n):
    # row order into an output that is not 16-byte aligned takes the
    # one-word stores; the sizes end the last vector inside a 4-row group
    torch = T.torch_cuda()
    x = column_values(n, n + 3)
    col = encode(x, kind)
    buf = torch.full((n + 8,), -1, dtype=torch.int32, device="cuda")
    fls.decode_column(col, n, fls.ORDER_ROWS, out=buf[1:n + 1])
    got = T.from_dev(buf)
    np.testing.assert_array_equal(got[1:n + 1], x)
    assert got[0] == 0xFFFFFFFF and np.all(got[n + 1:] == 0xFFFFFFFF)
    aligned = T.from_dev(fls.decode_column(col, n, fls.ORDER_ROWS))
    np.testing.assert_array_equal(aligned, x)


@pytest.mark.parametrize("kind", ["bitpack_t", "delta", "rle"])
def test_decode_stored_order_into_an_unaligned_output(kind):
    # stored order into an output that is not 16-byte aligned takes the
    # one-word stores; the aligned output takes the LDS stage and 16-byte
    # stores: both hold the same words
    torch = T.torch_cuda()
    n = 3 * 1024 + 300
    x = column_values(n, n + 5)
    col = encode(x, kind)
    aligned = T.from_dev(fls.decode_column(col, n, fls.ORDER_STORED))
    buf = torch.full((4 * 1024 + 8,), -1, dtype=torch.int32, device="cuda")
    fls.decode_column(col, n, fls.ORDER_STORED, out=buf[1:4 * 1024 + 1])
    got = T.from_dev(buf)
    np.testing.assert_array_equal(got[1:4 * 1024 + 1], aligned)
    assert got[0] == 0xFFFFFFFF and np.all(got[4 * 1024 + 1:] == 0xFFFFFFFF)


@pytest.mark.parametrize("kind", KINDS)
def test_decode_stored_order(kind):
    n = 9 * 1024 + 500
    x = column_values(n, 77)
    col = encode(x, kind)
    got = T.from_dev(fls.decode_column(col, n, fls.ORDER_STORED))
    assert got.size == 10 * 1024
    if kind == "bitpack":
        np.testing.assert_array_equal(got[:n], x)
        return
    # transposed storage: transpose_o of each stored vector gives the rows back
    rows = np.concatenate([T.o_perm("orc_transpose_o_u32", got[1024 * v:1024 * (v + 1)]) for v in range(10)])
    np.testing.assert_array_equal(rows[:n], x)


def test_full_size_delta_date_column():
    # 120M-row orderdate of the Q1.1 table, delta-encoded on the GPU: the
    # row-order materialization equals the generated column on the device
    torch = T.torch_cuda()
    n = 120_000_000
    od = fls.gen_c2(5, n)[0]
    w, vm, bs = fls.delta_encode_device(od, n)
    col = fls.Column(fls.ENC_DELTA, n, w, vmeta=vm, bases=bs)
    out = fls.decode_column(col, n, fls.ORDER_ROWS)
    assert bool(torch.equal(out, od[:n]))
    st = fls.decode_column(col, n, fls.ORDER_STORED)
    back = fls.transpose_vectors(st, (n + 1023) // 1024, inverse=True)
    assert bool(torch.equal(back[:n], od[:n]))


def test_errors():
    x = column_values(3000, 1)
    col = encode(x, "delta")
    with pytest.raises(fls.FlsError):
        fls.decode_column(col, 3000, order=7)
    with pytest.raises(fls.FlsError):  # in place is not a permutation
        d = T.to_dev(np.arange(1024, dtype=np.uint32))
        fls.transpose_vectors(d, 1, out=d)
    with pytest.raises(fls.FlsError):  # vectors are moved 16 bytes at a time
        d = T.to_dev(np.arange(2048, dtype=np.uint32))
        fls.transpose_vectors(d[1:1025], 1)


def rle_vector_column(run_counts, ibw=1, vbw=32):
    """An RLE column made by hand: vector v has run_counts[v] runs, index deltas
    packed at ibw bits, run values at vbw bits (reference words only)."""
    words, vmeta, rmeta, bases, rows, off = [], [], [], [], [], 0
    for nr in run_counts:
        starts = np.zeros(1024, np.int64)
        starts[1 + RNG.choice(1023, nr - 1, replace=False)] = 1
        idx = np.cumsum(starts).astype(np.uint32)
        vals = RNG.integers(0, 2**vbw, nr, dtype=np.uint64).astype(np.uint32)
        vbase = np.uint32(RNG.integers(0, 2**32 - 2**vbw + 1, dtype=np.uint64))
        t = fls.transpose_i(idx)
        index_words = fls.pack(fls.unrsum(t), ibw)
        bits = np.zeros(-(-nr * vbw // 32) * 32, np.uint8)
        bits[: nr * vbw] = ((vals[:, None] >> np.arange(vbw, dtype=np.uint32)) & 1).ravel()
        value_words = np.packbits(bits, bitorder="little").view(np.uint32)
        words += [index_words, value_words]
        vmeta.append(off << 8 | ibw)
        rmeta.append(int(vbase) | nr << 32 | vbw << 48 | ibw << 56)
        bases.append(t[:32])
        rows.append((vals[idx] + vbase).astype(np.uint32))
        off += index_words.size + value_words.size
    host = fls.HostColumn(fls.ENC_RLE, 1024 * len(run_counts), np.concatenate(words + [np.zeros(2, np.uint32)]),
                          vmeta=np.array(vmeta, np.uint64), bases=np.concatenate(bases),
                          aux=np.array(rmeta, np.uint64))
    return host.to_device(), np.concatenate(rows)


@pytest.mark.parametrize("ibw,vbw", [(1, 32), (1, 7), (3, 20), (32, 1)])
def test_decode_rle_run_counts(ibw, vbw):
    """Run counts around a half-wave, a load step (128) and the stage (512),
    and index deltas wider than a bit, in both orders, aligned and not."""
    torch = T.torch_cuda()
    counts = [1, 2, 31, 32, 33, 127, 128, 129, 511, 512, 513, 700, 1023, 1024, 5]
    col, rows = rle_vector_column(counts, ibw, vbw)
    stored = T.transpose_vectors(rows)
    n = rows.size - 300  # the last vector is partial in row order
    for shift in (0, 1):
        buf = torch.full((rows.size + 8,), -1, dtype=torch.int32, device="cuda")
        fls.decode_column(col, n, fls.ORDER_ROWS, out=buf[shift:shift + n])
        got = T.from_dev(buf)
        np.testing.assert_array_equal(got[shift:shift + n], rows[:n])
        assert np.all(got[shift + n:] == 0xFFFFFFFF)
        buf.fill_(-1)
        fls.decode_column(col, rows.size, fls.ORDER_STORED, out=buf[shift:shift + rows.size])
        np.testing.assert_array_equal(T.from_dev(buf)[shift:shift + rows.size], stored)
        buf.fill_(-1)
        fls.rle_decode(col.words, col.vmeta, col.aux, col.bases, len(counts), buf[shift:shift + rows.size])
        got = T.from_dev(buf)
        np.testing.assert_array_equal(got[shift:shift + rows.size], stored)
        assert np.all(got[shift + rows.size:] == 0xFFFFFFFF)


@pytest.mark.parametrize("ibw", [1, 3])
def test_decode_rle_vectors_beside_one_with_more_runs(ibw):
    """The two vectors of a wave on either side of the stage's 512 runs, and one
    with index deltas wider than a bit, in both orders, aligned and not; the
    last vector is partial in row order."""
    torch = T.torch_cuda()
    col, rows = rle_vector_column([600, 5, 512, 513, 1, 1024, 1024, 30, 513, 511], ibw, 17)
    stored = T.transpose_vectors(rows)
    n = rows.size - 1001
    for shift in (0, 1, 2):
        buf = torch.full((rows.size + 8,), -1, dtype=torch.int32, device="cuda")
        fls.decode_column(col, n, fls.ORDER_ROWS, out=buf[shift:shift + n])
        got = T.from_dev(buf)
        np.testing.assert_array_equal(got[shift:shift + n], rows[:n])
        assert np.all(got[shift + n:] == 0xFFFFFFFF)
        fls.decode_column(col, rows.size, fls.ORDER_STORED, out=buf[shift:shift + rows.size])
        np.testing.assert_array_equal(T.from_dev(buf)[shift:shift + rows.size], stored)


def test_decode_mixed_column_with_rle_vectors():
    """RLE vectors of every run count beside other encodings in one column."""
    import fastlanesgpu_amd.selector as sel
    torch = T.torch_cuda()
    parts = []
    for k, runs in enumerate([3, 600, 0, 512, 513, 0, 1024, 40, 0]):
        if runs:
            cuts = np.sort(RNG.choice(1023, runs - 1, replace=False)) + 1
            parts.append(np.repeat(RNG.integers(0, 2**20, runs), np.diff(np.concatenate([[0], cuts, [1024]]))))
        else:
            parts.append(np.arange(1024) * (k + 1) + RNG.integers(0, 3, 1024))
    x = np.concatenate(parts).astype(np.uint32)[:-77]
    ws = sel.MixedWorkspace(x.size)
    ws.cls[:] = torch.tensor([30 if r else 20 for r in [3, 600, 0, 512, 513, 0, 1024, 40, 0]], dtype=torch.uint8)
    sel.mixed_encode_classes(T.to_dev(x), x.size, ws)
    col = ws.column(x.size)
    padded = np.full(9 * 1024, x[-1], np.uint32)
    padded[: x.size] = x
    stored = T.transpose_vectors(padded)
    for shift in (0, 1):
        buf = torch.full((9 * 1024 + 8,), -1, dtype=torch.int32, device="cuda")
        fls.decode_column(col, x.size, fls.ORDER_ROWS, out=buf[shift:shift + x.size])
        got = T.from_dev(buf)
        np.testing.assert_array_equal(got[shift:shift + x.size], x)
        assert np.all(got[shift + x.size:] == 0xFFFFFFFF)
        sel.mixed_decode(col, out=buf[shift:])
        np.testing.assert_array_equal(T.from_dev(buf)[shift:shift + 9 * 1024], stored)
