"""GPU encoders (bit-pack, FastLanes delta, FastLanes RLE) against the host
encoders / the oracle, word for word, plus decode round trips."""
import numpy as np
import pytest

import fastlanesgpu_amd as fls
import fls_testlib as T

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(99)


def u32(t):
    return T.from_dev(t, np.uint32)


@pytest.mark.parametrize("transposed", [False, True])
def test_pack_column_device_matches_host(transposed):
    for bw in range(33):
        n = 5 * 1024 + 333
        x = RNG.integers(0, 2**bw, n, dtype=np.uint64).astype(np.uint32)
        want = fls.pack_column(x, bw, transpose=transposed)
        got = u32(fls.pack_column_device(T.to_dev(x), n, bw, transposed=transposed))[: want.size]
        np.testing.assert_array_equal(got, want, err_msg=f"bw={bw}")
    # frame of reference
    x = RNG.integers(1000, 1000 + 2**9, 3000).astype(np.uint32)
    want = fls.pack_column((x - 1000).astype(np.uint32), 9)
    np.testing.assert_array_equal(u32(fls.pack_column_device(T.to_dev(x), x.size, 9, base=1000))[: want.size], want)


@pytest.mark.parametrize("kind", ["sorted", "random", "dates", "constant", "small"])
def test_delta_device_matches_host(kind):
    n = 9 * 1024 + 100
    if kind == "sorted":
        x = np.sort(RNG.integers(0, 2**31, n)).astype(np.uint32)
    elif kind == "random":
        x = RNG.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    elif kind == "dates":
        x = T.o_gen_c2(3, n)[0]
    elif kind == "constant":
        x = np.full(n, 7, np.uint32)
    else:
        n = 5
        x = np.array([3, 9, 9, 10, 20], np.uint32)
    words, vmeta, bases = fls.delta_encode_column(x)
    dw, dv, db = fls.delta_encode_device(T.to_dev(x), n)
    np.testing.assert_array_equal(T.from_dev(dv, np.uint64)[: vmeta.size], vmeta)
    np.testing.assert_array_equal(u32(db)[: bases.size], bases)
    np.testing.assert_array_equal(u32(dw)[: words.size], words)


def rle_input(n, mean_run, bw):
    starts = RNG.random(n) < 1.0 / mean_run
    starts[0] = True
    vals = RNG.integers(0, 2**bw, n, dtype=np.uint64).astype(np.uint32)
    return vals[np.flatnonzero(starts)][np.cumsum(starts) - 1].astype(np.uint32)


@pytest.mark.parametrize("case", [(4 * 1024, 8, 13), (3 * 1024 + 77, 8, 32), (2048, 1, 5), (1024, 5000, 20),
                                  (7, 2, 3), (5 * 1024, 32, 0)])
def test_rle_device_matches_oracle(case):
    n, mean_run, bw = case
    x = rle_input(n, mean_run, bw) if bw else np.zeros(n, np.uint32)
    words, vmeta, rmeta, bases = fls.rle_encode_device(T.to_dev(x), n)
    words, vmeta = u32(words), T.from_dev(vmeta, np.uint64)
    rmeta, bases = T.from_dev(rmeta, np.uint64), u32(bases)
    n_vec = (n + 1023) // 1024
    for v in range(n_vec):
        seg = x[v * 1024:(v + 1) * 1024]
        hdr = T.OrcRle()
        ovals = np.zeros(1024, np.uint32)
        oidx = np.zeros(1024, np.uint32)
        T.oracle().orc_rle_encode_u32(np.ascontiguousarray(seg), seg.size, hdr, ovals, oidx)
        rm = int(rmeta[v])
        vbase, n_runs, vbw, ibw = rm & 0xFFFFFFFF, (rm >> 32) & 0xFFFF, (rm >> 48) & 0xFF, (rm >> 56) & 0xFF
        assert (vbase, n_runs, vbw, ibw) == (hdr.vbase, hdr.n_runs, hdr.vbw, hdr.ibw)
        off = int(vmeta[v]) >> 8
        assert int(vmeta[v]) & 0xFF == ibw
        np.testing.assert_array_equal(bases[32 * v:32 * v + 32], np.array(hdr.bases, np.uint32))
        np.testing.assert_array_equal(words[off:off + 32 * ibw], oidx[: 32 * ibw])
        nvw = (n_runs * vbw + 31) // 32
        np.testing.assert_array_equal(words[off + 32 * ibw:off + 32 * ibw + nvw], ovals[:nvw])


@pytest.mark.parametrize("case", [(6 * 1024 + 5, 8, 11), (2048, 1, 32), (1024, 100000, 7)])
def test_rle_roundtrip_gpu(case):
    torch = T.torch_cuda()
    n, mean_run, bw = case
    x = rle_input(n, mean_run, bw)
    words, vmeta, rmeta, bases = fls.rle_encode_device(T.to_dev(x), n)
    n_vec = (n + 1023) // 1024
    out = torch.empty(n_vec * 1024, dtype=torch.int32, device="cuda")
    fls.rle_decode(words, vmeta, rmeta, bases, n_vec, out)
    padded = np.full(n_vec * 1024, x[-1], np.uint32)
    padded[:n] = x
    np.testing.assert_array_equal(u32(out), T.transpose_vectors(padded))


@pytest.mark.parametrize("n", [1, 31, 33, 1023, 1024, 1025, 8 * 1024 - 1, 8 * 1024 + 1])
def test_encoders_at_vector_and_block_edges(n):
    """Sizes around a chain, a vector and a block of 8 vectors: bit-pack in both
    orders with a base, delta against the host encoder, RLE by round trip."""
    torch = T.torch_cuda()
    rng = np.random.default_rng(n)
    x = rng.integers(50, 50 + 2**13, n).astype(np.uint32)
    d = T.to_dev(x)
    for transposed in (False, True):
        want = fls.pack_column((x - 50).astype(np.uint32), 13, transpose=transposed)
        got = u32(fls.pack_column_device(d, n, 13, base=50, transposed=transposed))[: want.size]
        np.testing.assert_array_equal(got, want, err_msg=f"transposed={transposed}")
    words, vmeta, bases = fls.delta_encode_column(x)
    dw, dv, db = fls.delta_encode_device(d, n)
    np.testing.assert_array_equal(T.from_dev(dv, np.uint64)[: vmeta.size], vmeta)
    np.testing.assert_array_equal(u32(db)[: bases.size], bases)
    np.testing.assert_array_equal(u32(dw)[: words.size], words)
    x = np.repeat(x[: n // 3 + 1], 3)[:n]
    words, vmeta, rmeta, bases = fls.rle_encode_device(T.to_dev(x), n)
    n_vec = (n + 1023) // 1024
    out = torch.empty(n_vec * 1024, dtype=torch.int32, device="cuda")
    fls.rle_decode(words, vmeta, rmeta, bases, n_vec, out)
    padded = np.full(n_vec * 1024, x[-1], np.uint32)
    padded[:n] = x
    np.testing.assert_array_equal(u32(out), T.transpose_vectors(padded))


@pytest.mark.parametrize("n_vec", [1023, 1024, 1025, 2 * 4096 + 3])
def test_offsets_over_several_scan_blocks(n_vec):
    """Offsets, total and fallback count where the scan runs in one block, in
    exactly one, and in several (1,024 vectors each)."""
    import fastlanesgpu_amd.selector as sel
    torch = T.torch_cuda()
    n = n_vec * 1024 - 5
    g = torch.Generator(device="cuda")
    g.manual_seed(n_vec)
    # a width of its own for every vector: 1-bit to 16-bit steps between neighbours
    top = torch.randint(1, 17, (n_vec,), generator=g, device="cuda", dtype=torch.int32).repeat_interleave(1024)[:n]
    d = torch.randint(0, 1 << 30, (n,), generator=g, device="cuda", dtype=torch.int32) & ((1 << top) - 1)
    words, vmeta, _ = fls.delta_encode_device(d, n)
    vm = T.from_dev(vmeta, np.uint64)
    sizes = 32 * (vm & np.uint64(255))
    want = np.concatenate([[0], np.cumsum(sizes)])
    np.testing.assert_array_equal(vm >> np.uint64(8), want[:-1])
    assert words.numel() == want[-1]
    ws = sel.MixedWorkspace(n)
    conf = torch.rand(n_vec, generator=g, device="cuda")
    ws.cls.zero_()
    ws.fallbacks.zero_()
    sel.mixed_plan(d, n, ws, conf=conf, conf_min=0.3)
    assert int(ws.fallbacks.item()) == int((conf < 0.3).sum())
    sel.mixed_plan(d, n, ws, conf=conf, conf_min=0.3)  # the counter is added to
    assert int(ws.fallbacks.item()) == 2 * int((conf < 0.3).sum())


def test_offsets_over_more_scan_blocks_than_run_at_once():
    """More blocks than are resident together, which their tickets put in order,
    and more than 1,024 of them before the last, whose sums it adds in two trips:
    the delta plan's offsets against its widths, and the resolve's against the
    sizes of the exhaustive search (both plans only, nothing is packed)."""
    import fastlanesgpu_amd.selector as sel
    torch = T.torch_cuda()
    n_vec = 1024 * 1024 + 1025
    n = n_vec * 1024
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    step = torch.randint(0, 8, (n_vec,), generator=g, device="cuda", dtype=torch.int32)
    ramp = torch.arange(1024, device="cuda", dtype=torch.int32) & 31  # every chain 0, s, 2s, ..., 31s
    x = (step[:, None] * ramp[None, :]).reshape(-1)
    vmeta, aux, total = (torch.empty(k, dtype=torch.int64, device="cuda") for k in (n_vec, n_vec, 1))
    bases = torch.empty(32 * n_vec, dtype=torch.int32, device="cuda")
    scratch = torch.empty(int(fls.load().fls_encode_scratch_bytes(n)), dtype=torch.uint8, device="cuda")
    cls = torch.empty(n_vec, dtype=torch.uint8, device="cuda")

    def offsets(sizes):
        ends = torch.cumsum(sizes, 0)
        return ends - sizes, int(ends[-1])

    fls.call("fls_delta_plan_device", fls.dptr(x), n, fls.dptr(vmeta), fls.dptr(bases), fls.dptr(total),
             fls.dptr(scratch), fls.current_stream())
    width = torch.zeros_like(step) + (step >= 1) + (step >= 2) + (step >= 4)
    off, end = offsets(32 * width.long())
    assert torch.equal(vmeta & 255, width.long())
    assert torch.equal(vmeta >> 8, off)
    assert int(total.item()) == end
    _, sizes4 = sel.exhaustive_select(x, n)
    off, end = offsets((sizes4[:n_vec].min(1).values.long() - 16) // 4)
    fls.call("fls_mixed_stats_device", fls.dptr(x), n, None, fls.dptr(vmeta), fls.dptr(aux), fls.dptr(scratch),
             fls.current_stream())
    fls.call("fls_mixed_resolve_device", n, fls.dptr(cls), None, 0.0, 1, fls.dptr(vmeta), fls.dptr(aux),
             fls.dptr(total), None, fls.dptr(scratch), fls.current_stream())
    assert torch.equal(vmeta >> 8, off)
    assert int(total.item()) == end


@pytest.mark.parametrize("how", ["explicit", "current"])
def test_encodes_on_another_stream(how):
    """Encodes on a stream that has other work queued first: the size is read in
    that stream's order (delta, RLE), the column of a workspace is not read
    before its encode, and all equal the encodes on the default stream."""
    import contextlib

    import fastlanesgpu_amd.selector as sel
    torch = T.torch_cuda()
    n = 300 * 1024 + 5
    x = sel.gen_train_vectors(17, 0, 301)[:n]
    ws, want_ws = sel.MixedWorkspace(n, trial=True), sel.MixedWorkspace(n)
    sel.mixed_encode_exhaustive(x, n, want_ws)
    want = [fls.delta_encode_device(x, n), fls.rle_encode_device(x, n), want_ws.column(n)]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    arg = {"explicit": {"stream": side.cuda_stream}, "current": {}}[how]
    inside = contextlib.nullcontext if how == "explicit" else lambda: torch.cuda.stream(side)

    def busy():  # about 30 ms of other work on the side stream
        with torch.cuda.stream(side):
            torch.cuda._sleep(60_000_000)

    with inside():
        busy()
        got = [fls.delta_encode_device(x, n, **arg)]
        busy()
        got.append(fls.rle_encode_device(x, n, **arg))
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for a, b in zip(g, w):
            assert torch.equal(a, b)
    encoders = [sel.mixed_encode_exhaustive, sel.mixed_encode_classes, sel.mixed_encode, sel.mixed_encode_trial]
    for encode in encoders:
        ws.total.fill_(1)
        ws.words.zero_()
        torch.cuda.synchronize()
        with inside():
            busy()
            encode(x, n, ws, **arg)
        col = ws.column(n)
        assert col.n_words == want[2].n_words, encode.__name__
        for k in ("words", "vmeta", "aux"):
            assert torch.equal(getattr(col, k), getattr(want[2], k)), (encode.__name__, k)
    for stream in (0, torch.cuda.current_stream()):  # the stream that is current anyway, as an argument
        ws.words.zero_()
        sel.mixed_encode_exhaustive(x, n, ws, stream=stream)
        assert torch.equal(ws.column(n).words, want[2].words)
        with torch.cuda.stream(side):
            busy()
            assert torch.equal(ws.column(n).words, want[2].words)
    fresh = [fls.delta_encode_device(x, n, stream=0), fls.rle_encode_device(x, n, stream=torch.cuda.default_stream())]
    for g, w in zip(fresh, want):
        for a, b in zip(g, w):
            assert torch.equal(a, b)
