"""FSST decode of offsets and bytes in one call (sizes counted first, then segments joined) against the oracle, bit-exact: vocabulary strings, escape runs, empty and long strings, the reference's own FSST table,
repeated calls on one plan mixed with the two-step form, and the capacity error."""
import numpy as np
import pytest

import fastlanes_amd as fa
from fastlanes_amd import workloads as wl
from tests.test_gpu_decode import _mixed_strings, dev, empty, torch_cuda  # noqa: F401

pytestmark = pytest.mark.gpu


def _fused(torch, plan, d_in, n, cap):
    d_off = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
    d_bytes = empty(torch, cap)
    plan.decode_strings_fused(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), cap)
    plan.check()
    return d_off.cpu().numpy(), d_bytes.cpu().numpy()


def test_fused_vocabulary_strings(torch_cuda, oracle):
    torch = torch_cuda
    offs, data = wl.vocab_strings(40 * 1024, seed=11)
    enc = oracle.encode_str_column(offs, data)
    plan = fa.Plan(enc, "str")
    n = plan.n_values
    d_in = dev(torch, enc)
    for rep in range(3):  # new epoch per call; the status words of the previous call must not be taken as ready
        print(f"fsst fused vocabulary rep={rep}", flush=True)
        got_off, got = _fused(torch, plan, d_in, n, data.size)
        np.testing.assert_array_equal(got_off, offs.astype(np.int64))
        np.testing.assert_array_equal(got[: data.size], data)
    # the two-step form on the same plan afterwards
    d_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    plan.string_offsets(d_in.data_ptr(), d_off.data_ptr())
    np.testing.assert_array_equal(d_off.cpu().numpy(), offs.astype(np.int64))
    d_bytes = empty(torch, data.size)
    plan.decode_strings(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), data.size)
    plan.check()
    np.testing.assert_array_equal(d_bytes.cpu().numpy()[: data.size], data)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_fused_escapes_empty_and_long_strings(torch_cuda, oracle, seed):
    """Escape runs (0xFF bytes) across share boundaries, empty strings (equal start positions), and segments too
    large for the LDS image (per-string form)."""
    torch = torch_cuda
    print(f"fsst fused mixed seed={seed}", flush=True)
    offs, data = _mixed_strings(seed)
    enc = fa.encode_strings(offs.astype(np.uint32), data)
    n = offs.size - 1
    o2, d2 = oracle.decode_str_column(enc, n, data.size + 64)
    np.testing.assert_array_equal(d2, data)
    plan = fa.Plan(enc, "str")
    got_off, got = _fused(torch, plan, dev(torch, enc), n, data.size)
    np.testing.assert_array_equal(got_off, offs.astype(np.int64))
    np.testing.assert_array_equal(got[: data.size], data)


def _strs_from(rows):
    offs = np.zeros(len(rows) + 1, dtype=np.int64)
    offs[1:] = np.cumsum([len(r) for r in rows])
    return offs, np.frombuffer(b"".join(rows), dtype=np.uint8).copy()


@pytest.mark.parametrize("shape", ["all_empty", "one_long", "escapes_only", "tiny"])
def test_fused_segment_shapes(torch_cuda, oracle, shape):
    """Segments whose shares are empty, a segment of one 30 KB string among empty ones (byte-parallel count, too
    large for LDS), strings of escaped bytes only (every second byte a literal), one-byte strings."""
    torch = torch_cuda
    g = np.random.default_rng(7)
    rows = []
    for v in range(4):
        for i in range(1024):
            if shape == "all_empty":
                rows.append(b"" if v != 2 or i % 100 else b"abc")
            elif shape == "one_long":
                rows.append(bytes(g.integers(97, 100, 30_000, dtype=np.uint8).tobytes()) if i == 700 else b"")
            elif shape == "escapes_only":
                rows.append(bytes(g.integers(128, 256, int(g.integers(0, 9)), dtype=np.uint8).tobytes()))
            else:
                rows.append(bytes([97 + i % 26]))
    offs, data = _strs_from(rows)
    enc = fa.encode_strings(offs.astype(np.uint32), data)
    n = offs.size - 1
    o2, d2 = oracle.decode_str_column(enc, n, data.size + 64)
    np.testing.assert_array_equal(d2, data)
    print(f"fsst fused shape={shape} bytes={data.size} encoded={enc.size}", flush=True)
    plan = fa.Plan(enc, "str")
    got_off, got = _fused(torch, plan, dev(torch, enc), n, max(data.size, 1))
    np.testing.assert_array_equal(got_off, offs.astype(np.int64))
    np.testing.assert_array_equal(got[: data.size], data)


def test_fused_capacity_error(torch_cuda, oracle):
    torch = torch_cuda
    offs, data = wl.vocab_strings(4 * 1024, seed=3)
    enc = oracle.encode_str_column(offs, data)
    plan = fa.Plan(enc, "str")
    n = plan.n_values
    d_in = dev(torch, enc)
    d_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    d_bytes = empty(torch, data.size)
    plan.decode_strings_fused(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), data.size // 2)
    with pytest.raises(RuntimeError, match="capacity"):
        plan.check()
    np.testing.assert_array_equal(d_off.cpu().numpy(), offs.astype(np.int64))  # offsets are still whole


def test_fused_multi_page_column(torch_cuda):
    """A string column over the 128 MiB page limit (2^16 vocabulary strings repeated 96 times, ~182 MB encoded, two
    pages): each page is its own launch and its segments look back into the previous page's; the decode reproduces
    the input's offsets and bytes."""
    torch = torch_cuda
    o0, d0 = wl.vocab_strings(1 << 16, seed=13)
    reps = 96
    data = np.tile(d0, reps)
    offs = np.concatenate([[0], np.cumsum(np.tile(np.diff(o0).astype(np.int64), reps))])
    enc = fa.encode_strings(offs.astype(np.uint32), data)
    plan = fa.Plan(enc, "str")
    assert plan.n_pages >= 2
    n = plan.n_values
    print(f"fsst fused multi-page: {n} strings, {plan.n_pages} pages", flush=True)
    got_off, got = _fused(torch, plan, dev(torch, enc), n, data.size)
    np.testing.assert_array_equal(got_off, offs)
    np.testing.assert_array_equal(got[: data.size], data)


def test_fused_decode_in_a_graph(torch_cuda, oracle):
    """The fused decode captured in a HIP graph and replayed three times, with eager decodes of the same plan between
    the replays (they advance its ticket counter and epoch) and the outputs cleared before each replay: every replay
    decodes the column bit-exact, because each call's ticket base and epoch are taken on the device."""
    torch = torch_cuda
    offs, data = wl.vocab_strings(12 * 1024, seed=21)
    enc = oracle.encode_str_column(offs, data)
    plan = fa.Plan(enc, "str")
    n = plan.n_values
    d_in = dev(torch, enc)
    d_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    d_bytes = empty(torch, data.size)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):  # one eager call first, outside the capture
        plan.decode_strings_fused(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), data.size, s.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        plan.decode_strings_fused(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), data.size,
                                  torch.cuda.current_stream().cuda_stream)
    for rep in range(3):
        print(f"fsst graph replay {rep}", flush=True)
        d_off.zero_()
        d_bytes.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        plan.check()
        np.testing.assert_array_equal(d_off.cpu().numpy(), offs.astype(np.int64), err_msg=f"replay {rep}")
        np.testing.assert_array_equal(d_bytes.cpu().numpy()[: data.size], data, err_msg=f"replay {rep}")
        # eager work on the same plan between replays
        e_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        plan.string_offsets(d_in.data_ptr(), e_off.data_ptr())
        e_bytes = empty(torch, data.size)
        plan.decode_strings_fused(d_in.data_ptr(), e_off.data_ptr(), e_bytes.data_ptr(), data.size)
        plan.check()
        np.testing.assert_array_equal(e_bytes.cpu().numpy()[: data.size], data)


@pytest.mark.parametrize("length", ["short", "long"])
@pytest.mark.parametrize("symbols", ["pairs", "quads", "words"])
def test_fused_symbol_tables(torch_cuda, symbols, length):
    """Tables whose longest symbol has at most 3, at most 7 and 8 bytes (each has its own emission), with escapes in
    three strings of a hundred (runs of rare bytes, 0xFF among them, so that they fall on 32-byte and 8 KiB edges and across
    them), for strings short enough that a segment is one chunk and long enough that it is several, whose output takes
    several windows of the LDS image. Both call forms."""
    torch = torch_cuda
    g = np.random.default_rng(len(symbols) * 10 + len(length))
    words = wl.vocabulary(40, seed=3)
    rows = []
    for i in range(3 * 1024):
        n = int(g.integers(0, 21)) if length == "short" else int(g.integers(60, 500))
        if symbols == "pairs":
            b = bytearray(g.integers(97, 123, n, dtype=np.uint8).tobytes())
        elif symbols == "quads":
            b = bytearray(g.integers(97, 103, n, dtype=np.uint8).tobytes())
        else:
            b = bytearray(b" ".join(words[int(k)] for k in g.integers(0, 40, n // 6 + 1))[:n])
        if i % 100 < 3:
            p = int(g.integers(0, len(b) + 1))
            b[p:p] = (g.integers(160, 256, int(g.integers(1, 30)), dtype=np.uint8) | np.uint8(g.random() < 0.5)).tobytes()
        rows.append(bytes(b))
    offs, data = _strs_from(rows)
    enc = fa.encode_strings(offs.astype(np.uint32), data)
    longest = int(np.nonzero(enc[17:25])[0][-1]) + 1  # lenHisto of the serialized table: symbols of 1 .. 8 bytes
    print(f"fsst symbols={symbols} length={length} longest={longest}", flush=True)
    assert {"pairs": longest <= 3, "quads": 4 <= longest <= 7, "words": longest == 8}[symbols], longest
    plan, d_in = fa.Plan(enc, "str"), dev(torch, enc)
    got_off, got = _fused(torch, plan, d_in, offs.size - 1, data.size)
    np.testing.assert_array_equal(got_off, offs)
    np.testing.assert_array_equal(got[: data.size], data)
    d_off = torch.zeros(offs.size, dtype=torch.int64, device="cuda")
    plan.string_offsets(d_in.data_ptr(), d_off.data_ptr())
    np.testing.assert_array_equal(d_off.cpu().numpy(), offs)
    d_bytes = empty(torch, data.size + 3)
    plan.decode_strings(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr() + 3, data.size)  # unaligned output
    plan.check()
    np.testing.assert_array_equal(d_bytes.cpu().numpy()[3: 3 + data.size], data)


@pytest.mark.parametrize("vectors", [1, 1024, 1025])
def test_fused_segment_bases(torch_cuda, vectors):
    """Columns whose blocks sum the vectors' sizes themselves (up to 1024) and one that the scan kernel serves."""
    torch = torch_cuda
    print(f"fsst bases vectors={vectors}", flush=True)
    g = np.random.default_rng(vectors)
    lens = g.integers(0, 9, vectors * 1024)
    offs = np.concatenate([[0], np.cumsum(lens)])
    data = g.integers(97, 107, int(offs[-1]), dtype=np.uint8)
    enc = fa.encode_strings(offs.astype(np.uint32), data)
    got_off, got = _fused(torch, fa.Plan(enc, "str"), dev(torch, enc), offs.size - 1, data.size)
    np.testing.assert_array_equal(got_off, offs)
    np.testing.assert_array_equal(got[: data.size], data)


def _string_page(enc):
    """Symbols of a column's (single) FSST page, where its data page starts, and its two buffers' offsets in it."""
    lh = [int(x) for x in enc[17:25]]  # lenHisto: symbols of 1 .. 8 bytes
    zt, at, symbols = int(enc[16]) & 1, 25, [b"\0"] if int(enc[16]) & 1 else []
    lh[0] -= zt
    for k in (1, 2, 3, 4, 5, 6, 7, 0):
        for _ in range(lh[k]):
            symbols.append(enc[at: at + k + 1].tobytes())
            at += k + 1
    return symbols, at, enc[at + 8: at + 16].view(np.uint32).astype(np.int64)


def _decode_vector(symbols, bytes_, ends):
    """Strings of a vector: string i is the codes of bytes_[ends[i - 1] : ends[i]] (none where the end lies before)."""
    out = []
    for i, e in enumerate(ends):
        q, row = int(ends[i - 1]) if i else 0, []
        while q < e:
            c = int(bytes_[q])
            row.append(bytes([int(bytes_[q + 1]) if q + 1 < e else 0]) if c == 255 else symbols[c])
            q += 2 if c == 255 else 1
        out.append(b"".join(row))
    return out


@pytest.mark.parametrize("ends", ["lowered_at_segment_end", "lowered_inside", "lowered_to_zero", "raised", "shuffled"])
def test_ends_out_of_order(torch_cuda, ends):
    """End offsets that are not monotone in the middle one of three vectors: a segment that starts behind the one before it
    (well-formed by itself, over bytes that other segments hold too), one whose strings alone are out of order, one that
    starts past its first end. Every string is its own range of codes in all three call forms, its neighbours' vectors are
    untouched, and nothing is written past the capacity."""
    torch = torch_cuda
    g = np.random.default_rng(5)
    rows = [bytes(g.integers(97, 105, int(g.integers(0, 40)), dtype=np.uint8).tobytes()) for _ in range(3 * 1024)]
    for i in range(0, len(rows), 7):  # escapes
        rows[i] += bytes(g.integers(200, 256, 3, dtype=np.uint8).tobytes())
    offs, data = _strs_from(rows)
    enc = fa.encode_strings(offs.astype(np.uint32), data).copy()
    symbols, page, boff = _string_page(enc)
    eps = enc[page + 16: page + 32].view(np.uint32).astype(np.int64).reshape(2, 2)  # of vectors 1 and 2
    at = page + int(boff[1] + eps[0, 1])
    k = np.arange(1024)
    order = np.array([0, 4, 2, 6, 1, 5, 3, 7])
    place = 128 * (k % 8) + 16 * order[(k // 8) % 8] + k // 64  # string -> transposed position
    stored = enc[at: at + 4096].view(np.uint32).copy()
    e = stored[place].astype(np.int64)
    if ends == "lowered_at_segment_end":
        e[767] = 40
    elif ends == "lowered_inside":
        e[300] = e[290]
    elif ends == "lowered_to_zero":
        e[255:258] = 0
    elif ends == "raised":
        e[511] = e[600]
    else:
        e = g.permutation(e)
    stored[place] = e.astype(np.uint32)
    enc[at: at + 4096] = stored.view(np.uint8)
    start = page + int(boff[0] + eps[0, 0])
    rows[1024:2048] = _decode_vector(symbols, enc[start: page + int(boff[0] + eps[1, 0])], e)
    want_off, want = _strs_from(rows)
    print(f"fsst ends={ends} bytes={want.size}", flush=True)
    plan, d_in, n = fa.Plan(enc, "str"), dev(torch, enc), offs.size - 1
    got_off, got = _fused(torch, plan, d_in, n, want.size)
    np.testing.assert_array_equal(got_off, want_off)
    np.testing.assert_array_equal(got[: want.size], want)
    d_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    plan.string_offsets(d_in.data_ptr(), d_off.data_ptr())
    np.testing.assert_array_equal(d_off.cpu().numpy(), want_off)
    for cap, ok in ((want.size, True), (want.size - 1, False)):
        d_bytes = torch.full((want.size + 65536,), 171, dtype=torch.uint8, device="cuda")
        plan.decode_strings(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), cap)
        assert (d_bytes.cpu().numpy()[cap:] == 171).all()
        if ok:
            plan.check()
            np.testing.assert_array_equal(d_bytes.cpu().numpy()[:cap], want)


def _string_column(symbols_of, vectors):
    """A one-page column of given code streams (1024 rows of bytes a vector) under another column's symbol table."""
    _, page, _ = _string_page(symbols_of)
    k = np.arange(1024)
    place = 128 * (k % 8) + 16 * np.array([0, 4, 2, 6, 1, 5, 3, 7])[(k // 8) % 8] + k // 64
    data, ends, eps = [], [], []
    for v, rows in enumerate(vectors):
        if v:
            eps += [sum(len(d) for d in data), 4096 * v]
        data.append(b"".join(rows))
        e = np.zeros(1024, np.uint32)
        e[place] = np.cumsum([len(r) for r in rows])
        ends.append(e.tobytes())
    n, total = len(vectors), sum(len(d) for d in data)
    head = bytes([7, 1, 0, 0, n & 255, n >> 8, 0, 0]) + np.array([8 + 8 * n, 8 + 8 * n + total, *eps], np.uint32).tobytes()
    return np.frombuffer(symbols_of[:page].tobytes() + head + b"".join(data) + b"".join(ends), np.uint8).copy()


@pytest.mark.parametrize("shape", ["one_run", "dense", "denser", "aligned"])
def test_escape_runs(torch_cuda, shape):
    """Whether a 32-byte piece of a segment starts on an escape's literal depends on the run of 255 bytes before it: one run
    of 200 KB inside a string (and one of odd length), streams of mostly 255 over strings of all lengths, and runs that
    begin and end at string ends on 32-byte and 2 KiB places. All three call forms against the codes' definition."""
    torch = torch_cuda
    g = np.random.default_rng(len(shape))
    words, _ = wl.vocab_strings(1024, seed=2)
    table = fa.encode_strings(words.astype(np.uint32), wl.vocab_strings(1024, seed=2)[1])
    symbols, _, _ = _string_page(table)
    symbols += [bytes([(32774747032022883 >> (8 * b)) & 255 for b in range(8)])] * (255 - len(symbols))  # codes without one

    def stream(n, p):
        b = g.integers(0, 255, n, dtype=np.uint8)
        b[g.random(n) < p] = 255
        return b.tobytes()

    vectors = []
    for v in range(2):
        if shape == "one_run":
            rows = [stream(int(g.integers(0, 30)), 0.05) for _ in range(1024)]
            rows[300 + v], rows[700] = stream(37, 0.1) + b"\xff" * 200_000 + b"abc", b"\xff" * 70_001 + stream(50, 0.2)
        elif shape == "aligned":
            rows = [(b"\xff" if g.random() < 0.8 else b"a") * int(32 * g.integers(0, 4) * (64 if i % 97 == 0 else 1)) for i in range(1024)]
        else:
            p = 0.5 if shape == "dense" else 0.97
            rows = [stream(int(g.integers(0, 120 if i % 50 else 9000)), p) for i in range(1024)]
        vectors.append(rows)
    enc = _string_column(table, vectors)
    want_off, want = _strs_from([r for rows in vectors for r in _decode_vector(
        symbols, np.frombuffer(b"".join(rows), np.uint8), np.cumsum([len(r) for r in rows]))])
    print(f"fsst escape runs {shape}: {enc.size} bytes, {want.size} decoded", flush=True)
    plan, d_in, n = fa.Plan(enc, "str"), dev(torch, enc), want_off.size - 1
    got_off, got = _fused(torch, plan, d_in, n, want.size)
    np.testing.assert_array_equal(got_off, want_off)
    np.testing.assert_array_equal(got[: want.size], want)
    d_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    plan.string_offsets(d_in.data_ptr(), d_off.data_ptr())
    np.testing.assert_array_equal(d_off.cpu().numpy(), want_off)
    d_bytes = empty(torch, want.size)
    plan.decode_strings(d_in.data_ptr(), d_off.data_ptr(), d_bytes.data_ptr(), want.size)
    plan.check()
    np.testing.assert_array_equal(d_bytes.cpu().numpy()[: want.size], want)
