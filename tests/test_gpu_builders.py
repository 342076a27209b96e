"""GPU parity of the device graph builders (Graph.from_coo, Graph.transpose,
Graph.destination_index, the materialized Graph.cu_seqlens CSR) against the
CPU oracle.  Integer outputs: bit-exact, including the output dtypes the
reference constructors produce (row_ptr in dst's dtype, col_idx in src's).
"""

import ctypes

import numpy as np
import pytest
import torch

import tiga as tg
from tiga import _native
from oracle import ref

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _eq(t, a):
    return np.array_equal(t.cpu().numpy().astype(np.int64), np.asarray(a, dtype=np.int64))


@pytest.mark.parametrize("src_dtype,dst_dtype", [(torch.int32, torch.int32),
                                                 (torch.int64, torch.int64),
                                                 (torch.int32, torch.int64),
                                                 (torch.int64, torch.int32)])
@pytest.mark.parametrize("n_src,n_dst,E", [(7, 5, 0), (30, 20, 200), (1000, 70000, 300000),
                                           (5000, 3_000_000, 1_000_000)])
def test_from_coo_matches_oracle(src_dtype, dst_dtype, n_src, n_dst, E):
    print(f"from_coo {src_dtype} {dst_dtype} n_src={n_src} n_dst={n_dst} E={E}", flush=True)
    rng = np.random.default_rng(n_dst + E)
    src = rng.integers(0, n_src, E)
    dst = rng.integers(0, n_dst, E)
    dst[: E // 4] = dst[0] if E else 0          # a hub row with many duplicates
    g = tg.Graph.from_coo(torch.as_tensor(src, dtype=src_dtype, device=DEV),
                          torch.as_tensor(dst, dtype=dst_dtype, device=DEV),
                          num_src=n_src, num_dst=n_dst)
    rp, col = g.resolve_csr()
    erp, ecol, _ = ref.from_coo(src, dst, num_src=n_src, num_dst=n_dst)
    assert rp.dtype == dst_dtype and col.dtype == src_dtype
    assert _eq(rp, erp) and _eq(col, ecol)
    assert g.schema.num_src == n_src and g.schema.num_dst == n_dst


def test_from_coo_infers_sizes_and_rejects_out_of_range():
    src = torch.tensor([2, 0, 1, 2], device=DEV)
    dst = torch.tensor([1, 1, 0, 3], device=DEV)
    g = tg.Graph.from_coo(src, dst)
    erp, ecol, ns = ref.from_coo(src.cpu().numpy(), dst.cpu().numpy())
    rp, col = g.resolve_csr()
    assert _eq(rp, erp) and _eq(col, ecol) and g.schema.num_src == ns
    with pytest.raises(ValueError, match="out-of-range destination"):
        tg.Graph.from_coo(src, dst, num_dst=3)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_transpose_and_destination_index_match_oracle(dtype):
    print(f"transpose {dtype}", flush=True)
    rng = np.random.default_rng(11)
    n_src, n_dst, E = 40_000, 25_000, 400_000
    src = rng.integers(0, n_src, E)
    dst = np.sort(rng.integers(0, n_dst, E))
    erp, ecol, _ = ref.from_coo(src, dst, num_src=n_src, num_dst=n_dst)
    g = tg.Graph.from_csr(torch.as_tensor(erp, dtype=dtype, device=DEV),
                          torch.as_tensor(ecol, dtype=dtype, device=DEV), num_src=n_src)
    d = g.destination_index()
    assert d.dtype == torch.int64 and _eq(d, ref.destination_index(erp))
    t = g.transpose()
    trp, tcol, _ = ref.transpose(erp, ecol, n_src)
    rp, col = t.resolve_csr()
    assert rp.dtype == dtype and col.dtype == dtype
    assert _eq(rp, trp) and _eq(col, tcol)
    assert t.schema.num_src == n_dst and t.schema.num_dst == n_src
    # transposing twice sorts every row's sources (stable order by source)
    rp2, col2 = t.transpose().resolve_csr()
    erp2, ecol2, _ = ref.transpose(trp, tcol, n_dst)
    assert _eq(rp2, erp) and _eq(rp2, erp2) and _eq(col2, ecol2)
    order = np.lexsort((ecol, ref.destination_index(erp)))
    assert _eq(col2, ecol[order])


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_varlen_csr_matches_oracle(causal, dtype):
    print(f"varlen csr causal={causal} {dtype}", flush=True)
    rng = np.random.default_rng(5 + causal)
    lengths = rng.integers(0, 300, 24)
    lengths[[0, 5, 6, 23]] = 0                    # empty sequences, leading and trailing
    lengths[9] = 1
    cu = np.concatenate([[0], np.cumsum(lengths)])
    g = tg.Graph.cu_seqlens(torch.as_tensor(cu, dtype=dtype, device=DEV), causal=causal)
    rp, col = g.resolve_csr()
    erp, ecol = ref.cu_seqlens_csr(cu, causal=causal)
    assert rp.dtype == dtype and col.dtype == dtype
    assert _eq(rp, erp) and _eq(col, ecol)
    assert g.num_edges == ecol.size


def test_varlen_csr_single_and_empty():
    g = tg.Graph.triangular(1000, device=DEV)
    rp, col = g.resolve_csr()
    erp, ecol = ref.cu_seqlens_csr([0, 1000])
    assert _eq(rp, erp) and _eq(col, ecol)
    g0 = tg.Graph.cu_seqlens(torch.zeros(3, dtype=torch.int64, device=DEV))
    rp0, col0 = g0.resolve_csr()
    assert _eq(rp0, [0]) and col0.numel() == 0


def test_builders_do_not_use_torch_sorting(monkeypatch):
    """On the GPU the constructors run this library's kernels: the Torch ops
    the reference builds them from are never reached."""
    def refuse(*args, **kwargs):
        raise AssertionError("Torch graph-construction op called on the GPU path")

    src = torch.randint(0, 100, (5000,), device=DEV)
    dst = torch.randint(0, 100, (5000,), device=DEV)
    for name in ("argsort", "bincount", "repeat_interleave"):
        monkeypatch.setattr(torch, name, refuse)
    g = tg.Graph.from_coo(src, dst, num_src=100, num_dst=100)
    g.destination_index()
    g.transpose()
    tg.Graph.cu_seqlens(torch.tensor([0, 7, 20], device=DEV), causal=False).resolve_csr()


@pytest.mark.parametrize("n_rows,n_edges", [
    (1, 5),               # a key of no bits
    (2, 8191),            # one tile less one key
    (64, 8192),           # a full tile, a full 6-bit digit
    (65, 8193),           # a second tile of one key, a 7-bit digit
    (2048, 20_000),       # the widest single pass
    (2049, 64 * 8192 + 1),  # two passes, a second count segment
    (1 << 22, 30_000),    # two widest passes, most rows empty
    ((1 << 22) + 1, 30_000),  # three passes
])
@pytest.mark.parametrize("src_bits,dst_bits,n_src_known", [
    (64, 64, True), (64, 32, False), (32, 64, False), (32, 32, True)])
def test_coo_sort_at_tile_and_digit_edges(n_rows, n_edges, src_bits, dst_bits, n_src_known):
    """The radix sort against a stable argsort, bit for bit: sources as the
    sort's payload (32-bit ones, and 64-bit ones known to be in range) or
    gathered through the permutation; the permutation beside either."""
    print(f"coo sort rows={n_rows} edges={n_edges} {src_bits}/{dst_bits}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(n_edges)
    ints = {32: torch.int32, 64: torch.int64}
    skew = torch.rand(n_edges, device=DEV, generator=g, dtype=torch.float64) ** 3
    dst = (skew * n_rows).to(torch.int64).clamp_(max=n_rows - 1).to(ints[dst_bits])
    n_src = 2**31 - 1
    src = torch.randint(0, n_src, (n_edges,), device=DEV, generator=g).to(ints[src_bits])
    order = torch.argsort(dst, stable=True)
    want_ptr = torch.zeros(n_rows + 1, dtype=torch.int64, device=DEV)
    want_ptr[1:] = torch.cumsum(torch.bincount(dst.long(), minlength=n_rows), 0)
    row_ptr = torch.empty(n_rows + 1, dtype=dst.dtype, device=DEV)
    col = torch.empty_like(src)
    perm = torch.empty(n_edges, dtype=torch.int32, device=DEV)
    ws_bytes = ctypes.c_size_t()
    known = n_src if n_src_known else 0
    _native.call("tgx_coo_to_csr_workspace", known, n_rows, n_edges, ctypes.byref(ws_bytes))
    ws = torch.empty(ws_bytes.value, dtype=torch.uint8, device=DEV)
    for want_perm in (True, False):
        _native.call("tgx_coo_to_csr", src.data_ptr(), src_bits, dst.data_ptr(), dst_bits, known,
                     n_rows, n_edges, row_ptr.data_ptr(), col.data_ptr(),
                     perm.data_ptr() if want_perm else None, ws.data_ptr(), ws_bytes.value,
                     _native.stream_of(dst))
        assert torch.equal(row_ptr.long(), want_ptr)
        assert torch.equal(col, src[order])
        if want_perm:
            assert torch.equal(perm.long(), order)
    # The transpose of the CSR just built: row ids beside the permutation.
    graph = tg.Graph.from_csr(row_ptr, (col.long() % 5000).to(row_ptr.dtype), num_src=5000)
    t = graph._transposed()
    t_order = torch.argsort(graph._col_idx, stable=True)
    rows = torch.repeat_interleave(torch.arange(n_rows, device=DEV), want_ptr.diff())
    assert torch.equal(graph.destination_index(), rows)
    assert torch.equal(t.perm.long(), t_order) and torch.equal(t.col_t.long(), rows[t_order])
    assert torch.equal(t.inv_perm[t.perm.long()].long(), torch.arange(n_edges, device=DEV))
    tr_ptr, tr_col = graph.transpose().resolve_csr()
    assert torch.equal(tr_ptr, t.row_ptr_t.to(tr_ptr.dtype)) and torch.equal(tr_col, t.col_t.to(
        tr_col.dtype))


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_from_coo_range_checks_and_strided_edge_lists(dtype):
    print("from_coo range checks", flush=True)
    pairs = torch.tensor([[0, 3], [2, 1], [4, 3], [1, 0]], dtype=dtype, device=DEV)
    graph = tg.Graph.from_coo(pairs[:, 0], pairs[:, 1], num_src=5, num_dst=4)
    row_ptr, col = graph.resolve_csr()
    assert row_ptr.tolist() == [0, 1, 2, 2, 4] and col.tolist() == [1, 2, 0, 4]
    for src, dst, name in (([0, 5], [0, 1], "src"), ([0, -1], [0, 1], "src"),
                           ([0, 4], [0, 4], "dst"), ([0, 4], [-1, 0], "dst")):
        with pytest.raises(ValueError, match=f"{name} contains an out-of-range"):
            tg.Graph.from_coo(torch.tensor(src, dtype=dtype, device=DEV),
                              torch.tensor(dst, dtype=dtype, device=DEV), num_src=5, num_dst=4)


# Empty rows inside a tile of 2048 edges, to both sides of the 20480 rows from
# which a tile's edges search for their rows: between two of its edges, before
# the first, after the last, at a tile's end, and all over.
@pytest.mark.parametrize("n_rows,at", [
    (20_481, [0, 20_480]), (20_482, [0, 20_481]), (22_528, [4096] * 2048), (30_000, [29_999]),
    (30_000, [0, 0, 0]), (1_000_000, [7] * 2047 + [900_000] * 2 + [999_999]),
    (300_000, list(range(0, 300_000, 101))), (40_000, [5] * 2048 + [39_990] * 2048),
])
@pytest.mark.parametrize("row_bits,out_bits", [(32, 32), (64, 64), (64, 32), (32, 64)])
def test_destination_index_over_gaps(n_rows, at, row_bits, out_bits):
    print(f"destination index gaps rows={n_rows} edges={len(at)}", flush=True)
    ints = {32: torch.int32, 64: torch.int64}
    rows = torch.tensor(at, device=DEV)
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64, device=DEV)
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    row_ptr = row_ptr.to(ints[row_bits])
    out = torch.full((len(at) + 1,), -7, dtype=ints[out_bits], device=DEV)
    _native.call("tgx_destination_index", row_ptr.data_ptr(), row_bits, n_rows, len(at),
                 out.data_ptr(), out_bits, _native.stream_of(out))
    assert torch.equal(out[:-1].long(), rows) and int(out[-1]) == -7


def test_destination_index_does_not_walk_gaps():
    """Four million empty rows between two edges of one tile take a time of
    the order of what the same rows of 4 edges each take."""
    print("destination index gap time", flush=True)
    n_rows = 4_000_000
    times = []
    for gap in (False, True):
        degree = torch.zeros(n_rows, dtype=torch.int64, device=DEV)
        if gap:
            degree[0] = degree[-1] = 2_000
        else:
            degree += 4
        row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64, device=DEV)
        row_ptr[1:] = torch.cumsum(degree, 0)
        E = int(row_ptr[-1])
        out = torch.empty(E, dtype=torch.int64, device=DEV)
        best = float("inf")
        for _ in range(10):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            _native.call("tgx_destination_index", row_ptr.data_ptr(), 64, n_rows, E,
                         out.data_ptr(), 64, _native.stream_of(out))
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        times.append(best)
    print("   16M edges, 4,000 edges about a gap, ms:", times, flush=True)
    # (A hundred times as long before.)
    assert times[1] <= 5 * times[0]


def test_destination_index_of_more_rows_than_int32():
    """64-bit row ids past 2^31 - 1 rows; 32-bit ones are refused."""
    print("destination index past 2^31 rows", flush=True)
    n_rows = 2**31 + 5
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64, device=DEV)
    row_ptr[-2:] = torch.tensor([2, 5], device=DEV)
    out = torch.empty(5, dtype=torch.int64, device=DEV)
    args = (row_ptr.data_ptr(), 64, n_rows, 5, out.data_ptr())
    _native.call("tgx_destination_index", *args, 64, _native.stream_of(out))
    assert out.tolist() == [n_rows - 2] * 2 + [n_rows - 1] * 3
    with pytest.raises(RuntimeError, match="row ids overflow int32"):
        _native.call("tgx_destination_index", *args, 32, _native.stream_of(out))
    del row_ptr
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n_rows,n_edges", [(1, 3), (2048, 8193), ((1 << 22) + 1, 20_000)])
@pytest.mark.parametrize("src_bits", [32, 64])
def test_coo_sources_are_moved_as_they_are(n_rows, n_edges, src_bits):
    """tgx_coo_to_csr takes its n_src for nothing: any source, 64-bit ones past
    2^31 and negative ones among them, arrives whole.  tgx_coo_to_csr_in_range
    gives the same for sources in range."""
    print(f"coo sources rows={n_rows} edges={n_edges} {src_bits}", flush=True)
    ints = {32: torch.int32, 64: torch.int64}
    g = torch.Generator(device=DEV).manual_seed(n_edges)
    top = 2 ** (src_bits - 1) - 1
    dst = torch.randint(0, n_rows, (n_edges,), device=DEV, generator=g)
    order = torch.argsort(dst, stable=True)
    ws_bytes = ctypes.c_size_t()
    _native.call("tgx_coo_to_csr_workspace", 5, n_rows, n_edges, ctypes.byref(ws_bytes))
    ws = torch.empty(ws_bytes.value, dtype=torch.uint8, device=DEV)
    row_ptr = torch.empty(n_rows + 1, dtype=torch.int64, device=DEV)
    for name, low, high, n_src in (("tgx_coo_to_csr", -top - 1, top, 5),
                                   ("tgx_coo_to_csr", 0, 5, 0),
                                   ("tgx_coo_to_csr_in_range", 0, 2**31 - 1, 2**31 - 1),
                                   ("tgx_coo_to_csr_in_range", 0, top, top)):
        src = torch.randint(low, high, (n_edges,), device=DEV, generator=g).to(ints[src_bits])
        src[-1] = high - 1
        for perm in (None, torch.empty(n_edges, dtype=torch.int32, device=DEV)):
            col = torch.empty_like(src)
            _native.call(name, src.data_ptr(), src_bits, dst.data_ptr(), 64, n_src, n_rows,
                         n_edges, row_ptr.data_ptr(), col.data_ptr(),
                         None if perm is None else perm.data_ptr(), ws.data_ptr(),
                         ws_bytes.value, _native.stream_of(dst))
            assert torch.equal(col, src[order])
            assert perm is None or torch.equal(perm.long(), order)


def test_transpose_checks_what_a_caller_may_have_changed():
    """destination_index() hands out the graph's cached row ids, and a graph
    takes any integer as its source count: a transpose refuses row ids out of
    range and counts that from_coo refuses."""
    print("transpose checks", flush=True)
    row_ptr = torch.tensor([0, 2, 3], device=DEV)
    col = torch.tensor([0, 1, 1], device=DEV)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=2)
    graph.destination_index()[1] = 2**40
    with pytest.raises(ValueError, match="src contains an out-of-range"):
        graph.transpose()
    with pytest.raises(ValueError, match="num_dst must be a non-negative integer"):
        tg.Graph.from_csr(row_ptr, col, num_src=np.int64(2)).transpose()
    assert tg.Graph.from_csr(row_ptr, col, num_src=2).transpose().resolve_csr()[1].tolist() == \
        [0, 0, 1]
