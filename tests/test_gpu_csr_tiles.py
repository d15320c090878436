"""CSR products at the edges of their tiles, against the oracle and plain FP64 sums.

The kernel cuts the merged list of row ends and entries into tiles (1024 merged items below 2^22 of
them, 4096 from there on): rows that end on a tile's edge, rows over several tiles, tiles of empty
rows, one row in all, and more tiles than one block of the last kernel takes.  A sum of t terms in
any order differs by at most about t 2^-53 sum|terms|; 1e-13 covers the rows up to 1000 terms, the
longer ones (random signs off: all terms positive) are held to 1e-12 relative.
"""
import numpy as np
import pytest

import oracle
from networkit_amd import capi

pytestmark = pytest.mark.gpu


def csr_of(lengths, cols, seed):
    rng = np.random.default_rng(seed)
    ptr = np.zeros(len(lengths) + 1, np.uint64)
    ptr[1:] = np.cumsum(np.asarray(lengths, np.int64))
    nnz = int(ptr[-1])
    return oracle.CSR(len(lengths), cols, ptr, rng.integers(0, cols, nnz).astype(np.uint64),
                      rng.uniform(0.1, 1.0, nnz))


LENGTHS = {
    "one row": [5000],
    "one long row among empty ones": [0] * 1500 + [9000] + [0] * 1500,
    "all empty but one": [0] * 3000 + [1] + [0] * 3000,
    "ends on tile edges": [1023, 1023, 1022, 1, 0, 1023, 2047, 511, 511],
    "a row of one tile and of several": [1024, 4096, 1, 3 * 1024 - 1, 7],
    "around a wave's rows": [31, 32, 33, 63, 64, 65, 127, 128, 129, 2048, 2049] * 9,
    "short rows": [1] * 5000 + [2] * 5000,
}


@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_products_at_tile_edges(name):
    import torch
    lengths = LENGTHS[name]
    n = len(lengths)
    a = csr_of(lengths, n, 3)
    x = np.random.default_rng(4).random(n)
    ref = oracle.csr_spmv(a, x)
    d = capi.DeviceCSR(a.rows, a.cols, a.row_idx, a.col_idx, a.values)
    xd = torch.from_numpy(x).cuda()
    np.testing.assert_allclose(d.spmv(xd).cpu().numpy(), ref, rtol=1e-12, atol=0)
    y, sq = d.pagerank_step(xd, 0.25)
    np.testing.assert_allclose(y.cpu().numpy(), ref + 0.25, rtol=1e-12, atol=0)
    assert float(sq) == pytest.approx(float(((ref + 0.25 - x) ** 2).sum()), rel=1e-12)
    y2, sq2 = torch.empty_like(y), torch.empty_like(sq)
    d.pagerank_step_noalloc(xd, 0.25, y2, sq2)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(sq, sq2)


@pytest.mark.parametrize("rows,length", [(300000, 15), (1100000, 3), (1000, 70000), (1, 5000000)])
def test_large_tiles(rows, length):
    """Equal rows (so that torch can add them): 4096-item tiles; 70,000,000 entries take the fix
    kernel's many blocks."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows)
    nnz = rows * length
    col = torch.randint(rows, (nnz,), generator=g, device="cuda")
    val = torch.rand(nnz, generator=g, device="cuda", dtype=torch.float64)
    x = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    d = capi.DeviceCSR(rows, rows, torch.arange(rows + 1, device="cuda") * length, col, val)
    ref = (val * x[col]).reshape(rows, length).sum(1)
    y, sq = d.pagerank_step(x, 0.5)
    torch.cuda.synchronize()
    torch.testing.assert_close(y, ref + 0.5, rtol=1e-12, atol=0)
    want = float((ref + 0.5 - x).square().sum())
    assert float(sq) == pytest.approx(want, rel=1e-12)
    z = d.spmv(x)
    torch.cuda.synchronize()
    torch.testing.assert_close(z, ref, rtol=1e-12, atol=0)
    # every run adds in the same order
    y2, sq2 = d.pagerank_step(x, 0.5)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(sq, sq2)


# entries before the first offset and past the last one, in lists of less than a tile up to several
@pytest.mark.parametrize("before,after", [(0, 1), (0, 5000), (1, 0), (700, 0), (2500, 3000)])
@pytest.mark.parametrize("rows,length", [(1, 3), (700, 3), (1023, 1), (5, 2047), (40000, 110)])
def test_lists_longer_than_the_offsets(rows, length, before, after):
    """The offsets say which entries belong to the rows: some rows of a larger matrix, and lists with
    room to spare.  The spare entries would change every sum (values of 1e30), and the vectors lie
    between others that must stay as they are."""
    import torch
    rng = np.random.default_rng(rows + before + after)
    nnz = rows * length
    col, val = np.zeros(before + nnz + after, np.uint64), np.full(before + nnz + after, 1e30)
    col[before:before + nnz] = rng.integers(0, rows, nnz)
    val[before:before + nnz] = rng.uniform(0.1, 1.0, nnz)
    ptr = before + length * np.arange(rows + 1, dtype=np.uint64)
    x = rng.random(rows)
    ref = oracle.csr_spmv(oracle.CSR(rows, rows, ptr - before, col[before:before + nnz], val[before:before + nnz]), x)
    d = capi.DeviceCSR(rows, rows, ptr, col, val)
    room = torch.full((3 * rows,), -7.0, dtype=torch.float64, device="cuda")
    xd, y = torch.from_numpy(x).cuda(), room[rows:2 * rows]
    d.spmv(xd, y)
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy(), ref, rtol=1e-12, atol=0)
    y.fill_(-7.0)
    sq = torch.empty(1, dtype=torch.float64, device="cuda")
    for step in (d.pagerank_step, d.pagerank_step_noalloc):
        step(xd, 0.25, y=y, step_sq=sq)
        torch.cuda.synchronize()
        np.testing.assert_allclose(y.cpu().numpy(), ref + 0.25, rtol=1e-12, atol=0)
        assert float(sq) == pytest.approx(float(((ref + 0.25 - x) ** 2).sum()), rel=1e-12)
    assert torch.all(room[:rows] == -7.0) and torch.all(room[2 * rows:] == -7.0)


def test_rows_over_many_tiles():
    """Runs of carries around what one thread adds (8 tiles of 1024 items) and around a wave's turns
    (64 tiles a load, 256 a turn), each with an ordinary row behind it.  t positive terms in any order
    are within t 2^-53 of their sum, relatively; torch adds them pairwise (within 1e-15)."""
    import torch
    tiles = [6, 7, 8, 9, 10, 63, 64, 65, 66, 255, 256, 257, 258, 320, 511, 512, 513]
    lengths = np.array([x for k in tiles for x in (1024 * k, 3, 1024 * k + 1021)], np.int64)
    n = len(lengths)
    g = torch.Generator(device="cuda").manual_seed(5)
    nnz = int(lengths.sum())
    col = torch.randint(n, (nnz,), generator=g, device="cuda")
    val = torch.rand(nnz, generator=g, device="cuda", dtype=torch.float64)
    x = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    ref = torch.stack([(v * x[c]).sum() for v, c in zip(val.split(lengths.tolist()), col.split(lengths.tolist()))])
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    # below 2^22 items a tile has 1024 of them: the matrix in three parts
    for a, b in ((0, 39), (39, 45), (45, n)):
        k0, k1 = int(ptr[a]), int(ptr[b])
        assert k1 - k0 + b - a < 1 << 22
        d = capi.DeviceCSR(b - a, n, ptr[a:b + 1] - k0, col[k0:k1], val[k0:k1])
        y = d.spmv(x)
        torch.cuda.synchronize()
        tol = torch.from_numpy(lengths[a:b] * 2.0 ** -53 + 1e-15).cuda() * ref[a:b]
        assert torch.all((y - ref[a:b]).abs() <= tol)
    # the same rows in tiles of 4096 items
    d = capi.DeviceCSR(n, n, ptr, col, val)
    y, sq = d.pagerank_step(x, 0.5)
    y2, sq2 = d.pagerank_step(x, 0.5)
    torch.cuda.synchronize()
    assert torch.all((y - 0.5 - ref).abs() <= torch.from_numpy(lengths * 2.0 ** -53 + 1e-15).cuda() * (ref + 0.5))
    assert float(sq) == pytest.approx(float((ref + 0.5 - x).square().sum()), rel=2 * int(lengths.max()) * 2.0 ** -53)
    assert torch.equal(y, y2) and torch.equal(sq, sq2)
