"""The sparse layer's product and gradients at the edges of its forms: the
row form (few sources, or few of them active), the column form (64 rows of x
at a time), several destination tiles, ragged groups, values other than
spikes; bit for bit against the sequential CPU product, gradients against
float64."""

import numpy as np
import pytest
import scipy.sparse
import torch

from btorch_amd.models import SparseConn
from oracle import rsnn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _matrix(n_src, n_dst, degree, seed):
    rng = np.random.default_rng(seed)
    pre = np.repeat(np.arange(n_src), degree)
    post = rng.integers(0, n_dst, pre.size)
    keep = (pre % 7 != 3) & (post % 11 != 5)   # sources and destinations without edges
    key = np.unique(pre[keep] * n_dst + post[keep])
    w = rng.standard_normal(key.size).astype(np.float32)
    return scipy.sparse.coo_array((w, (key // n_dst, key % n_dst)), shape=(n_src, n_dst))


@pytest.mark.parametrize("n_src,n_dst,degree,rows,prob,backend", [
    (1, 5, 3, 1, 1.0, "native"),
    (200, 1000, 60, 700, 0.05, "native"),       # rows unasked: at most 1024 sources
    (1024, 333, 1500, 3, 0.5, "triton"),        # rows of W longer than a workgroup
    (1025, 40_000, 50, 2, 0.01, "native"),      # three destination tiles
    (1500, 97, 40, 64, 0.01, "native"),         # counted: few active
    (1500, 97, 40, 64, 1.0, "native"),          # counted: all active, columns
    (2000, 130, 70, 65, 0.9, "triton"),         # a second group of one row
    (3000, 16, 8, 1, 0.9, "native"),
    (3000, 777, 100, 129, 0.0, "native"),       # nothing active
])
def test_product_forms_match_sequential_sums(n_src, n_dst, degree, rows, prob, backend):
    mat = _matrix(n_src, n_dst, degree, 5)
    rng = np.random.default_rng(6)
    x = (rng.random((rows, n_src)) < prob) * rng.standard_normal((rows, n_src))
    x = torch.from_numpy(x.astype(np.float32))
    if rows > 1:
        x[rows // 2] = 0.0                       # a row with nothing active
    g = torch.from_numpy(rng.standard_normal((rows, n_dst)).astype(np.float32))
    conn = SparseConn(mat, enforce_dale=False, sparse_backend=backend, device=DEV)
    xd = x.to(DEV).requires_grad_(True)
    y = conn(xd)
    y.backward(g.to(DEV))
    ref = rsnn.NativeSparse(mat)(x)
    assert torch.equal(y.detach().cpu(), ref)
    with torch.no_grad():
        assert torch.equal(conn(xd).cpu(), ref)
    w64 = torch.from_numpy(mat.toarray().astype(np.float64))
    gx = g.double() @ w64.t()
    dst, src = conn.indices.cpu()
    gw = (x.double().t() @ g.double())[src, dst]
    # at most `degree` (gx) and `rows` (gw) products per sum: n * 2^-24 of the
    # sum of their magnitudes bounds a sequential float32 sum
    tol_x = (g.double().abs() @ w64.abs().t()) * (n_dst + 2) * 2.0**-24
    tol_w = (x.double().abs().t() @ g.double().abs())[src, dst] * (rows + 2) * 2.0**-24
    assert ((xd.grad.cpu().double() - gx).abs() <= tol_x).all()
    assert ((conn.magnitude.grad.cpu().double() - gw).abs() <= tol_w).all()


@pytest.mark.parametrize("n_src,n_dst,degree,rows,prob", [
    (1025, 301, 50, 1, 0.3),        # one row: a wavefront per destination
    (1025, 63, 130, 3, 1.0),
    (2100, 33_000, 10, 4, 0.02),    # more destinations than wavefronts
    (1025, 3, 2, 5, 0.01),          # a few rows, fewer destinations than a tile
    (8193, 5000, 300, 5, 0.002),    # tiles over the CUs, a second pass over x
    (8700, 2500, 1100, 6, 0.001),
])
def test_products_of_few_rows_match_sequential_sums(n_src, n_dst, degree, rows, prob):
    mat = _matrix(n_src, n_dst, degree, 7)
    rng = np.random.default_rng(8)
    x = (rng.random((rows, n_src)) < prob) * rng.standard_normal((rows, n_src))
    x = torch.from_numpy(x.astype(np.float32))
    x[:, -1] = 1.5
    conn = SparseConn(mat, enforce_dale=False, device=DEV)
    with torch.no_grad():
        y = conn(x.to(DEV)).cpu()
    assert torch.equal(y, rsnn.NativeSparse(mat)(x))


@pytest.mark.parametrize("n_src,rows", [(1000, 2), (1030, 2)])
def test_product_of_edges_past_int32(n_src, rows):
    # 2^31 edges and more: row offsets past int32 (the arrays are as long, only
    # the last few edges of them, of the last two sources, are read), for rows
    # of x read 1024 and 8192 values at a time; by destination there are none
    from btorch_amd import _lib
    first, n_dst = 2**31 + 5, 8
    row_ptr = torch.full((n_src + 1,), first, dtype=torch.int64, device=DEV)
    row_ptr[-2:] += torch.tensor([3, 5], device=DEV)
    col = torch.empty(first + 5, dtype=torch.int32, device=DEV)
    perm = torch.empty(first + 5, dtype=torch.int64, device=DEV)
    col[first:] = torch.tensor([1, 4, 6, 0, 4], dtype=torch.int32, device=DEV)
    perm[first:] = torch.tensor([2, 0, 4, 1, 3], device=DEV)
    w = torch.tensor([0.5, -1.25, 2.0, 4.0, 8.0], device=DEV)
    x = torch.zeros((rows, n_src), device=DEV)
    x[:, -2:] = torch.tensor([1.0, 3.0], device=DEV)
    y = torch.empty((rows, n_dst), device=DEV)
    lib = _lib.load()
    scratch = torch.empty(lib.btx_product_scratch_bytes(rows, n_src), dtype=torch.uint8, device=DEV)
    csc_ptr = torch.zeros(n_dst + 1, dtype=torch.int64, device=DEV)
    csc_src = torch.zeros(1, dtype=torch.int32, device=DEV)
    _lib.check(lib.btx_product(row_ptr.data_ptr(), col.data_ptr(), perm.data_ptr(),
                               csc_ptr.data_ptr(), csc_src.data_ptr(), w.data_ptr(), n_src,
                               n_dst, first + 5, x.data_ptr(), n_src, rows, y.data_ptr(),
                               scratch.data_ptr(), scratch.numel(), _lib.stream_ptr()),
               "btx_product")
    assert y.cpu().tolist() == [[-3.75, 2.0, 0.0, 0.0, 12.5, 0.0, 8.0, 0.0]] * rows


def test_gradients_use_the_weights_of_the_forward():
    # the weights are edited in place between forward and backward, as by an
    # optimiser step for another loss of the same layer
    mat = _matrix(300, 400, 40, 9)
    rng = np.random.default_rng(10)
    x = torch.from_numpy(((rng.random((6, 300)) < 0.3) * 1.0).astype(np.float32)).to(DEV)
    g = torch.from_numpy(rng.standard_normal((6, 400)).astype(np.float32)).to(DEV)
    conn = SparseConn(mat, enforce_dale=False, device=DEV)

    def grads(edit):
        xd = x.clone().requires_grad_(True)
        conn.magnitude.grad = None
        y = conn(xd)
        if edit:
            with torch.no_grad():
                conn.magnitude.mul_(3.0)
        y.backward(g)
        return xd.grad, conn.magnitude.grad

    want, got = grads(False), grads(True)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])


def test_prepared_weights_stay_those_of_prepare():
    mat = _matrix(300, 400, 40, 9)
    x = torch.ones(2, 300, device=DEV)
    conn = SparseConn(mat, enforce_dale=False, device=DEV)
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            before, packed = conn(x).detach(), conn.packed_weight().detach().clone()
            conn.prepare_sparse()
            with torch.no_grad():
                conn.magnitude.mul_(2.0)
            assert torch.equal(conn(x).detach(), before)
            assert torch.equal(conn.packed_weight().detach(), packed)
            assert torch.equal(conn.effective_weight_f32()[conn._csr_perm], packed)
            conn.finish_sparse()
            assert torch.equal(conn(x).detach(), 2 * before)
    conn.magnitude.grad = None
    conn.prepare_sparse()
    (conn(x) + conn(x)).sum().backward()
    conn.finish_sparse()
    assert torch.equal(conn.magnitude.grad, torch.full_like(conn.magnitude, 4.0))


@pytest.mark.parametrize("n_src,n_dst,degree,rows,prob", [
    (300, 41, 8, 4, 1.0),        # a few rows of few sources, by destination
    (700, 900, 30, 6, 1.0),      # few sources, all active: columns
    (5000, 3, 2, 70, 0.5),       # long destinations, their weight gradient in pieces
    (1024, 2000, 25, 64, 0.004),
    (4097, 60, 5, 9, 0.01),      # counted by a workgroup a row
])
def test_product_forms_by_cost_match_sequential_sums(n_src, n_dst, degree, rows, prob):
    test_product_forms_match_sequential_sums(n_src, n_dst, degree, rows, prob, "native")


def test_product_of_groups_that_take_either_form():
    # 67 groups of 64 rows, every third with all sources active (the columns),
    # the others with a few (the rows), the last one ragged
    n_src, n_dst, rows = 900, 90, 66 * 64 + 5
    mat = _matrix(n_src, n_dst, 20, 11)
    rng = np.random.default_rng(12)
    prob = np.where((np.arange(rows) // 64) % 3 == 1, 1.0, 0.002)[:, None]
    x = (rng.random((rows, n_src)) < prob) * rng.standard_normal((rows, n_src))
    x = torch.from_numpy(x.astype(np.float32))
    conn = SparseConn(mat, enforce_dale=False, device=DEV)
    with torch.no_grad():
        y = conn(x.to(DEV)).cpu()
    assert torch.equal(y, rsnn.NativeSparse(mat)(x))


@pytest.mark.parametrize("n_src,n_dst,short,long,rows,prob", [
    (900, 4000, 200, 2600, 14, 0.02),    # short rows of x: 256 threads, edges left after 1280
    (1024, 1500, 300, 900, 7, 0.004),    # the longest short row
    (6000, 400, 20, 390, 130, 0.047),    # 64 threads, edges left after 320, more than a list
    (5001, 60, 20, 40, 130, 0.1),        # 64 threads, few destinations
    (5000, 500, 90, 490, 5, 0.07),       # 256 threads, more than a list
    (4000, 9000, 300, 6000, 6, 0.01),    # 1024 threads, edges left after 5120
    (4000, 400, 390, 390, 6, 0.3),       # 1024 threads, more than a list
    (700, 300, 5, 30, 6, 0.3),           # by destination, four rows and two
    (700, 300, 5, 30, 401, 0.3),         # by destination, the last row alone
])
def test_products_of_short_and_long_sources_match_sequential_sums(n_src, n_dst, short, long,
                                                                  rows, prob):
    rng = np.random.default_rng(13)
    length = np.where(np.arange(n_src) % 50 == 17, long, short)
    length[np.arange(n_src) % 50 == 18] = 0
    length = np.minimum(length, n_dst)
    pre = np.repeat(np.arange(n_src), length)
    post = np.concatenate([rng.permutation(n_dst)[:k] for k in length])
    w = rng.standard_normal(pre.size).astype(np.float32)
    mat = scipy.sparse.coo_array((w, (pre, post)), shape=(n_src, n_dst))
    x = (rng.random((rows, n_src)) < prob) * rng.standard_normal((rows, n_src))
    x = torch.from_numpy(x.astype(np.float32))
    x[:, 17] = 0.5                               # a long source in every row
    conn = SparseConn(mat, enforce_dale=False, device=DEV)
    with torch.no_grad():
        y = conn(x.to(DEV)).cpu()
    assert torch.equal(y, rsnn.NativeSparse(mat)(x))
