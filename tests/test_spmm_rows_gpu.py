"""GPU parity of the matrix-core product for any number of rows (nm_spmm_rows)
and of the gathers through LDS: against the oracle bar at ragged depths (a last
chunk shorter than 64 columns, a single chunk, fewer chunks than splits), row
counts at the edges of its 128-row tiles, every split count, groups of products
of different widths, the SiLU-product input, and masks that name positions of
another group or outside x; and infinite weights at the end of a ragged depth."""
import ctypes

import pytest
import torch

from conftest import say
from spmv_decode_amd import _lib, hip_spmv
from test_gemv_gpu import make_case
from test_spmm_gpu import check_rows

pytestmark = pytest.mark.gpu

# (K, [h...], nnz, m): w of 500, 24, 2048, 1024, 1280 columns
SHAPES = [(1000, [384], 4, 8), (48, [128, 256], 2, 4), (4096, [1024, 128, 384], 32, 64), (2048, [1280], 64, 128),
          (1792, [640], 5, 7)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_rows_products(gpu, dtype, shape):
    K, hs, nnz, m = shape
    cases = [make_case(K, h, nnz, m, seed=K + 5 * h + i, dtype=dtype) for i, h in enumerate(hs)]
    mats = [(md, mi) for _, md, mi in cases]
    w = mats[0][0].shape[0]
    for rows in (1, 17, 127, 128, 129, 200, 257):
        X = torch.randn(rows, K, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda").to(dtype)
        for splits in (0, 1, 2, 3, 8):
            say(f"spmm rows {dtype} K{K} h{hs} {nnz}:{m} rows {rows} splits {splits} "
                f"-> {_lib.spmm_rows_plan(rows, hs, w, nnz, m, splits)}")
            outs = [torch.full((rows, h), 7.0, dtype=dtype, device="cuda") for h in hs]
            hip_spmv._spmm_rows(X, mats, w, nnz, m, outs, splits=splits)
            first = [o.clone() for o in outs]
            hip_spmv._spmm_rows(X, mats, w, nnz, m, outs, splits=splits)
            for (md, mi), o, f in zip(mats, outs, first):
                check_rows(o, X, md, mi, nnz, m, f"rows {dtype} {K}x{md.shape[1]} r{rows} s{splits}")
                assert torch.equal(o, f)  # splits are summed in order


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_rows_products_tall_tiles(gpu, dtype, shape):
    """The 256-row tiles at their edges; both tile heights add a split's
    products in the same order, so their results are the same bits."""
    K, hs, nnz, m = shape
    cases = [make_case(K, h, nnz, m, seed=K + 5 * h + i, dtype=dtype) for i, h in enumerate(hs)]
    mats = [(md, mi) for _, md, mi in cases]
    w = mats[0][0].shape[0]
    for rows in (1, 129, 255, 256, 257, 500):
        X = torch.randn(rows, K, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda").to(dtype)
        for splits in (1, 2, 3, 8):
            say(f"spmm rows tall {dtype} K{K} h{hs} {nnz}:{m} rows {rows} splits {splits}")
            outs, short = ([torch.full((rows, h), 7.0, dtype=dtype, device="cuda") for h in hs] for _ in range(2))
            hip_spmv._spmm_rows(X, mats, w, nnz, m, outs, splits=_lib.NM_ROWS_TALL + splits)
            hip_spmv._spmm_rows(X, mats, w, nnz, m, short, splits=_lib.NM_ROWS_SHORT + splits)
            for (md, mi), o, f in zip(mats, outs, short):
                check_rows(o, X, md, mi, nnz, m, f"tall {dtype} {K}x{md.shape[1]} r{rows} s{splits}")
                assert torch.equal(o, f)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_rows_silu_product(gpu, dtype):
    """The product formed in the gather is PyTorch's fp32 one, bit for bit, on
    every path (library GEMM, nm_spmm_rows), so the outputs are those of the
    product formed first."""
    for K, h, nnz, m, rows in ((14336, 4096, 32, 64, 200), (3072, 1024, 16, 32, 300), (1000, 384, 4, 8, 140)):
        _, md, mi = make_case(K, h, nnz, m, seed=K + h, dtype=dtype)
        w = md.shape[0]
        gen = torch.Generator(device="cuda").manual_seed(rows)
        gate = (4 * torch.randn(rows, K, generator=gen, device="cuda")).to(dtype)
        up = torch.randn(rows, K, generator=gen, device="cuda").to(dtype)
        gate[0, :6] = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -120.0, 60000.0]).to(dtype)
        act = (torch.nn.functional.silu(gate.float()) * up.float()).to(dtype)
        wp = (w + 7) // 8 * 8
        got, ref = (torch.empty(rows, wp, dtype=dtype, device="cuda") for _ in range(2))
        lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
        code = 0 if dtype == torch.float16 else 1
        _lib.check(lib.nm_gather_columns_silu_mul(code, gate.data_ptr(), up.data_ptr(), K, rows, mi.data_ptr(), w, nnz,
                                                  m, got.data_ptr(), wp, st), "silu")
        _lib.check(lib.nm_gather_columns(code, act.data_ptr(), K, rows, mi.data_ptr(), w, nnz, m, ref.data_ptr(), wp,
                                         st), "gather")
        assert torch.equal(got.view(torch.int16)[1:], ref.view(torch.int16)[1:])
        assert torch.equal(torch.nan_to_num(got[0]), torch.nan_to_num(ref[0]))
        a, b = (hip_spmv.nmsparse_spmm_silu_mul_hip(gate[1:], up[1:], md, mi, w, h, nnz, m),
                hip_spmv.nmsparse_spmm_forward_hip(act[1:], md, mi, w, h, nnz, m))
        assert torch.equal(a, b)
        check_rows(a, act[1:], md, mi, nnz, m, f"silu rows {dtype} {K}x{h} r{rows}")


# (K, nnz, m, rows): through LDS (gathered elements >= 2^21, windows within its width, aligned rows) and its neighbours
GATHERS = [(4096, 32, 64, 1030), (5120, 2, 4, 900), (16384, 1, 4, 530), (4200, 5, 7, 800), (32768, 128, 256, 130),
           (8200, 4, 8, 520), (8196, 2, 4, 520), (1024, 64, 128, 4100)]


@pytest.mark.parametrize("case", GATHERS, ids=str)
def test_large_gathers_are_index_selects(gpu, case):
    K, nnz, m, rows = case
    w = K // m * nnz
    gen = torch.Generator(device="cuda").manual_seed(K)
    X = torch.randn(rows, K, generator=gen, device="cuda").half()
    masks = [torch.rand(K // m, m, generator=gen, device="cuda").argsort(1)[:, :nnz].sort(1).values.to(torch.uint8),
             torch.randint(0, 256, (K // m, nnz), generator=gen, device="cuda", dtype=torch.uint8)]  # foreign positions
    wp = (w + 7) // 8 * 8 + 72
    for mi in masks:
        for shift in (0, 1):  # a mask that does not start at an 8-byte boundary
            buf = torch.zeros(w + 8, dtype=torch.uint8, device="cuda")
            buf[shift:shift + w] = mi.reshape(-1)
            idx = buf[shift:shift + w]
            out = torch.full((rows, wp), 3.0, device="cuda").half()
            say(f"gather K{K} {nnz}:{m} rows {rows} shift {shift}")
            _lib.check(_lib.load().nm_gather_columns(0, X.data_ptr(), K, rows, idx.data_ptr(), w, nnz, m,
                                                     out.data_ptr(), wp, torch.cuda.current_stream().cuda_stream), "g")
            pos = (torch.arange(w, device="cuda") // nnz) * m + mi.reshape(-1).long()
            ref = torch.where(pos < K, X.index_select(1, pos.clamp(max=K - 1)), torch.zeros((), device="cuda").half())
            assert torch.equal(out[:, :w], ref)
            assert bool((out[:, w:] == 0).all())


def test_rows_route_and_arguments(gpu):
    """Routes agree with each other's results (the oracle bar on both sides of
    each line of rows_route), and what nm_spmm_rows refuses is refused."""
    for K, hs, rows, own in ((4096, [4096, 1024, 1024], 159, False), (4096, [4096, 1024, 1024], 160, True),
                             (4096, [14336, 14336], 512, True), (4096, [14336, 14336], 513, False),
                             (256, [18432, 18432], 512, True), (256, [18560, 18432], 512, False),
                             (14336, [4096], 768, True), (14336, [4096], 769, False), (4096, [1024], 300, False),
                             (4096, [4096], 300, False)):
        assert hip_spmv.rows_route(rows, K // 2, hs) == own
        mats = [make_case(K, h, 32, 64, seed=K + h + i)[1:] for i, h in enumerate(hs)]
        X = torch.randn(rows, K, device="cuda").half()
        for (md, mi), o in zip(mats, hip_spmv.nmsparse_spmm_group_hip(X, mats, 32, 64)):
            check_rows(o, X, md, mi, 32, 64, f"route {K} {hs} {rows}")
    lib = _lib.load()
    h = (ctypes.c_int * 1)(256)
    one = (ctypes.c_void_p * 1)(X.data_ptr())
    stride = (ctypes.c_longlong * 1)(256)
    need = lib.nm_spmm_rows_scratch_bytes(200, 1, h, 64, 2, 4, 0)
    assert need > 0 and lib.nm_spmm_rows_scratch_bytes(0, 1, h, 64, 2, 4, 0) == 0
    assert lib.nm_spmm_rows_scratch_bytes(200, 1, (ctypes.c_int * 1)(200), 64, 2, 4, 0) == 0

    def call(dtype=0, x=X.data_ptr(), up=None, stride_x=128, rows=200, n=1, out=one, scratch=X.data_ptr(), nbytes=need,
             ws=X.data_ptr(), w=64, splits=0):
        return lib.nm_spmm_rows(dtype, x, up, stride_x, rows, n, one, one, out, stride, h, scratch, nbytes, ws, 1 << 20,
                                w, 2, 4, splits, None)

    assert call(dtype=2) == -7 and call(x=None) == -1 and call(stride_x=127) == -2 and call(rows=0) == -2
    assert call(w=63) == -4 and call(splits=9) == -7 and call(nbytes=need - 1) == -6
    assert call(scratch=X.data_ptr() + 16) == -5 and call(out=(ctypes.c_void_p * 1)(X.data_ptr() + 2)) == -5


# compressed columns: last chunks of 8 and 32 columns behind 0 to 6 whole ones (every stage of both rings), and of 24 to 62
DEPTHS = [64 * k + r for k in range(7) for r in (8, 32)] + [24, 500, 62, 254]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("w", DEPTHS)
def test_ragged_last_chunks_of_an_infinite_last_row(gpu, dtype, w):
    """Rows of the last chunk past the split hold copies of its last weight row
    until they are cleared: an infinite one there, times the zero activations
    behind it, would turn the outputs to NaN. They are +-Inf, and the others
    the bits of finite weights."""
    rows, h = 150, 256
    _, md, mi = make_case(2 * w, h, 2, 4, seed=w, dtype=dtype)
    X = torch.randn(rows, 2 * w, generator=torch.Generator(device="cuda").manual_seed(w), device="cuda").to(dtype)
    last = X[:, (w - 1) // 2 * 4 + int(mi.view(-1)[-1])].float()
    assert bool((last != 0).all())
    bad = md.clone()
    bad[-1, ::7] = float("inf")
    finite = torch.ones(h, dtype=torch.bool, device="cuda")
    finite[::7] = False
    for height in (_lib.NM_ROWS_SHORT, _lib.NM_ROWS_TALL):
        for splits in (1, 2, 3):
            say(f"ragged {dtype} w {w} height {height} splits {splits}")
            plain, got = (torch.full((rows, h), 7.0, dtype=dtype, device="cuda") for _ in range(2))
            hip_spmv._spmm_rows(X, [(md, mi)], w, 2, 4, [plain], splits=height + splits)
            hip_spmv._spmm_rows(X, [(bad, mi)], w, 2, 4, [got], splits=height + splits)
            check_rows(plain, X, md, mi, 2, 4, f"ragged {dtype} {w}")
            assert torch.equal(got[:, finite], plain[:, finite])
            assert torch.equal(got[:, ~finite].float(), (last * float("inf"))[:, None].expand(-1, int((~finite).sum())))
