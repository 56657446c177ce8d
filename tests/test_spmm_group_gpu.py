"""GPU parity of the grouped small-batch SpMM (nm_spmm_group: bit for bit one
launch per product) and of nm_silu_mul (PyTorch's fp32 SiLU product, bit for
bit)."""
import ctypes

import pytest
import torch

from conftest import say
from spmv_decode_amd import _lib, hip_spmv
from test_gemv_gpu import make_case
from test_spmm_gpu import check_rows

pytestmark = pytest.mark.gpu

# (K, [h...], nnz, m, one launch): products of one kernel, of two configurations, and a lone one
GROUPS = [(4096, [14336, 14336], 32, 64, True), (4096, [4096, 1024, 1024], 32, 64, True),
          (1000, [384, 128, 256, 640], 4, 8, True), (4096, [8192, 1024], 32, 64, False), (12, [128, 256], 3, 4, True)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
def test_small_groups_are_bitwise_single_launches(gpu, dtype):
    code = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}[dtype]
    for K, hs, nnz, m, one in GROUPS:
        mats = [make_case(K, h, nnz, m, seed=K + 3 * h + i, dtype=dtype)[1:] for i, h in enumerate(hs)]
        w = mats[0][0].shape[0]
        for rows in (1, 2, 3, 4, 5, 8):
            say(f"spmm group {dtype} K{K} h{hs} {nnz}:{m} rows {rows}")
            need = _lib.load().nm_spmm_group_workspace_bytes(code, rows, len(hs), (ctypes.c_int * len(hs))(*hs), w,
                                                             nnz, m)
            assert (need > 0) == one
            X = torch.randn(rows, K, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda").to(dtype)
            for _ in range(2):  # the counters are left at zero
                outs = hip_spmv.nmsparse_spmm_group_hip(X, mats, nnz, m)
                for (md, mi), o in zip(mats, outs):
                    assert torch.equal(o, hip_spmv.nmsparse_spmm_forward_hip(X, md, mi, w, md.shape[1], nnz, m))
        check_rows(outs[-1], X, *mats[-1], nnz, m, f"group {dtype} {K}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_silu_mul_is_the_fp32_product(gpu, dtype):
    lib = _lib.load()
    code = 0 if dtype == torch.float16 else 1
    bits = torch.arange(-32768, 32768, device="cuda", dtype=torch.int32).to(torch.int16)
    gate = bits.view(dtype)  # every value of the type, the special ones among them
    for scale in (1.0, 0.37, -3.0, 2.0 ** -14):
        up = torch.full_like(gate, scale)
        for n in (8, 2048, 2056, 65536):
            out = torch.full_like(gate, 5.0)
            _lib.check(lib.nm_silu_mul(code, gate.data_ptr(), up.data_ptr(), out.data_ptr(), n,
                                       torch.cuda.current_stream().cuda_stream), "nm_silu_mul")
            ref = (torch.nn.functional.silu(gate.float()) * up.float()).to(dtype)
            nan = torch.isnan(ref[:n])
            assert torch.equal(torch.isnan(out[:n]), nan)
            assert torch.equal(out[:n][~nan].view(torch.int16), ref[:n][~nan].view(torch.int16))
            assert bool((out[n:] == 5.0).all())
    assert lib.nm_silu_mul(code, gate.data_ptr(), up.data_ptr(), out.data_ptr(), 12, None) == -2
    assert lib.nm_silu_mul(code, gate.data_ptr() + 2, up.data_ptr(), out.data_ptr(), 8, None) == -5
    assert lib.nm_silu_mul(2, gate.data_ptr(), up.data_ptr(), out.data_ptr(), 8, None) == -7


def test_group_refuses_a_vector(gpu):
    """Rows are [..., rows, K], as for one product."""
    mats = [make_case(128, 128, 2, 4, seed=i)[1:] for i in range(2)]
    x = torch.randn(128, device="cuda").half()
    with pytest.raises(ValueError):
        hip_spmv.nmsparse_spmm_forward_hip(x, *mats[0], 64, 128, 2, 4)
    for n in (1, 2):
        with pytest.raises(ValueError):
            hip_spmv.nmsparse_spmm_group_hip(x, mats[:n], 2, 4)
