"""GPU parity of the fused residual add and RMSNorm (nm_add_rms_norm): the sum
bit for bit PyTorch's, the norm against 64 bits, at every kernel's width range
and its edges."""
import pytest
import torch

from conftest import say
from spmv_decode_amd import _lib, hip_spmv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_add_rms_norm_matches_exact(gpu, dtype):
    for dim in (8, 1024, 2048, 2056, 4096, 4104, 5120, 6144, 6152, 8192):
        for rows in (1, 3, 301):
            gen = torch.Generator(device="cuda").manual_seed(dim + rows)
            x, d = (torch.randn(2, rows, dim, device="cuda", generator=gen) * 3).to(dtype)
            w = (1 + 0.1 * torch.randn(dim, device="cuda", generator=gen)).to(dtype)
            say(f"add rms norm {dtype} {rows}x{dim}")
            total, out = hip_spmv.nmsparse_add_rms_norm(x, d, w, 1e-6)
            assert torch.equal(total, x + d)
            s = total.double()
            ref = s * torch.rsqrt(s.square().mean(-1, keepdim=True) + 1e-6) * w.double()
            # fp32 arithmetic on sums of 42 and fewer terms, then one rounding
            bar = (torch.finfo(dtype).eps / 2 + 2.0 ** -18) * ref.abs() + 2.0 ** -25
            assert bool(((out.double() - ref).abs() <= bar).all()), (dim, rows)


def test_add_rms_norm_special_values_and_refusals(gpu):
    x = torch.ones(5, 1032, device="cuda").half()
    d, w = torch.zeros_like(x), torch.ones(1032, device="cuda").half()
    x[1, 1031], x[2, 0], x[3], d[3] = float("inf"), float("nan"), 60000.0, 60000.0
    total, out = hip_spmv.nmsparse_add_rms_norm(x, d, w, 1e-5)
    ref = torch.nn.functional.rms_norm(x + d, (1032,), w, 1e-5)
    assert torch.equal(total[0], x[0]) and torch.isinf(total[3]).all()
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(out[[0, 4]], ref[[0, 4]])
    for bad in ((x.float(), d.float(), w.float()), (x[:, :1028], d[:, :1028], w[:1028]), (x, d[:4], w),
                (x, d, w[:1024]), (x, d.bfloat16(), w), (x.cpu(), d.cpu(), w.cpu()), (x[:, :1024], d[:, :1024], w[:1024])):
        assert not hip_spmv.add_rms_norm_supported(*bad)
        with pytest.raises(ValueError):
            hip_spmv.nmsparse_add_rms_norm(*bad, 1e-5)
    args = (x.data_ptr(), d.data_ptr(), w.data_ptr(), 1e-5, total.data_ptr(), out.data_ptr())
    lib = _lib.load()
    assert lib.nm_add_rms_norm(0, *args, 5, 8200, None) == -2
    assert lib.nm_add_rms_norm(2, *args, 5, 1032, None) == -7
    assert lib.nm_add_rms_norm(0, None, *args[1:], 5, 1032, None) == -1
