"""GPU parity of the dense GEMV of the output head (nm_dense_gemv) against the
product in 64 bits, at every kernel's K range and its edges, and row counts
around a step of the grid."""
import pytest
import torch

from conftest import say
from spmv_decode_amd import _lib, hip_spmv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_dense_gemv_matches_exact(gpu, dtype):
    for K in (8, 504, 512, 520, 1024, 2048, 2056, 3072, 4096, 5120, 5128, 8192):
        for n in (1, 7, 33, 1000, 16391):
            gen = torch.Generator(device="cuda").manual_seed(K + n)
            pad = 8 if n == 33 else 0
            w = (torch.randn(n, K + pad, device="cuda", generator=gen) * K ** -0.5).to(dtype)[:, :K]
            x = torch.randn(1, K, device="cuda", generator=gen).to(dtype)
            say(f"dense gemv {dtype} {n}x{K}")
            y = hip_spmv.nmsparse_dense_gemv(x, w).double()
            ref = x.double() @ w.double().t()
            # fp32 sums of K products (4 sqrt(K) 2^-24 of their magnitudes), then one rounding
            bar = (4 * K ** 0.5 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
                   + torch.finfo(dtype).eps / 2 * ref.abs() + 2.0 ** -25)
            assert bool(((y - ref).abs() <= bar).all()), (K, n)


def test_dense_gemv_special_values_and_refusals(gpu):
    w = torch.ones(40, 1032, device="cuda").half()
    w[3, 5] = float("inf")
    w[4, 1031] = float("nan")
    y = hip_spmv.nmsparse_dense_gemv(torch.ones(1, 1032, device="cuda").half(), w)[0]
    assert torch.isinf(y[3]) and torch.isnan(y[4]) and bool((y[[0, 1, 2, 5, 39]] == 1032).all())
    w[:, :8] = float("inf")  # lanes past a short row read its start
    z = hip_spmv.nmsparse_dense_gemv(torch.cat([torch.ones(1, 8), torch.zeros(1, 1024)], 1).cuda().half(), w)
    assert bool(torch.isinf(z[0, :3]).all())
    x = torch.ones(1, 64, device="cuda").half()
    for xb, wb in ((x.float(), w[:, :64].float()), (x[:, :60], w[:, :60]), (x, w[:, 4:68]), (x.bfloat16(), w[:, :64]),
                   (x.expand(2, 64), w[:, :64]), (x.cpu(), w[:, :64].cpu())):
        assert not hip_spmv.dense_gemv_supported(xb, wb)
        with pytest.raises(ValueError):
            hip_spmv.nmsparse_dense_gemv(xb, wb)
    lib = _lib.load()
    assert lib.nm_dense_gemv(0, x.data_ptr(), w.data_ptr(), 1032, y.data_ptr(), 40, 8200, None) == -2
    assert lib.nm_dense_gemv(2, x.data_ptr(), w.data_ptr(), 1032, y.data_ptr(), 40, 64, None) == -7
    assert lib.nm_dense_gemv(0, None, w.data_ptr(), 1032, y.data_ptr(), 40, 64, None) == -1


def test_decode_step_keeps_the_heads_gradient(gpu):
    """Where autograd records the output head, a decode step takes the
    differentiable product: the weight gets its gradient, the logits are those
    of the step without gradients to fp16 rounding."""
    from dataclasses import replace

    from spmv_decode_amd.decode.model import CONFIGS, Decoder

    cfg = replace(CONFIGS["qwen3-0.6b"], n_layers=1, vocab=520)
    torch.manual_seed(0)
    model = Decoder(cfg).to("cuda", torch.float16).requires_grad_(False)
    model.lm_head.weight.requires_grad_(True)
    model.setup_cache(64, torch.device("cuda"))
    assert model.head_kernel
    token, pos = torch.tensor([[3]], device="cuda"), torch.tensor([0], device="cuda")
    with torch.no_grad():
        plain = model.forward_step(token, pos).double()
    hidden = {}
    model.norm.register_forward_hook(lambda m, a, out: hidden.setdefault("x", out.detach()))
    logits = model.forward_step(token, pos)
    # one rounding each
    assert float((logits.double() - plain).norm() / plain.norm()) <= 2 * 2.0 ** -11
    seed = torch.randn_like(logits)
    grad, = torch.autograd.grad(logits, model.lm_head.weight, seed)
    ref = seed.double().t() @ hidden["x"].double().view(1, -1)
    assert float((grad.double() - ref).norm() / ref.norm()) <= 2.0 ** -10


def test_head_takes_a_replaced_weight(gpu):
    """A head whose weight the kernel does not take goes to the general product."""
    from spmv_decode_amd.decode.model import project_head

    head = torch.nn.Linear(64, 24, bias=False, device="cuda", dtype=torch.float16).requires_grad_(False)
    head.weight.data = torch.randn(64, 24, device="cuda", dtype=torch.float16).t()
    x = torch.randn(1, 1, 64, device="cuda", dtype=torch.float16)
    y, ref = project_head(head, x, True).double(), x.view(1, -1).double() @ head.weight.double().t()
    assert float((y - ref).norm() / ref.norm()) <= 2.0 ** -10
