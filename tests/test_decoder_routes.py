"""Routes of the decoder between the library's kernels and the general path:
what a layer, a norm or a head that differs from the ones setup_cache saw
computes."""
import copy

import pytest
import torch

from spmv_decode_amd.decode.model import Decoder, RMSNorm, tiny_config

# two fp16 paths of a few layers: rounding in another order, each below 2^-11 of its value, over about 40 roundings
REL = 2e-2


def decoder(device="cuda", dtype=torch.float16, seed=0, **cfg):
    torch.manual_seed(seed)
    return Decoder(tiny_config(**cfg)).to(device, dtype).requires_grad_(False)


def close(a, b, rel=REL):
    assert torch.isfinite(a).all() and float((a.double() - b.double()).norm() / b.double().norm()) <= rel


def steps(model, ids, device="cuda"):
    with torch.no_grad():
        return torch.cat([model.forward_step(t.view(1, 1), torch.tensor([i], device=device))
                          for i, t in enumerate(ids)])


def prompt(n=9):
    return torch.randint(0, 512, (n,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))


class Halved(RMSNorm):
    def forward(self, x):
        return super().forward(x) * 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["hook", "pre_hook", "global_hook", "class", "forward", "eps", "one_eps"])
def test_changed_head_norms_in_a_prompt(gpu, change):
    """A prompt's head norms are the modules: the queries and keys of a hooked,
    replaced or differently set one are those of the general path."""
    model = decoder(qk_norm=True)
    model.setup_cache(128, torch.device("cuda"))
    at, handle = model.layers[0].self_attn, None
    if change == "hook":
        at.q_norm.register_forward_hook(lambda m, args, out: out * 0.5)
    elif change == "pre_hook":
        at.k_norm.register_forward_pre_hook(lambda m, args: (args[0] + 1,))
    elif change == "global_hook":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda m, args, out: out * 0.5 if m is at.q_norm else None)
    elif change == "class":
        at.q_norm.__class__ = Halved
    elif change == "forward":
        at.k_norm.forward = lambda x: x * 0.5
    elif change == "eps":
        at.q_norm.eps = at.k_norm.eps = 10.0
    else:
        at.k_norm.eps = 10.0
    try:
        got, keys = model.prefill(prompt()), model.k_cache_t[0][:, :64, :9].clone()
        for blk in model.layers:
            blk.self_attn.decode_kernel = False
        ref = model.prefill(prompt())
    finally:
        if handle is not None:
            handle.remove()
    close(got, ref)
    close(keys, model.k_cache_t[0][:, :64, :9], 2.0 ** -9)  # two roundings against one


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [None, -1e-6])
def test_prompt_norms_of_an_eps_the_kernels_do_not_take(gpu, eps):
    model = decoder(qk_norm=True)
    model.setup_cache(128, torch.device("cuda"))
    for m in model.modules():
        if isinstance(m, RMSNorm):
            m.eps = eps
    got = model.prefill(prompt())
    for blk in model.layers:
        blk.self_attn.decode_kernel = False
    close(got, model.prefill(prompt()))


@pytest.mark.gpu
def test_a_layer_put_in_place_after_the_caches_attends_causally(gpu):
    """Its attention reads the mask rows, which the step then has to write."""
    model = decoder()
    model.setup_cache(128, torch.device("cuda"))
    ids = prompt()
    ref = steps(model, ids)
    layer = copy.deepcopy(model.layers[1])
    del layer.self_attn.decode_kernel  # as a newly made Block
    model.layers[1] = layer
    model.reset_cache()
    close(steps(model, ids), ref)
