"""Routes of the decoder between the library's kernels and the general path:
what a layer, a norm or a head that differs from the ones setup_cache saw
computes."""
import copy

import pytest
import torch

from spmv_decode_amd.decode.model import Decoder, tiny_config

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


@pytest.mark.gpu
def test_a_layer_put_in_place_after_the_caches_attends_causally(gpu):
    """Its attention reads the mask rows, which the step then has to write."""
    model = decoder()
    model.setup_cache(128, torch.device("cuda"))
    ids = torch.randint(0, 512, (9,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    ref = steps(model, ids)
    layer = copy.deepcopy(model.layers[1])
    del layer.self_attn.decode_kernel  # as a newly made Block
    model.layers[1] = layer
    model.reset_cache()
    close(steps(model, ids), ref)
