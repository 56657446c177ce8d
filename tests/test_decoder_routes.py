"""Routes of the decoder between the library's kernels and the general path:
what a layer, a norm or a head that differs from the ones setup_cache saw
computes."""
import copy

import pytest
import torch
import torch.autograd.forward_ad as fw

from spmv_decode_amd.decode.model import Attention, Decoder, RMSNorm, attend, rotate, tiny_config

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


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["step", "prefill"])
def test_forward_mode_tangents_of_the_head(gpu, call):
    """Logits are linear in the head's weight: its tangent 2 W gives 2 logits."""
    model = decoder()
    model.setup_cache(128, torch.device("cuda"))
    token, pos = torch.tensor([[3]], device="cuda"), torch.tensor([0], device="cuda")

    def run():
        with torch.no_grad():
            return model.forward_step(token, pos) if call == "step" else model.prefill(token.view(-1))

    plain, w = run(), model.lm_head.weight
    with fw.dual_level():
        del model.lm_head._parameters["weight"]
        model.lm_head.weight = fw.make_dual(w.detach().clone(), 2 * w.detach())
        tangent = fw.unpack_dual(run()).tangent
    assert tangent is not None
    close(tangent, 2 * plain)


@pytest.mark.gpu
def test_forward_mode_tangents_of_the_values(gpu):
    """The attention of a step is linear in its values, here those of a full
    cache's last position: their tangents 2 V give 2 y."""
    from spmv_decode_amd.decode.model import attention_core

    model = decoder(qk_norm=False)
    model.setup_cache(128, torch.device("cuda"))
    at, c = model.layers[0].self_attn, model.cfg
    qd, kvd = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    qkv = torch.randn(1, qd + 2 * kvd, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).half()
    pos = torch.tensor([127], device="cuda")  # every slot attended to: a mask row of zeros

    def run(qkv):
        with torch.no_grad():
            return attention_core(at, qkv, model.rope.index_select(0, pos), model.k_cache_t[0].clone(),
                                  model.v_cache_t[0].clone(), pos, model.q_pad.clone(), model.zero)

    plain = run(qkv)
    seed = torch.zeros_like(qkv)
    seed[:, qd + kvd:] = 2 * qkv[:, qd + kvd:]
    with fw.dual_level():
        tangent = fw.unpack_dual(run(fw.make_dual(qkv, seed))).tangent
    assert tangent is not None
    close(tangent, 2 * plain)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("form", ["transposed", "shifted"])
def test_compiled_step_with_a_head_the_kernel_does_not_take(request, device, form):
    """A head weight of other strides or alignment than setup_cache saw: a
    compiled step, which checks nothing when traced, multiplies it all the same."""
    if device == "cuda":
        request.getfixturevalue("gpu")
    model = decoder(device, torch.float32 if device == "cpu" else torch.float16)
    model.setup_cache(128, torch.device(device), model.lm_head.weight.dtype)
    assert model.head_kernel == (device == "cuda")
    model.head_kernel = True
    w = model.lm_head.weight
    if form == "transposed":
        w.data = w.data.t().contiguous().t()
    else:
        buf = torch.empty(w.numel() + 1, device=device, dtype=w.dtype)[1:].view_as(w)
        w.data = buf.copy_(w.data)
    token, pos = torch.tensor([[3]], device=device), torch.tensor([0], device=device)
    with torch.no_grad():
        ref = model.forward_step(token, pos)
        got = torch.compile(model.forward_step, backend="eager", fullgraph=True)(token, pos)
    close(got, ref)


class Wrapped(torch.nn.Module):
    def __init__(self, layer):
        super().__init__()
        self.layer = layer

    def forward(self, *args):
        return self.layer(*args)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("wrap", [Wrapped, lambda layer: torch.compile(layer, backend="eager")],
                         ids=["module", "compiled"])
def test_wrapped_layers_take_caches(request, device, wrap):
    if device == "cuda":
        request.getfixturevalue("gpu")
    dtype = torch.float32 if device == "cpu" else torch.float16
    model = decoder(device, dtype)
    model.setup_cache(128, torch.device(device), dtype)
    ids = torch.arange(9, device=device)
    ref = steps(model, ids, device)
    model.layers[0] = wrap(model.layers[0])
    model.setup_cache(128, torch.device(device), dtype)
    close(steps(model, ids, device), ref)


class MaskReader(Attention):
    """Attention written for the caches' documented layout, mask row included."""

    def forward(self, x, freqs, k_cache_t, v_cache_t, pos, q_pad, zero):
        c = self.cfg
        q, k, v = (p(x).view(-1, c.head_dim) for p in (self.q_proj, self.k_proj, self.v_proj))
        q_pad[:, :c.head_dim] = rotate(q, freqs)
        k_cache_t[:, :c.head_dim].index_copy_(2, pos, rotate(k, freqs).unsqueeze(-1))
        v_cache_t.index_copy_(2, pos, v.unsqueeze(-1))
        return self.o_proj(attend(q_pad, k_cache_t, v_cache_t, c, zero).view(1, 1, -1))


@pytest.mark.gpu
def test_an_attention_class_of_its_own_finds_the_mask_rows_written(gpu):
    model = decoder()
    model.setup_cache(128, torch.device("cuda"))
    ref = steps(model, prompt())
    for blk in model.layers:
        blk.self_attn.__class__ = MaskReader
    model.setup_cache(128, torch.device("cuda"))
    close(steps(model, prompt()), ref)


@pytest.mark.gpu
def test_a_decoder_without_layers(gpu):
    model = decoder(n_layers=0)
    model.setup_cache(128, torch.device("cuda"))
    token = torch.tensor([[3]], device="cuda")
    with torch.no_grad():
        y = model.forward_step(token, torch.tensor([0], device="cuda"))
        ref = model.norm(model.embed_tokens(token)).double().view(1, -1) @ model.lm_head.weight.double().t()
    close(y, ref, 2.0 ** -10)  # one rounding
    close(model.prefill(token.view(-1)), ref, 2.0 ** -10)


@pytest.mark.gpu
def test_a_dense_prompt_compiles_whole(gpu):
    model = decoder(qk_norm=True)
    model.setup_cache(128, torch.device("cuda"))
    ref, keys = model.prefill(prompt()), model.k_store.clone()
    got = torch.compile(model.prefill, backend="eager", fullgraph=True)(prompt())
    close(got, ref)
    close(model.k_store[:, :, :64, :9], keys[:, :, :64, :9])


@pytest.mark.gpu
@pytest.mark.parametrize("P", [3072, 3073])
def test_long_prompts_take_the_faster_attention(gpu, monkeypatch, P):
    """Both sides of the length at which PyTorch's attention is faster (4 heads
    over 2 of 64: 3072 positions) agree."""
    from spmv_decode_amd.decode import model as dm

    model = decoder(n_layers=1)
    model.setup_cache(3200, torch.device("cuda"))
    calls = []
    plain = dm.causal_attention
    monkeypatch.setattr(dm, "causal_attention", lambda *a: calls.append(1) or plain(*a))
    got = model.prefill(prompt(P))
    assert len(calls) == (P > 3072)
    monkeypatch.setattr(dm, "prompt_kernel_positions", lambda *a: 0 if P == 3072 else 1 << 20)
    close(got, model.prefill(prompt(P)))


@pytest.mark.gpu
def test_tuning_reports_the_products_that_run(gpu):
    """The head decodes in its own GEMV: neither BLAS form of it is timed or reported."""
    model = decoder()
    report = model.tune_dense_gemv(reps=2, warmup=1)
    assert report and "512x256" not in report
    with pytest.raises(KeyError):
        model.gemv_forms[512, 256]
    model.setup_cache(128, torch.device("cuda"))
    assert model.head_kernel
    odd = decoder()
    odd.lm_head.weight.data = odd.lm_head.weight.data.t().contiguous().t()
    assert "512x256" in odd.tune_dense_gemv(reps=2, warmup=1)
