"""Layers read the weights they are given: an edit through ``.data``, which moves neither a parameter's
address nor its version counter, reaches the next call of every projection whose weight is not kept as a
cast, and so do weights without a version counter (made in inference mode) and calls on other streams.
"""

from __future__ import annotations

import copy

import pytest
import torch

from nori_amd import ScalableSeqKV
from nori_amd.layer import EncoderBaseLayer, MultiheadAttention, QASSMaxScaling

pytestmark = pytest.mark.gpu


def _normal(module: torch.nn.Module, seed: int, device) -> torch.nn.Module:
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for p in module.parameters():
            p.copy_(torch.empty(p.shape).normal_(0.0, p.shape[-1] ** -0.5 if p.dim() > 1 else 0.1, generator=g))
    return module.eval().to(device)


def _dense_layer(seed, device, embed=128, heads=2):
    return _normal(EncoderBaseLayer(heads, embed, 3 * embed, pre_norm=True, activation="swiglu", norm_type="rmsnorm",
                                    deepnorm_alpha=0.25, layer_arch="smf", seq_attn_isolated=True,
                                    cross_share_all_kv_heads=False, use_qassmax=True, qass_mode="full"), seed, device)


def _after_edit(module, param, call, autocast=torch.float16):
    """(what ``call`` gives after ``param`` is edited through ``.data`` between two calls, what the
    first call gave, what an equal module that never saw the old value gives)."""
    with torch.inference_mode(), torch.autocast("cuda", dtype=autocast):
        before = call(module)
    with torch.no_grad():
        dict(module.named_parameters())[param].data.mul_(-1.5)
    fresh = copy.deepcopy(module)
    for m in fresh.modules():  # no kept cast comes along
        for name in ("_cast", "_stacked", "_mix", "_gate16", "_base16"):
            m.__dict__.pop(name, None)
    with torch.inference_mode(), torch.autocast("cuda", dtype=autocast):
        return call(module), before, call(fresh)


@pytest.mark.parametrize("rows", [60, 5000])
@pytest.mark.parametrize("autocast", [torch.float16, torch.bfloat16])
def test_feature_and_context_attention_read_the_edited_projection(cuda, rows, autocast):
    x = torch.randn(2, rows, 3, 128, generator=torch.Generator().manual_seed(1)).to(cuda)
    feat = _normal(MultiheadAttention(128, 2), 2, cuda)
    got, before, want = _after_edit(feat, "qkv_proj_weight", lambda m: m(x)[0], autocast)
    assert torch.equal(got, want) and not torch.equal(got, before)
    seq = _normal(MultiheadAttention(128, 2, qkv_combined=False), 3, cuda)
    rows_t = x.transpose(1, 2)
    got, before, want = _after_edit(seq, "qkv_proj_weight", lambda m: m.attend(rows_t, rows_t), autocast)
    assert torch.equal(got, want) and not torch.equal(got, before)
    got, before, want = _after_edit(seq, "qkv_proj_weight", lambda m: m.project_kv_cache(rows_t)["kv"], autocast)
    assert torch.equal(got, want) and not torch.equal(got, before)


@pytest.mark.parametrize("part", ["feature_attentions.0.qkv_proj_weight", "sequence_attentions.0.qkv_proj_weight"])
def test_dense_layer_reads_the_edited_projections(cuda, part):
    # the cached apply's feature projection and the cache build's context and feature projections
    x = torch.randn(1, 40, 5, 128, generator=torch.Generator().manual_seed(4)).to(cuda)
    layer = _dense_layer(5, cuda)

    def build(m):
        return m.forward_train_cache(x, quantize_kv_cache=True)[0]

    got, before, want = _after_edit(layer, part, build)
    assert torch.equal(got, want) and not torch.equal(got, before)
    if part.startswith("feature"):
        kv = torch.randn(5, 50, 2, 2, 64, generator=torch.Generator().manual_seed(6)).half().to(cuda)
        cache = {"seq_kv": ScalableSeqKV(kv, 1, 5, quantize=True)}
        got, before, want = _after_edit(layer, part, lambda m: m.forward_test_with_cache(x, cache))
        assert torch.equal(got, want) and not torch.equal(got, before)


def test_cache_projection_of_weights_without_a_version_counter(cuda):
    x = torch.randn(1, 3, 40, 128, generator=torch.Generator().manual_seed(7)).to(cuda)
    with torch.inference_mode():
        made = MultiheadAttention(128, 2, qkv_combined=False).to(cuda)
        plain = torch.nn.functional.linear(x.view(3, 40, 128), made.qkv_proj_weight[1:].reshape(256, 128))
        assert torch.equal(made.project_kv_cache(x)["kv"].view(3, 40, 256), plain)


def test_a_call_on_another_stream_does_not_read_the_first_ones_casts(cuda):
    # the first call's casts wait behind a long kernel on its own stream; a call on another stream
    # must not read what they have not written yet
    x = torch.randn(2, 60, 3, 128, generator=torch.Generator().manual_seed(8)).to(cuda).transpose(1, 2)
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        for call in (lambda m: m.attend(x, x), lambda m: m.project_kv_cache(x)["kv"]):
            attn = _normal(MultiheadAttention(128, 2, qkv_combined=False), 9, cuda)
            torch.cuda.synchronize()
            with torch.cuda.stream(busy):
                torch.cuda._sleep(200_000_000)
                want = call(attn)
            with torch.cuda.stream(other):
                got = call(attn)
            torch.cuda.synchronize()
            assert torch.equal(got, want)


@pytest.mark.parametrize("param", ["base_mlp.0.weight", "base_mlp.0.bias", "base_mlp.2.weight", "base_mlp.2.bias"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_qass_reads_the_edited_base_mlp(cuda, param, dtype):
    module = _normal(QASSMaxScaling(num_heads=2, head_dim=64, qass_mode="full"), 10, cuda).to(dtype)
    q = torch.randn(40, 3, 2, 64, generator=torch.Generator().manual_seed(11)).half().to(cuda)
    got, before, want = _after_edit(module, param, lambda m: m(q, 300))
    assert torch.equal(got, want) and not torch.equal(got, before)


def test_dense_layer_reads_the_edited_base_mlp(cuda):
    x = torch.randn(1, 40, 5, 128, generator=torch.Generator().manual_seed(12)).to(cuda)
    kv = torch.randn(5, 50, 2, 2, 64, generator=torch.Generator().manual_seed(13)).half().to(cuda)
    cache = {"seq_kv": ScalableSeqKV(kv, 1, 5, quantize=True)}
    got, before, want = _after_edit(_dense_layer(14, cuda), "sequence_attentions.1.qassmax.base_mlp.2.bias",
                                    lambda m: m.forward_test_with_cache(x, cache))
    assert torch.equal(got, want) and not torch.equal(got, before)
