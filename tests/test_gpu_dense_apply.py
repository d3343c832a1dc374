"""A dense layer's cached apply as one native call (nori_dense_apply) against the same layer's own calls.

Both run the same kernels, except that the projections of short operands go through
``nori_linear_f16`` in one and the library GEMM in the other: fp32 sums in another order, so a value
rounded to fp16 can land on its neighbour (2^-11 of it) and moves what follows by as much. Over the
few such roundings of a layer the 2-norm of the difference stays below 4 * 2^-11 of the update's.
"""

from __future__ import annotations

import pytest
import torch

from nori_amd import ScalableSeqKV
from nori_amd.layer import EncoderBaseLayer

pytestmark = pytest.mark.gpu


def _layer(embed, heads, shared, seed, device):
    torch.manual_seed(seed)
    layer = EncoderBaseLayer(heads, embed, 3 * embed, pre_norm=True, activation="swiglu", norm_type="rmsnorm",
                             deepnorm_alpha=0.25, layer_arch="smf", seq_attn_isolated=True,
                             cross_share_all_kv_heads=shared, use_qassmax=True, qass_mode="full")
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, p.shape[-1] ** -0.5 if p.dim() > 1 else 0.1)
    return layer.eval().to(device)


@pytest.mark.parametrize("embed,heads", [(128, 2), (128, 4), (256, 4)])
@pytest.mark.parametrize("tables,rows,groups,keys", [(1, 1, 1, 2), (1, 37, 9, 300), (3, 130, 5, 129), (2, 64, 33, 1024)])
@pytest.mark.parametrize("shared,quantized", [(False, True), (True, True), (False, False)])
def test_native_apply_equals_the_layers_calls(cuda, embed, heads, tables, rows, groups, keys, shared, quantized):
    layer = _layer(embed, heads, shared, embed + heads, cuda)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(tables, rows, groups, embed, generator=g).to(cuda)
    kv = torch.randn(tables * groups, keys, 2, 1 if shared else heads, embed // heads, generator=g).half().to(cuda)
    cache = {"seq_kv": ScalableSeqKV(kv, tables, groups, quantize=quantized)}
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        before = x.clone()
        taken = layer._apply_native(x, cache["seq_kv"], None) is not None
        assert taken == (embed == 128 or layer.mlp[0].fuses(x))
        got = layer.forward_test_with_cache(x, cache)
        layer.native_apply = False
        want = layer.forward_test_with_cache(x, cache)
        assert torch.equal(x, before)
    err = (got - want).double().norm() / (want - x).double().norm()
    assert float(err) <= 4 * 2.0**-11


def test_other_calls_keep_the_layers_own(cuda):
    # what is not the plain inference computation, or what a user watches, is not taken over
    layer = _layer(128, 2, False, 5, cuda)
    x = torch.randn(1, 20, 4, 128, device=cuda)
    kv = torch.randn(4, 50, 2, 2, 64, device=cuda).half()
    cache = ScalableSeqKV(kv, 1, 4, quantize=True)

    def taken(inp=x, c=cache, mask=None):
        return layer._apply_native(inp, c, mask) is not None

    with torch.inference_mode():
        assert not taken()  # fp32 projections
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not taken()
    with torch.autocast("cuda", dtype=torch.float16):
        assert not taken()  # gradients
        with torch.inference_mode():
            assert taken()
            assert not taken(x.half()) and not taken(x.transpose(1, 2)) and not taken(c={"kv": kv, "batch": 1, "groups": 4})
            assert not taken(x.expand(2, -1, -1, -1).contiguous())  # another batch than the cache's: the layer raises
            seen = []
            for module in (layer.mlp[0].w_down, layer.feature_attentions[0], layer.sequence_attentions[1].qassmax):
                hook = module.register_forward_hook(lambda *a: seen.append(1))
                assert not taken()
                hook.remove()
            assert taken()
            layer.train()
            assert not taken()


@pytest.mark.parametrize("embed,heads", [(128, 2), (256, 4), (352, 8)])
@pytest.mark.parametrize("tables,rows,groups", [(1, 40, 1), (1, 300, 9), (3, 701, 5)])
def test_fused_build_equals_the_modules_calls(cuda, embed, heads, tables, rows, groups):
    # the cache build's steps after its attention (residuals and norms inside the projections and the
    # SwiGLU kernel) against the modules' own calls, which a forward hook keeps; the cache does not
    # depend on them. Width 352 has no such kernels and takes the modules' calls both times.
    layer = _layer(embed, heads, False, embed, cuda)
    x = torch.randn(tables, rows, groups, embed, generator=torch.Generator().manual_seed(rows)).to(cuda)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        before = x.clone()
        fused = []
        real = layer._fused_after_attention
        layer._fused_after_attention = lambda *a: fused.append(real(*a)) or fused[-1]
        got, cache = layer.forward_train_cache(x, quantize_kv_cache=True)
        assert (len(fused) == 1 and fused[0] is not None) == (embed != 352)
        handle = layer.mlp[0].register_forward_hook(lambda *a: None)
        want, ref = layer.forward_train_cache(x, quantize_kv_cache=True)
        handle.remove()
        assert len(fused) <= 1 and torch.equal(x, before)
    assert torch.equal(cache["seq_kv"]["kv"], ref["seq_kv"]["kv"])
    assert float((got - want).double().norm() / (want - x).double().norm()) <= 4 * 2.0**-11


def test_sublayers_in_training_mode_keep_the_layers_own_calls(cuda):
    # dropout follows each attention's own mode, not the layer's: the feature attention drops out and
    # the cached attention refuses
    layer = _layer(128, 2, False, 6, cuda)
    x = torch.randn(1, 20, 4, 128, device=cuda)
    cache = ScalableSeqKV(torch.randn(4, 50, 2, 2, 64, device=cuda).half(), 1, 4, quantize=True)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        for attn in (layer.sequence_attentions[1], layer.feature_attentions[0]):
            attn.train()
            assert layer._apply_native(x, cache, None) is not None  # no dropout to apply
            attn.dropout = 0.5
            assert layer._apply_native(x, cache, None) is None
            if attn is layer.sequence_attentions[1]:
                with pytest.raises(RuntimeError, match="inference-only"):
                    layer.forward_test_with_cache(x, {"seq_kv": cache})
            attn.eval()
            assert layer._apply_native(x, cache, None) is not None


def test_parameters_on_another_device_or_of_another_shape_are_refused(cuda):
    # the native call passes pointers, so it leaves such a layer to the sublayers' own calls, which raise
    x = torch.randn(1, 20, 4, 128, device=cuda)
    cache = ScalableSeqKV(torch.randn(4, 50, 2, 2, 64, device=cuda).half(), 1, 4, quantize=True)

    def spoil_base(layer):
        layer.sequence_attentions[1].qassmax.base_mlp[-1].cpu()

    def spoil_gate(layer):
        layer.sequence_attentions[1].qassmax.gate_mlp[-1].cpu()

    def spoil_feature(layer):
        layer.feature_attentions[0].qkv_proj_weight.data = layer.feature_attentions[0].qkv_proj_weight.data.cpu()

    def shrink_base(layer):
        layer.sequence_attentions[1].qassmax.base_mlp[-1] = torch.nn.Linear(64, 64).to(cuda)

    for spoil in (spoil_base, spoil_gate, spoil_feature, shrink_base):
        layer = _layer(128, 2, False, 7, cuda)
        spoiled = _layer(128, 2, False, 7, cuda)
        spoil(spoiled)
        with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
            assert layer._apply_native(x, cache, None) is not None
            assert spoiled._apply_native(x, cache, None) is None, spoil.__name__
            with pytest.raises((RuntimeError, ValueError)):
                spoiled.forward_test_with_cache(x, {"seq_kv": cache})


@pytest.mark.parametrize("shared,quantized", [(False, True), (True, False)])
def test_native_apply_past_the_split_mlp(cuda, shared, quantized):
    # 11,700 tokens: the SwiGLU kernel of whole workgroups and projections of several blocks a workgroup
    test_native_apply_equals_the_layers_calls(cuda, 128, 2, 1, 1300, 9, 300, shared, quantized)
    test_native_apply_equals_the_layers_calls(cuda, 256, 4, 1, 1300, 9, 300, shared, quantized)
