"""The fused QASS gate (nori_qass_gate) on the GPU.

QASSMaxScaling.forward in "full" mode (ref src/synthefy_nori/model/layer.py:316-456) under fp16
autocast: q * base_scale * (1 + tanh(gate_mlp(q))), gate_mlp = Linear(d, 64) -> GELU ->
Linear(64, d). Checked against

* the same module's separate torch ops on the GPU under autocast (the reference's own
  execution): every output within 4 fp16 ulps
  of its own value plus 2 ulps of the gate (2^-10 at 1 + tanh in [1, 2)) times |q * base_scale|:
  the kernel's two GEMMs sum in another order than hipBLASLt's, a hidden activation one ulp off
  moves the gate by about an ulp, and where 1 + tanh(g) nearly cancels (g << 0) that ulp is a
  large part of the output. 99.98 % of the outputs come out bit-identical; the test asks for
  90 %. (torch's own ops on a strided view of the same queries take other GEMM kernels and
  match their contiguous run only to 83 %, so the reference runs on the contiguous copy.)
* the kernel's output for q as a strided view, bit for bit its output for the contiguous copy;
* the module in fp32 on the CPU: within 1e-2 of max |out| (the fp16 chain against fp32);
* head widths 8 / 44 / 56 / 64, 1 and 10 heads, a row count that is not a multiple of the
  kernel's 32-row tiles, q as a strided view into a [rows, 3, heads, d] projection, and that
  the fused path is the one taken.
"""
import math

import pytest
import torch

import nori_amd.layer as layer_mod
from nori_amd.layer import QASSMaxScaling

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _module(heads, d, seed):
    torch.manual_seed(seed)
    m = QASSMaxScaling(num_heads=heads, head_dim=d, qass_mode="full")
    with torch.no_grad():  # the reference zero-initializes the last layers: give the gate some work
        for mlp in (m.base_mlp, m.gate_mlp):
            for lin in (mlp[0], mlp[-1]):
                lin.weight.normal_(0.0, 1.0 / math.sqrt(lin.in_features))
                lin.bias.normal_(0.0, 0.3)
    return m.eval()


def _compare(got, ref, qbs):
    got, ref, qbs = got.double(), ref.double(), qbs.double()
    tol = 4 * 2.0**-11 * ref.abs() + 2 * 2.0**-10 * qbs.abs() + 4 * 2.0**-24
    worst = float(((got - ref).abs() / tol).max())
    same = float((got == ref).double().mean())
    return worst, same


@pytest.mark.parametrize("heads,d", [(10, 56), (1, 64), (4, 44), (2, 8)])
def test_fused_gate_against_the_separate_ops(monkeypatch, heads, d):
    m = _module(heads, d, seed=heads * 100 + d).to(DEV)
    g = torch.Generator().manual_seed(d)
    rows = 1000
    qkv = (torch.randn(rows, 3, heads, d, generator=g) * 2.0).half().to(DEV)
    calls = []
    real = layer_mod.qass_gate
    monkeypatch.setattr(layer_mod, "qass_gate", lambda *a: calls.append(1) or real(*a))
    contiguous = qkv[:, 0].contiguous().view(1, rows, heads, d)
    strided = qkv[:, 0].unsqueeze(0)
    print(f"qass gate heads {heads} d {d} q strides {tuple(strided.stride())}", flush=True)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        m.fused = True
        got = m(contiguous, 8192)
        got_strided = m(strided, 8192)
        m.fused = False
        ref = m(contiguous, 8192)
        m.qass_mode = "base_only"  # q * base_scale alone, for the error bound
        qbs = m(contiguous, 8192)
        m.qass_mode = "full"
    torch.cuda.synchronize()
    assert len(calls) == 2
    assert got.dtype == torch.float16 and got.shape == contiguous.shape
    worst, same = _compare(got, ref, qbs)
    print(f"  vs separate ops: worst {worst:.2f} of the bound, {same:.4f} bit-identical", flush=True)
    assert worst <= 1.0 and same >= 0.9
    assert torch.equal(got_strided, got)

    cpu = _module(heads, d, seed=heads * 100 + d)
    with torch.no_grad():
        exp = cpu(qkv[:, 0].unsqueeze(0).float().cpu(), 8192)
    err = float((got.float().cpu() - exp).abs().max() / exp.abs().max())
    print(f"  vs fp32 CPU: {err:.3e}", flush=True)
    assert err <= 1e-2


def test_fused_gate_at_the_config4_launch():
    """One config-4 build sub-batch's queries (8.4 M vectors: 102 x 8192 rows, 10 heads of 56):
    every output against the separate ops within the same bound, and the bit-identical share."""
    m = _module(10, 56, seed=7).to(DEV)
    q = torch.randn(102, 8192, 10, 56, device=DEV, dtype=torch.float16) * 2.0
    print("qass gate at [102, 8192, 10, 56]", flush=True)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        m.fused = True
        got = m(q, 8192)
        m.fused = False
        ref = m(q, 8192)
        m.qass_mode = "base_only"
        qbs = m(q, 8192)
        m.qass_mode = "full"
    torch.cuda.synchronize()
    worst, same = 0.0, 0
    for i in range(0, 102, 17):  # in slices: the float64 bound of the whole tensor is 6 GB per term
        w, sm = _compare(got[i:i + 17], ref[i:i + 17], qbs[i:i + 17])
        worst, same = max(worst, w), same + sm * 17 / 102
    print(f"  vs separate ops: worst {worst:.2f} of the bound, {same:.4f} bit-identical", flush=True)
    assert worst <= 1.0 and same >= 0.9


def test_single_key_and_fp32_queries_keep_the_torch_path(monkeypatch):
    m = _module(2, 32, seed=5).to(DEV)
    monkeypatch.setattr(layer_mod, "qass_gate", lambda *a: pytest.fail("fused gate taken"))
    q = torch.randn(64, 2, 32, device=DEV)
    with torch.inference_mode():
        assert torch.equal(m(q.half(), 1), q.half())  # one key: q unscaled
        out = m(q, 100)  # fp32 queries without autocast: the separate ops
    assert out.dtype == torch.float32


@pytest.mark.parametrize("heads,d", [(10, 56), (1, 64), (8, 44), (2, 8), (1, 4), (3, 128)])
@pytest.mark.parametrize("n_keys", [2, 300, 65536, 200000])
def test_base_scale_against_the_separate_ops(heads, d, n_keys):
    # nori_qass_base against the module's torch ops under fp16 autocast: the hidden layer rounds at
    # the same points, and its 64-term sum, in another order, can move the rounded delta by one fp16
    # ulp, which moves 1 + tanh by at most two (2^-10 in [1, 2)) and its product with T(log n) by a
    # last rounding: 3 * 2^-10 * T(log n) in all. Head counts fill a last workgroup only in part
    # (4, 352, 384 outputs).
    m = _module(heads, d, seed=heads + 7 * d).to(DEV)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
        log_n = torch.full((), math.log(float(n_keys)), device=DEV, dtype=torch.float16)
        want = log_n * (1.0 + torch.tanh(m.base_mlp(log_n.view(1, 1))))
        got = layer_mod.qass_base(math.log(float(n_keys)), *m._half_weights("_base16", m.base_mlp))
        assert got.dtype == torch.float16 and got.shape == (heads * d,)
        assert float((got.double() - want.view(-1).double()).abs().max()) <= 3 * 2.0**-10 * float(log_n)
        m.base_mlp[-1].bias.add_(1.0)  # in place: the fp16 copies follow
        assert not torch.equal(layer_mod.qass_base(math.log(float(n_keys)), *m._half_weights("_base16", m.base_mlp)), got)


@pytest.mark.parametrize("offset", [1, 4])
def test_base_scale_of_weights_in_a_flat_buffer(offset):
    # an fp16 module whose parameters are views into one buffer: rows of w2 on 2- and 8-byte
    # boundaries, which the separate ops took. Against them: the base scale's bar of 3 * 2^-10 * T(log n)
    # times the gate's factor (below 2), 2 ulps of the gate times |q * base| (base below 2 log n) and
    # 4 ulps of the output (below 4 log n |q|): 18 * 2^-10 * log n * |q|
    m = _module(2, 64, seed=3).to(DEV).half()
    with torch.no_grad():
        flat = torch.empty(offset + sum(p.numel() for p in m.parameters()), dtype=torch.float16, device=DEV)
        at = offset
        for p in m.parameters():
            view = flat[at : at + p.numel()].view(p.shape)
            view.copy_(p)
            p.data = view
            at += p.numel()
    q = torch.randn(40, 3, 2, 64, generator=torch.Generator().manual_seed(2)).half().to(DEV)
    with torch.inference_mode():
        got = m(q, 300)
        m.fused = False
        want = m(q, 300)
    assert bool(((got.float() - want.float()).abs() <= 18 * 2.0**-10 * math.log(300.0) * q.float().abs() + 2.0**-14).all())


def test_base_scale_rounds_its_weights_as_autocast_does():
    # fp32 and bf16 parameters read by the kernel: bit for bit its result on their fp16 casts
    for dtype in (torch.float32, torch.bfloat16):
        m = _module(3, 44, seed=5).to(DEV).to(dtype)
        params = [p.detach() for lin in (m.base_mlp[0], m.base_mlp[-1]) for p in (lin.weight, lin.bias)]
        got = layer_mod.qass_base(math.log(777.0), *params)
        assert torch.equal(got, layer_mod.qass_base(math.log(777.0), *[p.half() for p in params]))
        mixed = [params[0].half(), params[1], params[2].t().contiguous().t(), params[3].half()]
        assert torch.equal(got, layer_mod.qass_base(math.log(777.0), *mixed))


def test_base_scale_follows_the_dtype_its_linears_compute_in():
    # fp16 parameters under bf16 autocast compute in bf16, and the scaled queries come out as torch
    # promotes them; parameters of two dtypes without autocast are refused
    q = torch.randn(40, 3, 2, 64, generator=torch.Generator().manual_seed(4)).half().to(DEV)
    m = _module(2, 64, seed=6).to(DEV).half()
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
        got = m(q, 300)
        m.fused = False
        want = m(q, 300)
    assert got.dtype == want.dtype and torch.equal(got, want)
    m.fused = True
    m.base_mlp[-1].float()
    with torch.inference_mode(), pytest.raises(RuntimeError):
        m(q, 300)


def test_base_scale_of_other_modules_calls_them():
    # a layer of another class, or another activation, in the base MLP: the module's own call
    class Shifted(torch.nn.Linear):
        def forward(self, x):
            return super().forward(x) + 1.0

    q = torch.randn(40, 3, 2, 64, generator=torch.Generator().manual_seed(8)).half().to(DEV)
    for at, other in ((0, Shifted(1, 64)), (1, torch.nn.GELU(approximate="tanh")), (1, torch.nn.Tanh()), (2, Shifted(64, 128))):
        m = _module(2, 64, seed=9)
        m.base_mlp[at] = other
        m = m.to(DEV)
        with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):
            got = m(q, 300)
            log_n = torch.full((), math.log(300.0), device=DEV, dtype=torch.float16)
            scale = log_n.view(1, 1, 1, 1) * (1.0 + torch.tanh(m.base_mlp(log_n.view(1, 1)).view(1, 1, 2, 64)))
            assert torch.equal(got, layer_mod.qass_gate(q, *m._gate_weights(), scale))
