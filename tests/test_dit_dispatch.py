"""What the DiT call shims dispatch: one op of this library a call. On fake tensors (shapes
without storage, so no GPU is needed), and compiled on a GPU."""
from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode


class Calls(TorchDispatchMode):
    """Records the names of the joyomni_ops ops that run under it."""

    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.namespace == "joyomni_ops":
            self.names.append(func._opname)
        return func(*args, **(kwargs or {}))


def _qk_args(q_contiguous, k_contiguous, table_dtype=torch.float32):
    new = lambda *s, dt=torch.bfloat16: torch.empty(*s, dtype=dt, device="cuda")  # noqa: E731
    qkv = new(1, 9, 3, 4, 64)
    q, k = qkv[:, :, 0], qkv[:, :, 1]
    tables = (new(1, 9, 64, dt=table_dtype), new(1, 9, 64, dt=table_dtype))
    return (q.contiguous() if q_contiguous else q, k.contiguous() if k_contiguous else k,
            new(64), new(64)), tables


@pytest.mark.parametrize("table_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("q_contiguous,k_contiguous", [(True, True), (True, False), (False, True)])
def test_contiguous_qk_is_one_call_in_place(q_contiguous, k_contiguous, table_dtype):
    from joyomni_ops import dit_ops
    with FakeTensorMode(), Calls() as calls:
        args, tables = _qk_args(q_contiguous, k_contiguous, table_dtype)
        q, k = dit_ops.fused_qk_norm_rope_3d(*args, tables)
    assert calls.names == ["qk_norm_rope_inplace"]
    assert (q is args[0]) == q_contiguous and (k is args[1]) == k_contiguous


def test_kstage_is_one_call():
    from joyomni_ops import dit_ops
    with FakeTensorMode(), Calls() as calls:
        args, tables = _qk_args(False, False, torch.bfloat16)
        q, k, stage = dit_ops.fused_qk_norm_rope_3d_kstage(*args, tables)
    assert calls.names == ["qk_norm_rope_kstage"]
    assert q is args[0] and k is args[1] and stage.is_contiguous()


@pytest.mark.parametrize("name", ["fused_qk_norm_rope_3d", "fused_qk_norm_rope_3d_kstage"])
def test_freqs_are_a_pair_of_any_kind(name):
    from joyomni_ops import dit_ops
    with FakeTensorMode():
        args, (cos, sin) = _qk_args(True, True)
        getattr(dit_ops, name)(*args, iter((cos, sin)))
        getattr(dit_ops, name)(*args, torch.stack((cos, sin)))
        with pytest.raises(ValueError):
            getattr(dit_ops, name)(*args, (cos, sin, sin))


def _calls(dit_ops, new):
    """(function, arguments) of the calls that trace, and their arguments' [B, L, D]."""
    B, L, D = 2, 8, 256
    x, mod = (lambda: new(B, L, D)), (lambda: new(B, D))
    qk = lambda: new(1, L, 3, 4, 64).unbind(2)[:2]  # noqa: E731
    tables = lambda: (new(1, L, 64, dt=torch.float32), new(1, L, 64, dt=torch.float32))  # noqa: E731
    return {
        "quantize": (dit_ops.quantize_activation_fp8, (x(),)),
        "gelu_quantize": (dit_ops.gelu_quantize_activation_fp8, (x(),)),
        "norm_fp8": (dit_ops.layernorm_modulate_fp8, (x(), mod(), mod())),
        "add_norm_fp8": (dit_ops.fused_add_gate_layernorm_modulate_fp8,
                         (x(), x(), mod(), mod(), mod())),
        "qk_rope": (dit_ops.fused_qk_norm_rope_3d, (*qk(), new(64), new(64), tables())),
        "qk_rope_kstage": (dit_ops.fused_qk_norm_rope_3d_kstage,
                           (*qk(), new(64), new(64), tables())),
    }


TRACED = ["quantize", "gelu_quantize", "norm_fp8", "add_norm_fp8", "qk_rope", "qk_rope_kstage"]


@pytest.mark.parametrize("name", TRACED)
def test_result_shapes_without_a_launch(name):
    from joyomni_ops import dit_ops
    with FakeTensorMode(), Calls() as calls:
        fn, args = _calls(dit_ops, lambda *s, dt=torch.bfloat16: torch.empty(
            *s, dtype=dt, device="cuda"))[name]
        out = fn(*args)
    assert len(calls.names) == 1
    forms = [(tuple(t.shape), t.dtype, t.is_contiguous()) for t in out]
    fp8 = [((16, 256), torch.float8_e4m3fn, True), ((16, 1), torch.float32, True)]
    qk = [((1, 8, 4, 64), torch.bfloat16, name == "qk_rope")] * 2
    assert forms == {
        "add_norm_fp8": [((2, 8, 256), torch.bfloat16, True)] + fp8,
        "qk_rope": qk, "qk_rope_kstage": qk + [((1, 8, 4, 64), torch.bfloat16, True)],
    }.get(name, fp8)


@pytest.mark.gpu
@pytest.mark.parametrize("name", TRACED)
def test_compiled_without_a_graph_break(dev, name):
    from joyomni_ops import dit_ops
    g = torch.Generator().manual_seed(3)
    new = lambda *s, dt=torch.bfloat16: torch.randn(*s, generator=g).to(dt).to(dev)  # noqa: E731
    fn, args = _calls(dit_ops, new)[name]
    copy = lambda a: (tuple(map(copy, a)) if isinstance(a, tuple) else  # noqa: E731
                      torch.empty_strided(a.shape, a.stride(), dtype=a.dtype, device=dev).copy_(a))
    want = fn(*copy(args))
    for _ in range(2):
        got = torch.compile(fn, backend="aot_eager", fullgraph=True)(*copy(args))
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("name,grad_on", [(n, "x") for n in TRACED + ["fp8_linear"]] +
                         [(n, "vector") for n in TRACED[2:] + ["fp8_linear"]])
def test_results_claim_no_gradient(dev, name, grad_on):
    """What these calls write through quantized or in-place results has no gradient, whatever
    the inputs ask for; q and k rotated in place keep the history of what they were, and an
    Fp8Linear's output that of its bias."""
    from joyomni_ops import dit_ops
    new = lambda *s, dt=torch.bfloat16: torch.ones(*s, dtype=dt, device=dev)  # noqa: E731
    if name == "fp8_linear":
        args = (new(2, 8, 256), new(64, 256).to(torch.float8_e4m3fn).t(),
                new(64, dt=torch.float32), new(64))
        fn, wanted = dit_ops.fp8_linear, args[0] if grad_on == "x" else args[3]
    else:
        fn, args = _calls(dit_ops, new)[name]
        wanted = args[{"x": 1 if name == "add_norm_fp8" else 0, "vector": 2}[grad_on]]
    out = fn(*(a.requires_grad_() if a is wanted else a for a in args))
    flags = [t.requires_grad for t in (out if isinstance(out, tuple) else (out,))]
    if grad_on == "x" and name.startswith("qk_rope"):
        assert flags == [True, False, False][:len(flags)]
    else:
        assert flags == [name == "fp8_linear" and grad_on == "vector"] * len(flags)
