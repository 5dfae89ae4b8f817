"""What the DiT call shims dispatch, on fake tensors (shapes without storage, so no GPU is
needed): one op of this library a call."""
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
