"""torch.compile of the public functions on GPU tensors, traced without a GPU (fake tensors
with device "cuda"): every function is one node, its custom op, whether or not the native
extension is loaded in the process."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from tinytrain_amd import _lib
from tinytrain_amd.kernels.decode import flash_attn_decode
from tinytrain_amd.kernels.flash_attn import flash_attn, flash_attn_varlen
from tinytrain_amd.kernels.qk_prologue import qk_norm_rope

BF, F32 = torch.bfloat16, torch.float32


def _t(*shape, dtype=BF):
    return torch.empty(*shape, dtype=dtype, device="cuda")


CALLS = {
    "flash_attn_fwd": (flash_attn, lambda: [_t(2, 4, 70, 64), _t(2, 2, 70, 64), _t(2, 2, 70, 64)]),
    "flash_attn_varlen_fwd": (lambda q, k, v, cu: flash_attn_varlen(q, k, v, cu, 60),
                              lambda: [_t(4, 100, 64), _t(2, 100, 64), _t(2, 100, 64),
                                       _t(3, dtype=torch.int32)]),
    "flash_attn_decode": (flash_attn_decode,
                          lambda: [_t(2, 4, 1, 64), _t(2, 2, 90, 64), _t(2, 2, 90, 64),
                                   _t(2, dtype=torch.int32)]),
    "qk_norm_rope_fwd": (qk_norm_rope,
                         lambda: [_t(2, 30, 4, 64), _t(2, 30, 2, 64), _t(2, 30, 2, 64),
                                  _t(64, dtype=F32), _t(64, dtype=F32), _t(40, 64, dtype=F32),
                                  _t(40, 64, dtype=F32)]),
}


@pytest.mark.parametrize("loaded", [False, True])
@pytest.mark.parametrize("name", CALLS)
def test_fullgraph_trace_is_one_op(name, loaded, monkeypatch):
    fn, args = CALLS[name]
    if loaded:
        if not (_lib.LIB_PATH.exists() and _lib.NATIVE_PATH.exists()):
            pytest.skip("the libraries are not built")
        _lib.native()
    else:
        monkeypatch.setattr(_lib, "_lib", None)
        monkeypatch.setattr(_lib, "_native", None)
    ops = []

    def backend(gm, _):
        ops.extend(str(n.target) for n in gm.graph.nodes if n.op == "call_function")
        return gm.forward

    torch._dynamo.reset()
    with FakeTensorMode():
        torch.compile(lambda *a: fn(*a), backend=backend, fullgraph=True)(*args())
    assert [o for o in ops if "tinytrain" in o] == [f"tinytrain.{name}.default"], ops
