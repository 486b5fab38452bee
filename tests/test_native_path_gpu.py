"""GPU tests of the native eager path (csrc/torch_native.cpp) behind the public functions.

Plain eager calls must give exactly what the custom ops give, gradients included, and
everything else must still reach the custom ops: dispatch modes, functorch, forward-mode
tangents, recorded backwards and inputs outside the contract.  Tracing by torch.compile is
covered without a GPU in test_compile_host.py.
"""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from helpers import announce
from tinytrain_amd import _lib
from tinytrain_amd.attention import precompute_rope
from tinytrain_amd.kernels import flash_attn as fa
from tinytrain_amd.kernels.decode import flash_attn_decode
from tinytrain_amd.kernels.qk_prologue import qk_norm_rope, qk_norm_rope_fwd

pytestmark = pytest.mark.gpu
DEV = "cuda"
OPS = torch.ops.tinytrain


def _rand(*shape, seed=0, dtype=torch.bfloat16):
    g = torch.Generator(DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _attn(dtype=torch.bfloat16, T=70):
    ins = [_rand(2, 4, T, 64, dtype=dtype), _rand(2, 2, T, 64, seed=1, dtype=dtype),
           _rand(2, 2, T, 64, seed=2, dtype=dtype)]
    return ins, fa.flash_attn, lambda *a: fa.flash_attn_fwd(*a)[0]


def _varlen():
    cu = torch.tensor([0, 33, 33, 150], dtype=torch.int32, device=DEV)
    ins = [_rand(4, 150, 64), _rand(2, 150, 64, seed=1), _rand(2, 150, 64, seed=2)]
    return (ins, lambda *a: fa.flash_attn_varlen(*a, cu, 117),
            lambda *a: fa.flash_attn_varlen_fwd(*a, cu, 117)[0])


def _prologue():
    cos, sin = (t.to(DEV) for t in precompute_rope(64, 40, 1e6))
    ins = [_rand(2, 33, 4, 64), _rand(2, 33, 2, 64, seed=1), _rand(2, 33, 2, 64, seed=2),
           _rand(64, seed=3, dtype=torch.float32), _rand(64, seed=4, dtype=torch.float32)]
    return (ins, lambda *a: qk_norm_rope(*a, cos, sin, 1e-6),
            lambda *a: qk_norm_rope_fwd(*a, cos, sin, 1e-6)[:3])


PATHS = {"attn": _attn, "attn_fp32": lambda: _attn(torch.float32), "varlen": _varlen,
         "prologue": _prologue}


def _grads(f, ins, strided=False):
    ins = [t.clone().requires_grad_() for t in ins]
    out = f(*ins)
    outs = out if isinstance(out, (tuple, list)) else (out,)
    gs = [_rand(*o.shape, seed=7 + i, dtype=o.dtype) for i, o in enumerate(outs)]
    if strided:
        gs = [g.transpose(1, 2).contiguous().transpose(1, 2) for g in gs]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, ins, gs))


@pytest.mark.parametrize("path", PATHS)
@pytest.mark.parametrize("strided", [False, True])
def test_same_bits_as_the_ops(path, strided):
    announce(f"native path {path} strided={strided}")
    ins, native, op = PATHS[path]()
    for a, b in zip(_grads(native, ins, strided), _grads(op, ins, strided)):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            a, b = native(*ins), op(*ins)
            for x, y in zip(a if isinstance(a, tuple) else (a,), b if isinstance(b, tuple) else (b,)):
                assert torch.equal(x, y) and not x.requires_grad


def test_decode_same_bits_and_errors():
    announce("native path decode")
    q, k, v = _rand(3, 4, 2, 64), _rand(3, 2, 600, 64, seed=1), _rand(3, 2, 600, 64, seed=2)
    lens = torch.tensor([600, 1, 77], dtype=torch.int32, device=DEV)
    for a, b in zip(flash_attn_decode(q, k, v, lens), OPS.flash_attn_decode(q, k, v, lens)):
        assert torch.equal(a, b)
    with pytest.raises(fa.FlashAttnInputError, match="int32"):
        flash_attn_decode(q, k, v, lens.long())
    with pytest.raises(fa.FlashAttnInputError, match="contiguous"):
        flash_attn_decode(q, k.transpose(0, 1).contiguous().transpose(0, 1), v, lens)
    o, _ = flash_attn_decode(q.requires_grad_(), k, v, lens)  # recorded: the op's error
    with pytest.raises(RuntimeError, match="no autograd formula"):
        o.float().sum().backward()


def test_inputs_outside_the_contract_raise_as_before():
    announce("native path errors")
    (q, k, v), _, _ = _attn()
    with pytest.raises(fa.FlashAttnInputError, match="contiguous"):
        fa.flash_attn(q.transpose(1, 2).contiguous().transpose(1, 2), k, v)
    with pytest.raises(fa.FlashAttnInputError, match="dtype"):
        fa.flash_attn(q, k.float(), v)
    with pytest.raises(fa.FlashAttnInputError, match="ROCm GPU"):
        fa.flash_attn(q, k.cpu(), v.cpu())
    flat = torch.empty(q.numel() + 1, device=DEV, dtype=q.dtype)
    with pytest.raises(_lib.TTFAError, match="aligned"):
        fa.flash_attn(flat[1:].view(q.shape), k, v)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_modes_transforms_and_recorded_backwards_reach_the_ops():
    announce("native path hand-over")
    (q, k, v), native, op = _attn()
    with _Seen() as seen:
        native(q, k, v)
    assert any("flash_attn_fwd" in n for n in seen.names)
    q1 = q.clone().requires_grad_()
    o = native(q1, k, v)
    with _Seen() as seen:
        torch.autograd.grad(o, q1, torch.ones_like(o), retain_graph=True)
    assert any("flash_attn_bwd" in n for n in seen.names)
    # create_graph: the gradient is recorded, and differentiating it raises as the op does
    g, = torch.autograd.grad(o, q1, torch.ones_like(o), create_graph=True)
    assert g.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(g.float().sum(), q1)
    stacked = torch.vmap(native)(*(torch.stack([t, t]) for t in (q, k, v)))
    assert torch.equal(stacked[0], op(q, k, v)) and torch.equal(stacked[0], stacked[1])
    import torch.autograd.forward_ad as fw
    with fw.dual_level(), pytest.raises(NotImplementedError, match="forward mode AD"):
        native(fw.make_dual(q1, torch.ones_like(q)), k, v)


def test_saved_tensors_hooks_and_version_checks():
    announce("native path saved tensors")
    (q, k, v), native, _ = _attn()
    want = _grads(native, (q, k, v))
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        got = _grads(native, (q, k, v))
    assert len(packed) == 5
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    q1, k1 = q.clone().requires_grad_(), k.clone()
    o = native(q1, k1, v)
    k1.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.float().sum().backward()


@pytest.mark.parametrize("path", PATHS)
def test_saved_tensors_handed_back_strided(path):
    """Saved-tensor hooks may hand the forward's results back with other strides: the
    gradients are those of the values, as the ops give them."""
    announce(f"native path strided saved tensors {path}")
    ins, native, _ = PATHS[path]()
    want = _grads(native, ins)
    n = []

    def pack(t):
        n.append(t)
        return len(n) - 1, t

    def unpack(it):
        i, t = it
        of_forward = i >= 6 if path == "prologue" else i in (3, 4)   # rq, rk / o, M
        return t.transpose(0, 1).contiguous().transpose(0, 1) if of_forward else t

    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        got = _grads(native, ins)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_calls_on_a_side_stream_and_in_threads():
    """Each call runs on its caller's current stream; concurrent threads do not disturb one
    another's results."""
    from concurrent.futures import ThreadPoolExecutor

    announce("native path streams and threads")
    ins, native, _ = _attn(T=300)
    want = _grads(native, ins)

    def work(_):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            got = _grads(native, ins)
        s.synchronize()
        return all(torch.equal(a, b) for a, b in zip(got, want))

    torch.cuda.synchronize()
    with ThreadPoolExecutor(4) as ex:
        assert all(ex.map(work, range(12)))
