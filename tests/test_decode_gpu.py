"""GPU tests of KV-cache decode attention against the CPU oracle and the forward kernel.

* outputs match oracle.eager_attention.decode_reference (the last Tq rows of causal
  attention, fp64) within the attention tolerances, for MHA / GQA, both head dims,
  Tq = 1 and Tq > 1, per-batch cache lengths including lengths shorter than Tq (rows
  that see no key: O = 0, LSE = -inf), 1, and the full cache;
* decoding the last rows of a sequence agrees with the batched forward kernel on the
  whole sequence;
* run-to-run bitwise determinism and the torch.library op checks;
* every bound of the rule that splits a call, and rows that do not depend on other caches;
* NaN keys, which reach exactly the rows that see them;
* a workspace reused across shapes with leftovers in it, and HIP-graph replays with new
  inputs, both bitwise equal to fresh eager calls.
"""

import pytest
import torch

from helpers import announce, assert_close_abs
from oracle.eager_attention import TOL, TOL_LSE, decode_reference
from tinytrain_amd.kernels.decode import flash_attn_decode
from tinytrain_amd.kernels.flash_attn import _forward

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # B, Hq, Hkv, Tq, Lmax, D, lens
    (4, 16, 8, 1, 4096, 128, [4096, 1, 33, 2500]),
    (2, 8, 2, 4, 300, 64, [300, 5]),
    (3, 4, 4, 3, 1000, 128, [2, 999, 64]),
    (1, 32, 4, 4, 128, 64, [128]),          # 8 * 4 = 32 query rows per KV head
    (8, 12, 12, 1, 2048, 64, [2048, 1500, 1024, 511, 64, 33, 32, 31]),
]


def _inputs(B, Hq, Hkv, Tq, Lmax, D, seed=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hq, Tq, D, generator=g)
    q = q / q.pow(2).mean(-1, keepdim=True).sqrt()
    k = torch.randn(B, Hkv, Lmax, D, generator=g)
    k = k / k.pow(2).mean(-1, keepdim=True).sqrt()
    v = torch.randn(B, Hkv, Lmax, D, generator=g)
    return [t.to(torch.bfloat16) for t in (q, k, v)]


@pytest.mark.parametrize("B,Hq,Hkv,Tq,Lmax,D,lens", CASES)
def test_decode_matches_oracle(B, Hq, Hkv, Tq, Lmax, D, lens):
    announce(f"decode B={B} Hq={Hq} Hkv={Hkv} Tq={Tq} Lmax={Lmax} D={D} lens={lens}")
    q, k, v = _inputs(B, Hq, Hkv, Tq, Lmax, D)
    lens_t = torch.tensor(lens, dtype=torch.int32)
    want_o, want_lse = decode_reference(q, k, v, lens)
    o, lse = flash_attn_decode(q.to(DEV), k.to(DEV), v.to(DEV), lens_t.to(DEV))
    torch.cuda.synchronize()
    assert_close_abs("O", o.cpu(), want_o, TOL[torch.bfloat16])
    fin = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), fin)
    assert_close_abs("LSE", lse.cpu()[fin], want_lse[fin], TOL_LSE)


def _uneven(B, L, step):
    return [max(L - step * i, 0) for i in range(B)]


@pytest.mark.parametrize("B, Hq, Hkv, Tq, Lmax, D, lens, chunks", [
    (3, 4, 2, 1, 512, 128, [512, 33, 0], 1),            # 16 blocks: one launch
    (2, 2, 1, 1, 512, 64, [511, 480], 1),
    (2, 4, 2, 3, 513, 128, [513, 2], 9),                # 17: a block for every wave of a chunk
    (1, 2, 1, 2, 545, 64, [545], 5),
    (2, 32, 1, 1, 1000, 128, [1000, 65], 16),           # 32 query columns fill the merge stage
    (1, 16, 8, 1, 5000, 128, [4999], 32),               # one sequence: 256 workgroups
    (2, 16, 8, 1, 5000, 128, [4999, 31], 32),           # two: 512
    (1, 8, 2, 8, 16500, 64, [16391], 129),              # many chunks of few blocks per head
    (16, 4, 2, 1, 1000, 128, _uneven(16, 1000, 61), 16),    # 32 heads: chunks of two blocks
    (17, 4, 2, 1, 1000, 128, _uneven(17, 1000, 61), 15),    # 34: of a share each, 3 blocks
    (17, 4, 2, 2, 11500, 128, _uneven(17, 11500, 767), 15),  # a share of 24: four waves
    (17, 4, 2, 1, 11000, 128, _uneven(17, 11000, 733), 15),  # of 23: two
    (26, 4, 2, 1, 1200, 128, _uneven(26, 1200, 47), 9),  # 468 of 512 slots
    (32, 24, 3, 1, 700, 64, _uneven(32, 700, 22), 5),    # 480
    (54, 8, 2, 1, 700, 64, _uneven(54, 700, 13), 4),     # 432
    (65, 6, 3, 1, 800, 128, _uneven(65, 800, 12), 3),    # 390 would leave a fifth empty: 585
    (102, 4, 4, 1, 2048, 64, _uneven(102, 2048, 20), 2),  # 408 heads of 64 blocks: two chunks
    (102, 4, 4, 1, 2016, 64, _uneven(102, 2016, 20), 1),  # of 63: one, eight waves
    (103, 4, 4, 1, 2048, 64, _uneven(103, 2048, 20), 1),  # 412 heads
    (103, 4, 4, 1, 1504, 64, _uneven(103, 1504, 15), 1),  # 47 blocks: four waves
    (40, 8, 8, 4, 700, 128, _uneven(40, 700, 17), 1),
])
def test_decode_splits_match_oracle(B, Hq, Hkv, Tq, Lmax, D, lens, chunks):
    """Both sides of every rule that picks a call's workgroups per head and waves per
    workgroup, with uneven and empty caches, every second head group's last column among them."""
    from tinytrain_amd import _lib

    announce(f"decode splits B={B} Hq={Hq} Hkv={Hkv} Tq={Tq} Lmax={Lmax} D={D} lens={lens[:4]}")
    nbytes = _lib.load().ttfa_decode_workspace_bytes(B, Hq, Hkv, Tq, Lmax, D)
    assert nbytes == B * Hq * Tq * chunks * (D + 2) * 4
    q, k, v = _inputs(B, Hq, Hkv, Tq, Lmax, D)
    lens_t = torch.tensor(lens, dtype=torch.int32)
    want_o, want_lse = decode_reference(q, k, v, lens)
    o, lse = flash_attn_decode(q.to(DEV), k.to(DEV), v.to(DEV), lens_t.to(DEV))
    assert_close_abs("O", o.cpu(), want_o, TOL[torch.bfloat16])
    torch.cuda.synchronize()
    seen = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), seen)
    assert_close_abs("lse", lse.cpu()[seen], want_lse[seen], TOL_LSE)


@pytest.mark.parametrize("B, Hkv, L, D", [(17, 2, 2500, 128), (40, 2, 4000, 64), (8, 8, 8000, 128)])
def test_decode_rows_do_not_depend_on_the_other_caches(B, Hkv, L, D):
    """A sequence's bits are a function of the call's shape and of its own cache: the same
    beside full, short or empty caches, whose unused workgroups leave no trace."""
    announce(f"decode neighbours B={B} Hkv={Hkv} L={L} D={D}")
    q, k, v = (t.to(DEV) for t in _inputs(B, 2 * Hkv, Hkv, 1, L, D, seed=9))
    own = [L, L - 1, 33 * 32, 32, 1]

    def run(rest):
        lens = torch.tensor(own + [rest] * (B - len(own)), dtype=torch.int32, device=DEV)
        return [t[:len(own)] for t in flash_attn_decode(q, k, v, lens)]

    want = run(L)
    for rest in (L // 3, 40, 0):
        for a, b in zip(run(rest), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("Hkv, L, D, lens, at", [
    (2, 512, 128, [512, 20], [300, 3]),      # one chunk: a NaN in one wave of four, and in the
    (2, 512, 64, [500, 32], [499, 0]),       # only wave with keys
    (2, 2000, 128, [2000, 65], [1999, 64]),  # split, two waves per workgroup
    (8, 9000, 128, [9000, 40], [5000, 39]),  # split, four waves
    (2, 2000, 64, [1999, 40], [0, 7]),
])
@pytest.mark.parametrize("whole_block", [False, True])
def test_decode_nan_keys_reach_the_result(Hkv, L, D, lens, at, whole_block):
    """A NaN key makes O and LSE of exactly the rows that see it NaN, whichever workgroup and
    wave reads it (alone among finite keys, or with its whole 32-key block); every other row
    keeps its bits."""
    announce(f"decode NaN Hkv={Hkv} L={L} D={D} lens={lens} at={at} block={whole_block}")
    Tq = 2
    q, k, v = (t.to(DEV) for t in _inputs(2, 2 * Hkv, Hkv, Tq, L, D, seed=5))
    lens_t = torch.tensor(lens, dtype=torch.int32, device=DEV)
    clean = flash_attn_decode(q, k, v, lens_t)
    first = [a // 32 * 32 if whole_block else a for a in at]
    for b in range(2):
        k[b, 1, first[b]:at[b] + 1] = float("nan")
    o, lse = flash_attn_decode(q, k, v, lens_t)
    torch.cuda.synchronize()
    pos = torch.tensor(lens)[:, None] + torch.arange(-Tq, 0)            # last key a row sees
    bad = torch.zeros(2, 2 * Hkv, Tq, dtype=torch.bool)
    bad[:, 2:4] = (torch.tensor(first)[:, None] <= pos)[:, None]        # KV head 1: q heads 2, 3
    bad = bad.to(DEV)
    assert torch.equal(torch.isnan(lse), bad)
    assert torch.equal(torch.isnan(o), bad[..., None].expand_as(o))
    assert torch.equal(o[~bad], clean[0][~bad]) and torch.equal(lse[~bad], clean[1][~bad])


def test_decode_agrees_with_forward_kernel():
    announce("decode vs batched forward last rows")
    B, Hq, Hkv, T, D, Tq = 2, 8, 2, 700, 128, 2
    g = torch.Generator().manual_seed(1)
    q = torch.randn(B, Hq, T, D, generator=g).to(torch.bfloat16).to(DEV)
    k = torch.randn(B, Hkv, T, D, generator=g).to(torch.bfloat16).to(DEV)
    v = torch.randn(B, Hkv, T, D, generator=g).to(torch.bfloat16).to(DEV)
    o_full, lse_full = _forward(q, k, v)
    lens = torch.full((B,), T, dtype=torch.int32, device=DEV)
    o, lse = flash_attn_decode(q[:, :, T - Tq:].contiguous(), k, v, lens)
    torch.cuda.synchronize()
    assert_close_abs("O", o, o_full[:, :, T - Tq:], TOL[torch.bfloat16])
    assert_close_abs("LSE", lse, lse_full[:, :, T - Tq:], TOL_LSE)


@pytest.mark.parametrize("B, L", [(32, 4096), (1, 16384), (128, 1024)])
def test_decode_bench_shapes_match_forward(B, L):
    """At the decode bench's shapes (Hq 16, Hkv 8, D 128; hundreds of key splits per row
    at B=1), the decoded row of every batch equals row cache_len-1 of the batched forward
    kernel over the whole cache, for per-batch cache lengths."""
    announce(f"decode bench shape B={B} L={L}")
    Hq, Hkv, D = 16, 8, 128
    g = torch.Generator(device=DEV).manual_seed(3)

    def unit_rms(t):
        return (t / t.pow(2).mean(-1, keepdim=True).sqrt()).to(torch.bfloat16)

    q = unit_rms(torch.randn(B, Hq, L, D, device=DEV, generator=g))
    k = unit_rms(torch.randn(B, Hkv, L, D, device=DEV, generator=g))
    v = torch.randn(B, Hkv, L, D, device=DEV, generator=g).to(torch.bfloat16)
    lens = torch.randint(1, L + 1, (B,), device=DEV, generator=g, dtype=torch.int32)
    lens[0] = L
    o_full, lse_full = _forward(q, k, v)
    rows = (lens.long() - 1).view(B, 1, 1, 1).expand(B, Hq, 1, D)
    qd = torch.gather(q, 2, rows).contiguous()
    o, lse = flash_attn_decode(qd, k, v, lens)
    want_o = torch.gather(o_full, 2, rows)
    want_lse = torch.gather(lse_full, 2, (lens.long() - 1).view(B, 1, 1).expand(B, Hq, 1))
    torch.cuda.synchronize()
    assert_close_abs("O", o, want_o, TOL[torch.bfloat16])
    assert_close_abs("LSE", lse, want_lse, TOL_LSE)


def test_decode_deterministic_and_opcheck():
    announce("decode determinism + opcheck")
    q, k, v = (t.to(DEV) for t in _inputs(4, 8, 2, 2, 1024, 64, seed=2))
    lens = torch.tensor([1024, 700, 3, 1], dtype=torch.int32, device=DEV)
    a = flash_attn_decode(q, k, v, lens)
    b = flash_attn_decode(q, k, v, lens)
    torch.cuda.synchronize()
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    torch.library.opcheck(flash_attn_decode, (q, k, v, lens),
                          test_utils=("test_schema", "test_faketensor"))


def test_decode_shared_workspace_with_leftovers():
    """One workspace reused by calls of different shapes through the C ABI, first filled
    with random bits: every call equals a call of the op on a fresh workspace, bitwise
    (nothing a call reads from the workspace was left there by another)."""
    import math

    from tinytrain_amd import _lib

    announce("decode shared workspace with leftovers")
    lib = _lib.load()
    shapes = [(1, 16, 8, 1, 16384, 128, [16384]), (4, 8, 2, 2, 1024, 64, [1024, 700, 3, 1]),
              (128, 16, 8, 1, 1024, 128, None), (2, 12, 12, 1, 5000, 64, [4999, 2048])]
    need = max(lib.ttfa_decode_workspace_bytes(B, Hq, Hkv, Tq, L, D)
               for B, Hq, Hkv, Tq, L, D, _ in shapes)
    ws = torch.randint(-2**62, 2**62, (need // 8 + 2,), dtype=torch.int64, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    for rep in range(2):
        for i, (B, Hq, Hkv, Tq, L, D, lens) in enumerate(shapes):
            q, k, v = (t.to(DEV) for t in _inputs(B, Hq, Hkv, Tq, L, D, seed=10 * i + rep))
            if lens is None:
                lens = [L - 7 * j for j in range(B)]
            lens_t = torch.tensor(lens, dtype=torch.int32, device=DEV)
            want_o, want_lse = flash_attn_decode(q, k, v, lens_t)
            o, lse = torch.empty_like(q), torch.empty(B, Hq, Tq, device=DEV)
            _lib.check(lib.ttfa_decode_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                           lens_t.data_ptr(), o.data_ptr(), lse.data_ptr(),
                                           ws.data_ptr(), B, Hq, Hkv, Tq, L, D, _lib.TTFA_BF16,
                                           1.0 / math.sqrt(D), stream))
            torch.cuda.synchronize()
            assert torch.equal(o, want_o), (rep, i)
            assert torch.equal(lse, want_lse), (rep, i)


def test_decode_graph_replays():
    """flash_attn_decode captured in a HIP graph (16 key splits per row) and replayed with
    new cache contents and lengths between the replays (eager work and synchronisations in
    between): each replay equals the eager op on the same inputs, bitwise."""
    announce("decode graph replays")
    B, Hq, Hkv, Tq, L, D = 2, 16, 8, 1, 8192, 128
    q_s, k_s, v_s = (t.to(DEV) for t in _inputs(B, Hq, Hkv, Tq, L, D, seed=20))
    lens_s = torch.tensor([L, 5000], dtype=torch.int32, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        flash_attn_decode(q_s, k_s, v_s, lens_s)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o_s, lse_s = flash_attn_decode(q_s, k_s, v_s, lens_s)
    for r in range(4):
        q, k, v = (t.to(DEV) for t in _inputs(B, Hq, Hkv, Tq, L, D, seed=21 + r))
        q_s.copy_(q)
        k_s.copy_(k)
        v_s.copy_(v)
        lens_s.copy_(torch.tensor([L - 100 * r, 3000 + 7 * r], dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        want_o, want_lse = flash_attn_decode(q_s, k_s, v_s, lens_s)
        torch.cuda.synchronize()
        assert torch.equal(o_s, want_o), r
        assert torch.equal(lse_s, want_lse), r
