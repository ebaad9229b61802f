"""Leaving out the tiles without weight keeps the results: the C ABI called with the scratch that finds them
(sa_reach_bytes) and without it -- every bit of the forward, and of the backward but for what the exempt
keys' separate sums touch (_compare_backward) -- on inputs whose histories outgrow their logits, on inputs whose histories
do not, and on inputs that are not finite or too large for the bound. The kernels' results against the
oracle are the other tests' matter."""

from __future__ import annotations

import math

import pytest
import torch

from selective_attention import _lib, kernels

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.contiguous().view(torch.int16 if t.element_size() == 2 else torch.int32)


def _inputs(cuda, b, h, t, d, dtype, kind, seed=11):
    g = torch.Generator(device=cuda).manual_seed(seed)
    q, k, v, do = (torch.randn(b, h, t, d, device=cuda, generator=g) for _ in range(4))
    if kind == "sparse":      # few positive selector logits: no tile can be left out
        q[:, 0] += math.sqrt(3.0 * math.sqrt(d) / d)
        k[:, 0] -= math.sqrt(3.0 * math.sqrt(d) / d)
    elif kind == "holes":     # a few keys that nobody selects among selected ones: short and long runs
        k[:, 0, torch.arange(5, t, 97, device=cuda)] = 0.0
    elif kind == "groups":    # nobody selects the keys of every second workgroup of the key side
        k[:, 0, (torch.arange(t, device=cuda) // 128) % 2 == 1] = 0.0
    elif kind == "random":    # ... or of a random half of them
        some = torch.rand((t + 127) // 128, device=cuda, generator=g) < 0.5
        k[:, 0, some.repeat_interleave(128)[:t]] = 0.0
    elif kind == "special":   # values a zero weight does not silence, keys and queries beyond the bound
        v[:, -1, 3] = float("inf")
        v[:, 0, 200] = float("nan")
        k[:, -1, 70] = 3e18
        q[:, 0, t - 3] = 1e19
        do[:, -1, t - 5, 0] = float("inf")
    return tuple(x.to(dtype) for x in (q, k, v, do))


def _forward(q, k, v, exempt, reach, chunk=0, group=0):
    """sa_forward over the last `chunk` queries (0: all) with or without the scratch of sa_reach_bytes."""
    lib = _lib.load()
    b, h, tk, d = k.shape
    tq = chunk or tk
    dev, code = q.device, kernels._code_of(q)
    qs = q[:, :, tk - tq:].contiguous()
    out, rmax, rden = (torch.empty(b, h, tq, *s, device=dev) for s in ((d,), (), ()))
    carry = torch.empty(b, (tq + 31) // 32, tk, device=dev)
    g = torch.Generator(device=dev).manual_seed(3)
    pos = torch.arange(tk, device=dev)
    state = (0.4 * (tk - tq - 1 - pos).clamp_min(0)).expand(b, tk) + torch.rand(b, tk, device=dev, generator=g)
    state[:, :exempt] = 0.0
    base = lib.sa_forward_workspace_bytes(b, h, tk, d, code, group)
    size = base + (lib.sa_reach_bytes(b, h, tk, d, 0) if reach else 0)
    ws = torch.empty(max(size, 1), dtype=torch.uint8, device=dev)
    _lib.check(lib.sa_forward(qs.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), rmax.data_ptr(),
                              rden.data_ptr(), carry.data_ptr(), state.data_ptr() if chunk else None, state.data_ptr(), tk,
                              ws.data_ptr(), size, b, h, tq, tk, tk - tq, 0, d, 1 / math.sqrt(d), code, exempt, group, 0, 0,
                              torch.cuda.current_stream().cuda_stream))
    return out, rmax, rden, carry, state


# (B, H, T, D, dtype): both widths of the head-dim-64 forward and odd head counts, the other head dims and
# group widths, fp32; lengths around tiles, workgroups and mask words
SHAPES = [(1, 2, 1024, 64, "bf16"), (2, 3, 2081, 64, "bf16"), (1, 16, 8200, 64, "bf16"), (3, 1, 4127, 64, "bf16"),
          (1, 4, 1500, 32, "bf16"), (1, 2, 2049, 128, "bf16"), (1, 2, 1377, 64, "f32"), (1, 1, 1111, 32, "f32"),
          (1, 2, 1056, 128, "f32"),
          # fp32 backward on the split kernels: one tile past 1024, the longest and widest grid; unsplit beside them
          (1, 3, 1025, 32, "f32"), (1, 8, 2048, 64, "f32"), (1, 12, 1411, 64, "f32"),
          (1, 2, 4129, 64, "f32")]


@pytest.mark.parametrize("kind", ["normal", "holes", "groups", "sparse", "special"])
@pytest.mark.parametrize("b,h,t,d,dtype", SHAPES)
def test_forward_keeps_its_bits(cuda, b, h, t, d, dtype, kind):
    print(f"case forward {b} {h} {t} {d} {dtype} {kind}", flush=True)
    q, k, v, _ = _inputs(cuda, b, h, t, d, torch.bfloat16 if dtype == "bf16" else torch.float32, kind)
    for exempt, chunk in ((1, 0), (16, 0), (40, 0), (3, 77), (1, 300)):
        for got, want in zip(_forward(q, k, v, exempt, True, chunk), _forward(q, k, v, exempt, False, chunk)):
            assert torch.equal(_bits(got), _bits(want)), (exempt, chunk)


def test_forward_past_the_mask_keeps_its_bits(cuda):
    """More key tiles than a workgroup's mask holds (128 words of 64): the oldest are all visited."""
    t = 64 * 32 * 128 + 3000
    q, k, v, _ = _inputs(cuda, 1, 1, t, 64, torch.bfloat16, "normal")
    for got, want in zip(_forward(q, k, v, 1, True, 500), _forward(q, k, v, 1, False, 500)):
        assert torch.equal(_bits(got), _bits(want))


def _backward(q, k, v, do, aux, exempt, reach, grad_bf16):
    lib = _lib.load()
    b, h, t, d = q.shape
    code = kernels._code_of(q)
    out, rmax, rden, carry = aux
    grads = [torch.empty(q.shape, device=q.device, dtype=torch.bfloat16 if grad_bf16 else torch.float32) for _ in range(3)]
    size = lib.sa_backward_workspace_bytes(b, h, t, d, code, 0) + (lib.sa_backward_reach_bytes(b, h, t, d, exempt) if reach else 0)
    # (the rows of the checkpoint planes that no sweep writes are read as NaN if anything takes them)
    ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=q.device)
    _lib.check(lib.sa_backward(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), do.data_ptr(), rmax.data_ptr(),
                               rden.data_ptr(), carry.data_ptr(), *(x.data_ptr() for x in grads), ws.data_ptr(), size, b, h,
                               t, d, 1 / math.sqrt(d), code, _lib.DTYPE_BF16 if grad_bf16 else _lib.DTYPE_F32, exempt, 0,
                               torch.cuda.current_stream().cuda_stream))
    return grads


def _compare_backward(q, k, v, do, exempt, half):
    bf16 = q.dtype == torch.bfloat16
    aux = _forward(q, k, v, exempt, True)[:4]
    got = _backward(q, k, v, do, aux, exempt, True, half)
    want = _backward(q, k, v, do, aux, exempt, False, half)
    first = 128 if exempt <= 32 else 0
    for x, y in zip(got[1:], want[1:]):
        assert torch.equal(_bits(x[:, :, first:]), _bits(y[:, :, first:])), exempt
    # dQ: every bit, but for head 0 at bf16 head dim 64 beside keys taken apart. There a suffix sum of the first
    # workgroup may round elsewhere, which can turn the bf16 rounding of an element of dz + g: 2e-7 of all of dQ
    # and 1.3e-5 of a row seen
    d64 = bf16 and q.shape[-1] == 64 and first
    same = slice(1, None) if d64 else slice(None)
    assert torch.equal(_bits(got[0][:, same]), _bits(want[0][:, same])), exempt
    if d64:
        x, y = got[0][:, 0].double(), want[0][:, 0].double()
        rows = y.isfinite().all(-1)
        off, size = (x - y)[rows].norm(dim=-1), y[rows].norm(dim=-1)
        assert (off <= (2.0 ** -7 if half else 2.0 ** -13) * size).all(), exempt
        assert off.norm() <= (2.0 ** -9 if half else 2.0 ** -20) * size.norm(), exempt
    if first == 0:
        return
    for x, y in zip(got, want):
        x, y = x.double(), y.double()
        assert torch.equal(x.isnan(), y.isnan())
        fine = y.isfinite()
        # dK, dV of the exempt keys: split bf16 operands (2^-16 each) or fp32 products summed in another order;
        # a bf16 gradient's own rounding beside that
        tol = 2.0 ** -8 if half else 2.0 ** -14 if bf16 else 2.0 ** -18
        assert (x - y)[fine].norm() <= tol * y[fine].norm() + 1e-30, exempt


@pytest.mark.parametrize("kind", ["normal", "holes", "groups", "sparse", "special"])
@pytest.mark.parametrize("b,h,t,d,dtype", SHAPES)
def test_backward_keeps_its_bits(cuda, b, h, t, d, dtype, kind):
    """With more than 32 exempt keys the same instances of the kernels run: every bit. Up to 32 of them the
    exempt keys' dK, dV are summed by row segments, and the first 128 keys' tiles run an instance of their own,
    whose suffix sums the compiler may round elsewhere (one fp32 ulp seen, in head 0's dQ too): every bit of
    the later keys' dK, dV and of dQ but head 0's at bf16 head dim 64, the rest to rounding."""
    print(f"case backward {b} {h} {t} {d} {dtype} {kind}", flush=True)
    bf16 = dtype == "bf16"
    q, k, v, do = _inputs(cuda, b, h, t, d, torch.bfloat16 if bf16 else torch.float32, kind)
    for exempt in (1, 16, 32, 40):
        _compare_backward(q, k, v, do, exempt, bf16 and exempt == 1)


# More runs of kept 128-key groups than the query side's list holds (64): bwd_dq64_kernel with several heads and
# one, bwd_dq_kernel at one and two heads per wavefront, head dim 128, fp32
@pytest.mark.parametrize("kind", ["groups", "random"])
@pytest.mark.parametrize("b,h,t,d,dtype", [(1, 2, 20001, 64, "bf16"), (1, 1, 40000, 64, "bf16"), (1, 2, 40001, 32, "bf16"),
                                           (1, 1, 20001, 32, "bf16"), (1, 1, 33000, 128, "bf16"), (1, 1, 24001, 64, "f32")])
def test_backward_past_the_run_list_keeps_its_bits(cuda, b, h, t, d, dtype, kind):
    print(f"case backward runs {b} {h} {t} {d} {dtype} {kind}", flush=True)
    q, k, v, do = _inputs(cuda, b, h, t, d, torch.bfloat16 if dtype == "bf16" else torch.float32, kind)
    for exempt in (1, 40):
        _compare_backward(q, k, v, do, exempt, False)


def test_key_norms_of_more_sequences_than_a_grid_extent_holds_beside_them(cuda):
    """60000 sequences of 1024 keys, head dim 32, the last 32 queries: the key norms' workgroups no longer fit beside
    the column sums' (65535 in z). One sequence's rows, read by all of them."""
    lib = _lib.load()
    n, tq, tk, d = 60000, 32, 1024, 32
    q, k, v, _ = _inputs(cuda, 1, 1, tk, d, torch.bfloat16, "normal")
    q = q[:, :, tk - tq:].contiguous()
    before = (0.4 * (tk - tq - 1 - torch.arange(tk, device=cuda)).clamp_min(0)).float()[None]
    state = before.repeat(n, 1)
    out, rmax, rden = (torch.empty(n, 1, tq, *s, device=cuda) for s in ((d,), (), ()))
    carry = torch.empty(n, tq // 32, tk, device=cuda)
    size = lib.sa_forward_workspace_bytes(n, 1, tk, d, _lib.DTYPE_BF16, 0) + lib.sa_reach_bytes(n, 1, tk, d, 0)
    ws = torch.empty(size, dtype=torch.uint8, device=cuda)
    one = _lib.ViewStrides(0, 0, d)
    _lib.check(lib.sa_forward_strided(q.data_ptr(), one, k.data_ptr(), one, v.data_ptr(), one, out.data_ptr(), None, None,
                                      rmax.data_ptr(), rden.data_ptr(), carry.data_ptr(), state.data_ptr(), state.data_ptr(),
                                      tk, ws.data_ptr(), size, n, 1, tq, tk, tk - tq, d, 1 / math.sqrt(d), _lib.DTYPE_BF16, 1,
                                      0, 0, 0, torch.cuda.current_stream().cuda_stream))
    want = kernels.selective_attention_prefill(q, k, v, before, tk - tq)   # (before: the state after it)
    assert torch.equal(out, want.expand_as(out))
    assert torch.equal(state, before.expand_as(state))
