"""Decode attention around its segments' edges against fp32 attention.

The number of workgroups picks 1, 2 or 4 query heads per workgroup; each
choice is run at live lengths around the rows of a wave (64) and of a segment
(256), with the window wrapped in its ring, on a large workspace and on the
least one.  Tolerance: a bf16 output of weights that sum to one, so one
rounding (2^-9 relative to the largest value) plus fp32 summation.
"""

from __future__ import annotations

import math

import pytest
import torch

import kvm_testlib as T

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _reference(q, ka, va, rk, rv, start, R, ts, tf, group):
    idx = (start + torch.arange(R, device=DEV)) % rk.size(1)
    B, Hq, D = q.shape
    Hkv = Hq // group
    k = torch.cat([ka, rk[:, idx]], 1).float().view(B, Hkv, -1, D).repeat_interleave(group, 1)
    v = torch.cat([va, rv[:, idx]], 1).float().view(B, Hkv, -1, D).repeat_interleave(group, 1)
    tau = torch.cat([ts.view(-1, 1).expand(Hq, ka.size(1)), tf.view(-1, 1).expand(Hq, R)], 1)
    s = (q.float().unsqueeze(2) * k).sum(-1) * tau / math.sqrt(D)
    return (s.softmax(-1).unsqueeze(-1) * v).sum(2)


@pytest.mark.parametrize("B,Hq,Hkv,D,S,W", [
    (1, 32, 8, 128, 256, 512),   # one of four heads per workgroup
    (8, 32, 8, 128, 256, 512),   # two of four
    (24, 16, 4, 128, 200, 600),  # all four
    (5, 6, 6, 64, 100, 300),     # 64-wide heads
    (40, 12, 6, 64, 1024, 512),  # two heads of 64
    (1, 4, 4, 128, 4000, 512),   # more segments than the combine kernel loads at once
])
def test_decode_attention_segments(B, Hq, Hkv, D, S, W):
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    from kvm_amd import _lib

    lib = _lib.load()
    rows, group = B * Hkv, Hq // Hkv
    gen = torch.Generator(device=DEV).manual_seed(B * 1000 + S)
    ka, va, rk, rv = (torch.randn(rows, n, D, device=DEV, generator=gen).bfloat16() for n in (S, S, W, W))
    q = torch.randn(B, Hq, D, device=DEV, generator=gen).bfloat16()
    ts, tf = (1 + 0.1 * torch.randn(Hq, device=DEV, generator=gen) for _ in range(2))
    m = T.make_mixer(T.mixer_config(Hq, Hkv, D, 64), torch.ones(D), torch.zeros(D), tf, ts)
    ts, tf = m.state_head_temp.detach().float(), m.front_head_temp.detach().float()  # as the mixer holds them
    layer = m._layer_struct(B, torch.device(DEV))
    st = _lib.state_struct(ka, va, torch.ones(rows, S, device=DEV), ka, va, S)
    for active, R, start in ((S, W, W - 1), (S, 1, 0), (0, 65, W - 3), (S - 1, 64, W - 64), (S, 129, W - 128),
                             (S, 257, 7), (63, W - 1, 5)):
        T.log(f"[decode segments] B{B} Hq{Hq} Hkv{Hkv} D{D} active {active} window {R} from {start} of {W}")
        want = _reference(q, ka[:, :active], va[:, :active], rk, rv, start, R, ts, tf, group)
        for nws in (int(lib.kvm_decode_workspace_bytes(layer.ref(), active + R)),
                    4 * int(lib.kvm_decode_workspace_bytes(layer.ref(), S + W))):
            ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
            out = torch.full((B, Hq, D), float("nan"), device=DEV, dtype=torch.bfloat16)
            _lib.check(lib.kvm_decode_attention(
                layer.ref(), q.data_ptr(), q.stride(0), q.stride(1), st, active, rk.data_ptr(), rv.data_ptr(), W,
                start, R, out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(), nws, 0), "kvm_decode_attention")
            err = (out.float() - want).abs()
            bound = 2.0 ** -8 * want.abs() + 2.0 ** -16 * float(want.abs().max())
            assert bool((err <= bound).all()), f"max error {float(err.max())} at {active}+{R}, workspace {nws}"


@pytest.mark.parametrize("B,Hq,Hkv,D,S,W", [
    (8, 32, 8, 128, 256, 512),   # two heads per workgroup together, one alone
    (24, 16, 4, 128, 200, 600),  # four together
    (40, 6, 6, 64, 300, 300),
])
def test_decode_attention_bits_depend_on_the_rows_alone(B, Hq, Hkv, D, S, W):
    """A sequence's output has the same bits in a batch and alone, and whatever
    the workspace's size and the state's and the ring's capacity are."""
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    from kvm_amd import _lib

    lib = _lib.load()
    gen = torch.Generator(device=DEV).manual_seed(B)
    ka, va, rk, rv = (torch.randn(B, Hkv, n, D, device=DEV, generator=gen).bfloat16() for n in (S, S, W, W))
    q = torch.randn(B, Hq, D, device=DEV, generator=gen).bfloat16()
    ts, tf = (1 + 0.1 * torch.randn(Hq, device=DEV, generator=gen) for _ in range(2))
    m = T.make_mixer(T.mixer_config(Hq, Hkv, D, 64), torch.ones(D), torch.zeros(D), tf, ts)

    def attend(q, ka, va, rk, rv, active, R, start, scale):
        n, cap, ring = q.size(0), ka.size(2), rk.size(2)
        layer = m._layer_struct(n, torch.device(DEV))
        st = _lib.state_struct(ka, va, torch.ones(n * Hkv, cap, device=DEV), ka, va, cap)
        nws = scale * int(lib.kvm_decode_workspace_bytes(layer.ref(), active + R))
        ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
        out = torch.empty(n, Hq, D, device=DEV, dtype=torch.bfloat16)
        _lib.check(lib.kvm_decode_attention(
            layer.ref(), q.data_ptr(), q.stride(0), q.stride(1), st, active, rk.data_ptr(), rv.data_ptr(), ring,
            start, R, out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(), nws, 0), "kvm_decode_attention")
        return out

    for active, R in ((S, W), (S, 65), (0, 129), (S - 1, 257)):
        T.log(f"[decode bits] B{B} Hq{Hq} Hkv{Hkv} D{D} active {active} window {R} of {W}")
        want = attend(q, ka, va, rk, rv, active, R, 0, 1)
        assert torch.equal(attend(q, ka, va, rk, rv, active, R, 0, 4), want), "workspace size"
        assert torch.equal(attend(q, ka, va, rk.roll(7, 2), rv.roll(7, 2), active, R, 7, 1), want), "ring position"
        wide = [torch.cat([x, x, x, x, x], 2) for x in (ka, va, rk, rv)]
        assert torch.equal(attend(q, *wide, active, R, 0, 4), want), "capacity"
        for b in (0, B - 1):
            one = [x[b:b + 1].contiguous() for x in (q, ka, va, rk, rv)]
            assert torch.equal(attend(*one, active, R, 0, 1), want[b:b + 1]), f"sequence {b} alone"
