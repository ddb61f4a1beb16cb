"""Dense expert weight gradients (usaf_hip_moe_weight_grad) where its tiles end:
experts without slots, with 1, 63, 64, 65 and 130, rows and columns that are not
whole 128 x 128 tiles, expert counts that do and do not divide over the dies,
gathered and plain rows.  Operands are integers in [-4, 4]: the sums are exact in
fp32, so every output type must hold the 64-bit product rounded once, bit for bit.
"""
import pytest
import torch

from usaf_amd import _native as N
from usaf_amd import moe as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,R,C,counts,dt,out_dt,gathered", [
    (5, 136, 72, [0, 1, 65, 64, 130], torch.bfloat16, torch.bfloat16, True),
    (8, 256, 128, [63, 0, 2], torch.float16, torch.float16, False),
    (16, 128, 264, [7, 128], torch.bfloat16, torch.float32, True),
    (3, 8, 8, [1, 0, 9], torch.float16, torch.float32, False),
    (8, 128, 128, [0], torch.bfloat16, torch.bfloat16, False),
])
def test_weight_grad(gpu_device, E, R, C, counts, dt, out_dt, gathered):
    gen = torch.Generator().manual_seed(E + R + C)
    counts = [counts[e % len(counts)] for e in range(E)]
    S, T = sum(counts), 50
    print(f"[gpu-case] weight grad E={E} R={R} C={C} S={S} {dt} -> {out_dt} gathered={gathered}", flush=True)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    dy = torch.randint(-4, 5, (max(S, 1), R), generator=gen).to(dt)
    x = torch.randint(-4, 5, (T if gathered else max(S, 1), C), generator=gen).to(dt)
    rows = torch.randint(0, T, (max(S, 1),), generator=gen).to(torch.int32) if gathered else None
    d = lambda t: None if t is None else t.to(gpu_device)
    ddy, dx, drows, doffs = d(dy), d(x), d(rows), d(offs)
    out = torch.full((E, R, C), float("nan"), dtype=out_dt, device=gpu_device)
    N.call("usaf_hip_moe_weight_grad", ddy.data_ptr(), dx.data_ptr(), N.ptr(drows), doffs.data_ptr(), E, R, C,
           N.dtype_code(dt), out.data_ptr(), N.dtype_code(out_dt), N.stream_ptr(gpu_device))
    torch.cuda.synchronize()
    xs = x if rows is None else x[rows.long()]
    for e in range(E):
        a, b = int(offs[e]), int(offs[e + 1])
        assert torch.equal(out[e].cpu(), (dy[a:b].double().t() @ xs[a:b].double()).to(out_dt)), e


def test_weight_grad_of_saved_tensors_in_another_layout(gpu_device):
    """A saved-tensor hook may hand the activations back in another memory order."""
    print("[gpu-case] weight grad with saved hidden states and activations as transposed views", flush=True)
    gen = torch.Generator().manual_seed(1)
    E, H, I, T, dt = 4, 256, 128, 40, torch.bfloat16
    d = lambda *s: (torch.randn(s, generator=gen) * 0.1).to(dt).to(gpu_device)
    hs, dout, wg, wd = d(T, H), d(T, H), d(E, 2 * I, H), d(E, H, I)
    w = (torch.rand(T, E, generator=gen) * (torch.rand(T, E, generator=gen) < 0.5)).to(dt).to(gpu_device)
    grads = []
    # hs [T, H] and act [S, I]; gu and y as they are
    turn = lambda t: t.t().contiguous().t() if t.shape[1] == I or t.shape[0] == T else t
    for unpack in (lambda t: t, turn):
        p = [wg.clone().requires_grad_(True), wd.clone().requires_grad_(True)]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = G.routed_experts(hs.clone().requires_grad_(True), w, G.ExpertWeights(*p), weight_params=tuple(p))
        out.backward(dout)
        torch.cuda.synchronize()
        grads.append([q.grad for q in p])
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])


@pytest.mark.parametrize("counts,R,C,out_dt", [
    ([9000, 0, 5001], 72, 136, torch.bfloat16),  # 4 parts of each expert's slots
    ([16411], 128, 64, torch.float32),  # 16 parts
    ([4095], 64, 64, torch.float32),  # one slot short of 4 parts
])
def test_weight_grad_in_parts(gpu_device, counts, R, C, out_dt):
    print(f"[gpu-case] weight grad in parts counts={counts} R={R} C={C} -> {out_dt}", flush=True)
    gen = torch.Generator().manual_seed(R + C)
    S, E = sum(counts), len(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    # integers in [-4, 4]: sums of up to 16 * 16,411 are exact in fp32 in any order
    dy = torch.randint(-4, 5, (S, R), generator=gen).to(torch.bfloat16)
    x = torch.randint(-4, 5, (S, C), generator=gen).to(torch.bfloat16)
    b = G.Buckets(None, offs.to(gpu_device), None, None, None, S)
    out = G._dense_weight_grad(dy.to(gpu_device), x.to(gpu_device), None, b, out_dt)
    torch.cuda.synchronize()
    assert out.shape == (E, R, C) and out.dtype == out_dt and out.is_contiguous()
    for e in range(E):
        s = slice(int(offs[e]), int(offs[e + 1]))
        assert torch.equal(out[e].cpu(), (dy[s].double().t() @ x[s].double()).to(out_dt)), e
