"""Kernels of short calls at the sizes where they can go wrong: the sampled
gradient with a thread per position (runs of 0, 16 and more slots, and an average
on either side of its limit)."""
import pytest
import torch

from usaf_amd import moe as G
from usaf_amd.moe_loader import SparseGradStore

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[0, 1, 16, 17], [33, 5, 0], [72, 64, 80], [80, 81, 64], [300, 0, 2, 1]])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("accumulate", [False, True])
def test_sampled_gradient_short_runs(gpu_device, counts, dt, accumulate):
    # integers: the sums are exact in fp32, so each result is the 64-bit one rounded once to dt
    E, R, C = 2 * len(counts), 96, 136
    counts = counts * 2
    print(f"[gpu-case] sampled gradient counts={counts} {dt} accumulate={accumulate}", flush=True)
    gen = torch.Generator().manual_seed(sum(counts))
    S = sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    dy = torch.randint(-3, 4, (S, R), generator=gen).to(dt)
    x = torch.randint(-3, 4, (S, C), generator=gen).to(dt)
    idx = torch.randperm(E * R * C, generator=gen)[:5000]  # not sorted: through the position map
    store = SparseGradStore({"w": idx}, {"w": (E, R, C)}, device=gpu_device)
    old = torch.randint(-9, 10, (idx.numel(),), generator=gen).float()
    if accumulate:
        store.compact["w"].copy_(old)
    else:
        store.zero_()
    d_offs = offs.to(gpu_device)
    table = G.blocked_layout(d_offs, S)
    store.add_sampled("w", G.slot_blocked(dy.to(gpu_device), d_offs, S, table=table),
                      G.slot_blocked(x.to(gpu_device), d_offs, S, table=table), d_offs, dt)
    torch.cuda.synchronize()
    full = torch.stack([dy[offs[e]:offs[e + 1]].double().t() @ x[offs[e]:offs[e + 1]].double() for e in range(E)])
    want = full.reshape(-1)[idx].to(dt).float() + (old if accumulate else 0)
    assert torch.equal(store.compact["w"].cpu(), want)
