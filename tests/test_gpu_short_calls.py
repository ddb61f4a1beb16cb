"""Kernels of short calls at the sizes where they can go wrong: the one-launch
bucketing (one thread's 16 tokens, one expert, experts that do not divide the
block, the most tokens it takes and the next one) and the sampled gradient with
a thread per position (runs of 0, 16 and more slots, slices whose average run is
on either side of its limit, and both kinds in one call)."""
import pytest
import torch

from oracle import moe as M
from usaf_amd import moe as G
from usaf_amd.moe_loader import SparseGradStore

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (64, 1, 1), (65, 1, 1), (1, 128, 8), (17, 12, 3), (192, 128, 8),
                                   (193, 128, 8), (64, 384, 5), (24, 1000, 2), (3072, 8, 2), (63, 48, 48),
                                   (128, 128, 8), (129, 128, 8), (1024, 8, 2), (1025, 8, 2), (16, 1000, 4), (1024, 1, 1)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_bucket_small(gpu_device, T, E, k, dt):
    print(f"[gpu-case] bucket T={T} E={E} k={k} {dt}", flush=True)
    gen = torch.Generator().manual_seed(T + E)
    w, _, _ = M.route(torch.randn(T, E, generator=gen), k, False, dt)
    counts, offsets, tok, sw = M.bucket(w)
    S = int(offsets[-1])
    ovf = torch.zeros(1, dtype=torch.int32, device=gpu_device)
    for cap in (None, S + 5, max(S - 3, 0)):
        b = G.bucket_by_expert(w.to(gpu_device)) if cap is None else G.bucket_by_expert(w.to(gpu_device), cap, ovf)
        torch.cuda.synchronize()
        kept = S if cap is None else min(S, cap)
        assert torch.equal(b.counts.cpu().long(), counts)
        assert torch.equal(b.offsets.cpu().long(), offsets.clamp(max=kept))
        assert torch.equal(b.token_idx.cpu()[:kept].long(), tok[:kept])
        assert torch.equal(b.slot_w.cpu()[:kept], sw[:kept])
        assert not b.token_idx.cpu()[kept:].any() and not b.slot_w.cpu()[kept:].any()
        if cap is not None:
            assert int(ovf) == (cap < S)
        # slots in expert-major, token-ascending order; pairs past the capacity are dropped
        want = torch.full((T, E), -1, dtype=torch.int32)
        order = (w.t() != 0).nonzero()
        want[order[:kept, 1], order[:kept, 0]] = torch.arange(kept, dtype=torch.int32)
        assert torch.equal(b.pair_slot.cpu(), want)


@pytest.mark.parametrize("counts", [[0, 1, 16, 17], [33, 5, 0], [72, 64, 80], [80, 81, 64], [300, 0, 2, 1],
                                    [48, 56, 49], [400, 30, 7, 0, 12, 1, 3, 0, 16]])
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
