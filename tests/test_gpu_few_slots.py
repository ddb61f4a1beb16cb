"""The grouped 4-bit GEMMs at few slots per expert (moe_few.hip), where their
tiles end: experts without slots, with 1, 31, 32, 33 and 65, one expert only,
255 experts, widths that leave waves without rows (unsplit and split in two),
every split of the contraction, four weight-row units a wave.

Weights and activations are small integers (scale 1, zero -8; activations in
[-2, 2]), so every sum is exact in fp32 in any order and the outputs that are
rounded once must equal the 64-bit product rounded to the dtype, bit for bit.
act and dgu go through the hardware exp2 and reciprocal (about 1 ulp of fp32
each) and up to three roundings to the dtype, each of which may fall the other
way: 3 half-ulp steps, 3 * 2^-8 of the value in bf16 and 3 * 2^-11 in fp16.  A
value below the dtype's smallest normal may vanish on the way, the result
itself or the sigmoid (or silu) that is then multiplied by g and u: that normal
times 1 + |g u| more.
"""
import pytest
import torch

from usaf_amd import _native as N
from usaf_amd import moe as G

pytestmark = pytest.mark.gpu
EPS = {torch.bfloat16: 3 * 2.0 ** -8, torch.float16: 3 * 2.0 ** -11}


def _weight(E, rows, cols, gen, dev):
    n = E * rows * cols
    q = torch.randint(-128, 128, (n // 128, 64), generator=gen, dtype=torch.int8)
    one = torch.ones(n // 128, dtype=torch.float16)
    raw = q.view(torch.uint8)
    vals = torch.stack([raw & 15, raw >> 4], 2).double().view(E, rows, cols) - 8
    return G.Q4Tensor(q.to(dev), one.to(dev), (-8 * one).to(dev), torch.Size((E, rows, cols)), 128), vals


CASES = [  # E, H, I, slots of the experts in turn, dtype, overlay
    (3, 128, 128, [0, 1, 33], torch.bfloat16, False),
    (4, 384, 384, [31, 0, 32, 1], torch.float16, True),
    (6, 256, 640, [1, 2, 65, 0, 5, 17], torch.bfloat16, True),
    (1, 2048, 768, [20], torch.float16, False),
    (255, 128, 128, [1, 0, 3], torch.bfloat16, False),
    (128, 2048, 768, [16, 9, 33, 2], torch.bfloat16, True),
    (128, 2048, 768, [16, 30, 0], torch.float16, False),
    (2, 4096, 384, [19, 1], torch.bfloat16, False),
    (128, 640, 896, [16, 9, 33, 2], torch.bfloat16, False),  # down, d(act): unsplit blocks with two idle waves
]


@pytest.mark.parametrize("E,H,I,slots,dt,overlay", CASES, ids=lambda v: None if isinstance(v, list) else str(v))
def test_few_slots(gpu_device, E, H, I, slots, dt, overlay):
    dev = gpu_device
    gen = torch.Generator().manual_seed(E * 7 + H + I)
    counts = [slots[e % len(slots)] for e in range(E)]
    S, T = sum(counts), 64
    assert 0 < S <= 20 * E  # few enough for both directions
    print(f"[gpu-case] few slots E={E} H={H} I={I} S={S} {dt} overlay={overlay}", flush=True)
    qg, wg = _weight(E, 2 * I, H, gen, dev)
    qd, wd = _weight(E, H, I, gen, dev)
    ew = G.ExpertWeights(qg, qd)
    if overlay:
        for which, vals in (("gate_up", wg), ("down", wd)):
            idx = (torch.rand(vals.numel(), generator=gen) < 0.005).nonzero().reshape(-1)
            masters = torch.randint(-16, 17, (idx.numel(),), generator=gen).float()
            vals.view(-1)[idx] = masters.double()
            ew.set_overlay(which, idx.to(dev), masters.to(dev), dt)
    ints = lambda *s: torch.randint(-2, 3, s, generator=gen).to(dt)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    tok = torch.randint(0, T, (S,), generator=gen).to(torch.int32)
    # x with about 32 non-zeros a row: gate * up stays below fp16's largest value
    x = ints(T, H) * (torch.rand(T, H, generator=gen) < 32 / H).to(dt)
    act_in, dcur, dgu_in = ints(S, I), ints(S, H), ints(S, 2 * I)
    gu_in = torch.randn(S, 2 * I, generator=gen).to(dt)
    rows = [slice(int(offs[e]), int(offs[e + 1])) for e in range(E)]

    d = {n: t.to(dev) for n, t in (("x", x), ("act", act_in), ("dcur", dcur), ("dgu", dgu_in), ("gu", gu_in),
                                   ("tok", tok), ("offs", offs))}
    empty = lambda *s: torch.full(s, float("nan"), dtype=dt, device=dev)
    gu, act, y, dgu, dx = empty(S, 2 * I), empty(S, I), empty(S, H), empty(S, 2 * I), empty(S, H)
    table = G.blocked_layout(d["offs"], S)
    blk = empty(int(N.load().usaf_hip_blocked_elems(S, E, I)))
    code, st = N.dtype_code(dt), N.stream_ptr(dev)
    q, sz, _ = ew._ptrs("gate_up", dt)
    N.call("usaf_hip_moe_gate_up_fwd", d["x"].data_ptr(), T, H, d["tok"].data_ptr(), d["offs"].data_ptr(), S, E, I, q,
           sz, None, code, gu.data_ptr(), act.data_ptr(), blk.data_ptr(), table.data_ptr(), *ew._ovl("gate_up_fwd", dt), st)
    q, sz, _ = ew._ptrs("down", dt)
    N.call("usaf_hip_moe_down_fwd", d["act"].data_ptr(), I, d["offs"].data_ptr(), S, E, H, q, sz, None, code,
           y.data_ptr(), *ew._ovl("down_fwd", dt), st)
    N.call("usaf_hip_moe_down_bwd_t", d["dcur"].data_ptr(), H, d["gu"].data_ptr(), d["offs"].data_ptr(), S, E, I,
           *ew._ptrs_t("down"), code, dgu.data_ptr(), *ew._ovl("down_bwd", dt), st)
    N.call("usaf_hip_moe_gate_up_bwd_t", d["dgu"].data_ptr(), I, d["offs"].data_ptr(), S, E, H, *ew._ptrs_t("gate_up"),
           code, dx.data_ptr(), *ew._ovl("gate_up_bwd", dt), st)
    torch.cuda.synchronize()

    exact = lambda a, w, t: torch.cat([a[r].double() @ (w[e].t() if t else w[e]) for e, r in enumerate(rows)]).to(dt)
    assert torch.equal(gu.cpu(), exact(x[tok.long()], wg, True))
    assert torch.equal(y.cpu(), exact(act_in, wd, True))
    assert torch.equal(dx.cpu(), exact(dgu_in, wg, False))
    # act of the kernel's own gu; its blocked copy bit for bit
    tiny = float(torch.finfo(dt).tiny)
    def close(got, ref, gu):
        return bool(((got.double() - ref).abs() <= EPS[dt] * ref.abs() + tiny * (1 + gu)).all())
    g, u = gu.cpu().double().split(I, 1)
    assert close(act.cpu(), g * torch.sigmoid(g) * u, (g * u).abs())
    want = G.slot_blocked(act, d["offs"], S, table=table).data
    ld = (offs[1:] - offs[:-1] + 15) // 16 * 16
    n = int(ld.sum()) * I
    assert torch.equal(blk[:n].view(torch.int16), want[:n].view(torch.int16))
    # dgu from d(act) rounded once
    g, u = gu_in.double().split(I, 1)
    da, sig = exact(dcur, wd, False).double(), torch.sigmoid(g)
    assert close(dgu.cpu(), torch.cat([da * u * sig * (1 + g * (1 - sig)), da * g * sig], 1),
                 torch.cat([(da * u).abs(), (da * g).abs()], 1))


@pytest.mark.parametrize("gemm,E,cols,K,slots", [
    ("gate_up", 255, 160, 1536, [1, 0, 3]),  # split in two: the last block's second pair of waves has no rows
    ("gate_up", 8, 3008, 3072, [28, 33, 20]),  # four units a wave, split in four
    ("down", 8, 6016, 3072, [28, 33, 20]),
    ("d_act", 128, 2048, 1536, [16, 5, 33]),  # four units a wave, transposed, through the SwiGLU backward
])
def test_few_slots_one_gemm(gpu_device, gemm, E, cols, K, slots):
    """cols columns from a contraction of K (gate_up: cols gate and cols up rows; d_act:
    the gradients of gate and up from the transposed copy of a [K, cols] weight)."""
    dev, dt = gpu_device, torch.bfloat16
    gen = torch.Generator().manual_seed(E + cols + K)
    counts = [slots[e % len(slots)] for e in range(E)]
    S, rows, k = sum(counts), {"gate_up": 2 * cols, "down": cols, "d_act": K}[gemm], cols if gemm == "d_act" else K
    assert 0 < S <= (20 if gemm == "d_act" else 28) * E
    print(f"[gpu-case] few slots {gemm} E={E} cols={cols} K={K} S={S}", flush=True)
    q = torch.randint(-128, 128, (E, rows * k // 2), generator=gen, dtype=torch.int8)
    one = torch.ones(E * rows * k // 128, dtype=torch.float16)
    w = G.Q4Tensor(q.view(-1, 64).to(dev), one.to(dev), (-8 * one).to(dev), torch.Size((E, rows, k)), 128)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    x = torch.randint(-2, 3, (S, K), generator=gen).to(dt)
    gu = torch.randn(S, 2 * cols, generator=gen).to(dt)
    d_x, d_offs, d_rows, d_gu = x.to(dev), offs.to(dev), torch.arange(S, dtype=torch.int32, device=dev), gu.to(dev)
    out = torch.full((S, cols if gemm == "down" else 2 * cols), float("nan"), dtype=dt, device=dev)
    code, st = N.dtype_code(dt), N.stream_ptr(dev)
    if gemm == "gate_up":
        act = torch.empty(S, cols, dtype=dt, device=dev)
        N.call("usaf_hip_moe_gate_up_fwd", d_x.data_ptr(), S, K, d_rows.data_ptr(), d_offs.data_ptr(), S, E, cols,
               w.q.data_ptr(), w.scale_zero().data_ptr(), None, code, out.data_ptr(), act.data_ptr(), None, None,
               None, 0, st)
    elif gemm == "down":
        N.call("usaf_hip_moe_down_fwd", d_x.data_ptr(), K, d_offs.data_ptr(), S, E, cols, w.q.data_ptr(),
               w.scale_zero().data_ptr(), None, code, out.data_ptr(), None, 0, st)
    else:
        wt, szt = w.transposed()
        N.call("usaf_hip_moe_down_bwd_t", d_x.data_ptr(), K, d_gu.data_ptr(), d_offs.data_ptr(), S, E, cols,
               wt.data_ptr(), szt.data_ptr(), code, out.data_ptr(), None, 0, st)
    torch.cuda.synchronize()
    got = out.cpu()
    for e in range(E):
        a, b = int(offs[e]), int(offs[e + 1])
        if a == b:
            continue
        raw = q[e].view(torch.uint8)
        vals = torch.stack([raw & 15, raw >> 4], 1).double().view(rows, k) - 8
        if gemm != "d_act":
            assert torch.equal(got[a:b], (x[a:b].double() @ vals.t()).to(dt)), e
            continue
        da = (x[a:b].double() @ vals).to(dt).double()
        g, u = gu[a:b].double().split(cols, 1)
        sig = torch.sigmoid(g)
        ref = torch.cat([da * u * sig * (1 + g * (1 - sig)), da * g * sig], 1)
        tiny = float(torch.finfo(dt).tiny) * (1 + torch.cat([(da * u).abs(), (da * g).abs()], 1))
        assert bool(((got[a:b].double() - ref).abs() <= EPS[dt] * ref.abs() + tiny).all()), e
