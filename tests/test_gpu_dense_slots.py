"""The grouped GEMMs on dense weights at short m-tiles (moe_dense.hip), in all
three weight orders, where their tiles end: experts without slots, with 1, 31, 32,
33, 95 to 97 and 127 to 129, one expert only, 255 experts, widths that leave waves
without columns, one and odd counts of k-steps, weights behind a slot table; and the
persistent kernels (moe_gemm.hip) past the line of each order.

Weights in [-8, 7] and activations in [-2, 2] are integers: every sum is exact in
fp32 in any order, and outputs rounded once must equal the 64-bit product rounded
to the dtype, bit for bit.  act and dgu go through a sigmoid of a few ulp of fp32
and up to three roundings to the dtype, each of which may fall the other way:
3 half-ulp steps, 3 * 2^-8 of the value in bf16 and 3 * 2^-11 in fp16; a value
below the smallest normal may vanish on the way: that normal times 1 + |g u|.
"""
import pytest
import torch

from usaf_amd import _native as N
from usaf_amd import moe as G
from usaf_amd.expert_cache import frag_chunk_index

pytestmark = pytest.mark.gpu
EPS = {torch.bfloat16: 3 * 2.0 ** -8, torch.float16: 3 * 2.0 ** -11}


def _arena(w, inter, slot_of, n_slots):
    """[E, rows, K] weights as fragment-order slots (NaN where nothing is stored)."""
    E, rows, k = w.shape
    idx = frag_chunk_index(rows, k, inter)
    out = torch.full((n_slots, idx.numel(), 8), float("nan"), dtype=w.dtype)
    for e in range(E):
        out[slot_of[e], idx >= 0] = w[e].reshape(-1, 8)[idx[idx >= 0]]
    assert out[0].numel() == int(N.load().usaf_hip_frag_slot_elems(rows, k, inter))
    return out


CASES = [  # E, H, I, slots of the experts in turn, dtype
    (3, 128, 128, [0, 1, 129], torch.bfloat16),
    (5, 384, 128, [31, 0, 32, 33, 97], torch.float16),
    (6, 256, 640, [1, 128, 65, 0, 127, 95], torch.bfloat16),
    (1, 2048, 768, [80], torch.float16),
    (255, 128, 128, [1, 0, 3], torch.bfloat16),
    (2, 1152, 384, [96, 64], torch.bfloat16),
]


@pytest.mark.parametrize("E,H,I,slots,dt", CASES, ids=lambda v: None if isinstance(v, list) else str(v))
def test_dense_slots(gpu_device, E, H, I, slots, dt):
    counts = [slots[e % len(slots)] for e in range(E)]
    assert 0 < sum(counts) <= 80 * E  # few enough for every order
    _run(gpu_device, E, H, I, counts, dt)


# slots per expert on either side of each order's line: rows 80, fragment 96, [K, N] 128
@pytest.mark.parametrize("slots", [81, 96, 97, 128, 129, 321])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_dense_slots_lines(gpu_device, slots, dt):
    _run(gpu_device, 3, 256, 384, [slots + 7, slots - 7, slots], dt)


@pytest.mark.parametrize("H,I", [(64, 128), (192, 128), (128, 32), (256, 96), (128, 160)])
def test_dense_slots_odd_k_steps(gpu_device, H, I):
    """One and odd counts of 64-wide k-steps, and widths that leave waves without columns
    (the GEMMs whose shapes take them)."""
    _run(gpu_device, 3, H, I, [33, 0, 65], torch.bfloat16)


def _run(gpu_device, E, H, I, counts, dt):
    """Every GEMM whose shape allows H and I, against the 64-bit products."""
    dev = gpu_device
    gen = torch.Generator().manual_seed(E * 7 + H + I)
    S, T = sum(counts), 64
    print(f"[gpu-case] dense slots E={E} H={H} I={I} S={S} {dt}", flush=True)
    ints = lambda lo, hi, *s: torch.randint(lo, hi + 1, s, generator=gen).to(dt)
    wg, wd = ints(-8, 7, E, 2 * I, H), ints(-8, 7, E, H, I)
    slot_of = torch.randperm(E + 3, generator=gen)[:E]
    wide_h, wide_i = H % 128 == 0, I % 128 == 0  # contraction (gate_up; down) and down's activations
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    tok = torch.randint(0, T, (S,), generator=gen).to(torch.int32)
    # x with about 32 non-zeros a row: gate * up stays below fp16's largest value
    x = ints(-2, 2, T, H) * (torch.rand(T, H, generator=gen) < 32 / H).to(dt)
    act_in, dcur, dgu_in = ints(-2, 2, S, I), ints(-2, 2, S, H), ints(-2, 2, S, 2 * I)
    gu_in = torch.randn(S, 2 * I, generator=gen).to(dt)
    rows = [slice(int(offs[e]), int(offs[e + 1])) for e in range(E)]
    exact = lambda a, w, t: torch.cat(
        [a[r].double() @ (w[e].double().t() if t else w[e].double()) for e, r in enumerate(rows)]).to(dt)
    tiny = float(torch.finfo(dt).tiny)

    def close(got, ref, gu):
        return bool(((got.double() - ref).abs() <= EPS[dt] * ref.abs() + tiny * (1 + gu)).all())

    d = {n: t.to(dev) for n, t in (("x", x), ("act", act_in), ("dcur", dcur), ("dgu", dgu_in), ("gu", gu_in),
                                   ("tok", tok), ("offs", offs), ("wg", wg), ("wd", wd),
                                   ("slot", slot_of.to(torch.int32)))}
    if wide_h and wide_i:
        d["ag"], d["ad"] = _arena(wg, I, slot_of, E + 3).to(dev), _arena(wd, 0, slot_of, E + 3).to(dev)
    empty = lambda *s: torch.full(s, float("nan"), dtype=dt, device=dev)
    code, st = N.dtype_code(dt), N.stream_ptr(dev)
    table = G.blocked_layout(d["offs"], S)
    blk = empty(int(N.load().usaf_hip_blocked_elems(S, E, I)))
    for order in ("rows", "fragment"):
        if order == "fragment" and not (wide_h and wide_i):
            continue
        gu, act, y = empty(S, 2 * I), empty(S, I), empty(S, H)
        if order == "rows":
            if wide_h:
                N.call("usaf_hip_moe_gate_up_fwd", d["x"].data_ptr(), T, H, d["tok"].data_ptr(), d["offs"].data_ptr(),
                       S, E, I, None, None, d["wg"].data_ptr(), code, gu.data_ptr(), act.data_ptr(), blk.data_ptr(),
                       table.data_ptr(), None, 0, st)
            if wide_i:
                N.call("usaf_hip_moe_down_fwd", d["act"].data_ptr(), I, d["offs"].data_ptr(), S, E, H, None, None,
                       d["wd"].data_ptr(), code, y.data_ptr(), None, 0, st)
        else:
            N.call("usaf_hip_moe_gate_up_fwd_slots", d["x"].data_ptr(), T, H, d["tok"].data_ptr(), d["offs"].data_ptr(),
                   S, E, I, d["ag"].data_ptr(), d["slot"].data_ptr(), E + 3, code, gu.data_ptr(), act.data_ptr(), st)
            N.call("usaf_hip_moe_down_fwd_slots", d["act"].data_ptr(), I, d["offs"].data_ptr(), S, E, H,
                   d["ad"].data_ptr(), d["slot"].data_ptr(), E + 3, code, y.data_ptr(), st)
        torch.cuda.synchronize()
        if wide_i:
            assert torch.equal(y.cpu(), exact(act_in, wd, True)), order
        if wide_h:
            assert torch.equal(gu.cpu(), exact(x[tok.long()], wg, True)), order
            g, u = gu.cpu().double().split(I, 1)
            assert close(act.cpu(), g * torch.sigmoid(g) * u, (g * u).abs()), order
        if wide_h and order == "rows":  # act's blocked copy (a transpose behind the GEMM), bit for bit
            want = G.slot_blocked(act, d["offs"], S, table=table).data
            n = int(((offs[1:] - offs[:-1] + 15) // 16 * 16).sum()) * I
            assert torch.equal(blk[:n].view(torch.int16), want[:n].view(torch.int16))

    dgu, dx = empty(S, 2 * I), empty(S, H)
    if wide_i:
        N.call("usaf_hip_moe_down_bwd", d["dcur"].data_ptr(), H, d["gu"].data_ptr(), d["offs"].data_ptr(), S, E, I, None,
               None, d["wd"].data_ptr(), code, dgu.data_ptr(), st)
    if wide_h:
        N.call("usaf_hip_moe_gate_up_bwd", d["dgu"].data_ptr(), I, d["offs"].data_ptr(), S, E, H, None, None,
               d["wg"].data_ptr(), code, dx.data_ptr(), st)
    torch.cuda.synchronize()
    if wide_h:
        assert torch.equal(dx.cpu(), exact(dgu_in, wg, False))
    if wide_i:
        g, u = gu_in.double().split(I, 1)
        da, sig = exact(dcur, wd, False).double(), torch.sigmoid(g)
        assert close(dgu.cpu(), torch.cat([da * u * sig * (1 + g * (1 - sig)), da * g * sig], 1),
                     torch.cat([(da * u).abs(), (da * g).abs()], 1))
