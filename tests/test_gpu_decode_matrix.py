"""The matrix-core form of the decode step at the edges of its tiling: 64-token tiles, 512- and 1 024-token rounds of a
workgroup, and the fixed-point operands' range."""
import math

import numpy as np
import pytest
import torch

from oracle import cq_oracle as O
from tests.test_gpu_decode import _oracle, _run
from tests.test_gpu_token_mode import _token_case
from tests.util import make_case, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from calibquant_amd import ops
    return ops


def _close(got, want, rounding=2.0 ** -11):
    # fp16 results: one rounding (2^-11 of the value; bf16: 2^-8) on sums kept in 32 bits (a few 1e-6 of the largest, times the
    # logits' size in the exponent: logits of about 10)
    assert np.isfinite(got).all()
    bound = rounding * np.abs(want) + 1e-4 * np.abs(want).max()
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("case", [
    # B, Hq, Hkv, T: few units (1 024 threads) around a tile, a round and two rounds; one, two, three, four heads
    (1, 8, 8, 2), (1, 4, 4, 63), (1, 8, 4, 64), (1, 12, 4, 65), (2, 32, 8, 1023), (2, 32, 8, 1025), (1, 24, 4, 2049),
    # more units than compute units (512 threads): below and above a tile and a round
    (33, 32, 8, 63), (33, 32, 8, 129), (33, 32, 8, 513), (65, 24, 4, 577),
])
def test_tile_edges(ops, case, bits):
    B, Hq, Hkv, T = case
    print(f"case matrix {case} bits={bits}", flush=True)
    c = make_case(B, Hq, Hkv, 128, T, 0, bits, "fp16", seed=T)
    _close(_run(ops, c, "fp16", 0, bits), _oracle(c, 0, bits))


@pytest.mark.parametrize("bits", [1, 2])
def test_masked_tiles(ops, bits):
    """A mask that leaves out whole tiles, single tokens and the ragged end."""
    B, T = 3, 331
    c = make_case(B, 32, 8, 128, T, 0, bits, "fp16", seed=5)
    mask = np.zeros((B, T), np.float32)
    mask[0, :130] = mask[1, 1::2] = mask[2, 300:] = -1e4
    _close(_run(ops, c, "fp16", 0, bits, mask=mask), _oracle(c, 0, bits, mask=mask))


def test_query_of_any_scale(ops):
    """Queries far from 1 move the fixed-point grid; a query of zeros has no largest value to take it from."""
    for scale in (0.0, 2.0 ** -12, 2.0 ** 4):
        c = make_case(1, 32, 8, 128, 200, 0, 1, "fp16", seed=11)
        c["q"] = O.round_to(c["q"] * np.float32(scale), "fp16")
        _close(_run(ops, c, "fp16", 0, 1, calibrate=False), _oracle(c, 0, 1, calibrate_logits=False))


def test_infinity_in_one_head_stays_there(ops):
    c = make_case(1, 32, 8, 128, 200, 0, 1, "fp16", seed=12)
    want = _oracle(c, 0, 1)
    c["q"][0, 5, 17] = np.inf
    c["q"][0, 9, 3] = np.nan
    got = _run(ops, c, "fp16", 0, 1)
    hit = np.zeros(32, bool)
    hit[[5, 9]] = True
    assert np.isnan(got[0, hit]).all()
    _close(got[0, ~hit], want[0, ~hit])


@pytest.mark.parametrize("bits", [1, 2])
def test_logits_keep_small_channels_beside_a_large_one(ops, bits):
    """One channel's q.s_k is about 2^16 (its codes are 0, it adds nothing to any logit), the others' are 7/16 of 2^-6,
    once for every position a channel can have in a byte.  Odd tokens have all small codes, even tokens none."""
    cpb = 8 // bits                                 # channels per byte
    T, big = 200, 3
    odd = np.arange(T) % 2 == 1
    for pos in range(cpb):
        c = make_case(1, 32, 8, 128, T, 0, bits, "fp16", seed=13)
        small = np.arange(128) % cpb == pos
        small[big] = False
        q = np.where(small, 0.4375 * 2.0 ** -6 * 128 ** 0.5, 0.0)[None, :] * (1 + np.arange(32)[:, None] / 64)
        q[:, big] = 512.0
        c["q"] = O.round_to(q[None].astype(np.float32), "fp16")
        c["sk"][:], c["zk"][:] = 1.0, 0.0
        c["sk"][..., big] = 2048.0
        code = np.where(odd[:, None] & small[None, :], 1, 0)
        c["ck"][:] = O.encode(np.broadcast_to(code, (1, 8, T, 128)), bits)
        c["cv"][:] = O.encode(np.broadcast_to(odd[:, None], (1, 8, T, 128)), bits)
        c["sv"][:], c["zv"][:] = 1.0, 0.5
        got = _run(ops, c, "fp16", 0, bits, calibrate=False)
        k = code.astype(np.float64)
        w = (c["q"][0].astype(np.float64) / 128 ** 0.5) @ k.T
        p = np.exp(w - w.max(-1, keepdims=True))
        want = (p[:, odd].sum(-1) / p.sum(-1) - 0.5)[None, :, None]
        # fp32's own step at the large value is 2^-7; a channel may be off by half of 1/8 of that at most.  The weight of
        # the odd tokens moves by a quarter of a logit's change; then one rounding of the result.
        bound = small.sum() * 2.0 ** -11 / 4 + 2.0 ** -11 * np.abs(want) + 1e-6
        assert (np.abs(got - want) <= bound).all(), (pos, float((np.abs(got - want) / bound).max()))


def _token_run(ops, c, bits, dtype="fp16", mask=None, calibrate=True):
    import torch
    from tests.util import case_to_gpu, to_np
    g = case_to_gpu(c, dtype)
    out = ops.decode_attn(g["q"], g["ck"], g["cv"], g["sk"], g["zk"], g["sv"], g["zv"], None, None, bits=bits, v_mode="token",
                          mask=None if mask is None else torch.from_numpy(mask).cuda(), calibrate=calibrate)
    want = O.decode_attention(c["q"], c["ck"], c["cv"], c["sk"], c["zk"], c["sv"], c["zv"], None, None, 0, bits, v_token_group=32,
                              mask=mask, calibrate_logits=calibrate)
    return to_np(out), want


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("case", [
    # one, two, three, four heads per unit; around a tile, a round (1 024 tokens), four rounds and, beyond, eight
    (1, 8, 8, 2), (1, 4, 4, 63), (1, 8, 4, 65), (1, 12, 4, 64), (2, 32, 8, 1023), (33, 32, 8, 1025), (1, 8, 2, 4095), (1, 8, 2, 4097), (1, 2, 1, 5001),
])
def test_token_values_tile_edges(ops, case, bits):
    B, Hq, Hkv, T = case
    print(f"case token matrix {case} bits={bits}", flush=True)
    _close(*_token_run(ops, _token_case(B, Hq, Hkv, T, 0, bits, "fp16", seed=T), bits))


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("values", ["channel", "token"])
def test_logits_far_from_zero(ops, values, bits):
    """A channel with the same code in every token moves all logits of a head by 2^25 to 2^27, where fp32 has steps of 4
    and 8: the largest weight is 1 all the same, and a constant in the exponent would be off by powers of two."""
    T, odd = 200, np.arange(200) % 2 == 1
    c = _token_case(1, 32, 8, T, 0, bits, "fp16", seed=14) if values == "token" else make_case(1, 32, 8, 128, T, 0, bits, "fp16", seed=14)
    q = np.zeros((32, 128))
    q[:, 3] = 2.0 ** 14 * (1 + np.arange(32) / 16)        # times 2^15: the same for all tokens
    q[:, 40:44] = 512.0                                   # odd tokens: about 181 more
    c["q"] = O.round_to(q[None].astype(np.float32), "fp16")
    c["sk"][:], c["zk"][:] = 1.0, 0.0
    c["sk"][..., 3] = 2.0 ** 15
    code = np.zeros((T, 128), np.int64)
    code[:, 3] = 1
    code[odd, 40:44] = 1
    c["ck"][:] = O.encode(np.broadcast_to(code, (1, 8, T, 128)), bits)
    if values == "token":
        c["cv"][:] = np.where(odd, -1 if bits == 1 else 0x55555555, 0)[:, None]
        c["sv"][:], c["zv"][:] = 1.0, -0.5
        got, _ = _token_run(ops, c, bits, calibrate=False)
    else:
        c["cv"][:] = O.encode(np.broadcast_to(odd[:, None], (1, 8, T, 128)), bits)
        c["sv"][:], c["zv"][:] = 1.0, 0.5
        got = _run(ops, c, "fp16", 0, bits, calibrate=False)
    assert np.abs(got - 0.5).max() <= 2.0 ** -11          # the odd tokens' value: one rounding


@pytest.mark.parametrize("T", [200, 5000])
def test_mask_of_the_lowest_value_over_every_packed_token(ops, T):
    """fp32's lowest value on all packed tokens of the first sample (a padded prompt): its window alone counts."""
    c = make_case(2, 32, 8, 128, T, 40, 1, "fp16", seed=15)
    mask = np.zeros((2, T + 40), np.float32)
    mask[0, 8:8 + T] = np.finfo(np.float32).min
    _close(_run(ops, c, "fp16", 8, 1, mask=mask), _oracle(c, 8, 1, mask=mask))


def test_token_values_scales_far_apart(ops):
    """Every wave takes a head's grid from its largest weight times scale of a group; a group of zero scales has none."""
    c = _token_case(1, 32, 8, 300, 0, 1, "fp16", seed=3)
    c["sv"][:, :, 64:128] *= np.float32(2.0 ** -8)
    c["sv"][:, :, :, 1] = 0.0
    c["sv"][:, :, 5, 2] *= np.float32(2.0 ** 6)
    c["sv"] = O.round_to(c["sv"], "fp16")
    _close(*_token_run(ops, c, 1))


def test_token_values_infinite_scale_stays_in_its_group(ops):
    c = _token_case(1, 32, 8, 200, 0, 1, "fp16", seed=4)
    got, want = _token_run(ops, c, 1)
    c["sv"][0, 3, 17, 2] = np.inf
    hit, _ = _token_run(ops, c, 1)
    assert not np.isfinite(hit[0, 12:16, 64:96]).any()
    rest = np.ones(hit.shape, bool)
    rest[0, 12:16, 64:96] = False
    assert np.array_equal(hit[rest], got[rest])


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("dtype, far", [("fp16", 2.0 ** 15), ("bf16", 2.0 ** 40)])
def test_token_values_large_scale_of_a_token_without_weight(ops, dtype, far, bits):
    """A token's value scale may be of any size where its weight is zero: in the first sample it is masked (left padding),
    in the second one head of the unit gives it weight and the others give it none."""
    T = 200
    c = _token_case(2, 32, 8, T, 0, bits, dtype, seed=6)
    c["sv"] = O.round_to(c["sv"] * np.float32(2.0 ** -8), dtype)
    c["zv"] = O.round_to(c["zv"] * np.float32(2.0 ** -8), dtype)
    c["sv"][:, :, 7, 1] = far
    mask = np.zeros((2, T), np.float32)
    mask[0, :9] = -1e4
    # second sample: channel 0 tells token 7 from the others, exp(-100 * 16 / sqrt(128)) is 0 in fp32
    first = 1 << (8 - bits)                      # code 1 of a byte's first channel
    c["ck"][1, :, :, 0] &= first - 1
    c["ck"][1, :, 7, 0] |= first
    c["sk"][1, :, 0], c["zk"][1, :, 0] = 16.0, 0.0
    c["q"][1, :, 0] = -100.0
    c["q"][1, ::4, 0] = 0.0
    got, want = _token_run(ops, c, bits, dtype, mask, calibrate=False)
    for b in range(2):
        for h in range(32):
            _close(got[b, h], want[b, h], 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8)


@pytest.mark.parametrize("bits, vals, G, option", [(1, "channel", 4, "none"), (1, "channel", 3, "device-rows"), (2, "channel", 4, "mask"),
                                                   (1, "token", 4, "none"), (2, "token", 2, "device-rows")])
def test_decode_attn_streamed_rows_equal_a_small_batch(ops, bits, vals, G, option):
    """Launches that read most of the memory-side cache (168 MiB; at 2 bits 228 MiB) take their packed rows with
    non-temporal loads: the same arithmetic, so the first rows of such a batch equal a batch of their own in units of
    the same form, bit for bit.  (2 bits with per-token values: large, without such loads.)"""
    per = 32 * bits + (16 if vals == "token" else 0)
    H, T, R, S = 8, 1800, 20, 3
    B = ((168 if bits == 1 else 228) << 20) // (per * H * T) + 2
    g = torch.Generator(device="cuda").manual_seed(B)
    k = torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16)
    ck, sk, zk = ops.quantize_pack(k, bits, 0.5)
    cv, sv, zv = ops.quantize_pack_token(v, bits) if vals == "token" else ops.quantize_pack(v, bits, 0.5)
    del k, v
    q = torch.randn((B, H * G, 128), generator=g, device="cuda").to(torch.bfloat16)
    kr, vr = (torch.randn((B, H, R, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    mask = torch.where(torch.rand((B, T + R), generator=g, device="cuda") < 0.1, -1e4, 0.0) if option == "mask" else None

    def run(n):
        r_dev = torch.full((1,), R - 1, dtype=torch.int32, device="cuda") if option == "device-rows" else None
        call = ops.DecodeCall(q[:n].contiguous(), ck[:n], cv[:n], sk[:n], zk[:n], sv[:n], zv[:n], kr[:n], vr[:n], sprompt_len=S, bits=bits,
                              mask=None if mask is None else mask[:n].contiguous(), r_dev=r_dev, v_mode=vals)
        out = call.run().clone()
        torch.cuda.synchronize()
        p = call.plan()
        return out, (p["threads"], p["heads_per_unit"], p["chunks"])
    big, form = run(B)
    small, form2 = run(40)
    assert form == form2 and form[2] == 1
    assert torch.equal(big[:40], small)


@pytest.mark.parametrize("form", ["single", "mask", "chunked"])
@pytest.mark.parametrize("log_scale", [-13, -11, -9, -6])
def test_logit_range_below_the_resolution_of_the_logits(ops, form, log_scale):
    """Keys that differ by little beside what they share: logits of about 560 (one last place of fp32: 6e-5) that range over
    1e-5 to 1.4e-3.  The calibration stretches that range, so it is taken from the differences, not from the rounded
    logits."""
    T = 40000 if form == "chunked" else 300
    B, Hq, Hkv = 1, 4, 1
    rng = np.random.default_rng(6)
    c = make_case(B, Hq, Hkv, 128, T, 0, 1, "fp16", seed=6)
    bit = np.zeros((B, Hkv, T, 128), np.uint8)
    bit[..., 0] = rng.integers(0, 2, size=(B, Hkv, T))
    c["ck"] = O.encode(bit, 1)
    c["q"] = np.ones_like(c["q"])
    c["sk"] = np.ones_like(c["sk"])
    c["sk"][..., 0] = 2.0 ** log_scale
    c["zk"] = np.full_like(c["zk"], 50.0)
    mask = np.zeros((B, T), np.float32) if form == "mask" else None
    got = _run(ops, c, "fp16", 0, 1, mask=mask)
    want = O.decode_attention(c["q"], c["ck"], c["cv"], c["sk"], c["zk"], c["sv"], c["zv"], None, None, 0, 1, mask=mask, ftype=np.float64)
    _close(got, want)


def _window_case(B, Hq, Hkv, T, rows, dtype, seed):
    c = make_case(B, Hq, Hkv, 128, max(T, 64), rows, 1, dtype, seed=seed)
    if T == 0:
        c["ck"], c["cv"] = c["ck"][:, :, :0], c["cv"][:, :, :0]
    return c


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 4, 1), (6, 32, 8), (30, 12, 4), (20, 16, 4), (40, 32, 8)])   # 1, 2, 3 and 4 heads in 1 024 threads, 4 in 512
def test_window_edges(ops, shape, dtype):
    """Windows around a wave's 8 or 16 rows, a tile's 128 and the first row of the next, with and without packed tokens."""
    B, Hq, Hkv = shape
    for T, rows in ((0, 1), (0, 129), (70, 7), (70, 9), (70, 16), (70, 17), (70, 127), (70, 128), (70, 257)):
        print(f"case window {shape} {dtype} T={T} rows={rows}", flush=True)
        c = _window_case(B, Hq, Hkv, T, rows, dtype, rows)
        _close(_run(ops, c, dtype, min(rows, 5), 1), _oracle(c, min(rows, 5), 1), 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8)


@pytest.mark.parametrize("batch", [1, 70, 300])   # 1 head in 1 024 threads, 4 in 1 024, 4 in 512
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_window_weights_of_all_sizes(ops, dtype, batch):
    """One row weighs 1, the others 2^-12 to 2^-22 each but have values of 512 times its size, which adds up: the parts a weight is held in
    keep small ones as exactly as large ones.  An infinite value in the row of weight 1 makes its channel infinite and no other."""
    B, Hq, Hkv, R = batch, 4, 1, 130
    c = _window_case(B, Hq, Hkv, 0, R, dtype, 3)
    c["q"][:] = 0
    c["q"][..., 0] = 8.0
    c["kr"][:] = 0
    c["kr"][:, 0, :, 0] = -np.linspace(12, 21, R)
    c["kr"][:, 0, 77, 0] = 0
    c["vr"] = np.where(np.arange(R)[:, None] == 77, 0.25, 128.0 * (1 + np.arange(R)[:, None] % 7) / 7) * np.ones_like(c["vr"])
    c["vr"] = O.round_to(c["vr"].astype(np.float32), dtype)
    rounding = 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8
    _close(_run(ops, c, dtype, 0, 1), _oracle(c, 0, 1), rounding)
    c["vr"][:, 0, 77, 3] = np.inf
    got, want = _run(ops, c, dtype, 0, 1), _oracle(c, 0, 1)
    assert (got[..., 3] == np.inf).all()   # (a weight of 1 on an infinite value, none on any other)
    _close(np.delete(got, 3, -1), np.delete(want, 3, -1), rounding)


@pytest.mark.parametrize("form", [(1, 1), (1, 4), (70, 4), (300, 4), (100, 3), (300, 2)])   # (batch, heads): units of 1, 4 (in 1 024 threads, in 512), 3 and 2 heads
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_infinite_value_of_a_row_of_small_weight(ops, dtype, form):
    """A row whose weight is no zero in 32 bits and whose value is infinite makes the channel infinite, however small the weight, in units of all
    widths; no other channel notices."""
    B, Hq = form
    rounding = 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8
    for octaves in (13, 24.5, 25.5, 40, 60, 120):
        print(f"case infinite value {form} {dtype} weight 2^-{octaves}", flush=True)
        c = _window_case(B, Hq, 1, 0, 130, dtype, 3)
        c["q"][:], c["kr"][:] = 0, 0
        c["q"][..., 0] = 8.0
        c["kr"][:, 0, :, 0] = -140.0                # e^-99 of the largest: adds nothing
        c["kr"][:, 0, 77, 0] = 0
        c["kr"][:, 0, 40, 0] = -octaves * math.log(2) * math.sqrt(128) / 8
        c["kr"] = O.round_to(c["kr"].astype(np.float32), dtype)
        want = _oracle(c, 0, 1)
        c["vr"][:, 0, 40, 3], c["vr"][:, 0, 40, 64] = np.inf, -np.inf
        got = _run(ops, c, dtype, 0, 1)
        assert (got[..., 3] == np.inf).all() and (got[..., 64] == -np.inf).all()
        _close(np.delete(got, (3, 64), -1), np.delete(want, (3, 64), -1), rounding)


def test_query_and_statistics_on_odd_addresses(ops):
    """q and the statistics are read two values at a time and need no alignment beyond their own."""
    def odd(t):
        o = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return o.copy_(t)
    g = torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.bfloat16)
    ck, sk, zk = ops.quantize_pack(r(2, 150, 4, 128), 1, 0.5)
    cv, sv, zv = ops.quantize_pack(r(2, 150, 4, 128), 1, 0.3)
    q = r(2, 16, 128)
    want = ops.decode_attn(q, ck, cv, sk, zk, sv, zv, None, None, sprompt_len=0, bits=1)
    got = ops.decode_attn(odd(q), ck, cv, odd(sk), odd(zk), odd(sv), odd(zv), None, None, sprompt_len=0, bits=1)
    assert torch.equal(got, want)


@pytest.mark.parametrize("splits", [0, 2])
@pytest.mark.parametrize("shape", [(1, 4, 4), (2, 8, 4), (3, 24, 8), (17, 32, 4), (40, 32, 8)])   # units of 1, 2, 3 and 4 heads, the last in 512 threads
@pytest.mark.parametrize("bits, vals", [(1, "channel"), (2, "channel"), (1, "token"), (2, "token")])
def test_mask_and_row_count_are_forms_of_one_call(ops, shape, bits, vals, splits):
    """The call without either, with the window's length on the device and with a mask, whole and in chunks: the row count changes no bit, a mask of
    zeros only the order in which a logit is put together, and a masked row of the window is as if it were not there."""
    B, Hq, Hkv = shape
    T, R, S = 700, 140, 5
    print(f"case forms {shape} bits={bits} {vals} splits={splits}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B * bits)
    r = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float16)
    ck, sk, zk = ops.quantize_pack(r(B, T, Hkv, 128), bits, 0.5)
    cv, sv, zv = ops.quantize_pack_token(r(B, T, Hkv, 128), bits) if vals == "token" else ops.quantize_pack(r(B, T, Hkv, 128), bits, 0.5)
    q, kr, vr = r(B, Hq, 128), r(B, Hkv, R, 128), r(B, Hkv, R, 128)
    run = lambda rows, **kw: ops.decode_attn(q, ck, cv, sk, zk, sv, zv, kr[:, :, :rows], vr[:, :, :rows], sprompt_len=S, bits=bits, v_mode=vals,
                                             force_splits=splits, **kw)
    plain, shorter = run(R), run(R - 3)
    assert torch.equal(run(R, r_dev=torch.full((1,), R, dtype=torch.int32, device="cuda")), plain)
    assert torch.equal(run(R, r_dev=torch.full((1,), R - 3, dtype=torch.int32, device="cuda")), shorter)
    mask = torch.zeros((B, T + R), device="cuda")
    _close(to_np(run(R, mask=mask)), to_np(plain), 2.0 ** -10)   # (both results are rounded to fp16: up to half a step, 2^-11 of them, each)
    mask[:, T + R - 3:] = -1e4
    _close(to_np(run(R, mask=mask)), to_np(shorter), 2.0 ** -10)
