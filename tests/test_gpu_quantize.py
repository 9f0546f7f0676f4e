"""GPU parity of the prefill quantise-and-pack kernels against the oracle:
bit-exact codes, scales and zero-points (through the C-ABI library)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import cq_oracle as O
from tests.util import CLIPS, TDT, same_bits, to_gpu, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from calibquant_amd import ops
    return ops


SHAPES = [(2, 257, 3, 128), (1, 1, 2, 128), (3, 63, 1, 64), (1, 1000, 2, 256), (2, 3328, 8, 128),
          (1, 1500, 1, 128), (1, 2100, 2, 128), (1, 5000, 2, 128)]   # one-pass kernel row counts; beyond its reach


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_quantize_pack_bit_exact(ops, shape, bits, dtype):
    B, T, H, D = shape
    print(f"case quantize_pack shape={shape} bits={bits} dtype={dtype}", flush=True)
    k, v = O.synth_kv(B, T, H, D, dtype, seed=B * 1000 + T)
    for x, clip in zip((k, v), CLIPS[bits]):
        codes, s, z = ops.quantize_pack(to_gpu(x, dtype), bits, clip)
        torch.cuda.synchronize()
        oc, os_, oz = O.quantize_pack(x, bits, clip, dtype)
        assert same_bits(to_np(s), os_)
        assert same_bits(to_np(z), oz)
        assert np.array_equal(codes.cpu().numpy(), oc)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_quantize_pack_reads_the_strided_wqkv_view(ops, dtype):
    """The reference quantises views of the fused wqkv output
    (patch_internvl.py:219-234, 284, 290): token stride (Hq+2Hkv)*D, head stride (G+2)*D."""
    B, N, Hkv, G, D, S, T = 2, 300, 2, 4, 128, 41, 200
    rng = np.random.default_rng(0)
    qkv = O.round_to(rng.standard_normal((B, N, Hkv, G + 2, D), dtype=np.float32), dtype)
    t = to_gpu(qkv, dtype)
    kview = t[:, S:S + T, :, G, :]
    vview = t[:, S:S + T, :, G + 1, :]
    assert not kview.is_contiguous()
    for view, ref, clip in ((kview, qkv[:, S:S + T, :, G], 0.5), (vview, qkv[:, S:S + T, :, G + 1], 0.3)):
        codes, s, z = ops.quantize_pack(view, 1, clip)
        oc, os_, oz = O.quantize_pack(ref, 1, clip, dtype)
        assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
        assert np.array_equal(codes.cpu().numpy(), oc)


@pytest.mark.parametrize("bits", [1, 2])
def test_quantize_pack_long_context_single_sequence(ops, bits):
    """One sequence of 32 768 tokens: few (batch, head) pairs, so the statistics of a channel are
    folded from 256 chunk partials and every threshold level is searched by its own threads."""
    B, T, H, D = 1, 32768, 2, 128
    print(f"case quantize_pack long context bits={bits}", flush=True)
    k, v = O.synth_kv(B, T, H, D, "bf16", seed=77)
    for x, clip in zip((k, v), CLIPS[bits]):
        codes, s, z = ops.quantize_pack(to_gpu(x, "bf16"), bits, clip)
        torch.cuda.synchronize()
        oc, os_, oz = O.quantize_pack(x, bits, clip, "bf16")
        assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
        assert np.array_equal(codes.cpu().numpy(), oc)


def test_quantize_pack_constant_channel_matches_ieee_reference(ops):
    x = np.random.default_rng(1).standard_normal((1, 64, 2, 128)).astype(np.float32)
    x = O.round_to(x, "bf16")
    x[0, :, 1, 5] = 1.5        # scale 0, zero -inf, codes NaN -> index 0
    x[0, :, 0, 9] = -2.0       # scale 0, zero +inf
    x[0, :, 0, 17] = 0.0       # scale 0, zero NaN
    codes, s, z = ops.quantize_pack(to_gpu(x, "bf16"), 1, 0.5)
    oc, os_, oz = O.quantize_pack(x, 1, 0.5, "bf16")
    assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
    assert np.array_equal(codes.cpu().numpy(), oc)
    assert to_np(s)[0, 1, 5] == 0 and np.isinf(to_np(z)[0, 1, 5])


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
def test_quant_and_encode_operators(ops, bits, dtype):
    """The unfused pair quant() + encode() gives the same bytes as the fused kernel."""
    B, T, H, D = 2, 130, 2, 128
    k, _ = O.synth_kv(B, T, H, D, dtype, seed=3)
    x = to_gpu(k, dtype)
    clip = CLIPS[bits][0]
    xq, s, z = ops.quant_codes(x, bits, clip)
    oxq, os_, oz = O.quant(k, bits, clip, dtype)
    assert same_bits(to_np(xq), oxq) and same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
    for idx in (xq.transpose(1, 2).contiguous(), xq.transpose(1, 2).long(), xq.transpose(1, 2).to(torch.int32),
                xq.transpose(1, 2).to(torch.uint8)):
        enc = ops.encode_indices(idx, bits)
        codes, _, _ = ops.quantize_pack(x, bits, clip)
        assert torch.equal(enc, codes)


@pytest.mark.parametrize("B", [4, 64])
@pytest.mark.parametrize("bits", [1, 2])
def test_quantize_pack_matches_torch_device_op_chain(ops, bits, B):
    """torch's own device kernels, run op by op on the 16-bit tensor, are the
    primitives the reference executes (calibquant.py:27-36).  At batch 64 (the benchmark's prefill
    tensor) every workgroup of the one-pass kernel walks four parts of pairs, whose rows it requests while it packs
    the part before."""
    T, H, D = 3328, 8, 128
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((B, T, H, D), generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)
    clip = CLIPS[bits][0]
    L = 2 ** bits - 1
    mn = x.amin(dim=1, keepdim=True) * clip
    mx = x.amax(dim=1, keepdim=True) * clip
    s = (mx - mn) / L
    z = -mn / s
    xq = torch.round(torch.clamp(x / s + z, 0, L))
    codes, ks, kz = ops.quantize_pack(x, bits, clip)
    assert torch.equal(ks, s[:, 0]) and torch.equal(kz, z[:, 0])
    enc = ops.encode_indices(xq.transpose(1, 2).contiguous(), bits)
    assert torch.equal(enc, codes)


@pytest.mark.parametrize("bits", [1, 2])
def test_quantize_pack_full_size_properties(ops, bits):
    """Prefill tensor of the long-context configuration (1, 32768, 8, 128):
    size-independent properties.  Codes lie in range, every channel attains
    code 0 and code L when clip == 1, and dequantising then re-quantising
    reproduces the bytes."""
    B, T, H, D = 1, 32768, 8, 128
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((B, T, H, D), generator=g, device="cuda").to(torch.bfloat16)
    codes, s, z = ops.quantize_pack(x, bits, 1.0)
    L = 2 ** bits - 1
    dpe = 8 // bits
    shifts = torch.tensor([bits * (dpe - 1 - i) for i in range(dpe)], device="cuda", dtype=torch.uint8)
    un = ((codes[..., None] >> shifts) & L).reshape(B, H, T, D)
    assert int(un.amin()) == 0 and int(un.amax()) == L
    assert torch.all(un.amin(dim=2) == 0) and torch.all(un.amax(dim=2) == L)
    # fixed point: re-quantising the dequantised tensor in fp32-exact levels keeps the codes
    deq = (s.float()[:, :, None] * (un.float() - z.float()[:, :, None])).to(torch.bfloat16)
    codes2, _, _ = ops.quantize_pack(deq.transpose(1, 2), bits, 1.0)
    un2 = ((codes2[..., None] >> shifts) & L).reshape(B, H, T, D)
    assert (un2 != un).float().mean().item() < 2e-3


# Token axes beyond what one workgroup's registers hold (832 rows, 3 328 of a quarter of the channels): several parts of a
# pair's rows, whose workgroups exchange their extremes.
LONG_SHAPES = [(2, 9984, 8, 128),    # the 26B prompt's token count
               (3, 3329, 2, 128),    # just beyond one workgroup
               (4, 13000, 1, 128),
               (2, 40000, 2, 128),
               (1, 40000, 1, 128),   # a single (batch, head) pair
               (9, 5000, 8, 128),    # more parts than workgroups
               (2, 7000, 8, 128)]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", LONG_SHAPES)
def test_quantize_pack_long_token_axis_bit_exact(ops, shape, bits, dtype):
    B, T, H, D = shape
    print(f"case quantize_pack long shape={shape} bits={bits} dtype={dtype}", flush=True)
    k, _ = O.synth_kv(B, T, H, D, dtype, seed=T + bits)
    clip = CLIPS[bits][0]
    codes, s, z = ops.quantize_pack(to_gpu(k, dtype), bits, clip)
    torch.cuda.synchronize()
    oc, os_, oz = O.quantize_pack(k, bits, clip, dtype)
    assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
    assert np.array_equal(codes.cpu().numpy(), oc)


def test_quantize_pack_long_token_axis_strided_view(ops):
    B, N, Hkv, G, D, S, T = 2, 10100, 2, 4, 128, 41, 9984
    rng = np.random.default_rng(5)
    qkv = O.round_to(rng.standard_normal((B, N, Hkv, G + 2, D), dtype=np.float32), "bf16")
    t = to_gpu(qkv, "bf16")
    view = t[:, S:S + T, :, G, :]
    assert not view.is_contiguous()
    codes, s, z = ops.quantize_pack(view, 1, 0.5)
    oc, os_, oz = O.quantize_pack(qkv[:, S:S + T, :, G], 1, 0.5, "bf16")
    assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
    assert np.array_equal(codes.cpu().numpy(), oc)


def test_quantize_pack_split_slices_give_up_and_the_host_reports_it(ops):
    """The parts of a pair wait for each other a bounded number of polls.  A bound of zero takes their exchange out of
    service: every part goes on alone (the kernel ends normally; its statistics are those of single parts, i.e. not
    valid), the call returns success, the next call on the device reports the failure once, and from then on shapes of
    several parts take the three-launch path - bit-exact - until the bound is set again."""
    from calibquant_amd import _lib
    lib = _lib.load()
    B, T, H, D = 2, 9984, 2, 128
    k, _ = O.synth_kv(B, T, H, D, "bf16", seed=31)
    x = to_gpu(k, "bf16")
    oc, os_, oz = O.quantize_pack(k, 1, 0.5, "bf16")

    def check():
        codes, s, z = ops.quantize_pack(x, 1, 0.5)
        torch.cuda.synchronize()
        assert same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
        assert np.array_equal(codes.cpu().numpy(), oc)
    check()
    before = lib.cq_quantize_pack_wait_polls(0)
    try:
        ops.quantize_pack(x, 1, 0.5)          # launched; every part gives up
        torch.cuda.synchronize()
        with pytest.raises(_lib.CalibQuantError):
            ops.quantize_pack(x, 1, 0.5)      # the host finds the word set
        check()                               # three launches from here on
    finally:
        lib.cq_quantize_pack_wait_polls(before)
    check()


# What the one-pass kernel makes of a shape: whole rows or quarters, one part or several, one id per workgroup or a walk.
# Edges of passes (16 and 64 rows), of the rows a thread holds, of the parts; pair counts that are no multiple of eight.
CUT_SHAPES = [(1, 1, 1), (1, 2, 8), (2, 63, 3), (3, 65, 5), (1, 255, 2), (2, 833, 3), (1, 3329, 4), (5, 832, 8), (70, 831, 2),
              (67, 16, 8), (90, 333, 8), (1, 4097, 8), (2, 6657, 7), (21, 1700, 8)]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", CUT_SHAPES)
def test_quantize_pack_one_pass_cuts_bit_exact(ops, shape, bits, dtype):
    """Codes and statistics equal the oracle's bit for bit; channels of one sign, of equal values, with zeros of
    both signs and with infinities among them."""
    B, T, H = shape
    print(f"case quantize_pack cut shape={shape} bits={bits} dtype={dtype}", flush=True)
    rng = np.random.default_rng(T * 31 + B)
    x = O.round_to(rng.standard_normal((B, T, H, 128), dtype=np.float32), dtype)
    x[..., 3] = np.abs(x[..., 3])
    x[..., 50] = -np.abs(x[..., 50])
    x[:, T // 2:, :, 51] = np.abs(x[:, T // 2:, :, 51])      # one sign in some threads' rows only
    x[..., 77] = 1.5
    x[..., 78] = -0.0
    x[:, ::2, :, 79] = 0.0
    x[:, T // 3, :, 90] = np.inf
    x[:, T - 1, :, 91] = -np.inf
    x[..., 127] *= O.round_to(np.float32(2.0 ** -12), dtype)
    x = O.round_to(x, dtype)
    with np.errstate(all="ignore"):
        oc, os_, oz = O.quantize_pack(x, bits, CLIPS[bits][0], dtype)
    codes, s, z = ops.quantize_pack(to_gpu(x, dtype), bits, CLIPS[bits][0])
    torch.cuda.synchronize()
    # (equal values: the sign of a zero minimum is the only one that min() over +0 and -0 leaves open)
    assert same_bits(to_np(s), os_) and np.array_equal(to_np(z), oz, equal_nan=True)
    assert np.array_equal(codes.cpu().numpy(), oc)


@pytest.mark.parametrize("shape", [(2, 3328, 8), (1, 20000, 2), (4, 300, 8)])
def test_quantize_pack_recorded_and_replayed(ops, shape):
    """A recorded pass whose parts exchange their extremes comes back with the same epoch: what an earlier replay left in
    the workspace must not be taken for this one's.  New inputs in place for each replay, eager work between them."""
    B, T, H = shape
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16)
    ops.quantize_pack(x, 1, 0.5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.quantize_pack(x, 1, 0.5)
    for k in range(4):
        x.copy_(torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16) * (3.0 if k == 0 else 1.0 / (k + 1)))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, ops.quantize_pack(x, 1, 0.5)):
            assert torch.equal(a, b)


def test_quantize_pack_takes_no_record_from_what_the_workspace_held(ops):
    """The parts' exchange records are recognised by their contents, and the workspace is whatever memory was free.  Here its
    words hold the coming call's epoch above extremes that no part has - half of them taken from the upper half of the
    first record's first word (what the minima stand below), half from that and the maxima."""
    from calibquant_amd import _lib
    lib = _lib.load()
    B, T, H, D = 4, 9984, 8, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((B, T, H, D), generator=g, device="cuda").to(torch.bfloat16)
    ws = torch.zeros(lib.cq_quantize_pack_workspace(B, T, H, D), dtype=torch.uint8, device="cuda")

    def call():
        codes = torch.empty((B, H, T, D // 8), dtype=torch.uint8, device="cuda")
        s, z = (torch.empty((B, H, D), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        _lib.check(lib.cq_quantize_pack(x.data_ptr(), 0, B, T, H, D, *x.stride()[:3], 1, 0.5, codes.data_ptr(), s.data_ptr(),
                                        z.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "cq_quantize_pack")
        torch.cuda.synchronize()
        return codes, s, z
    want = call()
    words = ws[:ws.numel() // 32 * 32].view(torch.int64)

    def first_record():
        lo, hi = (int(w) & (1 << 64) - 1 for w in words[:2])
        return lo >> 32, lo >> 32 ^ hi & 0xffffffff
    upper, epoch = first_record()
    assert epoch != 0, "several parts per pair leave their records in the workspace"
    for i, e in enumerate((upper, epoch, epoch, upper)):
        words[i::4] = torch.tensor(((e + 1) << 32 | 0x7f008080) - (1 << 64 if e >> 31 else 0), device="cuda")
    for a, b in zip(call(), want):
        assert torch.equal(a, b)
    assert first_record()[1] == epoch + 1


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", [(4, 9984, 8), (1, 9984, 8), (3, 3329, 2), (1, 40000, 1), (64, 1700, 8)])
def test_quantize_pack_parts_that_wait_in_vain_read_the_rows_themselves(ops, shape, bits, dtype):
    """With a bound of one poll nearly every part misses others' extremes and reads those rows again: the same result,
    nothing is reported, and the next call is an ordinary one."""
    from calibquant_amd import _lib
    lib = _lib.load()
    B, T, H = shape
    print(f"case quantize_pack in vain shape={shape} bits={bits} dtype={dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + B)
    x = torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16 if dtype == "bf16" else torch.float16)
    x[..., 3] = x[..., 3].abs()
    x[:, T // 2:, :, 50] = -x[:, T // 2:, :, 50].abs()
    x[:, T // 3, :, 90] = float("inf")
    x[..., 91] = 0.0
    x[:, ::2, :, 91] = -0.0
    want = ops.quantize_pack(x, bits, 0.5)
    torch.cuda.synchronize()
    before = lib.cq_quantize_pack_wait_polls(1)
    try:
        for _ in range(2):
            for a, b in zip(ops.quantize_pack(x, bits, 0.5), want):
                assert same_bits(to_np(a), to_np(b)) if a.is_floating_point() else torch.equal(a, b)
            torch.cuda.synchronize()
    finally:
        lib.cq_quantize_pack_wait_polls(before)
    for a, b in zip(ops.quantize_pack(x, bits, 0.5), want):
        assert same_bits(to_np(a), to_np(b)) if a.is_floating_point() else torch.equal(a, b)


def test_quantize_pack_on_two_streams(ops):
    """Two passes whose parts exchange their extremes share the device, with a chunked decode step of one launch on a
    third stream: the results are those of each alone."""
    B, T, H = 24, 2400, 8
    g = torch.Generator(device="cuda").manual_seed(12)
    xs = [torch.randn((B, T, H, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2)]
    want = [ops.quantize_pack(x, 1, 0.5) for x in xs]
    n = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    codes = [torch.randint(0, 256, (4, H, 32768, 16), generator=g, device="cuda", dtype=torch.uint8) for _ in range(2)]
    decode = ops.DecodeCall(n(4, 32, 128), *codes, *[n(4, H, 128).abs() for _ in range(4)], None, None, bits=1)
    assert decode.plan()["launches"] == 1 and decode.plan()["chunks"] > 1
    good = decode.run().clone()
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(6):
        got = []
        for x, s in zip(xs, streams):
            with torch.cuda.stream(s):
                got.append(ops.quantize_pack(x, 1, 0.5))
        with torch.cuda.stream(streams[2]):
            decode.run()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert all(torch.equal(u, v) for u, v in zip(a, b))
        assert torch.equal(decode.out, good)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", [(1, 70, 2, 128), (3, 333, 5, 128), (1, 4100, 2, 128), (20, 1700, 8, 128), (2, 300, 3, 64), (1, 500, 2, 256)])
def test_quantize_pack_of_nan(ops, shape, bits, dtype):
    """A NaN of either sign makes the statistics of its channel NaN and its codes 0, as the ops do, in the one-pass kernel (one
    part, several, whole rows and quarters) and in the three launches alike; other channels are what they were."""
    B, T, H, D = shape
    print(f"case quantize_pack nan shape={shape} bits={bits} dtype={dtype}", flush=True)
    x = O.round_to(np.random.default_rng(T).standard_normal(shape, dtype=np.float32), dtype)
    clip = CLIPS[bits][0]
    plain = ops.quantize_pack(to_gpu(x, dtype), bits, clip)
    g = to_gpu(x, dtype)
    raw = g.view(torch.int16)
    raw[0, T // 2, 0, 5] = 0x7fff                    # the largest pattern of a positive NaN, the smallest of a negative one
    raw[B - 1, T - 1, H - 1, 62] = -0x8000 | (0x7f81 if dtype == "bf16" else 0x7c01)
    raw[B - 1, 0, H - 1, 63] = 0x7f81 if dtype == "bf16" else 0x7c01
    hit = np.zeros((B, H, D), bool)
    hit[0, 0, 5] = hit[B - 1, H - 1, 62] = hit[B - 1, H - 1, 63] = True
    codes, s, z = ops.quantize_pack(g, bits, clip)
    xq, s2, z2 = ops.quant_codes(g, bits, clip)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        oc, os_, oz = O.quantize_pack(to_np(g), bits, clip, dtype)
    assert np.isnan(os_[hit]).all() and not np.isnan(os_[~hit]).any()
    assert np.array_equal(codes.cpu().numpy(), oc)
    for a, b, p in ((s, os_, plain[1]), (z, oz, plain[2])):
        assert np.array_equal(np.isnan(to_np(a)), hit) and same_bits(to_np(a)[~hit], b[~hit]) and same_bits(to_np(a)[~hit], to_np(p)[~hit])
    # quant(): NaN statistics make every value of the channel NaN
    assert np.array_equal(np.isnan(to_np(s2[:, 0])), hit) and np.array_equal(np.isnan(to_np(xq)), np.broadcast_to(hit[:, None], shape))
    _, st, zt = ops.quant_codes_tensor(g, bits, clip)
    assert bool(st.isnan()) and bool(zt.isnan())


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", [(2, 300, 3, 128), (2, 4100, 2, 128)])
def test_quantize_pack_of_a_negative_clip_factor(ops, shape, bits):
    """A negative factor gives a negative scale: the op chain still says what the codes are."""
    x = O.round_to(np.random.default_rng(2).standard_normal(shape, dtype=np.float32), "bf16")
    codes, s, z = ops.quantize_pack(to_gpu(x, "bf16"), bits, -0.5)
    oc, os_, oz = O.quantize_pack(x, bits, -0.5, "bf16")
    assert (os_ < 0).all() and same_bits(to_np(s), os_) and same_bits(to_np(z), oz)
    assert np.array_equal(codes.cpu().numpy(), oc)


# More parts than workgroups, so that a workgroup goes on to a second part whose rows it has requested while it packed the
# first, with the parts of some pairs on either side of a turn (the grid is no multiple of the part count) and ragged last
# parts.
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("shape", [(30, 2400, 8), (30, 2399, 8), (43, 3327, 3), (25, 3328, 8)])
def test_quantize_pack_parts_across_turns_bit_exact(ops, shape, bits, dtype):
    from calibquant_amd import _lib
    B, T, H = shape
    p = _lib.QuantizePlan()
    _lib.check(_lib.load().cq_quantize_pack_plan(B, T, H, 0, ctypes.byref(p)), "plan")
    assert p.channels == 128 and p.parts > 1 and B * H * p.parts > p.workgroups and p.workgroups % p.parts
    print(f"case quantize_pack across turns shape={shape} bits={bits} dtype={dtype}", flush=True)
    rng = np.random.default_rng(T)
    x = O.round_to(rng.standard_normal((B, T, H, 128), dtype=np.float32), dtype)
    # every part of a pair has the extremes of some channels
    for part in range(p.parts):
        x[:, part * p.part_rows, :, part] = 9.0
        x[:, min(T, (part + 1) * p.part_rows) - 1, :, 64 + part] = -9.0
    codes, s, z = ops.quantize_pack(to_gpu(x, dtype), bits, CLIPS[bits][0])
    torch.cuda.synchronize()
    oc, os_, oz = O.quantize_pack(x, bits, CLIPS[bits][0], dtype)
    for a, b in ((s, os_), (z, oz)):     # (no zero minimum here: bit for bit)
        assert np.array_equal(to_np(a).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
    assert np.array_equal(codes.cpu().numpy(), oc)
