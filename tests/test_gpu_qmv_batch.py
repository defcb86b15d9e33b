"""The batch QMV kernel (vpq_qmv_batch.h) where it can go wrong: K that ends inside a chunk of codes or a piece of x, N
that ends inside a tile of 16 rows or leaves a partial 16-byte piece of scales, every count of staged rows of x, two
tiles of rows of x, more chunks than wavefronts -- against the oracle of each format, through the C ABI."""
import numpy as np
import pytest
import torch

from tests import parity
from tests.test_oracle_pins import f16_pack
from vpipe_amd import capi, synth

pytestmark = pytest.mark.gpu

# K: below one chunk of 256 (128 for 8-bit codes), one more than a whole number of chunks, K / 64 odd (scales read in
# 2-byte pieces), more than eight chunks; N: one row, one short of / past a tile, more tiles than CUs
SHAPES = [(64, 1, 2), (192, 15, 3), (320, 17, 4), (832, 33, 5), (2112, 31, 8), (2304, 4133, 9), (3904, 48, 13), (4096, 65, 16)]


@pytest.mark.parametrize("K,N,M", SHAPES)
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "w8g64", "f16"])
def test_qmv_batch_edges(vpq, oracle, dev, D, fmt, K, N, M):
    seed = K + 3 * N + M
    if fmt == "f16":
        w, s, b = f16_pack(N, K, seed)
        x = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float16).view(np.uint16)
        y64, _ = oracle.matmul_f16(w, s, b, x, K, N, M, rounded=False)
        t16 = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.float16) for a in (s, b, x)]
        run, args = vpq.qmv_w4g64_f16, (D.u32(w, dev), *t16)
    else:
        make = {"w4g64": synth.make_weight, "w4g32": synth.make_weight_g32, "w8g64": synth.make_weight8}[fmt]
        w, s, b = make(N, K, seed)
        x = synth.make_act(M, K, seed + 1)
        if fmt == "w8g64":
            y64, _ = oracle.matmul8(w, s, b, x, K, N, M, rounded=False)
        else:
            y64, _ = (oracle.qmv if fmt == "w4g64" else oracle.qmv_g32)(w, s, b, x, K, N, M)
        run = {"w4g64": vpq.qmv_w4g64, "w4g32": vpq.qmv_w4g32, "w8g64": vpq.qmv_w8g64}[fmt]
        args = (D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev))
    f = run(*args, K, N, M, f32out=True)
    out = parity.Guarded((M, N), args[3].dtype, dev)
    run(*args, K, N, M, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    parity.check_f32(f.cpu().numpy(), y64)
    # the stored element is the fp32 result rounded once
    assert torch.equal(out.view, f.to(args[3].dtype))


@pytest.mark.parametrize("M", [17, 31, 32, 33, 50, 64])
@pytest.mark.parametrize("K,N", [(960, 80), (4352, 24)])
def test_a_row_of_x_has_the_same_bits_in_any_batch(vpq, oracle, dev, D, M, K, N):
    # plain and gated, through the size-based entrances: up to 64 rows in one launch, each row as in a batch of its own
    w, s, b = synth.make_weight(N, K, 5 + M)
    x = synth.make_act(M, K, 6 + M)
    y64, yb = oracle.qmv(w, s, b, x, K, N, M)
    wd, sd, bd, xd = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    out = parity.Guarded((M, N), torch.bfloat16, dev)
    vpq.linear_w4g64(wd, sd, bd, xd, K, N, M, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    parity.check_bf16(D.bits(out.view), y64, yb)
    gated = vpq.linear_swiglu_w4g64(wd, sd, bd, xd, K, N, M)
    for m0 in range(0, M - 2, 13):
        n = min(13, M - m0)
        part = xd[m0:m0 + n].contiguous()
        assert torch.equal(vpq.qmv_w4g64(wd, sd, bd, part, K, N, n), out.view[m0:m0 + n])
        assert torch.equal(vpq.qmv_swiglu_w4g64(wd, sd, bd, part, K, N, n), gated[m0:m0 + n])


# The forms of 9 rows and more: K ends inside a piece of x or a chunk, N inside a tile and a quad of outputs.  Three tiles and 48
# rows, two and 48, two and 64, three and 32 (all rows, two workgroups along M), long pieces of 16 rows with one and two tiles
# and two to four workgroups along M, four rows a workgroup.
FORMS = [(320, 8843, 43), (832, 4110, 34), (1088, 6851, 57), (704, 8903, 27), (1856, 4301, 55), (2112, 1067, 27), (4032, 2117, 14),
         (2560, 4189, 11), (896, 2341, 41), (896, 1813, 61), (1152, 3, 12), (448, 11, 15),
         (1088, 5443, 32), (512, 3409, 31), (1152, 2579, 62)]      # (8 bits: two and one tile and 32 rows in long pieces)


@pytest.mark.parametrize("K,N,M", FORMS)
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "w8g64", "f16"])
def test_every_form_gives_the_bits_of_few_rows(vpq, dev, D, fmt, K, N, M):
    # against the same rows in batches of eight, which the oracle checks above
    bits, group, dtype = {"w4g64": (4, 64, torch.bfloat16), "w4g32": (4, 32, torch.bfloat16), "w8g64": (8, 64, torch.bfloat16),
                          "f16": (4, 64, torch.float16)}[fmt]
    def same(a, b):                                           # (a NaN where the infinity meets a weight of zero)
        return torch.equal(*(torch.nan_to_num(t.float(), nan=1e30, posinf=2e30, neginf=-2e30) for t in (a, b)))

    gen = torch.Generator(device=dev).manual_seed(K + N + M)
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=gen)
    s = torch.empty((N, K // group), device=dev).uniform_(0.005, 0.02, generator=gen).to(dtype)
    b = (-8 * s.float()).to(dtype)
    M = min(M, 16) if fmt == "f16" else M
    firsts = list(range(0, M - 8, 8)) + [M - 8]
    x = torch.randn((M, K), device=dev, generator=gen).to(dtype)
    x[M - 1, K - 1] = float("inf")                            # the last row is summed again
    few = {"w4g64": vpq.qmv_w4g64, "w4g32": vpq.qmv_w4g32, "w8g64": vpq.qmv_w8g64, "f16": vpq.qmv_w4g64_f16}[fmt]
    out = parity.Guarded((M, N), dtype, dev)
    if M <= 16:
        few(w, s, b, x, K, N, M, out=out.view)
        f32 = few(w, s, b, x, K, N, M, f32out=True)
        assert same(f32.to(dtype), out.view)
        res = torch.randn((M, N), device=dev, generator=gen).to(dtype)
        added = few(w, s, b, x, K, N, M, residual=res)
        assert same(added, (out.view.float() + res.float()).to(dtype))
    elif fmt == "w4g64":
        vpq.linear_w4g64(w, s, b, x, K, N, M, out=out.view)
        if N % 2 == 0:
            gated = parity.Guarded((M, N // 2), dtype, dev)
            vpq.linear_swiglu_w4g64(w, s, b, x, K, N, M, out=gated.view)
            gated.assert_intact()
            for m in range(0, M, 8):
                assert same(vpq.qmv_swiglu_w4g64(w, s, b, x[m:m + 8].contiguous(), K, N, min(8, M - m)), gated.view[m:m + 8])
    else:
        vpq.linear_twin(fmt, w, s, b, x, K, N, M, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    assert torch.isinf(out.view[M - 1]).any()
    for m in firsts:
        assert same(few(w, s, b, x[m:m + 8].contiguous(), K, N, 8), out.view[m:m + 8])


@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "w8g64"])
def test_grouped_launch_of_the_batch_kernel(vpq, dev, D, fmt):
    # four packs of different heights, none a multiple of a workgroup's rows: the bits of the separate calls
    K, M, Ns = 1344, 7, (40, 1, 133, 16)
    make = {"w4g64": synth.make_weight, "w4g32": synth.make_weight_g32, "w8g64": synth.make_weight8}[fmt]
    xd = D.bf16(synth.make_act(M, K, 3), dev)
    packs, outs = [], [parity.Guarded((M, N), torch.bfloat16, dev) for N in Ns]
    for i, N in enumerate(Ns):
        w, s, b = make(N, K, 40 + i)
        packs.append((D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), N))
    {"w4g64": vpq.qmv_group_w4g64, "w4g32": vpq.qmv_group_w4g32, "w8g64": vpq.qmv_group_w8g64}[fmt](
        packs, xd, K, M, outs=[o.view for o in outs])
    single = {"w4g64": vpq.qmv_w4g64, "w4g32": vpq.qmv_w4g32, "w8g64": vpq.qmv_w8g64}[fmt]
    for (w, s, b, N), o in zip(packs, outs):
        o.assert_intact()
        assert torch.equal(o.view, single(w, s, b, xd, K, N, M))


# the K of the one-row kernel in 16-byte pieces, of its narrow form, of neither
@pytest.mark.parametrize("K,M", [(4096, 1), (2560, 2), (4096, 3), (2112, 1), (2112, 2), (1024, 1), (1344, 1), (1344, 2), (1344, 5)])
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "q4_0", "w8g64", "f16"])
def test_grouped_launch_with_a_pack_off_alignment(vpq, dev, fmt, K, M):
    # one pack with scales two bytes off a 16-byte boundary: every pack has the bits of its own call.  The second half of K
    # nearly cancels the first, so that another order of additions shows in the stored elements.
    bits, group, dtype = {"w4g64": (4, 64, torch.bfloat16), "w8g64": (8, 64, torch.bfloat16), "f16": (4, 64, torch.float16)}.get(
        fmt, (4, 32, torch.bfloat16))
    half = K // 128 * 64
    gen = torch.Generator(device=dev).manual_seed(K + M)
    packs = []
    for i, N in enumerate((1030, 610, 40)):
        w = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=gen)
        s = torch.empty((N, K // group), device=dev).uniform_(0.005, 0.02, generator=gen).to(dtype)
        for t, per in ((w, 32 // bits), (s, group)):
            t[:, half // per:2 * half // per] = t[:, :half // per]
        if i == 1:
            s = torch.cat([s.new_zeros(1), s.view(-1)])[1:].view(s.shape)
            assert s.data_ptr() % 16 == 2
        packs.append((w, s, (-8 * s.float()).to(dtype), N))
    x = torch.randn((M, K), device=dev, generator=gen)
    x[:, half:2 * half] = -x[:, :half] * (1 + torch.randn((M, half), device=dev, generator=gen) / 64)
    x[:, 2 * half:] /= 64
    x = x.to(dtype)
    outs = [parity.Guarded((M, p[3]), dtype, dev) for p in packs]
    so = {"scale_only": True} if fmt == "q4_0" else {}
    run, single = {"w4g64": (vpq.qmv_group_w4g64, vpq.qmv_w4g64), "w8g64": (vpq.qmv_group_w8g64, vpq.qmv_w8g64),
                   "f16": (vpq.qmv_group_w4g64_f16, vpq.qmv_w4g64_f16)}.get(fmt, (vpq.qmv_group_w4g32, vpq.qmv_w4g32))
    run(packs, x, K, M, outs=[o.view for o in outs], **so)
    torch.cuda.synchronize()
    for (w, s, b, N), o in zip(packs, outs):
        o.assert_intact()
        assert torch.equal(o.view, single(w, s, b, x, K, N, M, **so))


def _weight64(fmt, w, s, b, K):
    """The pack in float64, from its words."""
    bits, group = (8, 64) if fmt == "w8g64" else (4, 32 if fmt in ("w4g32", "q4_0") else 64)
    q = (w[:, :, None] >> (np.arange(32 // bits, dtype=np.uint32) * bits)) & np.uint32((1 << bits) - 1)
    q = q.reshape(w.shape[0], K).astype(np.float64)
    f = (lambda v: v.view(np.float16).astype(np.float64)) if fmt == "f16" else (lambda v: synth.bf16_bits_to_f32(v).astype(np.float64))
    return q * np.repeat(f(s), group, 1) + np.repeat(f(b), group, 1)


@pytest.mark.parametrize("K", [1344, 4096])
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "q4_0", "w8g64", "f16"])
def test_rows_of_x_that_are_not_finite(vpq, dev, D, fmt, K):
    # One infinity in a row gives +-inf by the weight's sign (NaN where the weight is zero), opposite infinities and a NaN
    # give NaN where the plain sum does, and a row whose values only overflow the kernel's offset sums keeps its finite
    # results.  The other rows of the batch do not notice.
    N, M = 70, 9
    rng = np.random.default_rng(K)
    if fmt == "f16":
        w, s, b = f16_pack(N, K, 3)
        x = rng.standard_normal((M, K)).astype(np.float16)
    else:
        w, s, b = {"w4g64": synth.make_weight, "w4g32": synth.make_weight_g32, "w8g64": synth.make_weight8,
                   "q4_0": lambda N, K, seed: synth.make_weight_g32(N, K, seed, q40=True)}[fmt](N, K, 3)
        x = synth.bf16_bits_to_f32(synth.make_act(M, K, 4))
    w.reshape(-1)[::3] &= np.uint32(0xff00ff0f)               # codes of zero too
    bad = x.copy()
    bad[1, 5] = np.inf
    bad[3, K - 1] = -np.inf
    bad[4, 7], bad[4, K // 2] = np.inf, -np.inf
    bad[6, 70] = np.nan
    bad[8] *= 1000 if fmt == "f16" else np.float32(2.0 ** 121)
    as_dev = (lambda a: torch.from_numpy(a.astype(np.float16)).to(dev)) if fmt == "f16" else (lambda a: torch.from_numpy(a).to(dev).bfloat16())
    sb = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.float16 if fmt == "f16" else torch.bfloat16) for a in (s, b)]
    run = {"w4g64": vpq.qmv_w4g64, "w4g32": vpq.qmv_w4g32, "w8g64": vpq.qmv_w8g64, "f16": vpq.qmv_w4g64_f16,
           "q4_0": lambda w, s, b, *a, **k: vpq.qmv_w4g32(w, s, None, *a, scale_only=True, **k)}[fmt]
    xb, xg = as_dev(bad), as_dev(x)
    got = run(D.u32(w, dev), *sb, xb, K, N, M, f32out=True).cpu().double()
    good = run(D.u32(w, dev), *sb, xg, K, N, M, f32out=True).cpu().double()
    W = _weight64(fmt, w, s, b, K)
    with np.errstate(invalid="ignore"):
        want = torch.from_numpy(np.stack([(r[None] * W).sum(1) for r in xb.cpu().double().numpy()]))
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert inf[1].any() and inf[3].any() and torch.equal(got[inf], want[inf]) and not torch.isinf(got[~inf]).any()
    for m in (0, 2, 5, 7):
        assert torch.equal(got[m], good[m])
    parity.check_f32(got[8].numpy(), want[8].numpy())
    if fmt == "w4g64":
        gated = vpq.qmv_swiglu_w4g64(D.u32(w, dev), *sb, xb, K, N, M).cpu().double()
        g, u = got[:, 0::2], got[:, 1::2]
        ref = (g / (1 + torch.exp(-g)) * u).bfloat16().double()
        assert torch.equal(torch.isnan(gated), torch.isnan(ref)) and torch.equal(torch.isinf(gated), torch.isinf(ref))


# K on either side of where one row leaves the batch kernel, in one part and in several, of two and of four weight rows a wavefront
@pytest.mark.parametrize("K,N", [(2112, 70), (3136, 70), (3136, 23001), (9664, 69), (17472, 2400)])
def test_one_row_of_binary16_that_is_not_finite(vpq, dev, K, N):
    # an infinity in x gives +-inf by the weight's sign, NaN where the weight is zero or infinities meet; a NaN gives NaN
    gen = torch.Generator(device=dev).manual_seed(K + N)
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int32, device=dev, generator=gen)
    s = torch.empty((N, K // 64), device=dev).uniform_(0.005, 0.02, generator=gen).half()
    b = (-8 * s.float()).half()
    q = torch.stack([(w[:, [0, K // 16, K // 8 - 1]] >> 4 * i) & 15 for i in range(8)], -1).float()     # codes of three words
    W = q * s[:, [0, K // 128, K // 64 - 1], None].float() + b[:, [0, K // 128, K // 64 - 1], None].float()
    x = torch.randn((K,), device=dev, generator=gen).half()
    for at, inf in (((0, 5),), (1.0,)), (((2, 7),), (-1.0,)), (((0, 5), (1, 3)), (1.0, -1.0)):
        bad = x.clone()
        want = torch.zeros((N,), device=dev)
        for (word, i), sign in zip(at, inf):
            bad[[0, K // 2, K - 8][word] + i] = sign * float("inf")
            want = want + sign * float("inf") * W[:, word, i]
        assert torch.isinf(want).any() and torch.isnan(want).any()
        got = vpq.qmv_w4g64_f16(w, s, b, bad[None], K, N, 1, f32out=True)[0]
        assert torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(want, nan=7.0))
        out = vpq.qmv_w4g64_f16(w, s, b, bad[None], K, N, 1, residual=x[None, :1].expand(1, N).contiguous())[0]
        assert torch.equal(torch.nan_to_num(out.float(), nan=7.0, posinf=1e9, neginf=-1e9), torch.nan_to_num(want, nan=7.0, posinf=1e9, neginf=-1e9))
        outs = vpq.qmv_group_w4g64_f16([(w[:40], s[:40], b[:40], 40), (w[40:], s[40:], b[40:], N - 40)], bad[None], K, 1)
        assert torch.equal(torch.nan_to_num(torch.cat(outs, 1)[0].float(), nan=7.0), torch.nan_to_num(want.half().float(), nan=7.0))
    bad = x.clone()
    bad[70] = float("nan")
    assert torch.isnan(vpq.qmv_w4g64_f16(w, s, b, bad[None], K, N, 1)).all()


@pytest.mark.parametrize("K", [960, 3840, 9664])
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "q4_0", "w8g64", "f16"])
def test_fp32_results_are_as_close_as_a_plain_sum(vpq, dev, D, fmt, K):
    # The fp32 output against float64.  A plain fp32 sum of x * (scale q + bias) over such K is 0.7 to 2.3e-7 away
    # (2-norm, measured on the one-row-a-wavefront kernel); a sum that cancels against a multiple of sum(x) larger
    # than the codes is 2 to 6e-7 away.  The bound lies between the two, at four roundings of 2^-24.
    N, M = 256, 7
    rng = np.random.default_rng(K)
    if fmt == "f16":
        w, s, b = f16_pack(N, K, 3)
        x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).to(dev)
    else:
        w, s, b = {"w4g64": synth.make_weight, "w4g32": synth.make_weight_g32, "w8g64": synth.make_weight8,
                   "q4_0": lambda N, K, seed: synth.make_weight_g32(N, K, seed, q40=True)}[fmt](N, K, 3)
        x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dev).bfloat16()
    sb = [torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(x.dtype) for a in (s, b)]
    run = {"w4g64": vpq.qmv_w4g64, "w4g32": vpq.qmv_w4g32, "w8g64": vpq.qmv_w8g64, "f16": vpq.qmv_w4g64_f16,
           "q4_0": lambda w, s, b, *a, **k: vpq.qmv_w4g32(w, s, None, *a, scale_only=True, **k)}[fmt]
    got = run(D.u32(w, dev), *sb, x, K, N, M, f32out=True).cpu().double().numpy()
    want = x.cpu().double().numpy() @ _weight64(fmt, w, s, b, K).T
    assert np.linalg.norm(got - want) <= 4 * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("M", [1, 2, 5])
def test_k_that_is_too_deep_for_the_batch_kernel(vpq, oracle, dev, D, M):
    # its scales do not fit the LDS: the automatic and the MFMA call, single and grouped, run on the ring kernel
    K, Ns = 131072, (33, 16)
    x = synth.make_act(M, K, 7)
    xd = D.bf16(x, dev)
    packs, singles = [], []
    for N in Ns:
        w, s, b = synth.make_weight(N, K, 8 + N)
        pack = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev)
        f = vpq.qmv_w4g64(*pack, xd, K, N, M, f32out=True)
        parity.check_f32(f.cpu().numpy(), oracle.qmv(w, s, b, x, K, N, M)[0])
        singles.append(vpq.qmv_w4g64(*pack, xd, K, N, M))
        assert torch.equal(singles[-1], f.bfloat16())
        for variant in (capi.VPQ_QMV_MFMA, capi.VPQ_QMV_RING):
            assert torch.equal(vpq.qmv_w4g64(*pack, xd, K, N, M, variant=variant), singles[-1])
        packs.append(pack + (N,))
    outs = [parity.Guarded((M, N), torch.bfloat16, dev) for N in Ns]
    vpq.qmv_group_w4g64(packs, xd, K, M, outs=[o.view for o in outs])
    torch.cuda.synchronize()
    for o, one in zip(outs, singles):
        o.assert_intact()
        assert torch.equal(o.view, one)


@pytest.mark.parametrize("K", [6144, 6464, 9664])
def test_eight_bit_codes_over_a_long_k_have_the_same_bits_in_few_workgroups(vpq, oracle, dev, D, K):
    # few weight rows over a long K: two or three chunks of a wavefront in flight (every count of x loads, wavefronts with one
    # chunk more than others, a last chunk that ends early), against many, whose workgroups keep one, and the oracle
    N, n = 8224, 33
    w, s, b = synth.make_weight8(n, K, K + 3)
    gen = torch.Generator(device=dev).manual_seed(K)
    wd = torch.randint(-2 ** 31, 2 ** 31, (N, K // 4), dtype=torch.int32, device=dev, generator=gen)
    sd = torch.empty((N, K // 64), device=dev).uniform_(0.0003, 0.0012, generator=gen).bfloat16()
    bd = -128 * sd
    wd[:n], sd[:n], bd[:n] = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev)
    x = synth.make_act(21, K, K + 4)
    xd = D.bf16(x, dev)
    y64, _ = oracle.matmul8(w, s, b, x, K, n, 21, rounded=False)
    few = [t[:n].contiguous() for t in (wd, sd, bd)]
    for M in (2, 3, 4, 5, 6, 7, 8, 9, 16):
        got = vpq.qmv_w8g64(*few, xd[:M], K, n, M, f32out=True)
        parity.check_f32(got.cpu().numpy(), y64[:M])
        assert torch.equal(got, vpq.qmv_w8g64(wd, sd, bd, xd[:M], K, N, M, f32out=True)[:, :n])
    for M in (17, 21):
        got = vpq.linear_twin("w8g64", *few, xd[:M], K, n, M)
        assert torch.equal(got, vpq.linear_twin("w8g64", wd, sd, bd, xd[:M], K, N, M)[:, :n])


@pytest.mark.parametrize("K", [6144, 6176, 9664])
def test_eight_bit_codes_in_groups_of_32_over_a_long_k(vpq, oracle, dev, D, K):
    # as above, every count of rows of x of the forms that keep two or three chunks in flight
    N, n = 8224, 33
    w, s, b = synth.make_weight8(n, K, K + 5, group=32)
    gen = torch.Generator(device=dev).manual_seed(K)
    wd = torch.randint(-2 ** 31, 2 ** 31, (N, K // 4), dtype=torch.int32, device=dev, generator=gen)
    sd = torch.empty((N, K // 32), device=dev).uniform_(0.0003, 0.0012, generator=gen).bfloat16()
    bd = -128 * sd
    wd[:n], sd[:n], bd[:n] = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev)
    x = synth.make_act(16, K, K + 6)
    xd = D.bf16(x, dev)
    y64, yb = oracle.matmul8(w, s, b, x, K, n, 16, rounded=False, group=32)
    few = [t[:n].contiguous() for t in (wd, sd, bd)]
    for M in (2, 3, 4, 5, 6, 7, 8, 9, 13, 16):
        out = parity.Guarded((M, n), torch.bfloat16, dev)
        vpq.qmv_w8g32(*few, xd[:M], K, n, M, out=out.view)
        torch.cuda.synchronize()
        out.assert_intact()
        parity.check_bf16(D.bits(out.view), y64[:M], yb[:M])
        assert torch.equal(out.view, vpq.qmv_w8g32(wd, sd, bd, xd[:M], K, N, M)[:, :n])


@pytest.mark.parametrize("K", [6144, 9664])
@pytest.mark.parametrize("M", [2, 6, 16, 33, 50, 64])
def test_eight_bit_codes_over_a_long_k_gated_grouped_and_in_two_tiles_of_rows(vpq, dev, K, M):
    # the same bits from few workgroups, whose wavefronts keep several chunks in flight, as from many
    N, n = 8224, 34
    gen = torch.Generator(device=dev).manual_seed(K + M)
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 4), dtype=torch.int32, device=dev, generator=gen)
    s = torch.empty((N, K // 64), device=dev).uniform_(0.0003, 0.0012, generator=gen).bfloat16()
    b = -128 * s
    x = torch.randn((M, K), device=dev, generator=gen).bfloat16()
    few = [t[:n].contiguous() for t in (w, s, b)]
    if M > 16:
        out = parity.Guarded((M, n), torch.bfloat16, dev)
        vpq.linear_twin("w8g64", *few, x, K, n, M, out=out.view)
        torch.cuda.synchronize()
        out.assert_intact()
        assert torch.equal(out.view, vpq.linear_twin("w8g64", w, s, b, x, K, N, M)[:, :n])
        return
    out = parity.Guarded((M, n // 2), torch.bfloat16, dev)
    vpq.qmv_gated_w8g64(*few, x, K, n, M, out=out.view)
    many = vpq.qmv_w8g64(w, s, b, x, K, N, M)
    packs, outs, first = [], [], 0
    for rows in (17, 130, 48):
        packs.append(tuple(t[first:first + rows].clone() for t in (w, s, b)) + (rows,))
        outs.append(parity.Guarded((M, rows), torch.bfloat16, dev))
        first += rows
    vpq.qmv_group_w8g64(packs, x, K, M, outs=[o.view for o in outs])
    torch.cuda.synchronize()
    out.assert_intact()
    assert torch.equal(out.view, vpq.qmv_gated_w8g64(w, s, b, x, K, N, M)[:, :n // 2])
    first = 0
    for o, p in zip(outs, packs):
        o.assert_intact()
        assert torch.equal(o.view, many[:, first:first + p[3]])
        first += p[3]


# One row (8 bits from K = 2560 on, binary16 below K = 2048) and two rows of groups of 32: the oracle's sums, the
# bits of the same rows in a batch of three, a grouped launch the bits of the single ones; chunks in flight end with K
@pytest.mark.parametrize("fmt,M,K,N", [("w8g64", 1, 2496, 33), ("w8g64", 1, 2560, 33), ("w8g64", 1, 3072, 130), ("w8g64", 1, 9664, 17),
                                       ("w8g64", 2, 3840, 40), ("w8g64", 7, 3840, 40), ("f16", 1, 64, 3), ("f16", 1, 1088, 130),
                                       ("w4g32", 2, 96, 5), ("w4g32", 2, 4128, 130), ("w4g32", 1, 4128, 130)])
def test_one_and_two_rows(vpq, oracle, dev, D, fmt, M, K, N):
    seed = K + N + M
    if fmt == "f16":
        w, s, b = f16_pack(N, K, seed)
        x = np.random.default_rng(seed).standard_normal((3, K)).astype(np.float16).view(np.uint16)
        y64, _ = oracle.matmul_f16(w, s, b, x[:M], K, N, M, rounded=False)
        s, b, xd = (torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.float16) for a in (s, b, x))
        run, group = vpq.qmv_w4g64_f16, vpq.qmv_group_w4g64_f16
    else:
        w, s, b = (synth.make_weight8 if fmt == "w8g64" else synth.make_weight_g32)(N, K, seed)
        x = synth.make_act(max(M, 3), K, seed + 1)
        if fmt == "w8g64":
            y64, _ = oracle.matmul8(w, s, b, x[:M], K, N, M, rounded=False)
        else:
            y64, _ = oracle.qmv_g32(w, s, b, x[:M], K, N, M)
        s, b, xd = D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
        run, group = (vpq.qmv_w8g64, vpq.qmv_group_w8g64) if fmt == "w8g64" else (vpq.qmv_w4g32, vpq.qmv_group_w4g32)
    w, xm = D.u32(w, dev), xd[:M].contiguous()
    parity.check_f32(run(w, s, b, xm, K, N, M, f32out=True).cpu().numpy(), y64)
    out = parity.Guarded((M, N), xd.dtype, dev)
    run(w, s, b, xm, K, N, M, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    if (fmt, K) != ("w8g64", 2496) and (fmt, M) != ("w4g32", 1):   # (kernels of one row)
        assert torch.equal(out.view, run(w, s, b, xd[:max(M, 3)], K, N, max(M, 3))[:M])
    cut = N // 2
    packs = [tuple(t[i:j].clone() for t in (w, s, b)) + (j - i,) for i, j in ((0, cut), (cut, N))]
    assert torch.equal(torch.cat(group(packs, xm, K, M), dim=1), out.view)


# One row, scales and biases by 2-byte loads: K one group past a slice of 2048, odd counts of groups, one to four parts of K and
# the last K that is taken, N that ends inside a wavefront's rows; plain, with a residual, gated, and grouped
@pytest.mark.parametrize("fmt,N,K", [(f, n, k) for f, n in (("w4g64", 1), ("w4g64", 6), ("w4g32", 3), ("w4g32", 34), ("f16", 10),
                                                            ("w4g64", 2050))
                                     for k in (2080, 2112, 3840, 6080, 6208, 17344, 25024, 32704) if k % 64 == 0 or f == "w4g32"])
def test_one_row_with_narrow_scales(vpq, oracle, dev, D, fmt, N, K):
    seed = K + N
    if fmt == "f16":
        w, s, b = f16_pack(N, K, seed)
        x = np.random.default_rng(seed).standard_normal((1, K)).astype(np.float16).view(np.uint16)
        y64, _ = oracle.matmul_f16(w, s, b, x, K, N, 1, rounded=False)
        s, b, x = (torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.float16) for a in (s, b, x))
        run, group = vpq.qmv_w4g64_f16, vpq.qmv_group_w4g64_f16
    else:
        w, s, b = (synth.make_weight if fmt == "w4g64" else synth.make_weight_g32)(N, K, seed)
        x = synth.make_act(1, K, seed + 1)
        y64, _ = (oracle.qmv if fmt == "w4g64" else oracle.qmv_g32)(w, s, b, x, K, N, 1)
        s, b, x = D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
        run, group = (vpq.qmv_w4g64, vpq.qmv_group_w4g64) if fmt == "w4g64" else (vpq.qmv_w4g32, vpq.qmv_group_w4g32)
    w = D.u32(w, dev)
    f = run(w, s, b, x, K, N, 1, f32out=True)
    parity.check_f32(f.cpu().numpy(), y64)
    res = torch.randn((1, N), device=dev).to(x.dtype)
    out, added = parity.Guarded((1, N), x.dtype, dev), parity.Guarded((1, N), x.dtype, dev)
    run(w, s, b, x, K, N, 1, out=out.view)
    run(w, s, b, x, K, N, 1, out=added.view, residual=res)
    torch.cuda.synchronize()
    out.assert_intact()
    added.assert_intact()
    assert torch.equal(out.view, f.to(x.dtype))
    assert torch.equal(added.view, (out.view.float() + res.float()).to(x.dtype))
    if N % 2 == 0:
        gated = parity.Guarded((1, N // 2), x.dtype, dev)
        if fmt == "w4g64":
            vpq.qmv_swiglu_w4g64(w, s, b, x, K, N, 1, out=gated.view)
        else:
            run(w, s, b, x, K, N, 1, out=gated.view, activation=1)
        torch.cuda.synchronize()
        gated.assert_intact()
        g, u = f.double()[:, 0::2], f.double()[:, 1::2]
        want = g / (1 + torch.exp(-g)) * u
        # the result's own rounding (2^-8 bounds it for both elements) and a few steps of fp32 in the activation
        assert ((gated.view.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all()
    if N > 1:
        cuts = sorted({0, N // 3, N // 2, N})
        packs = [tuple(t[i:j].clone() for t in (w, s, b)) + (j - i,) for i, j in zip(cuts, cuts[1:])]
        assert torch.equal(torch.cat(group(packs, x, K, 1), dim=1), out.view)
