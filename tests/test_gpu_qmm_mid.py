"""The GEMM with 128-row weight tiles (vpq_qmm_mid.hip) where it can go wrong: K that ends inside a chunk of codes or
has an odd number of groups, fewer steps of K than x stages, N and M that end inside a tile, split shares of uneven
length -- against the oracle and, bit for bit, the 256 x 128 tile kernel; then every kernel that the size-based GEMM
chooses from (each count of rows of x per workgroup here, the 256 x 128 tile, each width of the large tile), in every
format it is built for, at shapes that take it, with M and N that end inside a tile."""
import numpy as np
import pytest
import torch

from tests import parity
from tests.test_oracle_pins import f16_pack
from vpipe_amd import synth

pytestmark = pytest.mark.gpu

# (K, N, M), all with 64 rows of x per workgroup: one step; two; an odd group count and a last chunk of one step; one to
# five tiles of rows with remainders
SHAPES = [(64, 130, 65), (128, 2, 17), (320, 258, 33), (1088, 262, 97), (3840, 200, 129), (2112, 1030, 300)]


@pytest.mark.parametrize("K,N,M", SHAPES)
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("fmt", ["w4g64", "w4g32", "w8g64", "f16"])
def test_qmm_mid_edges(vpq, oracle, dev, D, fmt, act, K, N, M):
    check_gemm(vpq, oracle, dev, D, fmt, act, K, N, M)


def check_gemm(vpq, oracle, dev, D, fmt, act, K, N, M):
    seed = K + 3 * N + M
    ms = np.unique(np.r_[0:3, M // 2, M - 3:M])
    if fmt == "f16":
        w, s, b = f16_pack(N, K, seed)
        x = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float16).view(np.uint16)
        args = (D.u32(w, dev), *(torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(dev).view(torch.float16) for a in (s, b, x)))
        y64, yb = oracle.matmul_f16(w, s, b, x[ms], K, N, len(ms), rounded=True)
        run = vpq.qmm_w4g64_f16
    else:
        make = {"w4g64": synth.make_weight, "w4g32": synth.make_weight_g32, "w8g64": synth.make_weight8}[fmt]
        w, s, b = make(N, K, seed)
        x = synth.make_act(M, K, seed + 1)
        args = (D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev))
        if fmt == "w8g64":
            y64, yb = oracle.matmul8(w, s, b, x[ms], K, N, len(ms), rounded=True)
        elif fmt == "w4g32":
            y64 = synth.bf16_bits_to_f32(x[ms]).astype(np.float64) @ synth.bf16_bits_to_f32(oracle.dequant_g32_bf16(w, s, b, K, N)).astype(np.float64).T
            yb = None
        else:
            y64, yb = oracle.qmm(w, s, b, x[ms], K, N, len(ms))
        run = {"w4g64": vpq.qmm_w4g64, "w4g32": vpq.qmm_w4g32, "w8g64": vpq.qmm_w8g64}[fmt]
    dt = args[3].dtype
    out = parity.Guarded((M, N // 2 if act else N), dt, dev)
    if act and fmt == "w4g64":
        vpq.qmm_swiglu_w4g64(*args, K, N, M, out=out.view)
    else:
        run(*args, K, N, M, out=out.view, **({"activation": 1} if act else {}))
    torch.cuda.synchronize()
    out.assert_intact()
    if act:
        # the store of the same sums: silu(gate) * up of the plain result's fp32 sums, to the element's rounding
        g, u = torch.from_numpy(np.asarray(y64)).double()[:, 0::2], torch.from_numpy(np.asarray(y64)).double()[:, 1::2]
        want = g / (1 + torch.exp(-g)) * u
        got = out.view.cpu()[torch.from_numpy(ms)].double()
        # sums differ by fp32 accumulation over K, the result by its own rounding (2^-9; 2^-11 in binary16)
        assert ((got - want).norm() / want.norm()).item() < 2.0 ** -8
        return
    got = out.view[torch.from_numpy(ms).to(dev)]
    if fmt == "f16":
        # binary16 rounding (2^-11 relative) and fp32 accumulation over K
        y = torch.from_numpy(np.asarray(y64)).reshape(len(ms), N).double()
        assert ((got.cpu().double() - y).norm() / y.norm()).item() < 2.0 ** -10
        return
    parity.check_bf16(D.bits(got), y64, yb)
    assert torch.equal(out.view, run(*args, K, N, M, tile_n=128))


ALL = ("w4g64", "w4g32", "w8g64", "f16")
# kernel (as vpq_qmm_plan), gated store, (K, N, M), formats
KERNELS = [
    (96, 0, (192, 24578, 80), ALL), (96, 1, (192, 24578, 80), ALL),
    (128, 0, (1088, 13314, 385), ("w4g64", "w4g32", "f16")), (128, 1, (1088, 13314, 385), ("w4g64", "w4g32", "f16")),
    (128, 0, (1088, 1026, 1541), ("w8g64",)), (128, 1, (1088, 1026, 1541), ("w8g64",)),
    (256, 0, (192, 1026, 4100), ALL), (256, 1, (320, 1026, 4100), ALL),
    (-128, 0, (512, 13314, 385), ALL), (-128, 1, (1024, 13314, 385), ("w8g64",)), (-128, 1, (4096, 1920, 4096), ("w4g64",)),
    (-192, 0, (512, 19970, 385), ("w4g64", "w8g64", "f16")),
    (-192, 1, (1024, 2306, 4100), ("w4g64", "f16")), (-192, 1, (512, 2306, 4100), ("w8g64",)),
    (-256, 0, (512, 21506, 517), ("w4g64", "w4g32", "f16")), (-256, 1, (1024, 3074, 4100), ("w4g64", "w4g32", "f16")),
]


@pytest.mark.parametrize("want,act,shape,fmt", [k[:3] + (f,) for k in KERNELS for f in k[3]])
def test_each_gemm_kernel_by_size(vpq, oracle, dev, D, want, act, shape, fmt):
    bits, group, f16 = {"w4g64": (4, 64, 0), "w4g32": (4, 32, 0), "w8g64": (8, 64, 0), "f16": (4, 64, 1)}[fmt]
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert vpq.load().vpq_qmm_plan(*shape, bits, group, f16, act, 1) == want
    check_gemm(vpq, oracle, dev, D, fmt, act, *shape)


# forced counts of shares: 64 rows a workgroup; 96; 128; the 256 x 128 tile (want, as vpq_qmm_plan)
@pytest.mark.parametrize("K,N,M,splits,want", [(1088, 131, 97, 3, 64), (1088, 132, 129, 2, 64), (640, 260, 48, 5, 64),
                                               (704, 5122, 129, 2, 96), (1088, 24578, 97, 2, 128),
                                               (704, 1026, 2049, 2, 256), (1088, 1027, 2049, 2, 256)])
def test_qmm_mid_uneven_shares(vpq, oracle, dev, D, K, N, M, splits, want):
    # shares that end inside a chunk of codes; a count of outputs that is and is not a multiple of four in the fold
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert vpq.load().vpq_qmm_plan(K, N, M, 4, 64, 0, 0, splits) == want
    w, s, b = synth.make_weight(N, K, 40 + M)
    x = synth.make_act(M, K, 41 + M)
    ms = np.arange(M) if M < 64 else np.unique(np.r_[0:3, 93:99, 126:130, 255:258, M // 2, M - 3:M] % M)
    y64, yb = oracle.qmm(w, s, b, x[ms], K, N, len(ms))
    args = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    out = parity.Guarded((M, N), torch.bfloat16, dev)
    vpq.qmm_splitk_w4g64(*args, K, N, M, splits=splits, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    parity.check_bf16(D.bits(out.view[torch.from_numpy(ms).to(dev)]), y64, yb)
    assert torch.equal(out.view, vpq.qmm_splitk_w4g64(*args, K, N, M, splits=splits))


@pytest.mark.parametrize("K,N,M,taken", [(5120, 12288, 333, True), (12288, 5120, 1024, True), (4096, 512, 128, False)])
def test_automatic_split_without_a_workspace(vpq, dev, K, N, M, taken):
    # 256 x 128 tiles that fill more than half of the chip by themselves need no workspace: the call runs unsplit;
    # a few tiles over a long K are refused without it
    gen = torch.Generator(device=dev).manual_seed(K + M)
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int32, device=dev, generator=gen)
    s = torch.empty((N, K // 64), device=dev).uniform_(0.005, 0.02, generator=gen).bfloat16()
    x = torch.randn((M, K), device=dev, generator=gen).bfloat16()
    b, y = -8 * s, torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    L, p = vpq.load(), [t.data_ptr() for t in (w, s, b, x, y)]
    status = L.vpq_qmm_splitk_w4g64_bf16(torch.cuda.current_stream().cuda_stream, *p, K, N, M, 0, None, 0)
    torch.cuda.synchronize()
    assert status == (0 if taken else -4)
    if taken:
        assert torch.equal(y, vpq.qmm_w4g64(w, s, b, x, K, N, M))


# 8 bits: two chunks of codes in LDS in turn, scales read every four steps: every remainder of K, for each count of rows of x
# per workgroup (want, as vpq_qmm_plan) that takes it
@pytest.mark.parametrize("want,N,M,steps", [(64, 262, 70, range(1, 14)), (96, 24578, 80, range(1, 10)), (128, 24578, 97, range(6, 14))])
def test_eight_bit_codes_over_every_remainder_of_k(vpq, dev, want, N, M, steps):
    gen = torch.Generator(device=dev).manual_seed(want)
    for K in (64 * t for t in steps):
        if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
            assert vpq.load().vpq_qmm_plan(K, N, M, 8, 64, 0, 0, 1) == want
        w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 4), dtype=torch.int32, device=dev, generator=gen)
        s = torch.empty((N, K // 64), device=dev).uniform_(0.0003, 0.0012, generator=gen).bfloat16()
        b = -128 * s
        x = torch.randn((M, K), device=dev, generator=gen).bfloat16()
        out = parity.Guarded((M, N), torch.bfloat16, dev)
        vpq.qmm_w8g64(w, s, b, x, K, N, M, out=out.view)
        torch.cuda.synchronize()
        out.assert_intact()
        # (the 256 x 128 tile, which the tests of 8-bit packs compare with the oracle)
        assert torch.equal(out.view, vpq.qmm_w8g64(w, s, b, x, K, N, M, tile_n=128)), K
