"""GPU parity of the gathered expert projections of an MoE block (one launch for all the
(token, expert) pairs), through the C ABI: each pair against the CPU oracle's QMV on that
expert's slab, and bit-identical to the plain kernel on the same slab -- the reference's own
contract for its gather kernels (gpu-kernels/metal/quant/affine_qmv.metal:918-921: "a gathered
expert is token-EXACT with the same expert run through the plain kernels")."""
import numpy as np
import pytest
import torch

from tests import parity
from vpipe_amd import capi, synth

pytestmark = pytest.mark.gpu


def expert_batch(E, N, K, seed):
    """E independent packs stacked into [E, N, ...] arrays."""
    packs = [synth.make_weight(N, K, seed + 13 * e) for e in range(E)]
    return tuple(np.stack([p[i] for p in packs]) for i in range(3))


def ids_for(E, npair, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, E, size=npair, dtype=np.int32)


# K, inner, E, top_k, M: one-pass and multi-pass K, K <= 1024 (two row groups per wavefront), K not a
# multiple of 512, odd inner, several tokens
GATED_SHAPES = [(2048, 96, 8, 4, 1), (2048, 768, 16, 8, 1), (4096, 33, 5, 2, 3), (768, 64, 4, 3, 2), (1984, 40, 3, 2, 2),
                (5120, 24, 6, 1, 4)]


@pytest.mark.parametrize("activation", [capi.VPQ_GATE_SWIGLU, capi.VPQ_GATE_GEGLU])
@pytest.mark.parametrize("K,inner,E,top_k,M", GATED_SHAPES)
def test_gathered_gate_up(vpq, oracle, dev, D, K, inner, E, top_k, M, activation):
    N = 2 * inner
    w, s, b = expert_batch(E, N, K, 4000 + K + inner)
    x = synth.make_act(M, K, 4100 + K + M)
    npair = M * top_k
    eid = ids_for(E, npair, 4200 + K)
    wd, sd, bd, xd = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    eidd = torch.from_numpy(eid).to(dev)
    out = parity.Guarded((npair, inner), torch.bfloat16, dev)
    vpq.gather_qmv_gated_w4g64(wd, sd, bd, xd, K, N, eidd, top_k, E, out=out.view, activation=activation)
    torch.cuda.synchronize()
    out.assert_intact()
    got = D.bits(out.view)
    act = oracle.swiglu if activation == capi.VPQ_GATE_SWIGLU else oracle.geglu
    want64 = np.empty((npair, inner))
    wantb = np.empty((npair, inner), dtype=np.uint16)
    for p in range(npair):
        e, t = int(eid[p]), p // top_k
        y64, _ = oracle.qmv(w[e], s[e], b[e], x[t:t + 1], K, N, 1)
        want64[p], wantb[p] = (a[0] for a in act(y64))
        plain = vpq.qmv_swiglu_w4g64(wd[e], sd[e], bd[e], xd[t:t + 1], K, N, 1, variant=capi.VPQ_QMV_ROWS,
                                     activation=activation)
        assert np.array_equal(got[p], D.bits(plain)[0]), "pair %d differs from the plain kernel on expert %d" % (p, e)
    parity.check_bf16(got, want64, wantb, mismatch_over_all=activation == capi.VPQ_GATE_SWIGLU)


# K (= inner), N (= hidden), E, npair
DOWN_SHAPES = [(768, 2048, 16, 8), (96 * 64 // 8, 256, 4, 5), (1024, 130, 3, 7), (2048, 64, 5, 1), (4608, 48, 2, 3)]


@pytest.mark.parametrize("K,N,E,npair", DOWN_SHAPES)
def test_gathered_down(vpq, oracle, dev, D, K, N, E, npair):
    w, s, b = expert_batch(E, N, K, 4300 + K + N)
    x = synth.make_act(npair, K, 4400 + K + npair)
    eid = ids_for(E, npair, 4500 + K)
    wd, sd, bd, xd = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    out = parity.Guarded((npair, N), torch.bfloat16, dev)
    vpq.gather_down_qmv_w4g64(wd, sd, bd, xd, K, N, torch.from_numpy(eid).to(dev), E, out=out.view)
    torch.cuda.synchronize()
    out.assert_intact()
    got = D.bits(out.view)
    want64 = np.empty((npair, N))
    wantb = np.empty((npair, N), dtype=np.uint16)
    for p in range(npair):
        e = int(eid[p])
        y64, yb = oracle.qmv(w[e], s[e], b[e], x[p:p + 1], K, N, 1)
        want64[p], wantb[p] = y64[0], yb[0]
        plain = vpq.qmv_w4g64(wd[e], sd[e], bd[e], xd[p:p + 1], K, N, 1, variant=capi.VPQ_QMV_ROWS)
        assert np.array_equal(got[p], D.bits(plain)[0]), "pair %d differs from the plain kernel on expert %d" % (p, e)
    parity.check_bf16(got, want64, wantb)


def test_gather_expert_id_out_of_range_gives_zeros(vpq, oracle, dev, D):
    K, inner, E, top_k = 1024, 32, 3, 2
    w, s, b = expert_batch(E, 2 * inner, K, 4600)
    x = synth.make_act(2, K, 4601)
    eid = np.array([1, -1, E, 2], dtype=np.int32)
    wd, sd, bd, xd = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    got = D.bits(vpq.gather_qmv_gated_w4g64(wd, sd, bd, xd, K, 2 * inner, torch.from_numpy(eid).to(dev), top_k, E))
    assert not got[1].any() and not got[2].any()
    assert got[0].any() and got[3].any()
    down = D.bits(vpq.gather_down_qmv_w4g64(wd, sd, bd, D.bf16(synth.make_act(4, K, 4602), dev), K, 2 * inner,
                                            torch.from_numpy(eid).to(dev), E))
    assert not down[1].any() and not down[2].any() and down[0].any() and down[3].any()


def test_gather_rejects_bad_arguments(vpq, dev):
    L = vpq.load()
    one = torch.zeros(4096, dtype=torch.int32, device=dev)
    p = one.data_ptr()
    assert L.vpq_gather_qmv_gated_w4g64_bf16(None, p, p, p, p, p, 64, 8, None, 1, 1, 1, capi.VPQ_GATE_SWIGLU) == -1
    assert L.vpq_gather_qmv_gated_w4g64_bf16(None, p, p, p, p, p, 64, 7, p, 1, 1, 1, capi.VPQ_GATE_SWIGLU) == -2   # odd N
    assert L.vpq_gather_qmv_gated_w4g64_bf16(None, p, p, p, p, p, 64, 8, p, 0, 1, 1, capi.VPQ_GATE_SWIGLU) == -2   # no pair
    assert L.vpq_gather_qmv_gated_w4g64_bf16(None, p, p, p, p, p, 64, 8, p, 1, 0, 1, capi.VPQ_GATE_SWIGLU) == -2   # top_k 0
    assert L.vpq_gather_qmv_gated_w4g64_bf16(None, p, p, p, p, p, 64, 8, p, 1, 1, 1, 7) == -2                      # activation
    assert L.vpq_gather_down_qmv_w4g64_bf16(None, p, p, p, p, p, 60, 8, p, 1, 1) == -2                             # K % 64
    assert L.vpq_gather_down_qmv_w4g64_bf16(None, p, p, p, p, p, 64, 8, p, 70000, 1) == -2                         # grid limit


# one group; half a wavefront's pass and just past it; one pass and two; odd group counts; the deepest that the gather kernel
# takes and the first that it leaves; N that ends inside a set of rows; enough pairs that a wavefront walks several sets
@pytest.mark.parametrize("K,N,pairs", [(64, 2, 3), (1024, 130, 2), (1088, 36, 3), (2048, 1026, 40), (2112, 70, 3), (4096, 34, 2), (4160, 34, 2)])
@pytest.mark.parametrize("bits", [4, 8])
def test_gathers_have_the_bits_of_the_plain_kernels(vpq, dev, D, bits, K, N, pairs):
    E, gen = 3, torch.Generator(device="cpu").manual_seed(4800 + K + N + bits)
    w = torch.randint(-2 ** 31, 2 ** 31, (E, N, K * bits // 32), dtype=torch.int32, generator=gen).to(dev)
    s = (torch.rand((E, N, K // 64), generator=gen) * 0.015 / (16 if bits == 8 else 1) + 0.001).bfloat16().to(dev)
    b = (-(2 ** (bits - 1)) * s.float() * 1.03).bfloat16()
    eid = torch.randint(0, E, (pairs,), dtype=torch.int32, generator=gen)
    eid[-1] = E                                          # no such expert: zeros
    x = torch.randn((pairs, K), generator=gen).bfloat16().to(dev)
    x[0, K // 2] = float("inf")
    act = parity.Guarded((pairs, N // 2), torch.bfloat16, dev)
    out = parity.Guarded((pairs, N), torch.bfloat16, dev)
    gated = vpq.gather_qmv_gated_w8g64 if bits == 8 else vpq.gather_qmv_gated_w4g64
    down = vpq.gather_down_qmv_w8g64 if bits == 8 else vpq.gather_down_qmv_w4g64
    gated(w, s, b, x, K, N, eid.to(dev), 1, E, out=act.view)
    down(w, s, b, x, K, N, eid.to(dev), E, out=out.view)
    torch.cuda.synchronize()
    act.assert_intact()
    out.assert_intact()
    assert not D.bits(act.view)[-1].any() and not D.bits(out.view)[-1].any()
    for p in range(0, pairs - 1, max(1, pairs // 5)):
        pack, xr = [t[int(eid[p])] for t in (w, s, b)], x[p:p + 1]
        if bits == 8:
            g = vpq.qmv_gated_w8g64(*pack, xr, K, N, 1, activation=1)
            d = vpq.qmv_w8g64(*pack, xr, K, N, 1)
        else:
            g = vpq.qmv_swiglu_w4g64(*pack, xr, K, N, 1, variant=capi.VPQ_QMV_ROWS)
            d = vpq.qmv_w4g64(*pack, xr, K, N, 1, variant=capi.VPQ_QMV_ROWS)
        assert np.array_equal(D.bits(act.view)[p], D.bits(g)[0])
        assert np.array_equal(D.bits(out.view)[p], D.bits(d)[0])
        if bits == 8:                                    # (and the sums, to their rounding)
            deq = (s[int(eid[p])].double().repeat_interleave(64, 1) * w[int(eid[p])].view(torch.uint8).view(N, K).double() +
                   b[int(eid[p])].double().repeat_interleave(64, 1))
            want = deq @ xr[0].double()
            got = out.view[p].double()
            if p == 0:
                assert not torch.isfinite(got).any()
            else:                                        # one bf16 rounding, and fp32 sums over K
                assert ((got - want).norm() / want.norm()).item() < 2.0 ** -8


# enough sets of rows that a wavefront walks several, in every form of the gather kernel (by K and code width), with an N that
# ends inside a set
@pytest.mark.parametrize("K,N,pairs", [(768, 2050, 48), (1024, 2050, 96), (2048, 1026, 40), (2112, 1026, 40), (2560, 1026, 40),
                                       (3072, 1026, 64), (4096, 1026, 40)])
@pytest.mark.parametrize("bits", [4, 8])
def test_gathers_whose_wavefronts_walk_several_sets(vpq, dev, D, bits, K, N, pairs):
    E, gen = 3, torch.Generator(device=dev).manual_seed(4900 + K + N + bits)
    sets = -(-N // (8 if bits == 4 and K <= 1024 else 4))
    walked = -(-sets * pairs // (32 * 256))              # sets of a wavefront (256 CUs)
    assert walked > 1
    w = torch.randint(-2 ** 31, 2 ** 31, (E, N, K * bits // 32), dtype=torch.int32, device=dev, generator=gen)
    s = (torch.rand((E, N, K // 64), device=dev, generator=gen) * 0.015 / (16 if bits == 8 else 1) + 0.001).bfloat16()
    b = (-(2 ** (bits - 1)) * s.float() * 1.03).bfloat16()
    eid = torch.randint(0, E, (pairs,), dtype=torch.int32, device=dev, generator=gen)
    x = torch.randn((pairs, K), device=dev, generator=gen).bfloat16()
    act = parity.Guarded((pairs, N // 2), torch.bfloat16, dev)
    out = parity.Guarded((pairs, N), torch.bfloat16, dev)
    gated = vpq.gather_qmv_gated_w8g64 if bits == 8 else vpq.gather_qmv_gated_w4g64
    down = vpq.gather_down_qmv_w8g64 if bits == 8 else vpq.gather_down_qmv_w4g64
    gated(w, s, b, x, K, N, eid, 1, E, out=act.view)
    down(w, s, b, x, K, N, eid, E, out=out.view)
    torch.cuda.synchronize()
    act.assert_intact()
    out.assert_intact()
    for p in sorted({0, 1, pairs // 2, pairs - 1}):
        e, xr = int(eid[p]), x[p:p + 1]
        pack = w[e], s[e], b[e]
        if bits == 8:
            g = vpq.qmv_gated_w8g64(*pack, xr, K, N, 1, activation=1)
        else:
            g = vpq.qmv_swiglu_w4g64(*pack, xr, K, N, 1, variant=capi.VPQ_QMV_ROWS)
            assert torch.equal(out.view[p], vpq.qmv_w4g64(*pack, xr, K, N, 1, variant=capi.VPQ_QMV_ROWS)[0])
        assert torch.equal(act.view[p], g[0])            # every row of the pair, whichever set of its wavefront
        # the plain store of 8 bits has no entry point of its own: one pair alone, where a wavefront has one set
        one = vpq.gather_down_qmv_w8g64 if bits == 8 else vpq.gather_down_qmv_w4g64
        alone = torch.empty((1, N), dtype=torch.bfloat16, device=dev)
        one(w, s, b, xr, K, N, eid[p:p + 1], E, out=alone)
        assert torch.equal(out.view[p], alone[0])


# One row of a gated 8-bit pack runs on the gathers' kernel: one to five passes over K and the first K past them, N that ends
# inside a set, wavefronts with several sets; against the oracle and the bits of the sorted form, which is another kernel
@pytest.mark.parametrize("K,N", [(64, 2), (1024, 10), (1088, 34), (2112, 70), (3136, 6), (4160, 130), (5120, 18), (5184, 18), (128, 65538)])
def test_one_gated_row_of_eight_bits(vpq, oracle, dev, D, K, N):
    w, s, b = synth.make_weight8(N, K, K + N)
    x = synth.make_act(1, K, K + N + 1)
    wd, sd, bd, xd = D.u32(w, dev), D.bf16(s, dev), D.bf16(b, dev), D.bf16(x, dev)
    out = parity.Guarded((1, N // 2), torch.bfloat16, dev)
    vpq.qmv_gated_w8g64(wd, sd, bd, xd, K, N, 1, out=out.view, activation=1)
    tile = torch.zeros((1,), dtype=torch.int32, device=dev)
    srow = torch.tensor([0, -1], dtype=torch.int32, device=dev)
    both = torch.empty((2, N // 2), dtype=torch.bfloat16, device=dev)
    vpq.qmv_grouped_gated_w8g64(wd[None], sd[None], bd[None], xd, K, N, tile, srow, 1, both)
    torch.cuda.synchronize()
    out.assert_intact()
    assert torch.equal(out.view[0], both[0])
    y64, _ = oracle.matmul8(w, s, b, x, K, N, 1, rounded=False)
    g64, gb = oracle.swiglu(np.asarray(y64).reshape(1, N))
    parity.check_bf16(D.bits(out.view), g64, gb)
