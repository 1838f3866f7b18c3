"""The grouped GEMM's tile variants, the prefill router and the grouping at the
sizes where their dispatch and remainders change, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from tests._util import log, max_rel, u16, u32
from trifuse_amd import moe as tmoe
from trifuse_amd import workload as wl

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16}
# A product's largest error over its largest value, in half steps u of the storage
# type (2^-8 of a bf16 value, 2^-11 of a half one). The result is rounded once:
# at most u of the largest. Its weights are rounded to about 0.4 u each (rms), which
# over a product adds up to 0.4 u of the result's rms, five times that at most over
# some 10^6 results, whose largest is about five times their rms: 0.4 u of the
# largest. The fp32 sums add 1e-6. So 1.4 u and a little.
STEP = {"bf16": 1.5 * 2.0 ** -8, "f16": 1.5 * 2.0 ** -11}


def _affine(shape, bits, dtype, key, device):
    *lead, width = shape
    q = wl.packed_nibbles((*lead, width * bits // 32), key, device)
    k = 16 / 2 ** bits
    s = wl.uniform_scales((*lead, width // 64), key + 1, device, lo=0.005 * k, hi=0.02 * k, dtype=DT[dtype])
    return q, s, (s.float() * -float(2 ** (bits - 1))).to(DT[dtype])


# Counts that end a 16-row block, a tile or its live-row steps exactly, one row
# early and one row late.
EDGES = [0, 1] + [c + d for c in (16, 32, 48, 64, 80, 96, 112, 128, 160, 192, 224, 256) for d in (-1, 0, 1)]


def _routes(T, E, K, seed):
    """T x K expert ids in random order: EDGES as the route counts of the first
    experts, as far as they take two thirds of the routes, the rest shared out
    evenly."""
    counts, left = np.zeros(E, dtype=np.int64), T * K
    for e, c in zip(range(E - 4), EDGES):
        if 3 * (T * K - left + c) > 2 * T * K:
            break
        counts[e] = c
        left -= c
    rest = E - 1 - e
    counts[e + 1:] = left // rest
    counts[E - 1] += left - left // rest * rest
    ids = np.repeat(np.arange(E, dtype=np.int32), counts)
    np.random.default_rng(seed).shuffle(ids)
    return ids.reshape(T, K)


# Two and a half half steps of the storage type, as for products: the result is
# rounded once (1), the K weighted expert outputs once each (less than 1), and the
# rounded weights and hidden rows of three products average out (0.4 each, in
# squares).
BLOCK_STEPS = {"bf16": 1e-2, "f16": 1e-2 / 8}

# Geometries with every input width an odd number of 128-wide super-steps or
# output columns off the tile: experts x columns that fill the compute units (down
# GEMM too), gate/up columns off the tile, and experts that do not fill them.
WIDE, RAGGED, NARROW = (1152, 640, 64, 8), (640, 704, 64, 8), (384, 512, 40, 8)
# Routes per expert on average, over the tile rule's lines: 64-, 96- and 128-row
# tiles, two 96-row tiles, 128 and 256 rows; for few columns also both sides of
# one round of 256-row tiles (128) and of the 64-weight-row tiles' fill (300).
CASES = [(WIDE, a) for a in (6, 30, 47, 60, 90, 105, 140, 200, 260, 450)] + [(RAGGED, a) for a in (60, 90, 140)] + \
    [(NARROW, a) for a in (10, 30, 58, 126, 130, 200, 300, 400, 500)]


@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("f16", 4), ("bf16", 8), ("f16", 8)])
@pytest.mark.parametrize("geom,a", CASES, ids=[f"{g[0]}x{g[1]}-{a}" for g, a in CASES])
def test_block_tiles(gpu, dtype, bits, geom, a):
    """Every token of a block against the per-expert fp64 reference."""
    H, I, E, K = geom
    T = a * E // K + 3
    log(f"block tiles {dtype} bits={bits} H={H} I={I} E={E} a={a} T={T}")

    class L:
        pass

    lay, w = L(), {}
    for i, (p, rows, width) in enumerate((("gate", I, H), ("up", I, H), ("down", H, I))):
        w[p] = _affine((E, rows, width), bits, dtype, 500 + 10 * i + bits, gpu)
        for n, t in zip("qsb", w[p]):
            setattr(lay, f"{p}_{n}", u32(t) if n == "q" else u16(t))
    x = wl.normal_bf16((T, H), 1.0, 60 + a, dtype=DT[dtype])
    idx = _routes(T, E, K, a)
    gates = np.random.default_rng(a + 1).random((T, K), dtype=np.float32) / K
    router = "affine" if dtype == "f16" else "dense"
    blk = tmoe.MoEBlock(H, I, E, K, route="olmoe", bits=bits, dtype=DT[dtype], router=router)
    wts = tmoe.ExpertWeights(None, *w["gate"], *w["up"], *w["down"])
    y = blk.experts(x.to(gpu), torch.from_numpy(idx).to(gpu), torch.from_numpy(gates).to(gpu), wts)
    torch.cuda.synchronize()
    ref = oracle.moe_reference_full(u16(x), idx, gates, lay, dtype=dtype)
    err = max_rel(oracle.st_to_f32(u16(y), dtype), ref)
    log(f"  max_rel {err:.2e}")
    assert err <= BLOCK_STEPS[dtype]


# Input widths: odd multiples of 64 (the LDS-dequantising kernel), one
# super-step, group counts not a multiple of 8 (4-byte scale copies), past
# 2048; output widths off the tile; rows around 16, 32, 64, 96 and 128; the
# lines between which 8-bit bf16 codes take the LDS-dequantising kernel (57, 384
# and not 480 to 528 rows an expert); few rows an expert at one, three and, past
# the scales that a tile keeps, five chunks of scales.
@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("f16", 4), ("bf16", 8), ("f16", 8)])
@pytest.mark.parametrize("E,N,Kin,rows", [(1, 64, 64, 200), (1, 192, 128, 177), (2, 320, 192, 500), (3, 128, 384, 401),
                                          (2, 192, 640, 290), (1, 256, 2304, 180), (40, 64, 1536, 41 * 17),
                                          (64, 1024, 128, 64 * 60), (64, 1024, 256, 64 * 110), (64, 1088, 128, 64 * 140),
                                          (64, 1024, 128, 64 * 250), (64, 2048, 128, 64 * 57), (16, 1536, 256, 16 * 383),
                                          (16, 1536, 256, 16 * 384), (16, 1536, 256, 16 * 500), (16, 1536, 256, 16 * 530),
                                          (64, 2048, 512, 64 * 5), (64, 2048, 1536, 64 * 7), (64, 2048, 2560, 64 * 5)])
def test_product_shapes(gpu, dtype, bits, E, N, Kin, rows):
    log(f"product {dtype} bits={bits} E={E} N={N} Kin={Kin} rows={rows}")
    q, s, b = _affine((E, N, Kin), bits, dtype, 7 * N + Kin + bits, gpu)
    x = wl.normal_bf16((rows, Kin), 1.0, rows, dtype=DT[dtype])
    rhs = np.random.default_rng(rows).integers(0, E, size=rows).astype(np.int32)
    out = tmoe.gather_qmm_rows(x.to(gpu), q, s, b, torch.from_numpy(rhs).to(gpu), bits=bits)
    torch.cuda.synchronize()
    pick = np.unique(np.linspace(0, rows - 1, 200).astype(np.int64))
    ref = oracle.gather_qmm_f64(u16(x)[pick], np.arange(pick.size), rhs[pick], u32(q), u16(s), u16(b), dtype=dtype)
    err = max_rel(oracle.st_to_f32(u16(out)[pick], dtype), ref)
    log(f"  max_rel {err:.2e}")
    assert err <= STEP[dtype]


def _shifted(t, elements):
    """t's values in an array that starts `elements` 2-byte elements past an aligned one."""
    buf = torch.zeros(t.numel() + elements, dtype=t.dtype, device=t.device)
    out = buf[elements:].view(t.shape)
    out.copy_(t)
    assert out.is_contiguous() and out.data_ptr() % 16 == (2 * elements) % 16
    return out


# Scales and biases that start at any element of an allocation: 2-byte
# boundaries (the LDS-dequantising kernel's 2-byte loads), 4-byte ones (dword
# copies) and 16-byte ones, on both sides of 2048 and at odd multiples of 64.
# Dword and 16-byte copies move the same values: the same bits.
@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("f16", 4), ("bf16", 8), ("f16", 8)])
@pytest.mark.parametrize("Kin", [192, 512, 2304, 3072])
def test_scale_alignment(gpu, dtype, bits, Kin):
    E, N, rows = 3, 128, 300
    q, s, b = _affine((E, N, Kin), bits, dtype, 11 * Kin + bits, gpu)
    x = wl.normal_bf16((rows, Kin), 1.0, Kin, dtype=DT[dtype])
    rhs = np.random.default_rng(Kin).integers(0, E, size=rows).astype(np.int32)
    ref = oracle.gather_qmm_f64(u16(x), np.arange(rows), rhs, u32(q), u16(s), u16(b), dtype=dtype)
    got = {}
    for shift in ((0, 0), (1, 1), (2, 2), (0, 1), (3, 0), (8, 2)):
        log(f"alignment {dtype} bits={bits} Kin={Kin} scales +{shift[0]} biases +{shift[1]}")
        out = tmoe.gather_qmm_rows(x.to(gpu), q, _shifted(s, shift[0]), _shifted(b, shift[1]),
                                   torch.from_numpy(rhs).to(gpu), bits=bits)
        torch.cuda.synchronize()
        got[shift] = u16(out)
        err = max_rel(oracle.st_to_f32(got[shift], dtype), ref)
        assert err <= STEP[dtype], (shift, err)
    for shift in ((2, 2), (8, 2)):
        np.testing.assert_array_equal(got[shift], got[0, 0])


# Around the router kernels' switches (64, 192 and 1024 tokens), token counts off 4
# and 16, every hidden width with a kernel, expert counts on both sides of 40
# and 48; infinite, NaN and subnormal rows. Bit for bit.
@pytest.mark.parametrize("T", [64, 65, 131, 192, 193, 1024, 1025, 1043])
@pytest.mark.parametrize("route,H,E", [("olmoe", 2048, 64), ("granite", 1536, 40), ("olmoe", 1024, 41),
                                       ("granite", 512, 7), ("olmoe", 512, 49)])
def test_prefill_router(gpu, route, H, E, T):
    log(f"prefill router {route} H={H} E={E} T={T}")
    I, K = 64, min(6, E)
    x = wl.normal_bf16((T, H), 1.0, T + H)
    x[1, 5] = float("inf")
    x[2, 7] = float("nan")
    x[3] = 1e-38
    x[4] = 0.0
    router = wl.normal_bf16((E, H), 0.02, E + T)
    router[0, :] = 1e-30
    lb = wl.zipf_bias(E, 3)
    blk = tmoe.MoEBlock(H, I, E, K, route=route)
    mk = [_affine((E, r, c), 4, "bf16", 900 + r, gpu) for r, c in ((I, H), (I, H), (H, I))]
    for bias in (None, lb):
        wts = tmoe.ExpertWeights(router.to(gpu), *mk[0], *mk[1], *mk[2],
                                 logit_bias=None if bias is None else bias.to(gpu))
        _, idx, gates = blk.forward(x.to(gpu), wts, return_routes=True)
        torch.cuda.synchronize()
        logits = oracle.router_logits(u16(x), u16(router), None if bias is None else bias.numpy())
        ridx, rg = oracle.route_olmoe(logits, K) if route == "olmoe" else oracle.route_granite(logits, K)
        np.testing.assert_array_equal(idx.cpu().numpy(), ridx)
        want = oracle.bf16_to_f32(rg) if route == "olmoe" else rg
        np.testing.assert_array_equal(gates.float().cpu().numpy(), want)


# The same kernels on half storage, whose router is affine and dequantised first:
# 4- and 16-token workgroups, half subnormals, infinities and NaN.
@pytest.mark.parametrize("T", [193, 1024, 1025, 1043])
@pytest.mark.parametrize("route,H,E,router_bits", [("olmoe", 2048, 64, 4), ("granite", 1536, 40, 4), ("olmoe", 1024, 49, 8),
                                                   ("granite", 512, 7, 8)])
def test_prefill_router_half(gpu, route, H, E, router_bits, T):
    log(f"prefill router half {route} H={H} E={E} T={T} router bits={router_bits}")
    I, K = 64, min(6, E)
    x = wl.normal_bf16((T, H), 1.0, T + H, dtype=torch.float16)
    x[1, 5] = float("inf")
    x[2, 7] = float("nan")
    x[3] = 5e-8  # one step of the half subnormals
    x[4] = 0.0
    x[5] = 3e-6
    rq, rs, rb = _affine((E, H), router_bits, "f16", E + T, gpu)
    rs, rb = rs * 0.3, rb * 0.3
    rs[0], rb[0] = 2e-7, -1.5e-6  # subnormal weights
    lb = wl.zipf_bias(E, 3)
    blk = tmoe.MoEBlock(H, I, E, K, route=route, dtype=torch.float16, router="affine")
    mk = [_affine((E, r, c), 4, "f16", 900 + r, gpu) for r, c in ((I, H), (I, H), (H, I))]
    for bias in (None, lb):
        wts = tmoe.ExpertWeights(None, *mk[0], *mk[1], *mk[2], router_q=rq, router_s=rs, router_b=rb, router_bits=router_bits,
                                 logit_bias=None if bias is None else bias.to(gpu))
        _, idx, gates = blk.forward(x.to(gpu), wts, return_routes=True)
        torch.cuda.synchronize()
        logits = oracle.router_logits_affine(u16(x), u32(rq), u16(rs), u16(rb), None if bias is None else bias.numpy(),
                                             dtype="f16")
        if route == "olmoe":
            ridx, rg = oracle.route_olmoe(logits, K, dtype="f16")
            rg = oracle.f16_to_f32(rg)
        else:
            ridx, rg = oracle.route_granite(logits, K, dtype="f16")
        np.testing.assert_array_equal(idx.cpu().numpy(), ridx)
        np.testing.assert_array_equal(gates.float().cpu().numpy(), rg)


# One workgroup up to 1024 routes, chunk histograms read whole up to 256
# chunks of 512, superblock sums past them; ids out of range go last.
@pytest.mark.parametrize("n", [63, 1000, 1024, 1025, 140003])
@pytest.mark.parametrize("E", [1, 40, 64])
def test_group_with_bad_ids(gpu, n, E):
    log(f"group n={n} E={E}, ids out of range")
    ids = np.random.default_rng(n + E).integers(-1, E + 2, size=n).astype(np.int32)
    order, inverse, offsets = tmoe.group(torch.from_numpy(ids).to(gpu), E)
    torch.cuda.synchronize()
    bucket = np.where((ids < 0) | (ids >= E), E, ids)
    want = np.argsort(bucket, kind="stable")
    np.testing.assert_array_equal(order.cpu().numpy(), want)
    np.testing.assert_array_equal(inverse.cpu().numpy()[want], np.arange(n))
    np.testing.assert_array_equal(offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(bucket, minlength=E + 1)[:E])]))
