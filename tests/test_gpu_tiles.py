"""The grouped GEMM's tile variants, the prefill router and the grouping at the
sizes where their dispatch and remainders change, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from tests._util import BLOCK_TOL, log, max_rel, u16, u32
from trifuse_amd import moe as tmoe
from trifuse_amd import workload as wl

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16}
# A product's largest error over its largest value. A weight and the result
# are each rounded to the storage type (half a step: 2^-9 of a bf16 value, 2^-12
# of a half one). Weight errors add up as a random walk and stay below half a
# step of the largest result; the fp32 sums add 1e-6. Twice the half step.
STEP = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}


def _affine(shape, bits, dtype, key, device):
    *lead, width = shape
    q = wl.packed_nibbles((*lead, width * bits // 32), key, device)
    k = 16 / 2 ** bits
    s = wl.uniform_scales((*lead, width // 64), key + 1, device, lo=0.005 * k, hi=0.02 * k, dtype=DT[dtype])
    return q, s, (s.float() * -float(2 ** (bits - 1))).to(DT[dtype])


def _routes(T, E, K, seed):
    """K distinct experts a token: expert 0 for every other token (more rows
    than one tile), expert 1 for none, the rest at random."""
    rng = np.random.default_rng(seed)
    score = rng.random((T, E))
    score[::2, 0] = 2.0
    score[:, 1] = -1.0
    return np.argsort(-score, axis=1)[:, :K].astype(np.int32)


# Routes per expert on average, over the tile rule's lines: 64-, 96- and
# 128-row tiles, two 96-row tiles, 128 and 256 rows.
@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("f16", 4), ("bf16", 8), ("f16", 8)])
@pytest.mark.parametrize("a", [6, 30, 60, 90, 105, 140, 200, 450])
def test_block_tiles(gpu, dtype, bits, a):
    H, I, E, K = 1024, 1024, 64, 8
    T = a * E // K + 3
    log(f"block tiles {dtype} bits={bits} a={a} T={T}")

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
    pick = np.unique(np.concatenate([np.arange(4), np.linspace(0, T - 1, 12).astype(np.int64), [T - 1]]))
    ref = oracle.moe_reference(u16(x)[pick], idx[pick], gates[pick], lay, dtype=dtype)
    err = max_rel(oracle.st_to_f32(u16(y)[pick], dtype), ref)
    log(f"  max_rel {err:.2e}")
    assert err <= BLOCK_TOL


# Input widths: odd multiples of 64 (the LDS-dequantising kernel), one
# super-step, group counts not a multiple of 8 (4-byte scale copies), past
# 2048; output widths off the tile; rows around 16, 32, 64, 96 and 128; the
# lines between which 8-bit bf16 codes take the LDS-dequantising kernel (57, 384
# and not 480 to 528 rows an expert).
@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("f16", 4), ("bf16", 8), ("f16", 8)])
@pytest.mark.parametrize("E,N,Kin,rows", [(1, 64, 64, 200), (1, 192, 128, 177), (2, 320, 192, 500), (3, 128, 384, 401),
                                          (2, 192, 640, 290), (1, 256, 2304, 180), (40, 64, 1536, 41 * 17),
                                          (64, 1024, 128, 64 * 60), (64, 1024, 256, 64 * 110), (64, 1088, 128, 64 * 140),
                                          (64, 1024, 128, 64 * 250), (64, 2048, 128, 64 * 57), (16, 1536, 256, 16 * 383),
                                          (16, 1536, 256, 16 * 384), (16, 1536, 256, 16 * 500), (16, 1536, 256, 16 * 530)])
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
    assert err <= BLOCK_TOL


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


# Around the router kernels' switches (64 and 1024 tokens), token counts off 4
# and 16, every hidden width with a kernel, expert counts on both sides of 40
# and 48; infinite, NaN and subnormal rows. Bit for bit.
@pytest.mark.parametrize("T", [64, 65, 131, 1024, 1025, 1043])
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
