"""Block outputs of a few fixed cases, for tests/test_gpu_knobs.py: run once
in the test process and once in a child process whose environment sets a
tuning override, so that the override's code path is checked for the same
bits. As a script: python -m tests._knob_cases OUT.npz"""
import sys

import numpy as np
import torch

from trifuse_amd import moe as tmoe
from trifuse_amd import workload as wl

# (geometry, tokens[, options]): one and two tokens take the streaming decode
# kernels (the down-weight copies when TFM_DS_PREFETCH=1); 300 and 400 OLMoE tokens
# and 64 and 1000 Granite tokens take the grouped GEMM at 32, 16, 12, 8 and 4
# super-steps (tile rows and waves: TFM_GGEMM_TILE, _DOWN_TILE and _WAVES; the
# router kernels: TFM_ROUTER_SPLIT_MAX_TOKENS), with half storage and 8-bit codes
# too; 8 tokens take the decode GEMV kernels (OLMoE with the published slot table,
# Granite with the grouping in every gate/up workgroup: TFM_DECODE_GROUPING swaps
# them); 32 tokens of either take 64-row tiles of at most 16 rows, which keep
# their weights two super-steps ahead (TFM_GGEMM_FEW_ROWS=0 one, as the other
# tiles do; =2 also runs the 300 OLMoE and 64 Granite tokens through that
# instance).
HALF = {"dtype": torch.float16, "affine_router": True}
CASES = [("olmoe", 1), ("olmoe", 2), ("granite", 1), ("olmoe", 300), ("granite", 64), ("olmoe", 8),
         ("granite", 8), ("olmoe", 32), ("granite", 32), ("olmoe", 400), ("granite", 1000), ("olmoe", 300, HALF),
         ("granite", 64, {"bits": 8}), ("olmoe", 300, {"bits": 8}), ("olmoe", 300, {"bits": 8, **HALF})]


def outputs(device="cuda:0"):
    out = {}
    for name, T, *opts in CASES:
        opt = opts[0] if opts else {}
        geom = wl.OLMOE if name == "olmoe" else wl.GRANITE
        layer = wl.make_layer(geom, 0, device, seed_tag=f"knob{name}", **opt)
        wts = tmoe.ExpertWeights.from_layer(layer)
        dtype = opt.get("dtype", torch.bfloat16)
        blk = tmoe.MoEBlock(geom.hidden, geom.intermediate, geom.experts, geom.top_k, route=geom.route,
                            bits=opt.get("bits", 4), dtype=dtype, router="affine" if "dtype" in opt else "dense")
        x = wl.make_x(geom, T, tag=f"knob{name}{T}").to(dtype).to(device)
        # The kernels a stage runs tell the router's two forms apart.
        with tmoe.StageProfiler() as prof:
            y = blk.forward(x, wts)
        torch.cuda.synchronize()
        key = f"{name}_{T}_{opt.get('bits', 4)}{'h' if 'dtype' in opt else ''}"
        out[key] = y.cpu().view(torch.int16).numpy()
        out["topk_" + key] = np.int32(prof.stage("topk")[1])
        prof.close()
    return out


if __name__ == "__main__":
    np.savez(sys.argv[1], **outputs())
