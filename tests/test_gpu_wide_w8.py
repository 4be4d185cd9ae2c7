"""The many-token tiles of the 8-bit weight-only formats: 128 x 256, which holds its packed weights in halves, and 128 x 128, which launches of few tiles take."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [128, 256, 384, 1408, 4096])
@pytest.mark.parametrize("gs,sym", [(128, False), (-1, True)])
@pytest.mark.parametrize("bn", [256, 128])
def test_wide_tile_of_8_bit_weights(k, gs, sym, bn):
    """One k block, an even and an odd number of them; 33 and 64 rows (half a tile: the shorter loop), 65, 128 and 200; channels that end inside a wave's 64, and
    waves without any.  Every weight is q * scale + zero rounded once to fp16; against the float64 product with those: the output's rounding
    is at most 2^-11 of it, and the fp32 sums of up to 4096 exact products, K * 2^-24 of the sum of their sizes at worst, stay an order below that."""
    from mxmoe_amd import _lib
    from mxmoe_amd.group_gemm import GroupGemmLaunch
    from mxmoe_amd.weights import quantize_and_pack

    lib = _lib.load()
    rng = np.random.default_rng(k)
    probs = []
    # (a launch of few tiles runs the slim tile, one problem of many makes it the wide one)
    for m, n in [(33, 144), (64, 256), (65, 16), (128, 528), (200, 272)] + [(129 * 128, 256)] * (bn == 256):
        x = rng.standard_normal((m if m <= 200 else 1, k)).astype(np.float16)
        w = (rng.standard_normal((n, k)) * 0.02).astype(np.float16)
        pw = quantize_and_pack(torch.from_numpy(w), (16, 8, gs, sym))
        if m > 200:
            probs.append((torch.from_numpy(x).cuda().expand(m, k).contiguous(), pw.data.cuda(), pw.scale.cuda(), (m, n, k), None))
            continue
        q, s, z = O.quant_minmax(w, 8, gs, sym)
        groups = k // 128 if gs > 0 else 1
        if sym:
            z = np.zeros_like(s)
        deq = q.reshape(n, groups, -1).astype(np.float64) * s.reshape(n, groups, 1).astype(np.float64) + z.reshape(n, groups, 1).astype(np.float64)
        ref = x.astype(np.float64) @ deq.reshape(n, k).astype(np.float16).astype(np.float64).T
        probs.append((torch.from_numpy(x).cuda(), pw.data.cuda(), pw.scale.cuda(), (m, n, k), ref))
    for kernel in ("groupgemm_hz_fused_wo8", "groupgemm_hz_fused_all"):
        kid = lib.mxmoe_find_kernel(kernel.encode())
        Cs = [torch.full(p[3][:2], float("nan"), dtype=torch.float16, device="cuda") for p in probs]
        g = GroupGemmLaunch([p[0] for p in probs], [p[1] for p in probs], [None] * len(probs), [p[2] for p in probs], Cs, [p[3] for p in probs], [(16, 8, gs, sym)] * len(probs), kernel_id=kid)
        info = (C.c_int32 * 8)()
        for (_, _, _, (m, _n, _k), _ref), b in zip(probs, g.plan()[1]):
            assert lib.mxmoe_kernel_branch(kid, b, info) == 0 and (info[1], info[2]) == (128, bn), (m, info[:3])
        g.run()
        for p, c in zip(probs, Cs):
            if p[4] is None:
                continue
            got = c.cpu().numpy().astype(np.float64)
            err = np.linalg.norm(got - p[4]) / np.linalg.norm(p[4])
            assert err <= 2.0 ** -11, (kernel, p[3], err)
