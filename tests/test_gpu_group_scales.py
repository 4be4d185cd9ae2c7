"""w4a4_g128 tiles: the products of token and channel scales come out of the matrix pipe."""
import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_g128", "groupgemm_hz_fused_all"])
@pytest.mark.parametrize("scale", ["as quantised", "subnormal", "largest", "zero and infinite"])
def test_scale_products_are_exact(kernel, scale):
    """Sums over the groups (bit patterns) and outputs equal the oracle's for scales over the whole range of fp16, at 1, 32, 33, 64 and 65 rows (both tile
    shapes and their edges), one group, an odd and an even number of groups, and channels that end inside a 32-channel block."""
    from mxmoe_amd import _lib, pack
    from mxmoe_amd.group_gemm import GroupGemmLaunch

    rng = np.random.default_rng(5)
    probs = []
    for m, n, k in [(1, 256, 128), (32, 264, 384), (33, 40, 256), (64, 512, 1408), (65, 256, 2048)]:
        qa, qb = rng.integers(-7, 8, (m, k)), rng.integers(-7, 8, (n, k))
        g = k // 128
        if scale == "subnormal":      # 2^-24 .. 2^-15, products down to 2^-38
            sa, sb = rng.integers(1, 1024, (m, g)), rng.integers(1, 1024, (n, g))
            sa, sb = sa.astype(np.uint16).view(np.float16), sb.astype(np.uint16).view(np.float16)
        elif scale == "largest":
            sa, sb = (rng.uniform(3e4, 6.5e4, s).astype(np.float16) for s in ((m, g), (n, g)))
        else:
            sa, sb = rng.uniform(0.01, 1.0, (m, g)).astype(np.float16), rng.uniform(1e-4, 1e-2, (n, g)).astype(np.float16)
        if scale == "zero and infinite":
            sa[0, 0] = 0
            sb[::7, 0] = 0
            sb[3, 0] = np.inf
        with np.errstate(all="ignore"):
            out, f32 = O.epilogue_grouped(O.int_gemm_grouped(qa, qb, 128), sa, sb)
        ta = pack.pack_int4_k(torch.from_numpy(qa.astype(np.int8))).cuda()
        tb = pack.pack_wxax_fragments(pack.pack_int4_k(torch.from_numpy(qb.astype(np.int8)))).cuda()
        probs.append((ta, tb, torch.from_numpy(sa.copy()).cuda(), torch.from_numpy(np.ascontiguousarray(sb.T)).cuda(), (m, n, k), out, f32))
    kid = _lib.load().mxmoe_find_kernel(kernel.encode())
    Cs = [torch.full(p[4][:2], float("nan"), dtype=torch.float16, device="cuda") for p in probs]
    acc = [torch.zeros(p[4][:2], dtype=torch.int32, device="cuda") for p in probs]
    GroupGemmLaunch([p[0] for p in probs], [p[1] for p in probs], [p[2] for p in probs], [p[3] for p in probs], Cs, [p[4] for p in probs], [(4, 4, 128, True)] * len(probs),
                    kernel_id=kid, acc=acc).run()
    for p, c, a in zip(probs, Cs, acc):
        got, want = a.cpu().numpy().view(np.float32), p[6]
        same = (got.view(np.int32) == want.view(np.int32)) | (np.isnan(got) & np.isnan(want))   # (which NaN is nobody's promise)
        assert same.all(), (p[4], np.argwhere(~same)[:3])
        got, want = c.cpu().numpy(), p[5]
        assert ((got.view(np.uint16) == want.view(np.uint16)) | (np.isnan(got) & np.isnan(want))).all(), p[4]
