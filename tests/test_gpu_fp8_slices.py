"""The fp8 tiles at the edges of their K slices and rows, against float64 sums of the codes' values."""
import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O
from test_gpu_group_gemm import DEV, F16, _launch

pytestmark = pytest.mark.gpu


# one to five slices of 64 values (the loop runs four at a time) and the lengths of a layer; rows on either side of each tile shape's edge.  A product of two codes
# has 8 bits and is aligned to the largest of its instruction's sum: the bound is that of the 16-deep instruction's test, 2e-4 of the largest sum.
@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 1408, 2048])
def test_fp8_tiles_at_the_edges_of_slices_and_rows(k):
    from mxmoe_amd import _lib, pack

    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_wxax_e4m3")
    rng = np.random.default_rng(k)
    probs = []
    for m, n in [(1, 264), (32, 512), (33, 256), (64, 512), (65, 256), (128, 512), (129, 264), (300, 768)]:
        ca, sa = O.quant_e4m3((rng.standard_normal((m, k)) * rng.uniform(0.1, 4, (m, 1))).astype(F16))
        cb, sb = O.quant_e4m3((rng.standard_normal((n, k)) * 0.02).astype(F16))
        probs.append(dict(A=torch.from_numpy(ca).to(DEV), B=pack.pack_wxax_fragments(torch.from_numpy(cb)).to(DEV), sa=torch.from_numpy(sa.reshape(-1)).to(DEV),
                          sb=torch.from_numpy(sb.reshape(-1)).to(DEV), acc32=O.fp8_gemm(ca, cb), size=(m, n, k), q=(8, 8, -1, True)))
    for _ in range(3):
        _, _, accs = _launch(probs, kernel_id=kid)
        for p, acc in zip(probs, accs):
            assert np.abs(acc.view(np.float32) - p["acc32"]).max() <= 2e-4 * np.abs(p["acc32"]).max(), p["size"]


# Small products beside large ones keep the fewest bits in an instruction that aligns 64 of them to the largest: rows with a few channels a hundred times the rest,
# on both sides and on one, and operands of one sign.  The sums are at most 7.1e-5 off the float64 ones in the 2-norm here (3.3e-6 with one sign), with 16 and with 64
# products to an instruction alike, to three digits; the bounds are 1.7 times that.
@pytest.mark.parametrize("k", [64, 1408, 4096])
@pytest.mark.parametrize("operands", ["outliers", "outliers on one side", "outliers in one slice", "positive"])
def test_fp8_sums_of_uneven_operands(k, operands):
    from mxmoe_amd import _lib, pack

    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_wxax_e4m3")
    rng = np.random.default_rng(k)
    probs = []
    for m, n in [(32, 512), (64, 512), (128, 512)]:
        x, w = rng.standard_normal((m, k)), rng.standard_normal((n, k)) * 0.02
        if operands == "positive":
            x, w = np.abs(x), np.abs(w)
        else:
            cols = slice(0, 3) if "slice" in operands else rng.choice(k, max(3, k // 100), replace=False)
            x[:, cols] *= 100
            if operands == "outliers":
                w[:, rng.choice(k, 3)] *= 60
        ca, sa = O.quant_e4m3(x.astype(F16))
        cb, sb = O.quant_e4m3(w.astype(F16))
        probs.append(dict(A=torch.from_numpy(ca).to(DEV), B=pack.pack_wxax_fragments(torch.from_numpy(cb)).to(DEV), sa=torch.from_numpy(sa.reshape(-1)).to(DEV),
                          sb=torch.from_numpy(sb.reshape(-1)).to(DEV), ref=O.e4m3_decode(ca).astype(np.float64) @ O.e4m3_decode(cb).astype(np.float64).T, size=(m, n, k), q=(8, 8, -1, True)))
    _, _, accs = _launch(probs, kernel_id=kid)
    errors = [np.linalg.norm(acc.view(np.float32) - p["ref"]) / np.linalg.norm(p["ref"]) for p, acc in zip(probs, accs)]
    print(operands, k, ["%.2e" % e for e in errors])
    assert max(errors) <= (6e-6 if operands == "positive" else 1.2e-4), errors
