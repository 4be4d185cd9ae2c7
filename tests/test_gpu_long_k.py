"""Problems whose K is above the smallest of their launch (a shared expert): the shape the planner gives them, and their results."""
import ctypes as C

import numpy as np
import pytest
import torch

CASES = [((16, 4, 128, False), [(33, 32), (128, 32), (201, 32), (513, 32), (20, 16), (2048, 128)]),
         ((4, 4, -1, True), [(32, 32), (100, 32), (128, 32), (129, 128)]),
         ((16, 16, -1, True), [(128, 32), (129, 128)])]


def _rows_of_tile(lib, m, n, k, q):
    from mxmoe_amd import _lib

    sizes = (_lib.Dim3 * 2)(_lib.Dim3(m, n, k), _lib.Dim3(5, n, k // 4))
    qs = (_lib.QParams * 2)(*[_lib.QParams(q[0], q[1], q[2], int(q[3]))] * 2)
    br = (C.c_int32 * 2)()
    rc = lib.mxmoe_group_gemm_plan(-1, sizes, qs, 2, br, None)
    assert rc >= 1000, lib.mxmoe_last_error()
    info = (C.c_int32 * 8)()
    assert lib.mxmoe_kernel_branch(rc - 1000, br[0], info) == 0
    return info[1]


@pytest.mark.parametrize("q,want", CASES)
def test_shape_of_a_long_problem(q, want):
    from mxmoe_amd import _lib

    lib = _lib.load()
    for m, rows in want:
        got = _rows_of_tile(lib, m, 2048, 5632, q)
        assert got <= 32 if rows <= 32 else got == rows, (m, got)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [33, 100, 128, 129, 201, 256, 420])
@pytest.mark.parametrize("mix", ["wo", "wo8", "wxax", "fp16", "fp8"])
def test_layer_with_a_wide_shared_expert(tokens, mix):
    """Device-planned and host-planned forwards pick the same tiles, so they agree bit for bit; the outputs stay within 1e-2 (2-norm) of the
    same layer through one row tile at a time, i.e. of its tokens in batches too small for any large tile."""
    from mxmoe_amd import synth as S
    from mxmoe_amd.layer import MxMoELayer

    f = {"wo": [(S.W4A16, S.W3A16), (S.W3A16, S.W4A16), (S.W2A16, S.W2A16)], "wo8": [((16, 8, 128, False),) * 2] * 3,
         "wxax": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W4A4, S.W4A4)], "fp16": [(S.FP16, S.FP16)] * 3,
         "fp8": [(S.W8A8, S.W8A8), (S.W4A4, S.W8A8), (S.W4A4, S.W4A4)]}[mix]
    cfg = S.MoEConfig("t", "test", 4, 2, 512, 1408, tokens, num_shared=4, rotate=1)
    layer = MxMoELayer(cfg, formats=[f[i % 3] for i in range(5)], fp8=mix == "fp8")
    hidden = S.make_hidden(cfg)
    ids, w = S.make_routing(cfg)
    got = layer(hidden, ids, w)
    want = layer.call_with_host_tables(hidden, ids, w)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    part = torch.cat([layer.call_with_host_tables(hidden[i:i + 16].contiguous(), ids[i:i + 16].contiguous(), w[i:i + 16].contiguous()) for i in range(0, tokens, 16)])
    a, b = got.double().cpu().numpy(), part.double().cpu().numpy()
    assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b)
