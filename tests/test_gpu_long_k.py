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


def _tables(lib, kid, probs):
    from mxmoe_amd import _lib

    n = len(probs)
    sizes = (_lib.Dim3 * n)(*[_lib.Dim3(*p[0]) for p in probs])
    qs = (_lib.QParams * n)(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for _, q in probs])
    if kid < 0:
        kid = lib.mxmoe_group_gemm_plan(-1, sizes, qs, n, None, None) - 1000
        assert kid >= 0, lib.mxmoe_last_error()
    out = (C.c_int32 * 1200)()
    assert lib.mxmoe_group_gemm_plan_tables(kid, sizes, qs, n, out, 1200) == 0, lib.mxmoe_last_error()
    return kid, np.array(out[:], np.int32)


def _tiles_of(lib, probs):
    from mxmoe_amd import _lib

    n = len(probs)
    sizes = (_lib.Dim3 * n)(*[_lib.Dim3(*p[0]) for p in probs])
    qs = (_lib.QParams * n)(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for _, q in probs])
    tiles = C.c_int32()
    assert lib.mxmoe_group_gemm_plan(-1, sizes, qs, n, None, C.byref(tiles)) >= 1000, lib.mxmoe_last_error()
    return tiles.value


@pytest.mark.parametrize("q,m", [((16, 4, 128, False), 64), ((16, 4, 128, False), 600), ((16, 8, 128, False), 200), ((4, 4, -1, True), 128), ((16, 16, -1, True), 128)])
def test_many_long_problems_keep_their_shapes(q, m):
    """Sixty problems of K = 4096 fill the chip: one of K = 2048 beside them is no reason for more and shorter tiles.  Nor is it for a few
    whose shorter tiles would together be the longer run; two small ones still take them."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    short = ((m, 2048, 2048), q)
    long = ((m, 2048, 4096), q)
    assert _tiles_of(lib, [long] * 60 + [short]) == _tiles_of(lib, [long] * 60) + _tiles_of(lib, [short])
    assert _tiles_of(lib, [long] * 200 + [short]) == _tiles_of(lib, [long] * 200) + _tiles_of(lib, [short])   # (two launches)
    few = ((100, 512, 4096), q)
    two = _tiles_of(lib, [few] * 2 + [((5, 512, 2048), q)])
    one = _tiles_of(lib, [few] + [((5, 512, 2048), q)])
    assert two - one == one - _tiles_of(lib, [((5, 512, 2048), q)]) > _tiles_of(lib, [few])


def test_problems_without_rows_have_no_say_in_the_shapes_of_others():
    """The device planner sees every expert, the operators leave out those without tokens: a problem without rows changes nothing."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    q = (16, 4, 128, False)
    live = [((201, 2048, 5632), q), ((40, 2048, 5632), q)]
    kid, alone = _tables(lib, -1, live)
    _, beside = _tables(lib, kid, live + [((0, 2048, 1408), q)])
    assert np.array_equal(alone, beside)


def test_plan_of_a_sequential_kernel_is_that_of_its_launches():
    """One launch per run of equal formats: the problem of smaller K is in another launch and makes nothing long."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    seq = lib.mxmoe_find_kernel(b"groupgemm_seq_launch_all")
    probs = [((201, 2048, 5632), (16, 4, 128, False)), ((201, 2048, 1408), (16, 16, -1, True))]
    sizes = (_lib.Dim3 * 2)(*[_lib.Dim3(*p[0]) for p in probs])
    qs = (_lib.QParams * 2)(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for _, q in probs])
    tiles = C.c_int32()
    assert lib.mxmoe_group_gemm_plan(seq, sizes, qs, 2, None, C.byref(tiles)) == 1000 + seq
    assert tiles.value == sum(int(_tables(lib, seq, [p])[1][1]) for p in probs)


LONG_LISTS = [  # (formats, N, K of each expert, rows of each expert, shared rows)
    ([(16, 4, 128, False), (16, 3, 128, False)], 2048, [4096] * 9 + [2048], [64] * 9 + [7], 0),
    ([(16, 4, 128, False)], 2048, [2048, 4096, 2048, 4096], [40, 100, 3, 0], 100),                  # two long ones, one without rows
    ([(16, 4, 128, False), (4, 4, -1, True)], 512, [4096] * 3 + [2048] * 100 + [4096] * 2, [90] * 105, 128),   # in both waves of the planner
    ([(4, 4, -1, True), (16, 16, -1, True)], 1024, [4096, 4096, 2048, 2048, 5632], [100, 128, 50, 1, 30], 60),
    ([(16, 8, 128, False)], 2048, [2048] * 5, [100] * 5, 300),                                      # long by the shared one alone
    ([(16, 4, 128, False)], 2048, [2048] * 120 + [4096] * 5, [20] * 125, 64),                      # two launches, one without a short problem
]


def _long_list(case):
    fmts, n, ks, rows, shared = case
    ks = ks + ([2 * max(ks)] if shared else [])
    return [fmts[i % len(fmts)] for i in range(len(ks))], n, ks, rows, shared


@pytest.mark.parametrize("case", range(len(LONG_LISTS)))
def test_grid_bound_covers_lists_of_long_problems(case):
    """The worst-case grid against the host's plan for random routings, where any number of problems may be the long ones of their launch."""
    import random

    from mxmoe_amd import _lib

    lib = _lib.load()
    qs, n, ks, rows, shared = _long_list(LONG_LISTS[case])
    e, et, total = len(rows), len(ks), sum(rows)
    desc = (_lib.BlockDesc * et)(*[_lib.BlockDesc(q[0], q[1], q[2], int(q[3]), (C.c_uint8 * 3)(), n, k, 0, 0) for q, k in zip(qs, ks)])
    kid = lib.mxmoe_plan_select_kernel(-1, desc, et)
    bound = lib.mxmoe_plan_grid_bound(kid, desc, e, total, shared)
    assert kid >= 0 and bound > 0, lib.mxmoe_last_error()
    rnd = random.Random(case)
    for trial in range(60):
        cuts = sorted(rnd.randint(0, total) for _ in range(e - 1))
        counts = rows if trial == 0 else [b - a for a, b in zip([0] + cuts, cuts + [total])]
        probs = [((m, n, k), q) for m, k, q in zip(counts + [shared] * (shared > 0), ks, qs)]
        for at in range(0, et, 120):
            _, host = _tables(lib, kid, probs[at:at + 120])
            assert host[3] <= bound, (trial, host[:4], bound)


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(LONG_LISTS)))
def test_device_planner_agrees_on_lists_of_long_problems(case):
    """Entries, phases and totals of the planning kernel against the host's (nothing is launched on them: the operands' addresses are not read)."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    qs, n, ks, rows, shared = _long_list(LONG_LISTS[case])
    e, et = len(rows), len(ks)
    desc = (_lib.BlockDesc * et)(*[_lib.BlockDesc(q[0], q[1], q[2], int(q[3]), (C.c_uint8 * 3)(), n, k, 0, 0) for q, k in zip(qs, ks)])
    kid = lib.mxmoe_plan_select_kernel(-1, desc, et)
    assert kid >= 0, lib.mxmoe_last_error()
    d_desc = torch.frombuffer(bytearray(bytes(desc)), dtype=torch.uint8).cuda()
    recv = torch.tensor(rows, dtype=torch.int64, device="cuda")
    plan = torch.zeros(lib.mxmoe_plan_bytes(et), dtype=torch.uint8, device="cuda")
    some = torch.zeros(16, dtype=torch.uint8, device="cuda")
    _lib.check(lib, lib.mxmoe_plan_block(kid, recv.data_ptr(), e, shared, d_desc.data_ptr(), desc, some.data_ptr(), some.data_ptr(), some.data_ptr(), plan.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
    got = plan.cpu().numpy()
    probs = [((m, n, k), q) for m, k, q in zip(rows + [shared] * (shared > 0), ks, qs)]
    for chunk, at in enumerate(range(0, et, 120)):
        _, host = _tables(lib, kid, probs[at:at + 120])
        ne, tiles, nph, _grid = host[:4]
        hdr = got[chunk * 4096:(chunk + 1) * 4096].view(np.int32)[14:]      # behind seven pointers
        assert list(hdr[:4]) == [at, ne, tiles, nph]
        assert np.array_equal(hdr[4:5 + nph], host[4:5 + nph]) and np.array_equal(hdr[13:14 + nph], host[13:14 + nph])
        assert np.array_equal(hdr[23:23 + 4 * ne], host[22:22 + 4 * ne])


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_few", "groupgemm_hz_fused_all_few"])
@pytest.mark.parametrize("n,experts,shared", [(4096, 8, 0), (4096, 9, 0), (2048, 7, 100), (512, 63, 33)])
def test_device_planner_agrees_on_launches_of_few_blocks(kernel, n, experts, shared):
    """The same comparison on the kernels with narrow tiles, at and past 128 blocks of 256 channels: problems of more than 32 rows."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    kid = lib.mxmoe_find_kernel(kernel.encode())
    fmts = [(4, 4, -1, True), (8, 8, -1, True)] + ([(16, 4, 128, False)] if "all" in kernel else [])
    rows = [(45, 30, 64, 1, 129, 33, 16, 100)[i % 8] for i in range(experts)]
    qs = [fmts[i % len(fmts)] for i in range(experts + (shared > 0))]
    ks = [2048] * experts + [4096] * (shared > 0)
    et = len(ks)
    desc = (_lib.BlockDesc * et)(*[_lib.BlockDesc(q[0], q[1], q[2], int(q[3]), (C.c_uint8 * 3)(), n, k, 0, 0) for q, k in zip(qs, ks)])
    d_desc = torch.frombuffer(bytearray(bytes(desc)), dtype=torch.uint8).cuda()
    recv = torch.tensor(rows, dtype=torch.int64, device="cuda")
    plan = torch.zeros(lib.mxmoe_plan_bytes(et), dtype=torch.uint8, device="cuda")
    some = torch.zeros(16, dtype=torch.uint8, device="cuda")
    _lib.check(lib, lib.mxmoe_plan_block(kid, recv.data_ptr(), experts, shared, d_desc.data_ptr(), desc, some.data_ptr(), some.data_ptr(), some.data_ptr(), plan.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
    _, host = _tables(lib, kid, [((m, n, k), q) for m, k, q in zip(rows + [shared] * (shared > 0), ks, qs)])
    ne, tiles, nph, grid = host[:4]
    hdr = plan.cpu().numpy()[:4096].view(np.int32)[14:]
    assert list(hdr[:4]) == [0, ne, tiles, nph] and grid <= lib.mxmoe_plan_grid_bound(kid, desc, experts, sum(rows), shared)
    assert np.array_equal(hdr[4:5 + nph], host[4:5 + nph]) and np.array_equal(hdr[13:14 + nph], host[13:14 + nph])
    assert np.array_equal(hdr[23:23 + 4 * ne], host[22:22 + 4 * ne])


@pytest.mark.gpu
@pytest.mark.parametrize("routed", [False, True])
def test_layer_whose_tokens_all_go_to_its_shared_expert(routed):
    """No expert id in range (or of one slot only): the shared expert is alone in its launches, in the device's plan and in the host's."""
    from mxmoe_amd import synth as S
    from mxmoe_amd.layer import MxMoELayer

    cfg = S.MoEConfig("t", "test", 4, 2, 512, 1408, 201, num_shared=4, rotate=1)
    layer = MxMoELayer(cfg, formats=[(S.W4A16, S.W3A16)] * 5)
    hidden = S.make_hidden(cfg)
    ids, w = S.make_routing(cfg)
    ids = torch.full_like(ids, -1)
    if routed:
        ids[17, 1] = 2
    got = layer(hidden, ids, w)
    assert torch.equal(got, layer.call_with_host_tables(hidden, ids, w)) and bool((got != 0).any())
