"""The order of a launch's tiles: which part of which problem each workgroup computes, on the host, through the functions the kernels call."""
import ctypes as C

import numpy as np
import pytest
import torch

W4, W8, FP, WO, WO8 = (4, 4, -1, True), (8, 8, -1, True), (16, 16, -1, True), (16, 4, 128, False), (16, 8, 128, False)


def _launch(lib, probs, kid=-1):
    from mxmoe_amd import _lib

    n = len(probs)
    sizes = (_lib.Dim3 * n)(*[_lib.Dim3(*p[:3]) for p in probs])
    qs = (_lib.QParams * n)(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for *_, q in probs])
    if kid < 0:
        kid = lib.mxmoe_group_gemm_plan(-1, sizes, qs, n, None, None) - 1000
        assert kid >= 0, lib.mxmoe_last_error()
    out = (C.c_int32 * 1200)()
    assert lib.mxmoe_group_gemm_plan_tables(kid, sizes, qs, n, out, 1200) == 0, lib.mxmoe_last_error()
    tab = np.array(out[:], np.int64)
    grid = int(tab[3]) + 64
    area = (C.c_int32 * (5 * grid))()
    assert lib.mxmoe_group_gemm_plan_tile_area(kid, sizes, qs, n, grid, area) == 0, lib.mxmoe_last_error()
    return tab, np.array(area[:], np.int64).reshape(grid, 5)


def _pairs(tab):
    entries = tab[22:22 + 4 * tab[0]].reshape(-1, 4)
    return [int(e[3]) & 0xFFFF for e in entries if (int(e[3]) >> 29) & 1]  # problems whose second segment runs beside the first


@pytest.mark.parametrize("q,rows,n,k", [
    (W8, 144, 2816, 2048), (W8, 192, 2816, 2048), (W8, 129, 2816, 2048), (W8, 546, 2048, 1408), (FP, 144, 2816, 2048), (FP, 300, 1288, 4096),
    (W4, 300, 28672, 4096), (W8, 1060, 28672, 4096),                  # activations of several groups of row tiles: the second segment goes with the last
    (W8, 160, 2824, 2048),                                            # the last column tile is 8 wide
    (WO, 140, 2816, 2048), (W4, 144, 2816, 2048),                     # two segments, no pairs
    (WO8, 140, 272, 2048), (WO8, 300, 16, 1408), (WO8, 140, 2816, 2048),  # slim tiles, wide tiles
])
def test_every_output_is_computed_once(lib, q, rows, n, k):
    """Every element of every output in exactly one workgroup's tile, for problems of two row segments next to empty and small ones."""
    probs = [((rows, rows + 1, rows - 1, 0, 7, 128)[i % 6], n, k, q) for i in range(60)]
    tab, area = _launch(lib, probs)
    assert bool(_pairs(tab)) == (q is W8 or q is FP or n == 28672)
    area = area[area[:, 0] >= 0]
    for p, (m, *_rest) in enumerate(probs):
        cover = np.zeros((m, n), np.int8)
        for _, r0, r1, c0, c1 in area[area[:, 0] == p]:
            cover[r0:r1, c0:c1] += 1
        assert (cover == 1).all(), (p, m)


def test_tiles_of_a_pair_that_share_weights_are_neighbours(lib):
    """All row tiles of both shapes against one block of channels come one after the other on an XCD (workgroup w runs on XCD w mod 8)."""
    tab, area = _launch(lib, [(192, 2816, 2048, W8)] * 64)
    assert len(_pairs(tab)) == 64
    area = area[area[:, 0] >= 0]
    order = np.concatenate([area[x::8] for x in range(8)])
    first = order[::2]
    assert (order[1::2, [0, 3, 4]] == first[:, [0, 3, 4]]).all() and set(map(tuple, first[:, 1:3])) == {(0, 128)} and set(map(tuple, order[1::2, 1:3])) == {(128, 192)}


@pytest.mark.parametrize("q,count,rows,n,k,pairs", [
    (W8, 64, 192, 2048, 1408, True), (W8, 8, 300, 4096, 14336, False),     # 1024 and 384 tiles: past and within what runs at a time
    (W8, 16, 144, 4096, 14336, True), (W8, 12, 144, 4096, 14336, False), (FP, 7, 180, 4096, 14336, False), (FP, 8, 256 + 10, 4096, 4096, False),  # 512 and 384, 224, 384
    (W8, 1, 546, 28672, 4096, False), (FP, 1, 546, 28672, 4096, True), (W8, 2, 290, 28672, 4096, True), (W8, 24, 290, 2048, 1408, False),  # 112, 224, 224, 48 columns
    (W8, 16, 420, 2816, 2048, True), (FP, 32, 144, 2048, 1408, False),     # 704 tiles; 512 of little weight
    (W4, 64, 192, 2816, 2048, False), (W4, 8, 300, 28672, 4096, True),     # int4: by what there is to fetch
    (W4, 24, 144, 4096, 14336, False), (W4, 32, 160, 4096, 14336, True),   # 768 and 1024 tiles
    (WO, 64, 140, 28672, 4096, False), ((4, 4, 128, True), 64, 90, 28672, 4096, False),
])
def test_when_segments_are_paired(lib, q, count, rows, n, k, pairs):
    tab, _ = _launch(lib, [(rows, n, k, q)] * count)
    assert (len(_pairs(tab)) == count) == pairs and (pairs or not _pairs(tab))
    # a problem without rows changes nothing
    tab2, _ = _launch(lib, [(rows, n, k, q)] * count + [(0, n, k, q)] * 8)
    assert (tab[:22] == tab2[:22]).all() and (tab[22:22 + 4 * tab[0]] == tab2[22:22 + 4 * tab[0]]).all()


def _device_plan_is_the_hosts(lib, q, counts, n, k):
    """Entries and phases of a block as the device planner leaves them against the host's; the host's tables."""
    from mxmoe_amd import _lib

    e = len(counts)
    qs, ks = (q if isinstance(q, list) else [q] * e), (k if isinstance(k, list) else [k] * e)
    desc = (_lib.BlockDesc * e)(*[_lib.BlockDesc(a, w, g, int(sym), (C.c_uint8 * 3)(), n, kk, 0, 0) for (a, w, g, sym), kk in zip(qs, ks)])
    kid = lib.mxmoe_plan_select_kernel(-1, desc, e)
    d_desc = torch.frombuffer(bytearray(bytes(desc)), dtype=torch.uint8).cuda()
    recv = torch.tensor(counts, dtype=torch.int64, device="cuda")
    plan = torch.zeros(lib.mxmoe_plan_bytes(e), dtype=torch.uint8, device="cuda")
    some = torch.zeros(16, dtype=torch.uint8, device="cuda")
    _lib.check(lib, lib.mxmoe_plan_block(kid, recv.data_ptr(), e, 0, d_desc.data_ptr(), desc, some.data_ptr(), some.data_ptr(), some.data_ptr(), plan.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
    tab, _ = _launch(lib, [(m, n, kk, qq) for m, kk, qq in zip(counts, ks, qs)], kid)
    ne, tiles, nph, grid = tab[:4]
    hdr = plan.cpu().numpy()[:4096].view(np.int32)[14:]
    assert list(hdr[:4]) == [0, ne, tiles, nph] and grid <= lib.mxmoe_plan_grid_bound(kid, desc, e, sum(counts), 0)
    assert np.array_equal(hdr[4:5 + nph], tab[4:5 + nph]) and np.array_equal(hdr[13:14 + nph], tab[13:14 + nph])
    assert np.array_equal(hdr[23:23 + 4 * ne], tab[22:22 + 4 * ne].astype(np.int32))
    return tab


# 8-bit weights, 128 rows: the 128 x 128 tile where a launch's 128 x 256 ones are up to 128, for up to 64 rows where they times K are up to 48 * 2048
@pytest.mark.parametrize("count,rows,n,k,bn", [
    (8, 96, 4096, 14336, 128), (8, 128, 4096, 4096, 128), (4, 192, 4096, 4096, 128), (2, 65, 4096, 4096, 128),          # 128 wide tiles and fewer
    (1, 128, 28672, 4096, 128), (1, 129, 28672, 4096, 256), (9, 96, 4096, 14336, 256), (1, 1100, 4096, 4096, 256),       # 112, 224, 144, 144
    (4, 64, 2816, 2048, 128), (5, 64, 2816, 2048, 256), (1, 33, 4096, 4096, 128), (2, 64, 4096, 4096, 256), (2, 65, 4096, 4096, 128), (1, 64, 4096, 14336, 256),
])
@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wo8", "groupgemm_hz_fused_all"])
def test_width_of_the_8_bit_weight_only_tile(lib, kernel, count, rows, n, k, bn):
    kid = lib.mxmoe_find_kernel(kernel.encode())

    def shapes(probs):
        tab, _ = _launch(lib, probs, kid)
        info, seen = (C.c_int32 * 8)(), {}
        for first, row0, m, pb in tab[22:22 + 4 * tab[0]].reshape(-1, 4):
            assert lib.mxmoe_kernel_branch(kid, int(pb) >> 16 & 31, info) == 0
            seen.setdefault(int(pb) & 0xFFFF, []).append((int(m), info[1], info[2]))
        return seen

    for tiles in shapes([(rows, n, k, WO8)] * count + [(0, n, k, WO8), (7, 256, k, WO8)]).values():
        assert all(t[1:] == (128, bn) if t[0] > 32 else t[1:] != (128, 384 - bn) for t in tiles), tiles
    # other formats' large tiles count too, those of problems of another K do not
    if kernel.endswith("all") and rows <= 128:
        assert shapes([(rows, n, k, WO8), (128, 33024, k, WO)])[0] == [(rows, 128, 256)]
        assert shapes([(rows, n, k, WO8)] * count + [(7, 256, k, WO8), (128, 33024, 2 * k, WO)])[0] == [(rows, 128, bn)]


@pytest.mark.gpu
@pytest.mark.parametrize("count,rows,n,k", [(8, 192, 2048, 1408), (16, 192, 2048, 1408), (17, 192, 2048, 1408), (60, 150, 2048, 1408), (4, 64, 2816, 2048), (5, 64, 2816, 2048), (1, 2000, 2048, 1408)])
def test_device_planner_takes_the_same_width(lib, count, rows, n, k):
    _device_plan_is_the_hosts(lib, WO8, [(rows, 0, 5)[i % 3] for i in range(count * 3)][:119], n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("other", [[WO8], [WO8, WO, W8, FP]])
@pytest.mark.parametrize("many,few", [(130, 1000), (20, 200), (300, 100), (130, 1100)])
def test_device_planner_takes_the_same_width_beside_problems_of_another_length(lib, other, many, few):
    """Few problems of K = 5632, and of K = 256, beside many of K = 1408: both waves of the planner hold some of each."""
    e = 90
    ks = [5632 if i % 29 == 7 else 1408 for i in range(e)]
    counts = [few if k > 1408 else (many, 0, many + 3, 40)[i % 4] for i, k in enumerate(ks)]
    _device_plan_is_the_hosts(lib, [other[i % len(other)] for i in range(e)], counts, 2048, ks)
    _device_plan_is_the_hosts(lib, [other[i % len(other)] for i in range(e)], counts, 2048, [256 if k > 1408 else k for k in ks])


@pytest.mark.gpu
@pytest.mark.parametrize("q,rows,n,k", [(W8, 192, 2816, 2048), (W4, 185, 28672, 4096), (FP, 150, 2048, 1408)])
def test_device_planner_makes_the_same_pairs(lib, q, rows, n, k):
    e = 8 if n == 28672 else 60
    counts = [(rows, rows + 1, rows - 1, 0, 7, 128)[i % 6] for i in range(e)]
    assert _pairs(_device_plan_is_the_hosts(lib, q, counts, n, k))


@pytest.mark.gpu
@pytest.mark.parametrize("q,k", [(W8, 128), (W4, 4096)])
def test_device_planner_with_as_many_tiles_as_its_sums_hold(lib, q, k):
    """64 problems of one wave, each with more tiles and columns than are told apart: the packed sum passes 2^31."""
    assert len(_pairs(_device_plan_is_the_hosts(lib, q, [1160] * 64, 28672 * 2, k))) == 64


@pytest.mark.parametrize("kernel,tiles", [("groupgemm_hz_fused_wxax", 8), ("groupgemm_hz_fused_wxax_b6", 5), ("groupgemm_hz_fused_all_b6", 5)])
def test_groups_of_row_tiles_by_the_bits_that_the_tile_reads(lib, kernel, tiles):
    """2 MB of activations to a group: 128 rows of 4096 values are 256 KB of int4 codes, 384 KB of bf6 fragments."""
    _, area = _launch(lib, [(1280, 28672, 4096, W4)] * 8, lib.mxmoe_find_kernel(kernel.encode()))
    first = area[::8][:tiles + 1]  # the first tiles of XCD 0
    assert first[:, 1].tolist() == [128 * i for i in range(tiles)] + [0] and first[:, 3].tolist() == [0] * tiles + [256]


@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_few", "groupgemm_hz_fused_all_few"])
@pytest.mark.parametrize("q", [W8, W4])
def test_kernels_for_few_rows_make_no_pairs(lib, kernel, q):
    """More rows than such a kernel is chosen for: its two shapes one after the other."""
    tab, _ = _launch(lib, [(96, 28672, 4096, q)] * 12, lib.mxmoe_find_kernel(kernel.encode()))
    assert tab[2] == 2 and not _pairs(tab)


@pytest.mark.parametrize("q,rows,shared,k", [(W8, 546, 8192, 5632), (WO, 192, 2049, 2816), (FP, 120, 1788, 5632), (W4, 4, 64, 5632)])
def test_tiles_of_a_long_problem_are_spread_over_the_xcds(lib, q, rows, shared, k):
    """A problem of two and four times the others' K: every XCD (workgroup w runs on XCD w mod 8) gets an eighth of its tiles of every shape, give or take one, and they run before the
    others of their shape; every tile is run once."""
    probs = [(rows, 2048, 1408, q)] * 60 + [(shared, 2048, k, q)]
    tab, area = _launch(lib, probs)
    long_of = [area[x::8] for x in range(8)]
    for shape in {(r1 - r0, c1 - c0) for p, r0, r1, c0, c1 in area if p == 60}:
        counts = [sum(1 for p, r0, r1, c0, c1 in a if p == 60 and (r1 - r0, c1 - c0) == shape) for a in long_of]
        assert max(counts) - min(counts) <= -(-sum(counts) // 8), (shape, counts)
        assert sum(counts) < 16 or min(counts) > 0, (shape, counts)
    live = area[area[:, 0] >= 0]
    for p, (m, n, *_r) in enumerate(probs):
        assert (live[live[:, 0] == p][:, [2, 4]] - live[live[:, 0] == p][:, [1, 3]]).prod(axis=1).sum() == m * n


@pytest.mark.gpu
@pytest.mark.parametrize("fmts", [[W8], [WO, W4], [W4, W8, FP, WO, WO8, (4, 4, 128, True), (16, 3, 128, False), (16, 2, 128, False)]])
@pytest.mark.parametrize("long_k", [2816, 256])
def test_device_planner_makes_the_same_phases(lib, fmts, long_k):
    """Problems of two lengths in one, two and eight formats: more phases than the table holds, most of the problems long or a few of them."""
    e = 96
    counts = [(150, 0, 40, 7, 300)[i % 5] for i in range(e)]
    _device_plan_is_the_hosts(lib, [fmts[i % len(fmts)] for i in range(e)], counts, 2048, [long_k if i % 9 == 4 else 1408 for i in range(e)])


@pytest.mark.parametrize("q,rows,shared,k", [(W8, 546, 8192, 5632), (WO, 192, 2049, 2816), (FP, 120, 1788, 5632), (W4, 4, 64, 5632), (W8, 300, 1300, 2816), (W8, 100, 136, 2816)])
def test_the_phase_of_a_long_problem_is_dealt_in_equal_runs(lib, q, rows, shared, k):
    """All tiles of its phases together: every XCD the same number, but for the last ones, which get what is left."""
    tab, area = _launch(lib, [(rows, 2048, 1408, q)] * 60 + [(shared, 2048, k, q)])
    live = area[area[:, 0] >= 0]
    bounds, seen = tab[13:14 + tab[2]], 0
    for lo, hi in zip(bounds, bounds[1:]):
        phase = area[lo:hi]
        if not (phase[:, 0] == 60).any():
            continue
        per_xcd = [int((phase[x::8, 0] >= 0).sum()) for x in range(8)]
        total = sum(per_xcd)
        run = -(-total // 8)
        if (phase[phase[:, 0] >= 0, 0] == 60).all():
            assert per_xcd == [min(run, max(0, total - run * x)) for x in range(8)]
            seen += total
    assert seen >= 0.8 * (live[:, 0] == 60).sum()
