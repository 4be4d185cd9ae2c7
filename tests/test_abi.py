"""CPU checks of the C-ABI boundary: the library loads, exports every symbol the header declares, and its host-only
entry points (registry, launch planning, error paths) behave.  No kernel is launched here."""
import ctypes as C
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_header_symbols_are_exported_and_bound(lib):
    from mxmoe_amd import _lib

    header = (ROOT / "include" / "mxmoe_amd.h").read_text()
    declared = set(re.findall(r"\b(mxmoe_[a-z0-9_]+)\s*\(", header))
    declared -= {"mxmoe_dim3", "mxmoe_qparams"}
    assert declared, "no declarations found"
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} declared in include/mxmoe_amd.h but not exported"
        assert name in _lib.SIGNATURES, f"{name} has no ctypes signature"
    assert set(_lib.SIGNATURES) == declared


def test_struct_layouts_match_the_reference_sizes():
    from mxmoe_amd import _lib

    assert C.sizeof(_lib.QParams) == 16 and C.sizeof(_lib.Dim3) == 12      # QParams quantize.cuh:14-25, dim3


def test_registry_names_follow_the_reference_format(lib):
    n = lib.mxmoe_num_kernels()
    assert n >= 4
    names = [lib.mxmoe_kernel_name(i).decode() for i in range(n)]
    assert any(re.match(r"\[w4a4_g-1_sym: \(\d+,\d+,\d+\) \(\d,\d,1\) \d\], ", s) for s in names)
    assert lib.mxmoe_find_kernel(b"groupgemm_hz_fused_wxax") == 0
    assert lib.mxmoe_find_kernel(b"nope") == -1
    out = (C.c_int32 * 8)()
    assert lib.mxmoe_kernel_branch(0, 0, out) == 0 and out[1] % 32 == 0 and out[2] % 64 == 0
    assert lib.mxmoe_kernel_branch(0, 99, out) != 0 and b"branch" in lib.mxmoe_last_error()


def _plan(lib, kernel, probs):
    from mxmoe_amd import _lib

    sizes = (_lib.Dim3 * len(probs))(*[_lib.Dim3(*p[0]) for p in probs])
    qs = (_lib.QParams * len(probs))(*[_lib.QParams(p[1][0], p[1][1], p[1][2], int(p[1][3])) for p in probs])
    br = (C.c_int32 * len(probs))()
    tiles = C.c_int32()
    rc = lib.mxmoe_group_gemm_plan(kernel, sizes, qs, len(probs), br, C.byref(tiles))
    return rc, list(br), tiles.value


def test_plan_counts_tiles_like_the_reference_launcher(lib):
    # kernel_sketch.py:89-101: total += cdiv(M, BM) * cdiv(N, BN) per problem with the tile of its qcfg
    probs = [((546, 2816, 2048), (4, 4, -1, True)), ((0, 2816, 2048), (8, 8, -1, True)), ((20, 2048, 1408), (8, 8, -1, True))]
    rc, br, tiles = _plan(lib, -1, probs)
    assert rc == 1000                                                     # first registered kernel covers w4a4 + w8a8
    out = (C.c_int32 * 8)()
    # 546 rows of w4a4 run as two segments: 4 whole 128 x 256 tile rows, then the 34 remaining rows with one 64 x 256 tile row
    lib.mxmoe_kernel_branch(0, br[0], out)
    assert (out[1], out[2]) == (128, 256)
    exp = 4 * (2816 // 256) + 1 * (2816 // 256) + 0 + 1 * (2048 // 256)
    assert tiles == exp
    lib.mxmoe_kernel_branch(0, br[2], out)
    assert out[0] == 1 and out[1] == 32                                  # 20 rows of w8a8 -> the 32-row w8a8 tile


def test_unsupported_format_message(lib):
    rc, _, _ = _plan(lib, -1, [((8, 256, 128), (8, 4, -1, True))])
    assert rc == 1 and lib.mxmoe_last_error() == b"quant type not supported"   # compose_kernel.py:433
    rc, _, _ = _plan(lib, -1, [((8, 256, 128), (16, 4, 128, False)), ((8, 256, 128), (4, 4, -1, True)), ((8, 256, 128), (16, 16, -1, True))])
    assert rc >= 1000 and b"fused_all" in lib.mxmoe_kernel_name(rc - 1000)


def test_missing_library_fails_loudly(tmp_path):
    from mxmoe_amd import _lib

    with pytest.raises(RuntimeError, match="no CPU fallback"):
        _lib.load(tmp_path / "libmissing.so")


def test_plan_bounds_on_random_problem_lists(lib):
    """Host planner on random problem lists (every format, empty problems, lists longer than one launch's table): it never fails, and
    the tile count lies between what the largest and the smallest tile shapes of the chosen kernel would need."""
    import random

    rnd = random.Random(7)
    fmts = [((4, 4, -1, True), 128), ((8, 8, -1, True), 64), ((16, 4, 128, False), 128), ((16, 3, 128, False), 128), ((16, 2, 128, True), 128),
            ((16, 16, -1, True), 32), ((4, 4, 128, True), 128)]
    out = (C.c_int32 * 8)()
    for trial in range(40):
        nprob = rnd.choice([1, 3, 17, 60, 121, 260])
        pick = rnd.sample(fmts, rnd.choice([1, 2, 3]))
        probs = []
        for _ in range(nprob):
            q, kmul = rnd.choice(pick)
            m = rnd.choice([0, 1, 7, 31, 32, 33, 100, 129, 546, 5000, 40000])
            n = 16 * rnd.randint(1, 400)
            k = kmul * rnd.randint(1, 40)
            probs.append(((m, n, k), q))
        rc, br, tiles = _plan(lib, -1, probs)
        assert rc >= 1000, (lib.mxmoe_last_error(), probs[:3])
        kid = rc - 1000
        shapes = []
        for b in range(lib.mxmoe_kernel_num_branches(kid)):
            assert lib.mxmoe_kernel_branch(kid, b, out) == 0
            shapes.append((out[0], out[1], out[2]))
        lo = hi = 0
        fmt_id = {(4, 4, -1): 2, (8, 8, -1): 1, (16, 4, 128): 3, (16, 3, 128): 4, (16, 2, 128): 5, (16, 16, -1): 0, (4, 4, 128): 6}
        for (m, n, k), q in probs:
            mine = [(bm, bn) for f, bm, bn in shapes if f == fmt_id[(q[0], q[1], q[2])]]
            assert mine, "the chosen kernel has a tile for every format of the list"
            if m == 0:
                continue
            lo += min(-(-m // bm) * -(-n // bn) for bm, bn in mine if bm == max(x for x, _ in mine))
            hi += max(-(-m // bm) * -(-n // bn) for bm, bn in mine)
        assert lo <= tiles <= hi, (trial, lo, tiles, hi)


def test_missing_arrays_are_refused_before_any_launch(lib):
    """A quantised problem without scale arrays, or a plan without its host arrays, fails on the host with code 5."""
    from mxmoe_amd import _lib

    sizes = (_lib.Dim3 * 1)(_lib.Dim3(8, 256, 128))
    q = (_lib.QParams * 1)(_lib.QParams(4, 4, -1, 1))
    one = (C.c_void_p * 1)(0)
    addr = C.addressof(one)
    rc = lib.mxmoe_group_gemm(0, addr, addr, None, None, addr, addr, None, None, None, None, addr, sizes, None, q, 1, None, None)
    assert rc == 5 and b"scale arrays" in lib.mxmoe_last_error()
    rc = lib.mxmoe_group_gemm(0, None, addr, addr, addr, addr, addr, None, None, None, None, addr, sizes, None, q, 1, None, None)
    assert rc == 5 and b"null argument" in lib.mxmoe_last_error()
    assert lib.mxmoe_group_gemm_plan(-1, None, None, 1, None, None) == 5


def test_ds_is_accepted_and_ignored(lib):
    """The reference's caller hands the kernels a second pointer array Ds with the same entries as Cs (test.cu:446-459) and its
    kernels store through Cs only (hz_fused.cuh:89,110): a distinct Ds array is no error here either.  Host-only: the call
    below passes every check up to the launch and is refused for its (missing) scale arrays, not for its Ds."""
    from mxmoe_amd import _lib

    sizes = (_lib.Dim3 * 1)(_lib.Dim3(8, 256, 128))
    q = (_lib.QParams * 1)(_lib.QParams(4, 4, -1, 1))
    one, other = (C.c_void_p * 1)(0), (C.c_void_p * 1)(0)
    a, b = C.addressof(one), C.addressof(other)
    rc = lib.mxmoe_group_gemm(0, a, a, None, None, a, b, None, None, None, None, a, sizes, None, q, 1, None, None)
    assert rc == 5 and b"scale arrays" in lib.mxmoe_last_error()
    empty = (_lib.Dim3 * 1)(_lib.Dim3(0, 256, 128))                       # no rows: nothing to launch, every check passed
    assert lib.mxmoe_group_gemm(0, a, a, a, a, a, b, None, None, None, None, a, empty, None, q, 1, None, None) == 0


def test_every_tile_is_run_by_exactly_one_workgroup_of_an_oversized_grid(lib):
    """A planned launch is enqueued with a grid sized for the worst routing.  The function the kernels call to find their tile,
    evaluated on the host over such a grid: every tile of the launch exactly once, every surplus workgroup without a tile
    (a surplus workgroup folded back into the last phase would run one of its tiles a second time)."""
    import random

    from mxmoe_amd import _lib

    rnd = random.Random(5)
    fmts = [((4, 4, -1, True), 128), ((8, 8, -1, True), 64), ((16, 4, 128, False), 128), ((16, 16, -1, True), 32)]
    for trial in range(30):
        pick = rnd.sample(fmts, rnd.choice([1, 2, 3]))
        probs = []
        for _ in range(rnd.choice([1, 5, 60, 120])):
            q, kmul = rnd.choice(pick)
            probs.append(((rnd.choice([0, 1, 31, 33, 100, 129, 546, 3000]), 16 * rnd.randint(1, 200), kmul * rnd.randint(1, 20)), q))
        if trial == 0:
            probs = [((0, 256, 128), (4, 4, -1, True))] * 3                # a launch without any tile
        rc, _, tiles = _plan(lib, -1, probs)
        assert rc >= 1000
        sizes = (_lib.Dim3 * len(probs))(*[_lib.Dim3(*p[0]) for p in probs])
        qs = (_lib.QParams * len(probs))(*[_lib.QParams(p[1][0], p[1][1], p[1][2], int(p[1][3])) for p in probs])
        grid = tiles + 8 * 9 + rnd.choice([0, 8, 200, 1000])
        out = (C.c_int32 * grid)()
        assert lib.mxmoe_group_gemm_plan_tile_map(rc - 1000, sizes, qs, len(probs), grid, out) == 0, lib.mxmoe_last_error()
        seen = sorted(t for t in out if t >= 0)
        assert seen == list(range(tiles)), (trial, tiles, len(seen))


def test_kernels_are_exported_with_the_reference_function_type(lib):
    """One function of the reference's FuncType per kernel, by index and by name; a failing call reports through
    mxmoe_last_status (the type returns void).  Host-only: the call below fails validation before any launch."""
    from mxmoe_amd import _lib

    n = lib.mxmoe_num_kernels()
    funcs = [lib.mxmoe_kernel_func(i) for i in range(n)]
    assert all(funcs) and len(set(funcs)) == n                              # every kernel its own function
    assert lib.mxmoe_kernel_func(n) is None and lib.mxmoe_get_kernel(b"nope") is None
    assert lib.mxmoe_get_kernel(b"groupgemm_hz_fused_wxax") == funcs[0]
    assert lib.mxmoe_get_kernel(lib.mxmoe_kernel_name(2)) == funcs[2]       # the full registry key works as well
    assert {lib.mxmoe_kernel_policy(i) for i in range(n)} == {0, 1, 2} and lib.mxmoe_kernel_policy(-1) == -1
    assert lib.mxmoe_get_stream() is None
    lib.mxmoe_set_stream(0x10)
    assert lib.mxmoe_get_stream() == 0x10
    lib.mxmoe_set_stream(None)
    fn = _lib.FUNC_TYPE(funcs[1])                                           # the fp16 kernel, asked to run a w4a4 problem
    sizes = (_lib.Dim3 * 1)(_lib.Dim3(8, 256, 128))
    q = (_lib.QParams * 1)(_lib.QParams(4, 4, -1, 1))
    one = (C.c_void_p * 1)(0)
    a = C.addressof(one)
    fn(a, a, a, a, a, a, None, None, None, None, a, sizes, None, q, 1)
    assert lib.mxmoe_last_status() == 1 and lib.mxmoe_last_error() == b"quant type not supported"
    fn(a, a, a, a, a, a, None, None, None, None, a, sizes, None, q, 0)      # an empty problem list is a successful no-op
    assert lib.mxmoe_last_status() == 0


def test_prologue_entry_points_validate_on_the_host(lib):
    one = (C.c_int64 * 8)()
    a = C.addressof(one)
    assert lib.mxmoe_quant_act(None, a, a, a, a, a, 256, 4, 2, 2, 0, 0, 1, 1, None, None) == 5 and b"null" in lib.mxmoe_last_error()
    assert lib.mxmoe_quant_act(a, a, a, None, a, a, 256, 4, 2, 2, 0, 0, 1, 1, None, None) == 5
    assert lib.mxmoe_quant_act(a, a, a, a, a, a, 256, -1, 2, 2, 0, 0, 1, 1, None, None) == 3
    assert lib.mxmoe_quant_act(a, a, a, a, a, a, 260, 4, 2, 2, 0, 0, 1, 1, None, None) == 3 and b"multiple of 8" in lib.mxmoe_last_error()
    assert lib.mxmoe_silu_mul_quant(a, None, a, a, a, a, 256, 256, 4, 2, 2, 1, 0, 1, 1, None, None) == 5
    assert lib.mxmoe_quant_act_tokens(None, a, a, a, a, a, 2048, 4, 2, 2, 0, 0, None) == 5 and b"null" in lib.mxmoe_last_error()
    assert lib.mxmoe_quant_act_tokens(a, a, a, a, a, a, 1408, 4, 2, 2, 0, 0, None) == 3 and b"512" in lib.mxmoe_last_error()
    assert lib.mxmoe_quant_act_tokens(a, a, a, a, a, a, 2048, 4, 9, 2, 0, 0, None) == 3 and b"8 slots" in lib.mxmoe_last_error()
    assert lib.mxmoe_quant_act_tokens(a, a, a, a, a, a, 2048, 4, 2, 2, 0, 4, None) == 3
    assert lib.mxmoe_quant_act_tokens(a, a, a, a, a, a, 2048, 0, 2, 2, 0, 0, None) == 0      # no tokens: nothing to launch
    assert lib.mxmoe_silu_mul_quant(a, a, a, a, a, a, 1408, 1408, 4, 2, 2, 0, 1, 176, 4, None, None) == 3 and b"sign table" in lib.mxmoe_last_error()
    assert lib.mxmoe_permute_plan_layer(a, 200, 2, 8, a, a, a, a, a, a, a, 0, None) == 3 and b"256" in lib.mxmoe_last_error()   # larger batches: the two separate calls
    assert lib.mxmoe_permute_plan_layer(a, 4, 2, 8, a, a, a, a, a, None, a, 0, None) == 5
    assert lib.mxmoe_permute_plan_layer_ws(a, 100000, 8, 256, a, a, a, a, a, a, a, 0, a, None) == 3 and b"16384" in lib.mxmoe_last_error()
    assert lib.mxmoe_permute_plan_layer_ws(a, 2000, 2, 8, a, a, a, a, a, a, a, 0, None, None) == 5             # no workspace
    assert lib.mxmoe_build_permutation(None, 4, 2, 8, a, a, a, a, a, None) == 5
    assert lib.mxmoe_route_topk(a, 1, 4, 8, 9, 0, a, a, None) == 3 and b"top-k" in lib.mxmoe_last_error()      # k > experts
    assert lib.mxmoe_route_topk(a, 1, 4, 5000, 2, 0, a, a, None) == 3
    assert lib.mxmoe_route_topk(a, 3, 4, 8, 2, 0, a, a, None) == 3                                              # unknown dtype
    assert lib.mxmoe_route_topk(a, 1, 4, 8, 2, 0, None, a, None) == 5
    assert lib.mxmoe_route_topk(None, 1, 0, 8, 2, 0, None, None, None) == 0                                     # no tokens: nothing to launch
    assert lib.mxmoe_build_permutation(a, 0, 2, 8, a, a, a, a, a, None) == 3


def test_planned_grid_bound_covers_every_routing(lib):
    """The worst-case grid of a planned launch against the tile count the host launcher plans for random routings of the same
    total: the bound must never be smaller (a smaller grid would silently drop tiles), and stays within a small factor."""
    import random

    from mxmoe_amd import _lib

    rnd = random.Random(11)
    cases = [([(4, 4, -1, True), (8, 8, -1, True)], 2816, 2048, 60, 32768, 0), ([(16, 4, 128, False), (16, 3, 128, False)], 2816, 2048, 64, 192, 32),
             ([(4, 4, -1, True), (8, 8, -1, True), (16, 4, 128, False)], 28672, 4096, 8, 16384, 0), ([(16, 16, -1, True)], 2816, 2048, 60, 2048, 0),
             ([(4, 4, 128, True), (4, 4, -1, True)], 2048, 1408, 17, 999, 7)]
    for fmts, n, k, e_cnt, routed, shared_rows in cases:
        et = e_cnt + (1 if shared_rows else 0)
        qs = [rnd.choice(fmts) for _ in range(et)]
        desc = (_lib.BlockDesc * et)(*[_lib.BlockDesc(q[0], q[1], q[2], int(q[3]), (C.c_uint8 * 3)(), n, k, 0, 0) for q in qs])
        kid = lib.mxmoe_plan_select_kernel(-1, desc, et)
        assert kid >= 0, lib.mxmoe_last_error()
        bound = lib.mxmoe_plan_grid_bound(kid, desc, e_cnt, routed, shared_rows)
        assert bound > 0, lib.mxmoe_last_error()
        worst = 0
        for trial in range(60):
            style = trial % 4
            if style == 0:                                          # everything on one expert
                counts = [0] * e_cnt
                counts[rnd.randrange(e_cnt)] = routed
            elif style == 1:                                        # as even as possible
                counts = [routed // e_cnt + (1 if i < routed % e_cnt else 0) for i in range(e_cnt)]
            elif style == 2:                                        # many experts just past a tile boundary
                unit = rnd.choice([1, 17, 33, 65, 129])
                counts = [0] * e_cnt
                left = routed
                for i in range(e_cnt):
                    take = min(left, unit)
                    counts[i] = take
                    left -= take
                counts[0] += left
            else:
                cuts = sorted(rnd.randint(0, routed) for _ in range(e_cnt - 1))
                counts = [b - a for a, b in zip([0] + cuts, cuts + [routed])]
            assert sum(counts) == routed
            rows = counts + ([shared_rows] if shared_rows else [])
            rc, _, tiles = _plan(lib, kid, [((m, n, k), q) for m, q in zip(rows, qs)])
            assert rc == 1000 + kid
            worst = max(worst, tiles)
            assert tiles + 8 * 9 <= bound, (fmts, counts[:6], tiles, bound)   # + the padding of every phase to the XCD count
        assert bound <= 2.5 * worst + 600, (fmts, worst, bound)
    bad = (_lib.BlockDesc * 1)(_lib.BlockDesc(8, 4, -1, 1, (C.c_uint8 * 3)(), 256, 128, 0, 0))
    assert lib.mxmoe_plan_select_kernel(-1, bad, 1) < 0 and lib.mxmoe_last_error() == b"quant type not supported"
    assert lib.mxmoe_plan_select_kernel(-1, desc, 4097) < 0               # checked before any entry is read
    assert lib.mxmoe_plan_bytes(130) >= 2 * 4096 + 130 * (32 + 40 + 12)   # a block of more than 120 experts: one table header per launch
    assert lib.mxmoe_plan_bytes(60) >= 4096 + 60 * (32 + 40 + 12)


@pytest.mark.parametrize("a_bits,rotate,refused", [(16, 1, True), (16, 2, False), (4, 1, False)])
def test_layer_run_wants_aligned_tokens_where_tiles_read_them_in_place(lib, a_bits, rotate, refused):
    """First blocks of 16-bit activations load `hidden` straight into LDS in 16-byte pieces.  Host-only: a handle over addresses that are
    never read, and calls that are refused before any launch (the accepted forms are not called)."""
    from mxmoe_amd import _lib

    def block(a, n, k):
        return (_lib.BlockDesc * 2)(*[_lib.BlockDesc(a, 16 if a == 16 else 4, -1, 1, (C.c_uint8 * 3)(), n, k, 0, 0)] * 2)

    gate_up, down = block(a_bits, 2 * 1024, 512), block(16, 512, 1024)
    page = (C.c_uint8 * 4096)()
    some = (C.addressof(page) + 255) & ~255
    d = _lib.LayerDesc(num_tokens=4, topk=2, num_experts=2, hidden=512, inter=1024, inter_shared=1024, rotate=rotate, had_k=1, had_f=1,
                       h_gate_up=C.cast(gate_up, C.c_void_p), h_down=C.cast(down, C.c_void_p), grid_gate_up=64, grid_down=64)
    d.kernel_gate_up, d.kernel_down = lib.mxmoe_plan_select_kernel(-1, gate_up, 2), lib.mxmoe_plan_select_kernel(-1, down, 2)
    for name in ("d_gate_up", "d_down", "act", "down_inp", "down_scales", "down_out", "plan_gate_up", "plan_down", "dst_exp", "token_of_row", "row_of_slot", "iota", "recv", "workspace"):
        setattr(d, name, some)
    for tag in range(6):
        d.token_store[tag] = d.token_scales[tag] = some
    assert lib.mxmoe_layer_supported(C.byref(d)) == 1
    handle = C.c_void_p()
    assert lib.mxmoe_layer_create(C.byref(d), C.byref(handle)) == 0, lib.mxmoe_last_error()
    try:
        if refused:
            for off in (2, 4, 8, 14):
                assert lib.mxmoe_layer_run(handle, some + off, some, some, some, None) == 3 and b"16-byte" in lib.mxmoe_last_error()
        assert lib.mxmoe_layer_run(handle, None, some, some, some, None) == 5
    finally:
        lib.mxmoe_layer_destroy(handle)


def test_lists_of_few_rows_take_the_kernels_with_narrow_tiles():
    """Up to 64 rows per problem, 24 on average (in launches of few blocks) and 768 blocks of 256 channels: on and past each limit; formats those kernels have no tile for; empty problems
    count for nothing."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    w4, w8, wo, fp = (4, 4, -1, True), (8, 8, -1, True), (16, 4, 128, False), (16, 16, -1, True)

    def picked(*probs):
        sizes = (_lib.Dim3 * len(probs))(*[_lib.Dim3(m, n, 2048) for m, n, _ in probs])
        qs = (_lib.QParams * len(probs))(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for *_, q in probs])
        rc = lib.mxmoe_group_gemm_plan(-1, sizes, qs, len(probs), None, None)
        assert rc >= 1000, lib.mxmoe_last_error()
        return lib.mxmoe_kernel_name(rc - 1000).decode().split("groupgemm_")[-1]

    few = [(5, 2816, w4), (1, 2816, w8)]
    assert picked(*few) == "hz_fused_wxax_few"
    assert picked(*few, (3, 2816, wo)) == "hz_fused_all_few"
    assert picked(*few, (0, 2816, fp)) != "hz_fused_wxax_few"          # (its format still has to be covered)
    assert picked(*few, (3, 2816, fp)) == "hz_fused_all"
    assert picked((3, 2816, wo), (2, 2816, wo)) == "hz_fused_wo_few"    # (64-channel tiles up to 6 rows on average)
    assert picked((6, 2816, wo), (6, 2816, wo), (0, 2816, wo)) == "hz_fused_wo_few" and picked((6, 2816, wo), (7, 2816, wo)) == "hz_fused_wo_skinny"
    assert picked((64, 2816, w4), (1, 2816, w8), (7, 2816, w8)) == "hz_fused_wxax_few"
    assert picked((65, 2816, w4), *[(1, 2816, w8)] * 9) == "hz_fused_wxax"
    assert picked((24, 2816, w4), (24, 2816, w8)) == "hz_fused_wxax_few"
    assert picked((24, 2816, w4), (25, 2816, w8)) == "hz_fused_wxax"
    assert picked(*[(1, 256, w4)] * 7) == "hz_fused_wxax" and picked(*[(1, 256, w4)] * 8) == "hz_fused_wxax_few"
    assert picked(*[(1, 2048, w4)] * 96) == "hz_fused_wxax_few" and picked(*[(1, 2048, w4)] * 97) == "hz_fused_wxax"


W4, W8, WO4, WO3, FP = (4, 4, -1, True), (8, 8, -1, True), (16, 4, 128, False), (16, 3, 128, False), (16, 16, -1, True)


# (problems, channels, K), formats, the most rows per problem that go to the narrow tiles
@pytest.mark.parametrize("count,n,k,formats,most", [
    (16, 2048, 1408, "48", 24), (17, 2048, 1408, "48", 8), (48, 2048, 1408, "4", 8), (49, 2048, 1408, "4", 5), (60, 2048, 1408, "48", 5), (48, 2048, 1408, "48o", 16), (60, 2048, 1408, "48o", 2),
    (60, 2816, 2048, "4", 12), (60, 2816, 2048, "8", 12), (60, 2816, 2048, "48", 16), (60, 2816, 2048, "48o", 16), (8, 14336, 4096, "8", 12), (8, 4096, 14336, "4", 24)])
def test_rows_up_to_which_lists_take_the_kernels_with_narrow_tiles(lib, count, n, k, formats, most):
    qs = [{"4": W4, "8": W8, "o": WO4}[f] for f in formats]

    def picked(rows):
        rc, _, _ = _plan(lib, -1, [((m, n, k), qs[i % len(qs)]) for i, m in enumerate(rows)])
        return lib.mxmoe_kernel_name(rc - 1000).decode().endswith("_few")

    assert picked([most] * count)
    assert not picked([most] * (count - 1) + [most + 1])
    if most < 24:                                                       # one problem above 32 rows: not among the launches that a 64-row tile would hold up
        few_blocks = count * -(-n // 256) <= 256
        assert picked([33] + [1] * (count - 1)) is not few_blocks and picked([32] + [1] * (count - 1))


def _blocks(formats, n, k, shared=None):
    """Host block descriptors: experts of the given formats, and a shared expert (format, N, K)."""
    from mxmoe_amd import _lib

    rows = [(q, n, k) for q in formats] + ([shared] if shared else [])
    return (_lib.BlockDesc * len(rows))(*[_lib.BlockDesc(q[0], q[1], q[2], int(q[3]), (C.c_uint8 * 3)(), nn, kk, 0, 0) for q, nn, kk in rows])


@pytest.mark.parametrize("formats", [[W4], [W8], [W4, W8], [WO4, WO3], [W4, W8, WO4], [FP], [W4, FP]])
@pytest.mark.parametrize("experts,topk,n,k,shared_n,shared_k", [(60, 4, 2816, 2048, 0, 0), (60, 4, 2048, 1408, 2048, 5632), (64, 6, 2816, 2048, 5632, 2048),
                                                                (8, 2, 4096, 14336, 0, 0), (8, 2, 28672, 4096, 0, 0), (4, 1, 256, 512, 0, 0)])
def test_planned_batches_take_the_kernel_that_the_launcher_takes_for_an_even_routing(lib, formats, experts, topk, n, k, shared_n, shared_k):
    """One rule for few rows, whoever asks: mxmoe_plan_select_kernel_rows against the automatic choice for a list with as even a routing as the batch has, up to
    the largest batch that any of those kernels is meant for, and the kernel by formats alone beyond."""
    qs = [formats[e % len(formats)] for e in range(experts)]
    shared = (formats[0], shared_n, shared_k) if shared_n else None
    desc = _blocks(qs, n, k, shared)
    for t in (1, 2, 3, 5, 8, 13, 16, 24, 32, 33, 48, 64, 65, 200):
        kid = lib.mxmoe_plan_select_kernel_rows(desc, experts, t, topk, t if shared else 0)
        live = min(experts, t * topk)
        counts = [t * topk // live + (e < t * topk % live) for e in range(live)] + [0] * (experts - live)
        assert kid >= 0, lib.mxmoe_last_error()
        if t > 64 or t * topk > 12 * experts and formats[0][0] == 16:
            assert kid == lib.mxmoe_plan_select_kernel(-1, desc, experts + (1 if shared else 0)), t
            continue
        rc, _, _ = _plan(lib, -1, [((c, n, k), q) for c, q in zip(counts, qs)] + ([((t, shared_n, shared_k), shared[0])] if shared else []))
        assert rc - 1000 == kid, (t, lib.mxmoe_kernel_name(rc - 1000), lib.mxmoe_kernel_name(kid))


def test_planned_batches_refuse_what_is_no_batch(lib):
    desc = _blocks([W4, W4], 256, 512)
    for args in ((0, 1, 1, 0), (2, 0, 1, 0), (2, 1, 0, 0), (2, 1, 1, -1)):
        assert lib.mxmoe_plan_select_kernel_rows(desc, *args) < 0
    assert lib.mxmoe_plan_select_kernel_rows(None, 2, 1, 1, 0) < 0
    assert lib.mxmoe_plan_select_kernel_rows(_blocks([(4, 2, -1, True)] * 2, 256, 512), 2, 1, 1, 0) < 0


@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_few", "groupgemm_hz_fused_all_few"])
def test_few_blocks_take_narrow_tiles_beyond_32_rows(lib, kernel):
    """Launches of up to 128 blocks of 256 channels with narrow tiles: problems of 33 .. 128 rows take them too (a 64-row tile would be what the launch waits
    for); one block more, or a weight-only problem, and they do not.  Problems without rows are no blocks of the launch."""
    kid = lib.mxmoe_find_kernel(kernel.encode())

    def tile(rows, probs):
        rc, br, _ = _plan(lib, kid, probs)
        assert rc == 1000 + kid
        info = (C.c_int32 * 8)()
        at = next(i for i, p in enumerate(probs) if p[0][0] == rows)
        assert lib.mxmoe_kernel_branch(kid, br[at], info) == 0
        return info[1], info[2]                                          # rows, channels of the tile

    def few(rows, q, blocks, empty=0):
        return [((rows, 4096, 14336), q)] + [((5, 4096, 14336), W4 if i % 2 else W8) for i in range(blocks // 16 - 1)] + [((7, 256, 14336), W4)] * (blocks % 16) \
            + [((0, 4096, 14336), W8)] * empty

    for q in (W4, W8):
        for rows in (33, 45, 64, 65, 100, 128):
            assert tile(rows, few(rows, q, 128, empty=4)) == (32, 64), (q, rows)
        assert tile(45, few(45, q, 129))[1] == 256 and tile(64, few(64, q, 129))[1] == 256 and tile(129, few(129, q, 64))[1] == 256
        assert tile(32, few(32, q, 128)) == (32, 64) and tile(32, few(32, q, 160)) == (32, 64)
    wide = lib.mxmoe_find_kernel(kernel.replace("_few", "").encode())
    rc, br, _ = _plan(lib, wide, few(45, W4, 64))                         # kernels without narrow tiles: as before
    assert rc == 1000 + wide
    if "all" in kernel:
        assert tile(45, few(45, WO4, 64)) == (128, 256)


def test_planned_grid_bound_with_narrow_tiles(lib):
    """The worst-case grid of planned launches on the kernels with narrow tiles against the tiles of the same launches planned on the host; few blocks count
    over all experts there (they are not known to be empty), so a list of all of them decides alike."""
    import random

    rnd = random.Random(5)
    for kernel, n, k, e, shared_rows, fmts in (("groupgemm_hz_fused_wxax_few", 4096, 14336, 8, 0, [W4, W8]), ("groupgemm_hz_fused_all_few", 4096, 14336, 8, 0, [W4, W8, WO4]),
                                               ("groupgemm_hz_fused_wxax_few", 512, 1024, 40, 64, [W4, W8]), ("groupgemm_hz_fused_wxax_few", 2048, 1408, 60, 48, [W4])):
        kid = lib.mxmoe_find_kernel(kernel.encode())
        qs = [rnd.choice(fmts) for _ in range(e)]
        desc = _blocks(qs, n, k, (fmts[0], n, 2 * k) if shared_rows else None)
        for routed in (1, 7, 64, 128, 200, 512):
            bound = lib.mxmoe_plan_grid_bound(kid, desc, e, routed, shared_rows)
            assert bound > 0, lib.mxmoe_last_error()
            for trial in range(60):
                counts = [0] * e
                if trial % 3 == 0:
                    unit = rnd.choice([1, 17, 32, 33, 40, 64, 65])
                    left = routed
                    for i in range(e):
                        counts[i] = min(unit, left)
                        left -= counts[i]
                    counts[rnd.randrange(e)] += left
                else:
                    for _ in range(routed):
                        counts[min(int(rnd.paretovariate(0.7 if trial % 3 == 1 else 3.0)) - 1, e - 1)] += 1
                rc, _, tiles = _plan(lib, kid, [((m, n, k), q) for m, q in zip(counts, qs)] + ([((shared_rows, n, 2 * k), fmts[0])] if shared_rows else []))
                assert rc == 1000 + kid and tiles + 8 * 9 <= bound, (kernel, n, routed, counts, tiles, bound)
