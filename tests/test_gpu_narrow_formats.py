"""Narrow tiles of the formats beside plain integers: fp8 (32 x 64, fp32 sums of four waves) and w4a4 with scales per 128 values (16 x 64, groups dealt to the waves)."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O
from test_gpu_group_gemm import DEV, F16, _grouped_problem, _launch


def _branches(g, kid):
    from mxmoe_amd import _lib

    info = (C.c_int32 * 8)()
    out = []
    for b in g.plan()[1]:
        assert _lib.load().mxmoe_kernel_branch(kid, b, info) == 0
        out.append((info[1], info[2]))
    return out


# slices of 64 values: fewer than waves, than the loads in flight, one more, many; rows and channels on either side of a tile's and a fragment block's edges
@pytest.mark.gpu
@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_e4m3_few", "groupgemm_hz_fused_all_e4m3_few"])
@pytest.mark.parametrize("k", [64, 192, 320, 1088, 1408, 5632])
def test_narrow_fp8_tile(kernel, k):
    """Within the bound of the wide tile's test (2e-4 of the largest sum), and in the 2-norm no further from the float64 sums than the wide tile's, whose one chain of
    sums is four times as long, but for the spread of such errors (1.1)."""
    from mxmoe_amd import _lib, pack

    lib = _lib.load()
    kid, wide = lib.mxmoe_find_kernel(kernel.encode()), lib.mxmoe_find_kernel(b"groupgemm_hz_fused_wxax_e4m3")
    rng = np.random.default_rng(k)
    probs = []
    for m, n in [(1, 64), (31, 72), (32, 264), (33, 96), (16, 2048)]:
        ca, sa = O.quant_e4m3((rng.standard_normal((m, k)) * rng.uniform(0.1, 4, (m, 1))).astype(F16))
        cb, sb = O.quant_e4m3((rng.standard_normal((n, k)) * 0.02).astype(F16))
        probs.append(dict(A=torch.from_numpy(ca).to(DEV), B=pack.pack_wxax_fragments(torch.from_numpy(cb)).to(DEV), sa=torch.from_numpy(sa.reshape(-1)).to(DEV),
                          sb=torch.from_numpy(sb.reshape(-1)).to(DEV), ref=O.e4m3_decode(ca).astype(np.float64) @ O.e4m3_decode(cb).astype(np.float64).T, size=(m, n, k), q=(8, 8, -1, True)))
    g, outs, accs = _launch(probs, kernel_id=kid)
    assert [b for b, p in zip(_branches(g, kid), probs) if p["size"][0] <= 32] == [(32, 64)] * 4
    _, _, wides = _launch(probs, kernel_id=wide)
    err = lambda acc, p: np.linalg.norm(acc.view(np.float32) - p["ref"])  # noqa: E731
    for p, out, acc in zip(probs, outs, accs):
        assert np.abs(acc.view(np.float32) - p["ref"]).max() <= 2e-4 * np.abs(p["ref"]).max(), p["size"]
        scaled = p["ref"] * p["sa"].cpu().numpy().astype(np.float64)[:, None] * p["sb"].cpu().numpy().astype(np.float64)
        assert np.linalg.norm(out.astype(np.float64) - scaled) <= 2.0 ** -10 * np.linalg.norm(scaled), p["size"]
    norm = np.sqrt(sum(np.linalg.norm(p["ref"]) ** 2 for p in probs))
    total = [np.sqrt(sum(err(a, p) ** 2 for a, p in zip(x, probs))) for x in (accs, wides)]
    print(k, ["%.2e" % (t / norm) for t in total])
    assert total[0] <= 1.1 * total[1]


# groups: one, fewer than waves, whole rounds, one more, more than are in flight, many
@pytest.mark.gpu
@pytest.mark.parametrize("k", [128, 384, 512, 640, 1408, 2176, 4096])
def test_narrow_group_scaled_tile_bit_exact(k):
    """fp32 group sums and outputs of the oracle, bit for bit; channels that end inside a tile, a fragment block and a 16-channel block; rows that end inside a tile, and more than a tile's."""
    from mxmoe_amd import _lib

    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_all_e4m3_few")
    rng = np.random.default_rng(k)
    probs = [_grouped_problem(rng, m, n, k) for m, n in [(1, 64), (5, 72), (16, 200), (15, 8), (17, 264), (2, 2048)]]
    g, outs, accs = _launch(probs, kernel_id=kid)
    assert [b for b, p in zip(_branches(g, kid), probs) if p["size"][0] <= 16] == [(16, 64)] * 5
    for p, out, acc in zip(probs, outs, accs):
        assert np.array_equal(acc, p["acc"]), p["size"]
        assert np.array_equal(out.view(np.uint16), p["out"].view(np.uint16)), p["size"]


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 16, 33])
def test_layer_of_four_formats_on_the_narrow_tiles(tokens):
    """Their gate_up form in a layer with fp8, against the forms with host tables and with stored gate_up rows on the same kernels: identical outputs."""
    from mxmoe_amd import _lib, synth as S
    from mxmoe_amd.layer import MxMoELayer

    W8A16 = (16, 8, 128, False)
    fm = [(S.W4A4G128, S.W8A8), (S.W8A8, S.W4A4G128), (W8A16, S.W2A16), (S.W2A16, W8A16), (S.W4A4, S.W4A4G128)]
    cfg = S.MoEConfig("t", "test", 14, 2, 512, 1408, tokens, num_shared=1, rotate=1)
    layer = MxMoELayer(cfg, formats=[fm[i % 5] for i in range(15)], fp8=True)
    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_all_e4m3_few")
    layer._planned_kernel = lambda *_, **__: kid
    layer.kid_gate_up = layer.kid_down = kid
    hidden = S.make_hidden(cfg).cuda()
    ids, w = S.make_routing(cfg)
    if tokens > 1:
        ids[0, 1], ids[:tokens // 2, 0] = -1, 0
    ids, w = ids.cuda(), w.cuda()
    got = layer(hidden, ids, w).clone()
    assert layer._short[(tokens, 2)] is not None
    assert torch.equal(layer.call_with_host_tables(hidden, ids, w), got)
    layer._short[(tokens, 2)] = None
    assert torch.equal(layer(hidden, ids, w), got)


def test_lists_with_fp8_take_the_kernels_with_narrow_tiles():
    """mxmoe_few_row_kernel: the sibling with the same operand variants for few rows, without many-token tiles; the kernel itself for many, for shapes and formats that no sibling takes."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    name = lambda kid: lib.mxmoe_kernel_name(kid).decode().split("groupgemm_hz_fused_")[-1]  # noqa: E731
    f8, w4, fp, g128 = (8, 8, -1, True), (4, 4, -1, True), (16, 16, -1, True), (4, 4, 128, True)

    def picked(kernel, *probs):
        sizes = (_lib.Dim3 * len(probs))(*[_lib.Dim3(m, n, 2048) for m, n, _ in probs])
        qs = (_lib.QParams * len(probs))(*[_lib.QParams(q[0], q[1], q[2], int(q[3])) for *_, q in probs])
        kid = lib.mxmoe_few_row_kernel(-1 if kernel is None else lib.mxmoe_find_kernel(kernel), sizes, qs, len(probs))
        return None if kid < 0 else name(kid)

    e4m3, whole = b"groupgemm_hz_fused_wxax_e4m3", b"groupgemm_hz_fused_all_e4m3"
    assert picked(e4m3, (4, 2816, f8), (3, 2816, w4)) == "wxax_e4m3_few" and picked(e4m3, (65, 2816, f8)) == "wxax_e4m3"
    assert picked(b"groupgemm_hz_fused_wxax", (4, 2816, f8)) == "wxax_few"                  # int8 codes: not the fp8 kernels
    assert picked(whole, (4, 2816, f8), (3, 2816, g128)) == "all_e4m3_few" and picked(whole, (4, 2816, f8), (3, 2816, fp)) == "all_e4m3"
    wo = (16, 4, 128, False)
    assert picked(None, (4, 2816, (8, 8, -1, True)), (3, 2816, wo)) == "mixed_few" and picked(None, (4, 2816, w4), (3, 2816, g128)) == "mixed_few"
    assert picked(None, (4, 2816, w4)) == "wxax_few" and picked(None, (4, 2816, wo)) == "wo_few" and picked(None, (65, 2816, w4)) is None
    assert lib.mxmoe_few_row_kernel(-1, None, None, 0) == -1 and lib.mxmoe_few_row_kernel(-3, None, None, 0) == -2 and lib.mxmoe_few_row_kernel(10 ** 6, None, None, 0) == -2
