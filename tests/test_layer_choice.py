"""Which kernels and which form a layer takes for a number of tokens (host only: layers of empty weights, handles that are never run)."""
import ctypes as C

import pytest
import torch

from mxmoe_amd import _lib, synth as S
from mxmoe_amd.layer import MxMoELayer
from mxmoe_amd.weights import PackedWeight

W8A16 = (16, 8, 128, False)


def _layer(formats, experts=60, topk=4, hidden=2048, inter=1408, num_shared=0, rotate=0, fp8=False, tokens=1):
    """`formats`: (gate_up, down) in turn over the experts, the shared one last."""
    n = experts + (num_shared > 0)
    cfg = S.MoEConfig("t", "test", experts, topk, hidden, inter, tokens, num_shared=num_shared, rotate=rotate)
    fm = [formats[i % len(formats)] for i in range(n)]
    width = [inter] * experts + [inter * num_shared] * (n - experts)

    def empty(q, rows, k):
        return PackedWeight(torch.empty(16, dtype=torch.uint8), torch.empty(16, dtype=torch.uint8), tuple(q), rows, k)

    return MxMoELayer(cfg, device="cpu", packed=([empty(f[0], 2 * w, hidden) for f, w in zip(fm, width)], [empty(f[1], hidden, w) for f, w in zip(fm, width)]), fp8=fp8)


def _name(kid):
    return _lib.load().mxmoe_kernel_name(kid).decode().split("groupgemm_hz_fused_")[-1]


def _starts(d):
    return bool(_lib.load().mxmoe_layer_starts_with_gate_up(C.byref(d)))


MIXES = {"w4a4": [(S.W4A4, S.W4A4)], "w4a4/w8a8": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4)], "w4a16/w3a16": [(S.W4A16, S.W3A16), (S.W3A16, S.W4A16)],
         "w8a16/w2a16": [(W8A16, S.W2A16), (S.W2A16, W8A16)], "fp16": [(S.FP16, S.FP16)], "w4a4/w8a8/w4a16": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A16), (S.W4A16, S.W4A4)]}


@pytest.mark.parametrize("mix", list(MIXES))
@pytest.mark.parametrize("experts", [8, 60, 128, 430, 512])
def test_kernel_and_form_are_chosen_together(mix, experts):
    """The first block's kernel is one that pays only without a head in front of it nowhere else than in a layer that has none: the handle and the choice of the kernel ask one rule."""
    lib = _lib.load()
    for topk in (2, 4, 6, 8):
        layer = _layer(MIXES[mix], experts=experts, topk=topk, hidden=512, inter=128)
        for tokens in (1, 16, 64, 65, 85, 100, 128, 129):
            d, gate_up, _ = layer._layer_desc(tokens, topk)
            assert not lib.mxmoe_layer_has_head(layer._short_setup(tokens, topk)._handle) == _starts(d)
            if not _starts(d):
                assert d.kernel_gate_up == lib.mxmoe_layer_kernel(gate_up, experts, tokens, topk, 0, 0), (tokens, topk)


def test_where_a_layer_starts_with_gate_up():
    """Either side of each limit: tokens, pairs, top-k, counters of many experts in LDS, hidden sizes, 16-bit tokens that are rotated."""
    def starts(tokens, topk=4, mix="w4a4", **kw):
        return _starts(_layer(MIXES[mix], topk=topk, **kw)._layer_desc(tokens, topk)[0])

    assert starts(1) and starts(128) and not starts(129)
    assert starts(85, 6) and not starts(86, 6) and starts(64, 8, experts=64) and not starts(65, 8, experts=64)
    assert starts(2, 64, experts=128, inter=256) and not starts(2, 65, experts=128, inter=256)
    assert starts(1, 4, mix="fp16") and starts(64, 4, mix="fp16") and not starts(65, 4, mix="fp16")
    assert starts(4, experts=200, inter=128, hidden=512) and not starts(4, experts=512, inter=128, hidden=512)
    assert starts(1, mix="fp16", hidden=512, inter=160) and not starts(1, hidden=1536)
    assert starts(1, mix="w4a16/w3a16", rotate=1) and not starts(1, mix="w4a16/w3a16", rotate=2) and starts(1, rotate=2)
    many = _layer(MIXES["w4a4"], experts=500, hidden=512, inter=256)  # (1000 blocks of channels: narrow tiles without a head only)
    d, gate_up, _ = many._layer_desc(128, 4)
    assert _name(_lib.load().mxmoe_layer_kernel(gate_up, 500, 128, 4, 0, 1)) == "wxax_few"
    assert not _starts(d) and _name(d.kernel_gate_up) == "wxax"


def test_a_layer_starts_with_gate_up_only_on_tiles_that_the_kernel_has():
    """A kernel named by the caller: one launch for each kernel of 64-channel tiles; none where the kernel's tables may name a tile with other sums, or a format has no such tile in it."""
    lib = _lib.load()

    def starts(kernel, formats, fp8=False):
        d, *keep = _layer([(f, S.FP16) for f in formats], fp8=fp8)._layer_desc(4, 4)
        d.kernel_gate_up = lib.mxmoe_find_kernel(b"groupgemm_hz_fused_" + kernel.encode())
        assert d.kernel_gate_up >= 0 and lib.mxmoe_layer_supported(C.byref(d))
        return _starts(d)

    assert starts("wxax_few", [S.W4A4, S.W8A8]) and starts("wxax_e4m3_few", [S.W4A4, S.W8A8], fp8=True)
    assert starts("wo_few", [S.W4A16, S.W3A16, S.W2A16]) and starts("a16_few", [S.FP16, W8A16, S.W2A16]) and starts("mixed_few", [S.W4A4, S.W4A4G128, W8A16, S.W3A16])
    assert starts("all_e4m3_few", [S.W4A4, S.W8A8, S.W4A4G128, W8A16], fp8=True)
    assert not starts("all_few", [S.W4A4, S.W4A16]) and not starts("all_few", [S.W8A8, W8A16])
    assert not starts("all", [S.W4A4]) and not starts("wxax", [S.W4A4]) and not starts("wo", [S.W4A16]) and not starts("fp16", [S.FP16])


# the layers that test_gpu_few_tokens.test_first_launch_without_a_head compares with the form that has a head, and the kernels that it names for them
def _compared():
    import test_gpu_few_tokens as T

    return next(m for m in T.test_first_launch_without_a_head.pytestmark if m.name == "parametrize").args[1]


@pytest.mark.parametrize("case", _compared(), ids=str)
def test_layers_compared_with_a_head_have_none(case):
    tokens, topk, experts, inter, num_shared, mix = case
    first = {"fp16": [S.FP16], "wo": [S.W4A16, S.W3A16, S.W2A16], "all": [W8A16, S.W4A16, S.FP16], "first": [W8A16, S.W4A16, S.W2A16], "behind": [S.W4A16, S.W3A16],
             "int": [S.W4A4, S.W8A8], "many": [S.W4A4, S.W4A4G128, W8A16, S.W8A8, S.W3A16]}
    kernel = {"wo": "wo_few", "behind": "wo_few", "int": "wxax_few", "many": "mixed_few", "fp8": "wxax_e4m3_few", "many fp8": "all_e4m3_few"}
    fp8 = "fp8" in mix
    form = "first" if inter % 128 and mix != "fp16" else {"fp8": "int", "many fp8": "many"}.get(mix, mix)
    kernel = "a16_few" if form == "first" else kernel.get(mix, "a16_few")
    layer = _layer([(f, S.FP16 if form == "first" else f) for f in first[form]], experts=experts, topk=topk, hidden=512, inter=inter, num_shared=num_shared, rotate=0, fp8=fp8)
    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_" + kernel.encode())
    planned = layer._planned_kernel
    layer._planned_kernel = lambda h, t, k, **_: kid if int(h[0].N) == 2 * inter else planned(h, t, k)
    assert not _lib.load().mxmoe_layer_has_head(layer._short_setup(tokens, topk)._handle)
