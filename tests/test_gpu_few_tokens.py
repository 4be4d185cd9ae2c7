"""The few-token tiles of fp16 and of 8-bit weights (16 x 64, groupgemm_hz_fused_a16_few): where their ranges end, and what is sent to them."""
import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O

FP16, W8A16 = (16, 16, -1, True), (16, 8, 128, False)


def _problem(rng, m, n, k, q):
    """Operands on the host and the product in float64 (8-bit weights: of the dequantised weights, not rounded)."""
    from mxmoe_amd.weights import quantize_and_pack

    x = rng.standard_normal((m, k)).astype(np.float16)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float16)
    if q == FP16:
        return x, torch.from_numpy(w), None, x.astype(np.float64) @ w.astype(np.float64).T
    pw = quantize_and_pack(torch.from_numpy(w), q)
    c, s, z = O.quant_minmax(w, 8, 128, False)
    deq = c.reshape(n, k // 128, 128).astype(np.float64) * s.reshape(n, -1, 1).astype(np.float64) + z.reshape(n, -1, 1).astype(np.float64)
    return x, pw.data, pw.scale, x.astype(np.float64) @ deq.reshape(n, k).T


@pytest.mark.gpu
@pytest.mark.parametrize("k", [128, 384, 512, 640, 2176])
def test_few_token_tiles_of_16_and_8_bit_weights(k):
    """K dealt to four waves: parts of no block, one, several, and unequal ones; 1 row, a whole row tile, one row more, several tiles; channels that end inside a tile's 64.
    The output's rounding is at most 2^-11 of it; the fp32 sums add, for 8 bits, those of terms that still carry the codes' bias (as in
    test_weight_only_streams_of_every_length): as much again."""
    from mxmoe_amd import _lib
    from mxmoe_amd.group_gemm import GroupGemmLaunch

    rng = np.random.default_rng(k)
    sizes = [(1, 64), (16, 144), (17, 16), (33, 80), (5, 256)]
    probs = [(*_problem(rng, m, n, k, q), (m, n, k), q) for m, n in sizes for q in (FP16, W8A16)]
    Cs = [torch.full(p[4][:2], float("nan"), dtype=torch.float16, device="cuda") for p in probs]
    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_a16_few")
    GroupGemmLaunch([torch.from_numpy(p[0]).cuda() for p in probs], [p[1].cuda() for p in probs], [None] * len(probs), [None if p[2] is None else p[2].cuda() for p in probs], Cs,
                    [p[4] for p in probs], [p[5] for p in probs], kernel_id=kid).run()
    for p, c in zip(probs, Cs):
        err = np.linalg.norm(c.cpu().numpy().astype(np.float64) - p[3]) / np.linalg.norm(p[3])
        assert err <= (2.0 ** -11 if p[5] == FP16 else 2.0 ** -10), (p[4], p[5], err)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 5, 33])
@pytest.mark.parametrize("q", [FP16, W8A16])
def test_layer_on_the_few_token_tiles(tokens, q):
    """Their gate_up form (rows gathered by token, several row tiles of one expert at 33 tokens, dropped ids) and the block behind it, against the layer in float64 on the same
    weights: three roundings to fp16 (silu * up of rounded gate and up, down, combine), each at most 2^-11 of its result, add up to less than 2^-9 of the norm."""
    from mxmoe_amd import _lib, synth
    from mxmoe_amd.layer import MxMoELayer

    cfg = synth.MoEConfig("t", "test", 6, 2, 512, 640, tokens, num_shared=1, rotate=0)
    layer = MxMoELayer(cfg, formats=[(q, q)] * 7)
    layer._planned_kernel = lambda *_, **__: _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_a16_few")
    hidden = synth.make_hidden(cfg)
    ids, w = synth.make_routing(cfg)
    ids[:, 0] = 1
    ids[-1, 1] = -1 if tokens > 1 else ids[-1, 1]
    got = layer(hidden.cuda(), ids.cuda(), w.cuda()).cpu().numpy().astype(np.float64)

    def dense(e):
        out = []
        for m in synth.expert_weights(cfg, e):
            m = m.numpy()
            if q == W8A16:
                c, s, z = O.quant_minmax(m, 8, 128, False)
                g = m.shape[1] // 128
                m = c.reshape(m.shape[0], g, 128).astype(np.float64) * s.reshape(-1, g, 1).astype(np.float64) + z.reshape(-1, g, 1).astype(np.float64)
            out.append(m.reshape(-1, m.shape[-1] if m.ndim == 2 else g * 128).astype(np.float64))
        return out

    def mlp(x, e):
        w13, w2 = dense(e)
        y = x @ w13.T
        gate, up = y[..., :y.shape[-1] // 2], y[..., y.shape[-1] // 2:]
        return (gate / (1 + np.exp(-gate)) * up) @ w2.T

    x = hidden.numpy().astype(np.float64)
    want = mlp(x, 6)
    for t in range(tokens):
        for k in range(2):
            if 0 <= int(ids[t, k]) < 6:
                want[t] += float(w[t, k]) * mlp(x[t], int(ids[t, k]))
    assert np.linalg.norm(got - want) <= 2.0 ** -9 * np.linalg.norm(want)


def test_lists_that_the_few_token_tiles_take():
    """fp16 problems up to 12 rows on average, with 8-bit weights among them up to 6; a K or N that the tiles' blocks do not divide, more than 64 rows and few blocks of channels go where they went."""
    from mxmoe_amd import _lib

    lib = _lib.load()
    fp, w8, w4 = FP16, W8A16, (16, 4, 128, False)

    def picked(*probs):
        sizes = (_lib.Dim3 * len(probs))(*[_lib.Dim3(*p[:3]) for p in probs])
        qs = (_lib.QParams * len(probs))(*[_lib.QParams(p[3][0], p[3][1], p[3][2], int(p[3][3])) for p in probs])
        rc = lib.mxmoe_group_gemm_plan(-1, sizes, qs, len(probs), None, None)
        assert rc >= 1000, lib.mxmoe_last_error()
        return lib.mxmoe_kernel_name(rc - 1000).decode().split("groupgemm_hz_fused_")[-1]

    assert picked((12, 2816, 2048, fp)) == "a16_few" and picked((13, 2816, 2048, fp)) == "fp16"
    assert picked((1, 2816, 2048, fp), (23, 2816, 2048, fp)) == "fp16"          # (more than a quarter of the problems exceed a row tile)
    assert picked((6, 2816, 2048, fp), (6, 2816, 2048, w8)) == "a16_few" and picked((6, 2816, 2048, fp), (7, 2816, 2048, w8)) == "all"
    assert picked((6, 2816, 2048, w8)) == "a16_few" and picked((7, 2816, 2048, w8)) == "all"
    assert picked((6, 2816, 2048, w8), (6, 2816, 2048, w4)) == "a16_few" and picked((6, 2816, 2048, w4)) == "wo_few"
    assert picked((4, 2816, 2080, fp)) == "fp16" and picked((4, 2824, 2048, fp)) == "fp16"
    assert picked((4, 2816, 2080, fp), (4, 2816, 2048, w8)) == "all" and picked((0, 2816, 2080, fp), (4, 2816, 2048, fp)) == "a16_few"
    assert picked((1, 1792, 2048, fp)) == "fp16" and picked((1, 2048, 2048, fp)) == "a16_few"
    assert picked(*[(4, 2816, 2048, fp)] * 20, (65, 2816, 2048, fp)) == "fp16"


# tokens, top-k, experts, inter, shared experts, formats: one token; a partial row tile; 256 and 512 entries, the most of one and two a thread, and a few more than 256; more experts than a wave has lanes and than one launch's tables hold;
# two and four row tiles of the shared expert and of one expert; shared columns that end inside the grid's rows; quantised and rotated second blocks
@pytest.mark.gpu
@pytest.mark.parametrize("tokens,topk,experts,inter,num_shared,mix", [
    (1, 1, 8, 1408, 0, "fp16"), (1, 6, 64, 1408, 2, "wo"), (17, 3, 70, 96, 3, "fp16"), (33, 6, 130, 160, 1, "all"), (64, 4, 60, 256, 4, "wo"), (64, 4, 60, 352, 0, "all"),
    (32, 8, 24, 1408, 1, "behind"), (5, 2, 66, 640, 2, "behind"), (16, 16, 8, 512, 1, "fp16"),
    (1, 4, 60, 1408, 4, "int"), (64, 4, 60, 1408, 1, "int"), (33, 2, 9, 640, 2, "many"), (64, 4, 130, 1408, 1, "many"), (1, 1, 10, 512, 0, "many"),
    (43, 6, 70, 96, 3, "fp16"), (64, 8, 64, 1408, 2, "wo"), (64, 6, 24, 1408, 1, "int"), (57, 7, 130, 640, 1, "many"), (128, 4, 60, 512, 1, "all"), (128, 4, 12, 1408, 1, "int"),
    (40, 6, 64, 1408, 1, "fp8"), (64, 2, 12, 512, 0, "many fp8"), (17, 6, 64, 1408, 2, "many fp8"),
])
def test_first_launch_without_a_head(tokens, topk, experts, inter, num_shared, mix):
    """gate_up that finds its problems from the ids, against the form with tables from launches in front on the same kernels: identical outputs.  Ids out of range,
    one expert with most of the tokens, an expert twice in a token's list; a second call on other ids (nothing of the first is left); a misaligned view of the tokens."""
    from mxmoe_amd import _lib, synth as S
    from mxmoe_amd.layer import MxMoELayer

    if inter % 128 and mix != "fp16":  # (their second block's K is in groups of 128)
        mix = "first"
    fm = {"fp16": [(FP16, FP16)], "wo": [(S.W4A16, S.W3A16), (S.W3A16, S.W2A16), (S.W2A16, S.W4A16)], "all": [(W8A16, FP16), (S.W4A16, W8A16), (FP16, S.W2A16)],
          "first": [(W8A16, FP16), (S.W4A16, FP16), (S.W2A16, FP16)], "behind": [(S.W4A16, S.W4A4), (S.W3A16, S.W8A8), (S.W4A16, S.W4A16)],
          "int": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W4A4, S.W4A4)], "many": [(S.W4A4, S.W8A8), (S.W4A4G128, S.W4A4), (W8A16, S.W4A4G128), (S.W8A8, S.W3A16), (S.W3A16, S.W4A4)]}
    fm["fp8"], fm["many fp8"] = fm["int"], fm["many"]
    fm = fm[mix]
    n = experts + (num_shared > 0)
    cfg = S.MoEConfig("t", "test", experts, topk, 512, inter, tokens, num_shared=num_shared, rotate=int(mix not in ("fp16", "wo", "all", "first")))
    layer = MxMoELayer(cfg, formats=[fm[i % len(fm)] for i in range(n)], fp8="fp8" in mix)
    kid = _lib.load().mxmoe_find_kernel(b"groupgemm_hz_fused_" + {"wo": b"wo_few", "behind": b"wo_few", "int": b"wxax_few", "many": b"mixed_few", "fp8": b"wxax_e4m3_few",
                                                                  "many fp8": b"all_e4m3_few"}.get(mix, b"a16_few"))
    planned = layer._planned_kernel
    layer._planned_kernel = lambda h, t, k, **_: kid if int(h[0].N) == 2 * inter else planned(h, t, k)
    gen = torch.Generator().manual_seed(tokens)
    store = torch.randn(tokens * 512 + 8, generator=gen).half().cuda()
    calls = []
    for call in range(3):
        ids = torch.stack([torch.randperm(experts, generator=gen)[torch.arange(topk) % experts] for _ in range(tokens)]).to(torch.int32)
        if tokens > 1:
            ids[:, 0] = call
            ids[0, -1], ids[tokens // 2, 0] = -1, experts + 3
            ids[-1, -1] = ids[-1, 0]
        w = torch.rand(tokens, topk, generator=gen)
        off = 1 if call == 2 else 0
        calls.append((store[off:off + tokens * 512].view(tokens, 512), ids.cuda(), w.cuda()))
    got = [layer(*c).clone() for c in calls]
    assert layer._short[(tokens, topk)] is not None
    layer._short[(tokens, topk)] = None                                  # the form with launches in front
    for c, g in zip(calls, got):
        assert torch.equal(layer(*c), g)


def test_first_block_of_a_layer_takes_the_narrow_tiles_up_to_more_experts():
    """896 blocks of 256 channels: up to 64 tokens, 512 pairs and 12 rows a problem where gate_up starts the layer, not at all elsewhere or in fp8; up to 768 blocks the same choice."""
    import ctypes as C

    from mxmoe_amd import _lib

    lib = _lib.load()

    def picked(tokens, n, variant=0, first=True, w=4):
        desc = (_lib.BlockDesc * 8)(*[_lib.BlockDesc(w, w, -1, 1, (C.c_uint8 * 3)(variant, 0, 0), n, 4096, 0, 0) for _ in range(8)])
        kid = lib.mxmoe_layer_kernel(desc, 8, tokens, 2, 0, int(first))
        return lib.mxmoe_kernel_name(kid).decode().split("groupgemm_hz_fused_")[-1]

    assert [picked(t, 28672) for t in (4, 48, 49, 64)] == ["wxax_few", "wxax_few", "wxax", "wxax"]
    assert picked(4, 28672, first=False) == "wxax" and picked(4, 32768 + 256) == "wxax" and picked(4, 28672, 2, w=8) == "wxax_e4m3"
    assert all(picked(t, 24576) == picked(t, 24576, first=False) for t in (1, 16, 64, 65))


def test_first_block_of_a_layer_takes_the_few_row_kernels_up_to_128_tokens():
    """Where gate_up starts the layer: 128 tokens, 512 pairs, 10 weight-only rows an expert (8 of a K above 2048), 64 tokens with fp16 weights among them; elsewhere 64 tokens and 6 rows."""
    import ctypes as C

    from mxmoe_amd import _lib

    lib = _lib.load()

    def picked(tokens, topk, formats, experts=60, shared=0, k=2048, first=True):
        n = experts + (shared > 0)
        desc = (_lib.BlockDesc * n)(*[_lib.BlockDesc(*formats[i % len(formats)], (C.c_uint8 * 3)(0, 0, 0), 2816, k, 0, 0) for i in range(n)])
        kid = lib.mxmoe_layer_kernel(desc, experts, tokens, topk, shared, int(first))
        assert kid >= 0, lib.mxmoe_last_error()
        return lib.mxmoe_kernel_name(kid).decode().split("groupgemm_hz_fused_")[-1]

    w4a4, w8a8, w4, w8, fp = (4, 4, -1, 1), (8, 8, -1, 1), (16, 4, 128, 0), (16, 8, 128, 0), (16, 16, -1, 1)
    assert [picked(t, 4, [w4a4]) for t in (64, 65, 128, 129)] == ["wxax_few", "wxax_few", "wxax_few", "wxax"]
    assert picked(85, 6, [w4a4]) == "wxax_few" and picked(86, 6, [w4a4]) == "wxax" and picked(65, 4, [w4a4], first=False) == "wxax"
    assert picked(128, 4, [w4a4, w8a8, w4]) == "mixed_few" and picked(64, 8, [w4]) == "wo_few" and picked(128, 4, [w8, w4]) == "a16_few"
    assert picked(80, 6, [w4], shared=80) == "wo_few" and picked(85, 6, [w4], experts=50) == "wo"
    assert picked(48, 4, [w4], experts=24, k=4096) == "wo_few" and picked(49, 4, [w4], experts=24, k=4096) != "wo_few"
    assert picked(64, 4, [fp]) == "a16_few" and picked(65, 4, [fp]) == "fp16" and picked(65, 4, [w4, fp]) != "a16_few"
    assert picked(65, 4, [w4], first=False) == "wo"


@pytest.mark.parametrize("kernel", ["groupgemm_hz_fused_wxax_e4m3_few", "groupgemm_hz_fused_all_e4m3_few"])
def test_fp8_problems_of_few_rows_have_one_tile(kernel):
    """Whatever the rows and the number of problems: the launch that starts a layer has that tile alone, and sums in another one are not the same to the bit."""
    import ctypes as C

    from mxmoe_amd import _lib

    lib = _lib.load()
    kid = lib.mxmoe_find_kernel(kernel.encode())
    for count, n, k in ((1, 4096, 14336), (8, 2816, 2048), (60, 2816, 2048), (60, 2048, 1408)):
        for m in (1, 31, 32, 33, 40, 64, 65, 128, 200):
            sizes = (_lib.Dim3 * count)(*[_lib.Dim3(m if i == 0 else 3, n, k) for i in range(count)])
            qs = (_lib.QParams * count)(*[_lib.QParams(8, 8, -1, 1)] * count)
            branch, tiles = (C.c_int32 * count)(), C.c_int32(0)
            assert lib.mxmoe_group_gemm_plan(kid, sizes, qs, count, branch, C.byref(tiles)) == 1000 + kid
            assert len(set(branch)) == 1, (count, m, list(branch)[:2])
            assert tiles.value == -(-n // 64) * (count - 1 + -(-m // 32))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [33, 40, 64])
@pytest.mark.parametrize("mix", ["fp8", "w4a4 and fp8"])
def test_fp8_layer_with_and_without_a_head(tokens, mix):
    """More than 32 rows of one expert and of the shared one, K = 2048, more than 256 blocks of channels, second blocks in fp16 (nothing is requantised behind the sums), tokens of values
    of many sizes (the sums of normal ones hardly ever hang on their order): identical outputs of the layer that starts with gate_up and of the one with launches in front, on the kernel that the layer takes by itself."""
    from mxmoe_amd import _lib, synth as S
    from mxmoe_amd.layer import MxMoELayer

    fm = [(S.W8A8, S.FP16)] if mix == "fp8" else [(S.W8A8, S.FP16), (S.W4A4, S.FP16)]
    cfg = S.MoEConfig("t", "test", 30, 2, 2048, 1408, tokens, num_shared=1, rotate=0)
    layer = MxMoELayer(cfg, formats=[fm[i % len(fm)] for i in range(31)], fp8=True)
    gen = torch.Generator().manual_seed(tokens)
    hidden = (torch.randn(tokens, 2048, generator=gen) * torch.exp(2 * torch.randn(tokens, 2048, generator=gen)) / 64).half().cuda()
    ids, w = S.make_routing(cfg)
    ids[:, 0] = 2
    ids, w = ids.cuda(), w.cuda()
    got = layer(hidden, ids, w).clone()
    assert torch.isfinite(got).all()
    kid = layer._planned_kernel(layer._block_descs(layer.qp_gate_up, [2816] * 31, [2048] * 31, layer.w13, False), tokens, 2, first=True)
    assert _lib.load().mxmoe_kernel_name(kid).endswith(b"groupgemm_hz_fused_wxax_e4m3_few")
    assert layer._short[(tokens, 2)] is not None
    layer._short[(tokens, 2)] = None
    assert torch.equal(layer(hidden, ids, w), got)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1408, 4096, 14336])
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
def test_weight_only_sums_are_as_close_as_those_of_the_many_token_tiles(bits, k):
    """The few-token tiles sum biased codes and take the bias out of the sum, the tiles of many tokens round every weight to fp16: in the 2-norm against float64 the former are no further off than the latter (but
    for the spread of such errors, 1.1), for tokens around zero and for tokens with a mean, whose biased sums are large."""
    from mxmoe_amd import _lib
    from mxmoe_amd.group_gemm import GroupGemmLaunch
    from mxmoe_amd.weights import quantize_and_pack

    lib, gen, n, q = _lib.load(), torch.Generator(device="cuda").manual_seed(k + bits), 512, (16, bits, 128, False)
    from mxmoe_amd.quant import quant_minmax

    w = (torch.randn(n, k, generator=gen, device="cuda") * 0.02).half()
    pw, (c, s, z) = quantize_and_pack(w, q), quant_minmax(w, bits, 128, False)
    deq = (c.reshape(n, -1, 128).double() * s.reshape(n, -1, 1).double() + z.reshape(n, -1, 1).double()).reshape(n, k)
    for mean, dev in ((0.0, 1.0), (0.7, 0.5)):
        x = (torch.randn(128, k, generator=gen, device="cuda") * dev + mean).half()
        ref = x.double() @ deq.T.contiguous()
        err = {}
        for kernel in ("a16_few", "all"):
            out, acc = torch.zeros(128, n, dtype=torch.float16, device="cuda"), torch.zeros(128, n, dtype=torch.int32, device="cuda")
            GroupGemmLaunch([x], [pw.data], [None], [pw.scale], [out], [(128, n, k)], [q], kernel_id=lib.mxmoe_find_kernel(b"groupgemm_hz_fused_" + kernel.encode()), acc=[acc]).run()
            err[kernel] = ((acc.view(torch.float32).double() - ref).norm() / ref.norm()).item()
        print(bits, k, mean, err)
        assert err["a16_few"] <= 1.1 * err["all"], (mean, err)


# tokens, top-k, experts, first of the experts that most tokens take, tokens that take others: up to four (32 rows each) and eight (16) row tiles of an expert over rows of the grid that no expert needs, as many of them as
# tiles, more, fewer and none; those experts behind the first 64; ids out of range
@pytest.mark.gpu
@pytest.mark.parametrize("mix", ["fp16", "wo", "int"])
@pytest.mark.parametrize("tokens,topk,experts,first,others", [(64, 4, 60, 0, 0), (128, 4, 60, 7, 0), (128, 4, 130, 66, 0), (128, 4, 130, 126, 9), (128, 2, 5, 1, 0), (128, 3, 6, 2, 1), (65, 2, 2, 0, 0), (97, 1, 70, 69, 0),
                                                              (128, 4, 60, 20, 64)])
def test_row_tiles_of_an_expert_that_most_tokens_take(tokens, topk, experts, first, others, mix):
    """Dealt to several workgroups where the grid has spare ones: identical outputs with the form that has launches in front."""
    from mxmoe_amd import _lib, synth as S
    from mxmoe_amd.layer import MxMoELayer

    fm = {"fp16": [(FP16, FP16)], "wo": [(S.W4A16, S.W2A16), (S.W2A16, S.W4A16)], "int": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4)]}[mix]
    cfg = S.MoEConfig("t", "test", experts, topk, 512, 256, tokens, num_shared=1, rotate=int(mix == "int"))
    layer = MxMoELayer(cfg, formats=[fm[i % len(fm)] for i in range(experts + 1)])
    lib = _lib.load()
    kid = lib.mxmoe_find_kernel(b"groupgemm_hz_fused_" + {"fp16": b"a16_few", "wo": b"wo_few", "int": b"wxax_few"}[mix])
    layer._planned_kernel = lambda *_, **__: kid
    gen = torch.Generator().manual_seed(tokens + experts)
    ids = (first + torch.arange(topk)).remainder(experts).repeat(tokens, 1).to(torch.int32)
    for t in range(others):
        ids[2 * t] = torch.randperm(experts, generator=gen)[:topk].to(torch.int32)
    ids[-1, 0], ids[-2, -1] = -1, experts
    ids, w = ids.cuda(), torch.rand(tokens, topk, generator=gen).cuda()
    hidden = torch.randn(tokens, 512, generator=gen).half().cuda()
    got = layer(hidden, ids, w).clone()
    assert not lib.mxmoe_layer_has_head(layer._short[tokens, topk]._handle)
    layer._short[tokens, topk] = None
    assert torch.equal(layer(hidden, ids, w), got)
