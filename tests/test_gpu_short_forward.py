"""The short form of the planned forward (mxmoe_layer_run: one head launch, rows gathered by token, silu(gate) * up as gate_up's output)
against the forward with host tables and stored gate_up rows: identical outputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

W8A16 = (16, 8, 128, False)


def _layer(tokens, topk, formats, hidden=512, inter=1408, num_shared=1, rotate=1, fp8=False):
    from mxmoe_amd import synth
    from mxmoe_amd.layer import MxMoELayer

    n = len(formats) - (1 if num_shared else 0)
    cfg = synth.MoEConfig("t", "test", n, topk, hidden, inter, tokens, num_shared=num_shared, rotate=rotate)
    return cfg, MxMoELayer(cfg, formats=formats, fp8=fp8)


def _check(cfg, layer, drop=True):
    from mxmoe_amd import synth

    assert layer._short_setup(cfg.tokens, cfg.topk) is not None
    hidden = synth.make_hidden(cfg)
    ids, w = synth.make_routing(cfg)
    if drop:
        ids[0, 0] = cfg.num_experts + 2
        ids[cfg.tokens // 2, cfg.topk - 1] = -1
    got = layer(hidden, ids, w)
    want = layer.call_with_host_tables(hidden, ids, w)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    again = layer(hidden, ids, w)                                       # (buffers of the previous call)
    assert torch.equal(again, want)


# tokens: one row, the edges of the 16 / 32 / 64 / 128-row tiles over a few experts, and past one chunk of 256 permuted entries
@pytest.mark.parametrize("tokens", [1, 2, 31, 33, 129, 700])
@pytest.mark.parametrize("mix", ["wxax", "wo", "fp16", "all", "fp8"])
def test_short_forward_equals_the_forward_with_host_tables(tokens, mix):
    from mxmoe_amd import synth as S

    fm = {"wxax": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W4A4, S.W4A4), (S.W8A8, S.W8A8)],
          "wo": [(S.W4A16, S.W3A16), (S.W3A16, S.W2A16), (S.W2A16, S.W4A16), (S.W4A16, S.W4A16)],
          "fp16": [(S.FP16, S.FP16)] * 4,
          "all": [(S.W4A4G128, S.W4A16), (S.FP16, S.W8A8), (W8A16, S.W4A4G128), (S.W4A4, S.FP16), (S.W8A8, W8A16), (S.W2A16, S.W4A4), (S.W4A16, S.W2A16)],
          "fp8": [(S.W8A8, S.W8A8), (S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W8A8, S.W8A8)]}[mix]
    cfg, layer = _layer(tokens, 2, fm, fp8=mix == "fp8")
    _check(cfg, layer, drop=tokens > 1)


def _few_layer(tokens, mix, inter, hidden=512):
    """A layer of ten to twelve experts and a shared one on the kernels made for few rows, its routing drawn to one expert (up to all of the tokens: several narrow row tiles)."""
    from mxmoe_amd import _lib
    from mxmoe_amd import synth as S

    fm = {"wxax": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W4A4, S.W4A4), (S.W8A8, S.W8A8)],
          "all": [(S.W4A4, S.W8A8), (S.W8A8, S.W4A16), (S.W4A16, S.W4A4), (S.W3A16, S.W8A8), (W8A16, S.W2A16)]}[mix]
    fm = fm * (12 // len(fm)) + fm[:1]
    cfg, layer = _layer(tokens, 2, fm, hidden=hidden, inter=inter)
    lib = _lib.load()
    desc = layer._block_descs(layer.qp_gate_up, [2 * inter] * len(fm), [hidden] * len(fm), layer.w13, False)
    kid = lib.mxmoe_plan_select_kernel_rows(desc, cfg.num_experts, tokens, cfg.topk, tokens)
    assert lib.mxmoe_kernel_name(kid).decode().endswith(f"groupgemm_hz_fused_{mix}_few")
    hidden_t = S.make_hidden(cfg).cuda()
    ids, w = S.make_routing(cfg)
    ids = ids.cuda()
    ids[:, 0] = 1                                                       # (expert 1 may be in a token's list twice: it gets both rows)
    ids[:tokens // 4, 0] = 0
    return cfg, layer, hidden_t, ids, w.cuda()


# tokens: one row; the last that fits one narrow row tile; one more (two row tiles of narrow tiles: few blocks); the most those kernels take
@pytest.mark.parametrize("tokens,inter", [(1, 1408), (24, 1408), (32, 1408), (33, 512), (64, 512)])
@pytest.mark.parametrize("mix", ["wxax", "all"])
def test_short_forward_on_the_kernels_for_few_rows(tokens, inter, mix):
    """Their gate_up form (rows gathered by token, silu(gate) * up as output) with every format that they hold beside each other."""
    cfg, layer, hidden, ids, w = _few_layer(tokens, mix, inter)
    assert layer._short_setup(cfg.tokens, cfg.topk) is not None
    want = layer.call_with_host_tables(hidden, ids, w)
    assert torch.equal(layer(hidden, ids, w), want)


@pytest.mark.parametrize("hidden,inter,num_shared,rotate", [(1024, 224, 0, 2), (2048, 64, 2, 0), (4096, 96, 1, 0), (512, 32, 0, 0)])
def test_short_forward_row_lengths_and_rotations(hidden, inter, num_shared, rotate):
    """Every row length of the head's token kernel; intermediate sizes that end inside a tile's gate half."""
    from mxmoe_amd import synth as S

    if inter % 128 == 0 or rotate:
        fm = [(S.W4A4, S.FP16), (S.W8A8, S.FP16), (S.FP16, S.FP16), (S.W4A4G128, S.FP16), (S.W4A16, S.FP16)]
    else:
        fm = [(S.W4A16, S.FP16), (S.W8A8, S.FP16), (S.FP16, S.FP16), (S.W4A4, S.FP16), (S.W3A16, S.FP16)]
    cfg, layer = _layer(70, 3, fm, hidden=hidden, inter=inter, num_shared=num_shared, rotate=rotate)
    _check(cfg, layer)


def test_short_forward_of_more_experts_than_one_launch_holds():
    from mxmoe_amd import synth as S

    cfg, layer = _layer(300, 3, [((S.W4A4, S.W8A8), (S.W8A8, S.FP16), (S.FP16, S.W4A4))[i % 3] for i in range(131)], inter=512)
    _check(cfg, layer)


@pytest.mark.parametrize("inter,had,down,num_shared,rotate", [(320, None, "W8A8", 2, 1), (480, None, "FP16", 4, 2), (1024, (64, 2), "W4A4", 2, 1), (1408, None, "W4A4", 4, 1),
                                                              (2048, (64, 4), "W8A8", 2, 1)])
def test_routed_and_shared_rows_of_two_lengths_in_one_launch(monkeypatch, inter, had, down, num_shared, rotate):
    """row_quant_pair_kernel at 1, 2, 3 and 4 chunks of 8 values per lane of a routed row.  Rows of 1024 and 2048 values are powers of two and
    would take no table of their own: they get one of kb x kb signs (the rotation's sums are exact for any signs) on both sides."""
    from mxmoe_amd import layer as L
    from mxmoe_amd import synth as S

    if had:
        kb, f = had
        signs = (1.0 - 2.0 * torch.randint(0, 2, (kb, kb), generator=torch.Generator().manual_seed(inter))).cuda()
        plain = L.device_signs
        monkeypatch.setattr(L, "device_signs", lambda n, dev: (kb * f, f, signs) if n % inter == 0 else plain(n, dev))
    fmt = getattr(S, down)
    cfg, layer = _layer(260, 2, [(S.W8A8, fmt), (S.W4A4, fmt), (S.FP16, fmt), (S.W8A8, fmt)], inter=inter, num_shared=num_shared, rotate=rotate)
    _check(cfg, layer)


@pytest.mark.parametrize("tokens,topk,num_shared", [(300, 2, 2), (300, 3, 2), (300, 2, 4), (2305, 1, 2), (4096, 2, 2), (4096, 3, 2), (4097, 2, 2)])
def test_short_forward_of_many_shared_rows_beside_routed_ones(tokens, topk, num_shared):
    """Work of the shared rows below, at and above the routed rows', which decides how the launch is shared out; the last number of shared rows in one launch with routed ones."""
    from mxmoe_amd import synth as S

    cfg, layer = _layer(tokens, topk, [(S.W4A4, S.W8A8), (S.W8A8, S.W4A4), (S.W4A4, S.W4A4), (S.W8A8, S.W4A4), (S.W4A4, S.W8A8)], num_shared=num_shared)
    _check(cfg, layer)


@pytest.mark.parametrize("tokens", [50, 1100])
def test_short_forward_of_the_most_experts_it_takes(tokens):
    """512 experts, the most LDS the head asks for, in workgroups of 256 and of 512 threads; five launches per block to plan."""
    from mxmoe_amd import synth as S

    cfg, layer = _layer(tokens, 4, [((S.W4A4, S.W8A8), (S.W8A8, S.FP16), (S.FP16, S.W4A4))[i % 3] for i in range(513)], inter=128, rotate=0)
    _check(cfg, layer)


def test_short_forward_counts_ids_in_a_launch_of_its_own():
    """More than 65536 (token, slot) entries: the per-chunk counting launch in front of the head."""
    from mxmoe_amd import synth as S

    cfg, layer = _layer(33001, 2, [(S.W4A4, S.FP16), (S.W8A8, S.W4A16), (S.FP16, S.FP16), (S.W4A16, S.FP16)], inter=128, num_shared=0, rotate=0)
    _check(cfg, layer)


@pytest.mark.parametrize("mix", ["fp16", "wo", "wxax"])
@pytest.mark.parametrize("offset", [1, 2, 4, 7])
def test_tokens_from_the_middle_of_a_buffer(mix, offset):
    """A contiguous view whose address is not a multiple of 16 bytes, with enough rows for the tiles that load tokens straight into LDS."""
    from mxmoe_amd import synth as S

    fm = {"fp16": (S.FP16, S.FP16), "wo": (S.W4A16, S.W3A16), "wxax": (S.W4A4, S.W8A8)}[mix]
    cfg, layer = _layer(300, 2, [fm] * 4)
    hidden = S.make_hidden(cfg).cuda()
    ids, w = S.make_routing(cfg)
    store = torch.zeros(hidden.numel() + 16, dtype=torch.float16, device="cuda")
    view = store[offset:offset + hidden.numel()].view(hidden.shape)
    view.copy_(hidden)
    assert view.is_contiguous() and view.data_ptr() % 16 == 2 * offset
    assert torch.equal(layer(view, ids, w), layer(hidden, ids, w))
    assert torch.equal(view, hidden)


def test_layers_the_short_form_does_not_take():
    from mxmoe_amd import synth as S

    for hidden in (256, 1536):                                          # rows below 512 values, or no power of two
        cfg, layer = _layer(20, 2, [(S.FP16, S.FP16)] * 3, hidden=hidden, num_shared=0, rotate=0)
        assert layer._short_setup(cfg.tokens, cfg.topk) is None
        hidden_t = S.make_hidden(cfg)
        ids, w = S.make_routing(cfg)
        assert torch.equal(layer(hidden_t, ids, w), layer.call_with_host_tables(hidden_t, ids, w))


@pytest.mark.parametrize("num_bytes", [4, 3584, 3588, 4032, 4036, 8064, 10000])
def test_upload_in_kernel_arguments(num_bytes):
    """Host tables of less than one, exactly one (4032 bytes) and several launches' arguments; the bytes behind them stay as they were."""
    import numpy as np

    from mxmoe_amd import _lib

    lib = _lib.load()
    host = np.random.default_rng(num_bytes).integers(0, 256, num_bytes, dtype=np.uint8)
    dst = torch.full((num_bytes + 8,), 7, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib, lib.mxmoe_upload(dst.data_ptr(), host.ctypes.data, num_bytes, stream))
    want = host.copy()
    host[:] = 0                                                         # the caller's array is free again at once
    assert np.array_equal(dst[:num_bytes].cpu().numpy(), want) and bool((dst[num_bytes:] == 7).all())
    assert lib.mxmoe_upload(dst.data_ptr(), host.ctypes.data, 3, stream) == 3 and lib.mxmoe_upload(None, host.ctypes.data, 4, stream) == 5


@pytest.mark.parametrize("topk,num_shared", [(1, 0), (8, 1), (9, 1), (17, 0)])
def test_combine_of_more_slots_than_it_loads_at_a_time(topk, num_shared):
    """gg_unpermute_out (combine_kernel takes eight slots at a time) against the oracle, ids out of range included."""
    import numpy as np

    from mxmoe_amd import ops
    from oracle import mxmoe_oracle as O

    rng = np.random.default_rng(topk)
    t, e, k = 13, 20, 136
    ids = np.stack([rng.permutation(e)[:topk] for _ in range(t)]).astype(np.int32)
    ids[4, 0] = e + 1
    w = rng.random((t, topk), dtype=np.float32)
    slots = np.argsort(ids.reshape(-1), kind="stable")
    slots = slots[ids.reshape(-1)[slots] < e]                           # sorted rows in (expert, token, slot) order
    rows = len(slots)
    down = rng.standard_normal((rows + (t if num_shared else 0), k)).astype(np.float16)
    want = O.unpermute_combine(down[:rows], slots, w, down[rows:] if num_shared else None)
    store = torch.from_numpy(down).cuda()
    got = ops.gg_unpermute_out(store, torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(), e, k, num_shared)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    with pytest.raises(RuntimeError, match="out_store holds"):
        ops.gg_unpermute_out(store[:-1], torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(), e, k, num_shared)
