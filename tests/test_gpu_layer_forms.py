"""The forms of a layer's forward (with and without a head, tables by the device and by the host, step by step) on the kernels that the layer takes by itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu

W8A16 = (16, 8, 128, False)


def _weights(experts, inter, hidden, num_shared, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    widths = [inter] * experts + ([inter * num_shared] if num_shared else [])
    return [tuple((torch.randn(n, k, generator=gen, device="cuda") * 0.02).half() for n, k in ((2 * w, hidden), (hidden, w))) for w in widths]


def _routing(tokens, experts, topk, skewed, gen):
    z = torch.rand(tokens, experts, generator=gen, device="cuda").clamp_(1e-6, 1 - 1e-6)
    z = -(-z.log()).log()
    if skewed:
        z = z - 1.2 * torch.arange(1, experts + 1, device="cuda").log()
    w, ids = torch.topk(z, topk, dim=1)
    return ids.to(torch.int32), torch.softmax(w, dim=1)


MIXES = {"fp16": ["FP16"], "w8a16/w2a16": ["W8A16", "W2A16"], "w4a16/w3a16": ["W4A16", "W3A16"], "w4a4/fp8": ["W4A4", "W8A8"], "w4a4/w8a8/w4a16": ["W4A4", "W8A8", "W4A16"],
         "w4a4g128/fp8/w8a16/w2a16": ["W4A4G128", "W8A8", "W8A16", "W2A16"]}


@pytest.mark.parametrize("num_shared", [0, 2])
@pytest.mark.parametrize("mix", list(MIXES))
def test_forms_of_a_layer_agree(mix, num_shared):
    """60 experts top-4 from 1 to 200 tokens, evenly routed and skewed: one choice of kernels for all forms, so identical outputs, also where the sums of two kernels differ in single bits (fp16 and
    weight-only blocks; fp8 ones, with tokens of values of many sizes).  The list's real row counts would choose otherwise in some of these cases (skewed: fewer experts of more rows; even: no more rows than on average)."""
    from mxmoe_amd import synth as S
    from mxmoe_amd.layer import MxMoELayer

    fm = [W8A16 if f == "W8A16" else getattr(S, f) for f in MIXES[mix]]
    n = 60 + (num_shared > 0)
    formats = [(fm[i % len(fm)], S.FP16 if "fp8" in mix and i % 2 else fm[(i + 1) % len(fm)]) for i in range(n)]
    gen = torch.Generator(device="cuda").manual_seed(5)
    rotate = int("fp8" not in mix)  # (a rotation would even the tokens out)
    base = S.MoEConfig("t", "test", 60, 4, 2048, 1408, 1, num_shared=num_shared, rotate=rotate)
    layer = MxMoELayer(base, formats=formats, weights=_weights(60, 1408, 2048, num_shared, 3), fp8="fp8" in mix)
    for tokens in (1, 16, 33, 64, 65, 96, 128, 200):
        layer.cfg = S.MoEConfig("t", "test", 60, 4, 2048, 1408, tokens, num_shared=num_shared, rotate=rotate)
        for skewed in (False, True):
            hidden = torch.randn(tokens, 2048, generator=gen, device="cuda")
            if "fp8" in mix:
                hidden = hidden * torch.exp(2 * torch.randn(tokens, 2048, generator=gen, device="cuda")) / 64
            hidden = hidden.half()
            ids, w = _routing(tokens, 60, 4, skewed, gen)
            got = layer(hidden, ids, w).clone()
            assert torch.isfinite(got).all()
            short, layer._short[tokens, 4] = layer._short[tokens, 4], None
            assert short is not None
            assert torch.equal(layer(hidden, ids, w), got), (tokens, skewed, "planned, with gate and up stored")
            layer._short[tokens, 4] = short
            assert torch.equal(layer.call_with_host_tables(hidden, ids, w), got), (tokens, skewed, "host tables")
            layer.forward(hidden, ids)
            assert torch.equal(layer.combine(w), got), (tokens, skewed, "step by step")


@pytest.mark.parametrize("tokens", [65, 100, 128])
@pytest.mark.parametrize("mix", ["fp16", "w8a16/w2a16", "w4a16/w3a16", "w8a16/w4a16/fp16"])
def test_layer_of_65_to_128_tokens_against_float64(mix, tokens):
    """On the same weights (dequantised, not rounded).  Roundings to fp16 of gate, up, their product, the second block's weights (in its tiles of many tokens), its output and the combined
    one: six errors of at most 2^-11 each, without correlation 2^-11 / sqrt(3) each, so less than 2^-10 together; the float32 sums add less than one more of those."""
    from mxmoe_amd import synth as S
    from mxmoe_amd.layer import MxMoELayer
    from mxmoe_amd.quant import quant_minmax

    fm = {"w8a16/w4a16/fp16": [W8A16, S.W4A16, S.FP16]}.get(mix) or [W8A16 if f == "W8A16" else getattr(S, f) for f in MIXES[mix]]
    cfg = S.MoEConfig("t", "test", 40, 4, 2048, 1408, tokens, num_shared=1, rotate=0)
    formats = [(fm[i % len(fm)], fm[(i + 1) % len(fm)]) for i in range(41)]
    weights = _weights(40, 1408, 2048, 1, 9)
    layer = MxMoELayer(cfg, formats=formats, weights=weights)
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    hidden = torch.randn(tokens, 2048, generator=gen, device="cuda").half()
    ids, w = _routing(tokens, 40, 4, True, gen)
    got = layer(hidden, ids, w).double()

    def dense(m, q):
        if q == S.FP16:
            return m.double()
        c, s, z = quant_minmax(m, q[1], 128, False)
        return (c.reshape(m.shape[0], -1, 128).double() * s.reshape(m.shape[0], -1, 1).double() + z.reshape(m.shape[0], -1, 1).double()).reshape(m.shape)

    want = torch.zeros(tokens, 2048, dtype=torch.float64, device="cuda")
    for e in range(41):
        rows, slot = (ids == e).nonzero(as_tuple=True) if e < 40 else (torch.arange(tokens, device="cuda"), None)
        if len(rows) == 0:
            continue
        y = hidden[rows].double() @ dense(weights[e][0], formats[e][0]).T.contiguous()
        gate, up = y[:, :y.shape[1] // 2], y[:, y.shape[1] // 2:]
        out = (gate / (1 + torch.exp(-gate)) * up) @ dense(weights[e][1], formats[e][1]).T.contiguous()
        want.index_add_(0, rows, out * (1.0 if slot is None else w[rows, slot].double()[:, None]))
    assert (got - want).norm() <= 1.5 * 2.0 ** -10 * want.norm()


@pytest.mark.parametrize("tokens", [1, 24, 64])
def test_layer_on_the_few_row_kernel_with_many_token_tiles(tokens):
    """groupgemm_hz_fused_all_few, which lists of w4a4 / w8a8 beside weight-only problems take: a layer of such lists takes the kernel without tiles for many tokens; named for both blocks, with a head and by host tables,
    identical outputs."""
    from mxmoe_amd import _lib, synth as S
    from mxmoe_amd.layer import MxMoELayer

    lib = _lib.load()
    name = lambda kid: lib.mxmoe_kernel_name(kid).decode().split("groupgemm_hz_fused_")[-1]  # noqa: E731
    fm = [(S.W4A4, S.W8A8), (S.W8A8, S.W4A16), (S.W4A16, S.W4A4), (S.W3A16, S.W8A8), (W8A16, S.W2A16)]
    cfg = S.MoEConfig("t", "test", 10, 2, 512, 512, tokens, num_shared=1, rotate=1)
    layer = MxMoELayer(cfg, formats=[fm[i % 5] for i in range(11)])
    assert "all_few" not in {name(k) for k in layer._kernels(tokens, 2)} and (tokens < 24 or name(layer._kernels(tokens, 2)[0]) == "mixed_few")
    kid = lib.mxmoe_find_kernel(b"groupgemm_hz_fused_all_few")
    layer = MxMoELayer(cfg, formats=layer.formats, packed=(layer.w13, layer.w2))
    layer._planned_kernel = lambda *_, **__: kid
    hidden, (ids, w) = S.make_hidden(cfg).cuda(), S.make_routing(cfg)
    ids[:, 0] = 1
    ids, w = ids.cuda(), w.cuda()
    got = layer(hidden, ids, w).clone()
    assert layer._kernels(tokens, 2) == (kid, kid) and lib.mxmoe_layer_has_head(layer._short[tokens, 2]._handle)
    assert torch.equal(layer.call_with_host_tables(hidden, ids, w), got)
    layer._short[tokens, 2] = None
    assert torch.equal(layer(hidden, ids, w), got)
