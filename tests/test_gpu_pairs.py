"""Launches whose problems' two row segments are dealt out as pairs, by what they compute: whole outputs against 64-bit products, for every format that takes pairs."""
import pytest
import torch

from test_tile_order import FP, W4, W8, _launch, _pairs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ints(gen, shape, top):
    return torch.randint(-top, top + 1, shape, generator=gen, device=DEV, dtype=torch.int8)


def _fp8(gen, shape):
    """e4m3 codes of all exponents and their values."""
    code = torch.randint(0, 256, shape, generator=gen, device=DEV, dtype=torch.uint8)
    code = torch.where((code & 0x7F) == 0x7F, code ^ 1, code)  # (no NaN)
    return code, code.view(torch.float8_e4m3fn).double()


# rows: some whole tiles and a remainder in each of the shorter shapes, next to problems of one segment; K of few slices keeps the references quick.
# w4a4 pairs only where there is much to fetch (pairs_pay): wide problems, which share their weights here.
@pytest.mark.parametrize("kernel,q,rows,n,k,count", [
    ("groupgemm_hz_fused_fp16", FP, (144, 190, 100, 300, 128, 7, 0, 257), 2824, 256, 64),
    ("groupgemm_hz_fused_all", FP, (144, 190, 100, 300, 128, 7, 0, 257), 2824, 256, 64),
    ("groupgemm_hz_fused_bf16", FP, (144, 190, 100, 300), 2816, 64, 64),
    ("groupgemm_hz_fused_wxax", W8, (144, 190, 100, 300, 128, 7, 0, 257), 2824, 320, 64),
    ("groupgemm_hz_fused_all", W8, (144, 190, 100, 300), 2816, 320, 64),
    ("groupgemm_hz_fused_wxax_e4m3", W8, (144, 190, 100, 300, 128, 7, 0, 257), 2824, 320, 64),
    ("groupgemm_hz_fused_all_e4m3", W8, (144, 190, 100, 300), 2816, 320, 64),
    ("groupgemm_hz_fused_wxax", W4, (185, 300, 128, 1060), 28672, 4096, 8),
    ("groupgemm_hz_fused_wxax_b6", W4, (185, 300, 128, 1060), 28672, 4096, 8),
])
def test_paired_launches_compute_every_output(lib, kernel, q, rows, n, k, count):
    from mxmoe_amd import pack
    from mxmoe_amd.group_gemm import GroupGemmLaunch

    kid = lib.mxmoe_find_kernel(kernel.encode())
    ms = [rows[i % len(rows)] for i in range(count)]
    tab, _ = _launch(lib, [(m, n, k, q) for m in ms], kid)
    assert len(_pairs(tab)) >= count // 4
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n + k)
    fp8, bf16, bf6 = "e4m3" in kernel, "bf16" in kernel, kernel.endswith("b6")
    A, B, va, vb = [], [], [], []
    for i, m in enumerate(ms):
        new_b = q is not W4 or i == 0
        if fp8:
            (ca, xa), (cb, xb) = _fp8(gen, (m, k)), _fp8(gen, (n, k))
            a, b = ca, pack.pack_wxax_fragments(cb)
        elif q is FP:  # small integers: sums of at most 1024 (bf16: 256), exact in the output's type
            xa, xb = _ints(gen, (m, k), 2), _ints(gen, (n, k), 2)
            a, b = (x.bfloat16().view(torch.float16) if bf16 else x.half() for x in (xa, xb))
        else:
            top = 127 if q is W8 else 7
            xa, xb = _ints(gen, (m, k), top), _ints(gen, (n, k), top) if new_b else None
            if bf6:
                a, b = pack.pack_bf6_fragments(xa) if m else xa, pack.pack_bf6_fragments(xb) if new_b else None
            else:
                a = xa if q is W8 else pack.pack_int4_k(xa)
                b = pack.pack_wxax_fragments(xb if q is W8 else pack.pack_int4_k(xb)) if new_b else None
        A.append(a)
        va.append(xa)
        B.append(b if b is not None else B[0])
        vb.append(xb.double() if xb is not None else vb[0])
    one = torch.ones(max(n, *ms), dtype=torch.float16, device=DEV) * 2.0**-10
    scales = None if q is FP else [one] * count
    Cs = [torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV) for m in ms]
    accs = None if q is FP else [torch.zeros((m, n), dtype=torch.int32, device=DEV) for m in ms]
    GroupGemmLaunch(A, B, scales, scales, Cs, [(m, n, k) for m in ms], [q] * count, kernel_id=kid, acc=accs).run()
    for i, m in enumerate(ms):
        if m == 0:
            continue
        ref = va[i].double() @ vb[i].t()
        if q is FP:
            got = Cs[i].view(torch.bfloat16) if bf16 else Cs[i]
            assert torch.equal(got.double(), ref), (i, m)
        elif fp8:  # (the bound of the fp8 tiles' own tests)
            assert (accs[i].view(torch.float32).double() - ref).abs().max() <= 2e-4 * ref.abs().max(), (i, m)
        else:
            assert torch.equal(accs[i], ref.to(torch.int32)), (i, m)
            assert torch.equal(Cs[i], (accs[i].float() * 2.0**-20).half()), (i, m)


@pytest.mark.parametrize("fmt", [W8, FP])
def test_paired_gate_up_form_equals_the_stored_rows(lib, fmt):
    """A layer whose first launch is paired: gathered rows and silu(gate) * up as output against the forward that stores the gate_up rows, token for token."""
    from mxmoe_amd import synth
    from mxmoe_amd.layer import MxMoELayer

    cfg = synth.MoEConfig("t", "test", 60, 4, 512, 1408, 2500, rotate=1, routing="zipf")
    layer = MxMoELayer(cfg, formats=[(fmt, fmt)] * 60)
    hidden = synth.make_hidden(cfg)
    ids, w = synth.make_routing(cfg)
    assert layer._short_setup(cfg.tokens, cfg.topk) is not None
    recv = torch.bincount(ids.reshape(-1).long(), minlength=60).tolist()
    tab, _ = _launch(lib, [(m, 2816, 512, fmt) for m in recv])
    assert len(_pairs(tab)) >= 4
    got = layer(hidden, ids, w)
    want = layer.call_with_host_tables(hidden, ids, w)
    assert torch.equal(got, want)
