"""Integer codes taken from packed halves: the arithmetic over every value and scale on the CPU, and the row quantisers at the ends of the fp16 range."""
import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O

F16, F32, F64 = np.float16, np.float32, np.float64


def _fma16(a, b, c):
    return (a.astype(F64) * b.astype(F64) + c.astype(F64)).astype(F16)  # exact in 64 bits: products of 22 bits beside terms at most 2^30 away


def _codes(v, s, upper):
    """The steps of HalfDiv (mxmoe_rows.hpp) on fp16 numbers."""
    e = np.maximum((s.view(np.uint16) >> 10).astype(int), 0) - 15
    f = F64(2.0) ** np.where(s < F16(2.0**-14), 15, -e)
    sn, x = (s * f).astype(F16), (v * f).astype(F16)
    r = (1.0 / sn.astype(F64)).astype(F16)
    q0 = (x * r).astype(F16)
    q = _fma16(_fma16(-q0, sn, x), r, q0)
    q = np.minimum(np.maximum(q, F16(-upper)), F16(upper))
    return (q + F16(1536)).view(np.uint16).astype(int) - 0x6600


@pytest.mark.parametrize("upper", [7, 127])
def test_codes_from_packed_halves_are_those_of_the_fp32_quotient(upper):
    """Every fp16 value that a row of that scale can hold (its largest magnitude is at most upper times the scale before the scale was rounded), every
    mantissa of a scale, every scale below the normal numbers and the largest ones."""
    vals = np.arange(0x0000, 0x7C00, dtype=np.uint16).view(F16)
    top = F16(65504 / upper).view(np.uint16)
    scales = np.concatenate([np.arange(0x3C00, 0x4000), np.arange(1, 0x440), np.arange(top - 40, top + 1)]).astype(np.uint16).view(F16)
    for s in scales:
        v = vals[vals.astype(F64) <= (F64(s) * (1 + 2.0**-11) + 2.0**-25) * upper]
        want = np.rint(np.clip((v.astype(F32) / F32(s)).astype(F16), F16(-upper), F16(upper))).astype(int)
        ss = np.full_like(v, s)
        assert np.array_equal(_codes(v, ss, upper), want), s
        assert np.array_equal(_codes(-v, ss, upper), -want), s


def test_reciprocal_of_a_scale_is_no_tie():
    """A reciprocal that is off by one part in 2^23 rounds to the fp16 number that the exact one rounds to."""
    r = 1.0 / (1.0 + np.arange(1024) / 1024.0)
    for off in (1 - 2.0**-23, 1 + 2.0**-23):
        assert np.array_equal((r * off).astype(F32).astype(F16), r.astype(F16))


# a row with an infinity has an infinite scale: codes 0, and the lowest one for the infinity itself
# one row per token and wave, per row and wave, per workgroup of 4 (few rows) and 8 waves, and any row; all three integer formats, as they are
@pytest.mark.gpu
@pytest.mark.parametrize("k,t", [(512, 40), (1408, 600), (1408, 40), (3072, 40), (14336, 40)])
def test_rows_at_the_ends_of_the_range_bit_exact(k, t):
    from mxmoe_amd import ops
    from test_gpu_prologue import DEV, _ids, _unpack

    rng = np.random.default_rng(k + t)
    tops = np.array([2.0**-24, 5 * 2.0**-24, 100 * 2.0**-24, 2.0**-14, 0.0061, 0.9, 7, 127, 896.5, 65504])[np.arange(t) % 10]
    x = (rng.uniform(-1, 1, (t, k)) * tops[:, None]).astype(F16)
    x[:, 5] = tops.astype(F16)
    x[:, 7:400:3] = ((rng.integers(-14, 15, (t, 131)) / 14) * tops[:, None]).astype(F16)  # halves of a code of four bits
    x[11, 9], x[12, 40] = np.inf, -np.inf
    ids = _ids(rng, t, 3, 1)
    qp = [(4, 4, -1, True), (8, 8, -1, True), (4, 4, 128, True)]
    inp, sc = ops.quant_inp_act(torch.from_numpy(x).to(DEV), torch.from_numpy(ids).to(DEV), 3, 256, 0, qp, rotate=0)[:2]
    torch.cuda.synchronize()
    _, perm, _, recv = O.permute_by_expert(ids, 3)
    st = 0
    for e in range(3):
        rows = perm[st:st + int(recv[e])]
        st += len(rows)
        assert len(rows)
        with np.errstate(invalid="ignore"):
            codes, s, _ = O.quant_minmax(x[rows], qp[e][0], qp[e][2], True)
        codes = np.where(np.isnan(codes), 1 - 2.0 ** (qp[e][0] - 1), codes).astype(np.int8)
        assert np.array_equal(sc[e].cpu().numpy().view(np.uint16).reshape(-1), s.reshape(-1).view(np.uint16)), e
        assert np.array_equal(_unpack(inp[e], O.act_tag(qp[e][0], qp[e][2]), k), codes), e
