"""The row quantisers by the kernel that a launch takes, against the CPU oracle bit for bit: which one it is depends on the row's length and rotation
and on the number of rows."""
import numpy as np
import pytest
import torch

from oracle import mxmoe_oracle as O
from test_gpu_prologue import DEV, F16, _bf6_rows, _check_rows, _ids, _unpack

pytestmark = pytest.mark.gpu

W4, W8, FP = (4, 4, -1, True), (8, 8, -1, True), (16, 16, -1, True)


def _order(monkeypatch, f, kb):
    """Rotations of order f * kb, Sylvester (f) kron the table of kb: lengths that no table order of its own leads to."""
    from mxmoe_amd import ops

    h = np.ones((1, 1), np.int8)
    while len(h) < f:
        h = np.block([[h, h], [h, -h]])
    table = O.had_table(kb)
    full = np.kron(h, table).astype(np.int8)
    real = O.had_table
    monkeypatch.setattr(O, "get_hadK", lambda n: (full, f * kb))
    monkeypatch.setattr(O, "had_table", lambda k: full if k == f * kb else real(k))
    signs = torch.from_numpy(table.astype(np.float32)).to(DEV)
    monkeypatch.setattr(ops, "device_signs", lambda n, device: (f * kb, f, signs))
    assert O.had_factor(f * kb)[:2] == (f, kb)


def _check(got, scales, y, q, variant, what):
    if variant == "bf6" and q == W4:
        codes, s, _ = O.quant_minmax(y, 4, -1, True)
        assert np.array_equal(_bf6_rows(got, *y.shape), codes.astype(np.int8)), (what, "codes")
    elif variant == "fp8" and q == W8:
        codes, s = O.quant_e4m3(y)
        assert np.array_equal(got.contiguous().view(torch.uint8).cpu().numpy().reshape(codes.shape), codes), (what, "codes")
    else:
        return _check_rows(got, scales, y, q, what)
    assert np.array_equal(scales.cpu().numpy().view(np.uint16), s.reshape(-1).view(np.uint16)), (what, "scales")


def _quant_inp(k, t, topk, variant, n_sh=0):
    from mxmoe_amd import ops

    rng = np.random.default_rng(k + t)
    e = 4
    x = (rng.standard_normal((t, k)) * rng.uniform(0.05, 20, (t, 1))).astype(F16)
    x[3] = 0
    ids = _ids(rng, t, e, topk)
    qp = [W4, W8, FP, W4] + [W8] * n_sh
    inp, sc = ops.quant_inp_act(torch.from_numpy(x).to(DEV), torch.from_numpy(ids).to(DEV), e, 256, n_sh, qp, rotate=1, **{v: True for v in (variant,) if v})[:2]
    torch.cuda.synchronize()
    _, o_perm, _, o_recv = O.permute_by_expert(ids, e)
    y = O.online_hadamard(x)
    st = 0
    for ex in range(e + n_sh):
        m = t if ex == e else int(o_recv[ex])
        rows = slice(None) if ex == e else o_perm[st:st + m]
        st += m if ex < e else 0
        _check(inp[ex], sc[ex], (y if qp[ex][0] < 16 else x)[rows], qp[ex], variant, ex)


def _silu(n, n_sh, t, variant, topk=2):
    from mxmoe_amd import ops

    rng = np.random.default_rng(n + n_sh + t)
    e = 4
    ids = _ids(rng, t, e, topk)
    o_dst, _, _, o_recv = O.permute_by_expert(ids, e)
    gu = (rng.standard_normal((t * topk, 2 * n)) * 2).astype(F16)
    gu_sh = (rng.standard_normal((t, 2 * n * n_sh)) * 2).astype(F16)
    qp = [W4, W8, FP, W4] + [W4 if variant == "bf6" else W8] * (n_sh > 0)
    inp, sc = ops.silu_mul_then_quant(torch.from_numpy(np.concatenate([gu.reshape(-1), gu_sh.reshape(-1)])).to(DEV), int((o_recv != 0).sum()), e, 2048, n, n_sh, t, topk,
                                      torch.from_numpy(o_dst).to(DEV), torch.from_numpy(o_recv), qp, rotate=1, **{v: True for v in (variant,) if v})[:2]
    torch.cuda.synchronize()
    st = 0
    for ex in range(e + (n_sh > 0)):
        m = t if ex == e else int(o_recv[ex])
        y = O.silu_mul(gu_sh if ex == e else gu[st:st + m])
        st += m if ex < e else 0
        _check(inp[ex], sc[ex], O.online_hadamard(y) if qp[ex][0] < 16 else y, qp[ex], variant, ex)


# one length with H_8, more rows than go one to a workgroup: one row per wave; one to four chunks of 512 values per row
@pytest.mark.parametrize("variant", ["", "bf6", "fp8"])
@pytest.mark.parametrize("k,order", [(224, None), (896, (4, 28)), (1408, None), (1920, (4, 60))])
def test_rows_by_waves_with_the_dense_stage_bit_exact(k, order, variant, monkeypatch):
    if order:
        _order(monkeypatch, *order)
    if variant == "bf6" and k % 64:
        pytest.skip("bf6 fragments are 64 values long")
    _quant_inp(k, 301, 2, variant, n_sh=1)
    if k <= 1408:
        _silu(k, 0, 301, variant)


# the same rows beside a shared expert's of twice the length, in one launch
@pytest.mark.parametrize("variant", ["", "bf6", "fp8"])
@pytest.mark.parametrize("n,order", [(224, None), (896, (4, 28)), (1408, None), (1920, (4, 60))])
def test_rows_by_waves_beside_shared_rows_bit_exact(n, order, variant, monkeypatch):
    if order:
        _order(monkeypatch, *order)
    if variant == "bf6" and n % 64:
        pytest.skip("bf6 fragments are 64 values long")
    _silu(n, 2, 270, variant)


# the last row count of the kernel with one row per workgroup and the first of its neighbour, for each limit that row lengths lead to
@pytest.mark.parametrize("k,rows", [(192, 256), (192, 257), (448, 512), (448, 513), (480, 256), (480, 257), (224, 16), (1408, 512), (1408, 513)])
def test_rows_at_the_limits_between_kernels_bit_exact(k, rows):
    _quant_inp(k, rows, 1, "")
    _silu(k, 0, rows, "", topk=1)


# tokens of two routed rows and a shared one of twice the length: one row of either kind per workgroup, routed rows by waves, launches after each other, any row
@pytest.mark.parametrize("n,t", [(1408, 85), (1408, 86), (480, 85), (480, 86), (480, 129), (224, 20), (224, 256), (224, 513), (448, 256)])
def test_shared_rows_at_the_limits_between_kernels_bit_exact(n, t):
    _silu(n, 2, t, "")


# table orders times H_64 and H_256, in the kernel that takes any row
@pytest.mark.parametrize("k,variant", [(3072, ""), (3072, "bf6"), (3072, "fp8"), (7168, ""), (11264, ""), (11264, "bf6")])
def test_rows_of_any_length_bit_exact(k, variant):
    _quant_inp(k, 21, 2, variant, n_sh=1)


@pytest.mark.parametrize("k,t", [(1408, 40), (1408, 520), (2816, 40), (3072, 40)])
def test_rows_with_infinities_and_nans_stay_by_themselves(k, t):
    """A rotated row with such a value has no specified codes; the rows that share its workgroup, wave or LDS have theirs, and rows that are
    copied as fp16 keep every bit."""
    from mxmoe_amd import ops

    rng = np.random.default_rng(k + t)
    e = 3
    x = rng.standard_normal((t, k)).astype(F16)
    bad = np.zeros(t, bool)
    bad[1::3] = True
    x[bad, rng.integers(0, k, bad.sum())] = rng.choice(np.array([np.inf, -np.inf, np.nan], F16), bad.sum())
    ids = _ids(rng, t, e, 1)
    qp = [W4, W8, FP]
    inp, sc = ops.quant_inp_act(torch.from_numpy(x).to(DEV), torch.from_numpy(ids).to(DEV), e, 256, 0, qp, rotate=1)[:2]
    torch.cuda.synchronize()
    _, o_perm, _, o_recv = O.permute_by_expert(ids, e)
    st = 0
    for ex in range(e):
        rows = o_perm[st:st + int(o_recv[ex])]
        st += len(rows)
        good = ~bad[rows]
        assert good.any() and not good.all()
        if qp[ex] == FP:
            assert np.array_equal(inp[ex].cpu().numpy().view(np.uint16), x[rows].view(np.uint16))
            continue
        codes, s, _ = O.quant_minmax(O.online_hadamard(x[rows][good]), qp[ex][0], -1, True)
        assert np.array_equal(sc[ex].cpu().numpy().view(np.uint16)[good], s.reshape(-1).view(np.uint16))
        assert np.array_equal(_unpack(inp[ex], 1 if qp[ex][0] == 8 else 2, k)[good], codes.astype(np.int8))
