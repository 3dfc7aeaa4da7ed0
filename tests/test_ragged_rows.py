"""Rows that are not whole 16-byte slots, or start off a 16-byte boundary: the
ragged form of the resident kernels (the row's last slot moved back to end with
the row, overlapping the one before it).

Every lanes-per-row and slots-per-lane shape at odd widths, against float64 on
the same inputs: y and inv_rms per element, dx against its row's scale, dgamma
against the sum of its terms' magnitudes (fp32 sums of `rows` terms in any order err
by at most rows * 2^-24 of it; column sums here add in fp64, fp32 only over aligned
rows).  bf16 results carry one rounding (2^-9 relative) more.
"""
import pytest

import cgadimpl_amd as agk
from gpu_util import device_inputs

pytestmark = pytest.mark.gpu

EPS = 1e-6
# one slot and an element more; each power of two of lanes; two and four slots per
# lane; just past the widest ragged backward (looped)
COLS = {
    "f32": [4, 5, 7, 9, 30, 61, 129, 253, 259, 515, 1030, 2051, 4095, 4097, 8193, 16383, 16387],
    "bf16": [8, 9, 15, 17, 61, 121, 253, 511, 1001, 2045, 4099, 8191, 8195, 16383, 16391],
}
CASES = [(dt, c) for dt in COLS for c in COLS[dt]]


def _ref(x, g, dy):
    x64, g64, d64 = x.double(), g.double(), dy.double()
    r = (x64.square().mean(-1, keepdim=True) + EPS).rsqrt()
    xh = x64 * r
    gy = d64 * g64
    dx = r * (gy - xh * (gy * xh).mean(-1, keepdim=True))
    terms = d64 * xh
    return xh * g64, r[:, 0], dx, terms.sum(0), terms.abs().sum(0)


def _check(x, g, dy, y, inv, dx, dg, label):
    ry, rr, rdx, rdg, mag = _ref(x, g, dy)
    one = 2.0 ** -8 if str(x.dtype).endswith("bfloat16") else 0.0  # a rounding to storage
    bar = 1e-5 + one
    assert ((y.double() - ry).abs() <= bar * ry.abs() + 1e-30).all().item(), (label, "y")
    assert ((inv.double().view(-1) - rr).abs() <= 1e-5 * rr).all().item(), (label, "inv_rms")
    scale = rdx.abs().amax(-1, keepdim=True) + (rr * dy.double().abs().amax(-1)).view(-1, 1)
    assert ((dx.double() - rdx).abs() <= bar * scale).all().item(), (label, "dx")
    assert ((dg.double() - rdg).abs() <= 1e-5 * mag + 1e-30).all().item(), (label, "dgamma")


@pytest.mark.parametrize("dtype,cols", CASES, ids=str)
@pytest.mark.parametrize("rows", [1, 37, 600, 1700])
def test_layer_matches_fp64(cuda, dtype, cols, rows):
    import torch
    print(f"{dtype} {rows}x{cols}", flush=True)
    x, g, dy = device_inputs((rows, cols), dtype, rows * 31 + cols, cuda)
    y, inv = agk.rmsnorm_fwd(x, g, EPS)
    dx, dg = agk.rmsnorm_bwd(x, g, inv, dy)
    torch.cuda.synchronize()
    _check(x, g, dy, y, inv, dx, dg, f"{dtype} {rows}x{cols}")
    # in place, gradients alone, no gamma, and repeats: the same bits
    x_in = x.clone()
    agk.rmsnorm_fwd(x_in, g, EPS, y=x_in)
    dx_only, _ = agk.rmsnorm_bwd(x, g, inv, dy, want_dgamma=False)
    _, dg_only = agk.rmsnorm_bwd(x, g, inv, dy, want_dx=False)
    h, inv2 = agk.rmsnorm_fwd(x, None, EPS)
    torch.cuda.synchronize()
    assert torch.equal(x_in, y) and torch.equal(dx_only, dx) and torch.equal(dg_only, dg)
    assert torch.equal(inv2, inv)
    # accumulation: the fresh gradient added once to every element
    pre_dx, pre_dg = torch.full_like(x, 0.25), torch.full((cols,), -0.5, device=cuda)
    adx, adg = agk.rmsnorm_bwd(x, g, inv, dy, dx=pre_dx.clone(), dgamma=pre_dg.clone(),
                               accumulate=True)
    torch.cuda.synchronize()
    assert torch.equal(adg, pre_dg + dg)
    if dtype == "f32":
        assert torch.equal(adx, pre_dx + dx)
    else:  # dx above is rounded to bf16 before the sum, the accumulated term is not
        assert ((adx.float() - (0.25 + dx.float())).abs()
                <= 2.0 ** -8 * (0.25 + dx.float().abs())).all().item()


@pytest.mark.parametrize("dtype,cols", CASES, ids=str)
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("rows", [600, 900])
def test_composition_equals_its_two_calls(cuda, dtype, cols, accumulate, rows):
    """agk_rms_mul_bwd against the multiply's VJP then the RMSNorm VJP of dr, bit for bit, and
    the column sums of a linear layer's bias."""
    import torch
    x, g, gy = device_inputs((rows, cols), dtype, cols, cuda)
    r, inv = agk.rmsnorm_fwd(x, None, EPS)
    y = agk.mul_rowbcast_fwd(r, g)
    assert torch.equal(y, r * g)
    dx0 = torch.full_like(x, 0.5)
    dg0 = torch.full((cols,), 2.0, device=cuda)
    flags = agk.AGK_ACCUM_ALL if accumulate else 0
    dr, dx, dg = agk.rms_mul_bwd(x, g, inv, gy, dx=dx0.clone(), dgamma=dg0.clone(),
                                 accumulate=flags)
    da, db = agk.mul_rowbcast_bwd(gy, r, g, db=dg0.clone(),
                                  accumulate=agk.AGK_ACCUM_DGAMMA if accumulate else 0)
    dx2, _ = agk.rmsnorm_bwd(x, None, inv, da, dx=dx0.clone(), want_dgamma=False,
                             accumulate=agk.AGK_ACCUM_DX if accumulate else 0)
    acc_da, _ = agk.mul_rowbcast_bwd(gy, r, g, da=dx0.clone(), want_db=False,
                                     accumulate=agk.AGK_ACCUM_DX)
    s = agk.sum_rows(gy)
    torch.cuda.synchronize()
    assert torch.equal(dr, da) and torch.equal(dx, dx2) and torch.equal(dg, db)
    if dtype == "f32":
        assert torch.equal(acc_da, dx0 + da)
    else:  # da above is rounded to bf16 before the sum, the accumulated term is not
        assert ((acc_da.float() - (0.5 + da.float())).abs()
                <= 2.0 ** -8 * (0.5 + da.float().abs())).all().item()
    assert ((s.double() - gy.double().sum(0)).abs() <= 1e-5 * gy.double().abs().sum(0)).all().item()


@pytest.mark.parametrize("dtype,cols", [("f32", 5), ("bf16", 9), ("f32", 129), ("bf16", 1001)],
                         ids=str)
def test_many_row_multiply(cuda, dtype, cols):
    """The row-vector multiply over enough rows for its ragged form: torch's product, bit for
    bit, also in place."""
    import torch
    a, b, _ = device_inputs((16411, cols), dtype, cols, cuda)
    want = a * b
    y = agk.mul_rowbcast_fwd(a, b)
    agk.mul_rowbcast_fwd(a, b, y=a)
    torch.cuda.synchronize()
    assert torch.equal(y, want) and torch.equal(a, want)


@pytest.mark.parametrize("dtype,cols", [("f32", 1024), ("bf16", 2048), ("f32", 100),
                                        ("bf16", 8192)], ids=str)
@pytest.mark.parametrize("shift", [1, 3])
def test_rows_off_a_boundary_match_aligned_rows(cuda, dtype, cols, shift):
    """Whole-slot rows whose tensors start `shift` elements off a 16-byte boundary (each at its
    own offset): y, inv_rms and dx are the aligned call's bits (the same lanes add the same
    slots); dgamma's partial rows too."""
    import torch
    rows = 600
    x, g, dy = device_inputs((rows, cols), dtype, cols + shift, cuda)

    def off(t, n):
        buf = torch.empty(t.numel() + n, dtype=t.dtype, device=cuda)[n:]
        return buf.copy_(t.reshape(-1)).view(t.shape)

    y, inv = agk.rmsnorm_fwd(x, g, EPS)
    dx, dg = agk.rmsnorm_bwd(x, g, inv, dy)
    xo, go, do = off(x, shift), off(g, shift + 1), off(dy, 2 * shift)
    yo, invo = agk.rmsnorm_fwd(xo, go, EPS, y=off(y * 0, shift))
    dxo, dgo = agk.rmsnorm_bwd(xo, go, invo, do, dx=off(dx * 0, shift + 2))
    torch.cuda.synchronize()
    for a, b in ((yo, y), (invo, inv), (dxo, dx), (dgo, dg)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,cols", [("f32", 1030), ("bf16", 1001)], ids=str)
def test_infinities_and_nans_stay_where_they_belong(cuda, dtype, cols):
    """An infinite or NaN dy or x in the overlapped columns (which two slots hold): the same
    NaN / infinity pattern as the formula in fp32, other rows and columns untouched."""
    import torch
    x, g, dy = device_inputs((700, cols), dtype, cols, cuda)
    _, _, clean_dx, clean_dg, _ = _ref(x, g, dy)
    dy[3, cols - 3] = float("inf")
    dy[5, cols - 1] = float("nan")
    dy[7, cols - 9] = float("-inf")
    y, inv = agk.rmsnorm_fwd(x, g, EPS)
    dx, dg = agk.rmsnorm_bwd(x, g, inv, dy)
    torch.cuda.synchronize()
    xf, gf, df, r = x.float(), g.float(), dy.float(), inv.view(-1, 1)
    gy = df * gf
    s = (r * r * (gy * xf).sum(-1, keepdim=True)) / cols
    want = r * (gy - xf * s)
    assert torch.equal(torch.isnan(dx), torch.isnan(want))
    assert torch.equal(torch.isinf(dx), torch.isinf(want))
    rows = [i for i in range(700) if i not in (3, 5, 7)]
    bar = (1e-5 + (2.0 ** -8 if dtype == "bf16" else 0.0)) * clean_dx.abs().amax()
    assert ((dx[rows].double() - clean_dx[rows]).abs() <= bar).all().item()
    bad = [cols - 9, cols - 3, cols - 1]
    assert not torch.isfinite(dg[bad]).any().item()
    good = torch.ones(cols, dtype=torch.bool, device=cuda)
    good[bad] = False
    assert torch.isfinite(dg[good]).all().item()


ROWOP_COLS = {"f32": [4, 5, 9, 61, 253, 515, 1001, 4099, 8195, 16383],
              "bf16": [8, 9, 121, 1001, 4099, 8195, 16391, 32767]}


# rows 4100: enough for the ragged form at every width that is looped in few rows
@pytest.mark.parametrize("dtype,cols,rows", [(d, c, r) for d in ROWOP_COLS for c in ROWOP_COLS[d]
                                             for r in (1, 541, 4100) if r < 4100 or c < 1025],
                         ids=str)
def test_row_ops_match_fp64(cuda, dtype, cols, rows):
    """LayerNorm, softmax and log-sum-exp, the RMSNorm JVP, with masked logits in the overlapped
    columns.  Bars: 1e-5 of the row's scale (fp32 sums and the hardware exponential's
    |z - max| 2^-24 ln 2), one storage rounding for bf16."""
    import torch
    print(f"{dtype} {rows}x{cols}", flush=True)
    x, g, dy = device_inputs((rows, cols), dtype, rows * 13 + cols, cuda)
    one = 2.0 ** -8 if dtype == "bf16" else 0.0
    bar = 1e-5 + one

    def close(got, want, scale, what):
        assert ((got.double() - want).abs() <= bar * scale + 1e-30).all().item(), what

    def accumulates(call, fresh, what):
        pre = torch.full_like(x, 0.25)
        got = call(pre.clone())
        torch.cuda.synchronize()
        if dtype == "f32":
            assert torch.equal(got, pre + fresh), what
        else:  # the accumulated term is not rounded to bf16 first
            f = fresh.float()
            assert ((got.float() - (0.25 + f)).abs() <= 2.0 ** -8 * (0.25 + f.abs())).all().item()

    x64, d64, g64 = x.double(), dy.double(), g.double()
    y, mean, rstd = agk.layernorm_fwd(x, 1e-5)
    dx = agk.layernorm_bwd(x, mean, rstd, dy)
    m = x64.mean(-1, keepdim=True)
    r = ((x64 - m).square().mean(-1, keepdim=True) + 1e-5).rsqrt()
    xh = (x64 - m) * r
    close(y, xh, xh.abs().amax(-1, keepdim=True), "layernorm")
    want = r * (d64 - d64.mean(-1, keepdim=True) - xh * (d64 * xh).mean(-1, keepdim=True))
    # |dx| <= r (2 + max|xh|) max|dy| (mean |xh| <= 1): the scale its rounding is relative to
    close(dx, want, r * (2 + xh.abs().amax(-1, keepdim=True)) * d64.abs().amax(-1, keepdim=True),
          "layernorm dx")
    accumulates(lambda o: agk.layernorm_bwd(x, mean, rstd, dy, dx=o, accumulate=True), dx, "ln acc")

    _, inv = agk.rmsnorm_fwd(x, g, EPS)
    ty = agk.rmsnorm_jvp(x, g, inv, dy, tgamma=g)
    ri = inv.double().view(-1, 1)
    want = g64 * ri * (d64 - x64 * ri.square() * (d64 * x64).mean(-1, keepdim=True)) + g64 * x64 * ri
    # the same bound for each of the rule's two terms
    xr = (x64 * ri).abs().amax(-1, keepdim=True)
    close(ty, want, 1.5 * (ri * (1 + xr) * d64.abs().amax(-1, keepdim=True) + 1.5 * xr), "jvp")

    z = (x * 3).contiguous()
    z[:, -2:] = float("-inf")   # columns that two slots hold
    z64 = z.double()
    for ws in (False, None):
        s = agk.softmax_fwd(z, workspace=ws)
        dz = agk.softmax_bwd(s, dy, workspace=ws)
        p = torch.softmax(z64, -1)
        close(s, p, p.amax(-1, keepdim=True), "softmax")
        s64 = s.double()
        want = s64 * (d64 - (s64 * d64).sum(-1, keepdim=True))
        close(dz, want, (s64 * d64.abs().amax(-1, keepdim=True)).amax(-1, keepdim=True) * 2, "softmax dz")
        dl = dy[:, :1].contiguous()
        lb = agk.logsumexp_bwd(z, dl, workspace=ws)
        close(lb, dl.double() * p, dl.double().abs() * p.amax(-1, keepdim=True), "lse dz")
    accumulates(lambda o: agk.softmax_bwd(s, dy, dz=o, accumulate=True), dz, "softmax acc")
    lse, keep = agk.logsumexp_fwd_keep(z)
    want = torch.logsumexp(z64, -1, keepdim=True)
    assert ((keep.double() - want).abs() <= 1e-5 * (1 + want.abs())).all().item()
    assert ((lse.double() - want).abs() <= bar * (1 + want.abs())).all().item()
    jv = agk.logsumexp_jvp(z, dy)
    want = (p * d64).sum(-1, keepdim=True)
    assert ((jv.double() - want).abs() <= bar * (p * d64.abs()).sum(-1, keepdim=True)).all().item()
    in_place = z.clone()
    agk.softmax_fwd(in_place, y=in_place)
    torch.cuda.synchronize()
    assert torch.equal(in_place, agk.softmax_fwd(z))


@pytest.mark.parametrize("dtype,rows,cols", [("f32", 60001, 131), ("f32", 30000, 2051),
                                             ("f32", 5000, 9001), ("bf16", 60001, 95),
                                             ("bf16", 9000, 4099)], ids=str)
def test_column_gradients_of_many_rows(cuda, dtype, rows, cols):
    """dgamma, the row-vector multiply's db and the column sums: fp64 sums in 256 partial rows,
    each rounded to fp32, and the total rounded again.  A rounding is at most 2^-24 relative,
    0.42 of that in the root mean square, so the two together stay under 2^-24 of the result in
    the 2-norm over the columns; dgamma's terms hold one rounding more each (x times inv_rms).
    fp32 sums of the same rows are two to four times further off."""
    import torch
    x, g, dy = device_inputs((rows, cols), dtype, rows + cols, cuda)
    _, inv = agk.rmsnorm_fwd(x, None, EPS)
    _, dg = agk.rmsnorm_bwd(x, g, inv, dy, want_dx=False)
    _, db = agk.mul_rowbcast_bwd(dy, x, g, want_da=False)
    s = agk.sum_rows(x)
    torch.cuda.synchronize()
    x64, d64 = x.double(), dy.double()
    for got, terms, roundings in ((dg, d64 * (x64 * inv.double().view(-1, 1)), 1), (db, d64 * x64, 0),
                                  (s, x64, 0)):
        want = terms.sum(0)
        bound = 2.0 ** -24 * (want.norm() + roundings * terms.norm())
        assert (got.double() - want).norm() <= bound
