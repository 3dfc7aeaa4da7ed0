"""Parity of the general broadcast multiply (agk_mul_bcast_fwd / _bwd) with the
pinned oracle (oracle/rowops.py: mul_bcast_fwd, mul_bcast_vjp).

Bars:
  - the forward and the gradient of an operand with the output's shape are one
    product (plus, when accumulating, one add) rounded to storage: bit-exact
    against the oracle's float32 arithmetic (bf16: rounded to bf16 bits);
  - the gradient of a broadcast operand is a float64 sum of exact products
    rounded to float32 once; the device sums in another order, so the result
    may differ in the last float32 place: relative error <= 2^-22 (two float32
    ulps) per element, against the oracle's float64 sum;
  - results are identical run to run.
Shapes cover every broadcast form (missing axes, extent-1 axes, both operands
reduced, 0-d scalars, long reductions that take the 256-lane reduction, empty
outputs) in fp32 and bf16.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import cgadimpl_amd as agk
from gpu_util import to_dev, to_host
from oracle import rowops as ro
from tolerances import TOL_F32

pytestmark = pytest.mark.gpu

PAIRS = [
    ((3, 4), (3, 4)),
    ((3, 4), (4,)),
    ((7, 1), (1, 9)),
    ((2, 3, 4), (2, 1, 4)),
    ((2, 3, 4), (3, 1)),
    ((1,), (5, 6)),
    ((), (5, 6)),
    ((2, 1, 3, 1), (1, 4, 1, 5)),
    ((4, 33, 130), (4, 1, 130)),
    ((6, 700, 3), (1, 700, 1)),        # long sums for b (256-lane reduction)
    ((1, 1), (5000, 3)),               # a summed over 15000 products
    ((64, 1, 96), (64, 40, 1)),
    ((8, 64, 96), (1, 1, 96)),         # column sums whose quarters cross outer positions
    ((6, 5, 4, 32), (6, 1, 1, 32)),    # two reduced axes between kept ones
    ((4, 33, 128), (4, 1, 128)),       # 16-byte forward in bf16 too
]
REL = 2.0 ** -22


def _operands(sa, sb, seed, dtype):
    g = np.random.default_rng(seed)
    out = np.broadcast_shapes(sa, sb)
    a = g.standard_normal(sa).astype(np.float32)
    b = g.standard_normal(sb).astype(np.float32)
    gy = g.standard_normal(out).astype(np.float32)
    if dtype == "bf16":  # (bf16_encode makes a 0-d array 1-d: reshape back)
        return tuple(oracle.bf16_encode(t).reshape(t.shape) for t in (gy, a, b))
    return gy, a, b


def _f32(t):  # (bf16_decode makes a 0-d array 1-d: reshape back)
    return oracle.bf16_decode(t).reshape(t.shape) if t.dtype == np.uint16 else t


def _check_grad(got, ref64, full, dtype, what):
    if full:  # product rounded to storage
        want = ref64.astype(np.float32)
        if dtype == "bf16":
            want = oracle.bf16_encode(want)
        assert got.dtype == want.dtype and got.shape == want.shape, what
        assert np.array_equal(got, want), what
    else:
        assert got.dtype == np.float32 and got.shape == ref64.shape, what
        err = np.abs(got.astype(np.float64) - ref64)
        assert np.all(err <= REL * np.abs(ref64) + 1e-30), (what, float(err.max()))


def _is_full(shape, out):
    return (1,) * (len(out) - len(shape)) + tuple(shape) == tuple(out)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("sa,sb", PAIRS, ids=lambda v: str(v))
def test_forward_and_vjp_match_oracle(cuda, sa, sb, dtype):
    gy, a, b = _operands(sa, sb, 11, dtype)
    out = np.broadcast_shapes(sa, sb)
    # (np.ascontiguousarray, inside to_dev, makes a 0-d array 1-d: reshape back)
    ad, bd, gyd = to_dev(a, cuda).reshape(sa), to_dev(b, cuda).reshape(sb), to_dev(gy, cuda)
    print(f"bcast {dtype} a{sa} b{sb}", flush=True)
    assert agk.mul_bcast_shape(sa, sb) == tuple(out)
    y = to_host(agk.mul_bcast_fwd(ad, bd))
    want = ro.mul_bcast_fwd(_f32(a), _f32(b))
    if dtype == "bf16":
        want = oracle.bf16_encode(want)
    assert y.shape == tuple(out) and np.array_equal(y, want)
    da, db = agk.mul_bcast_bwd(gyd, ad, bd)
    ra, rb = ro.mul_bcast_vjp(_f32(gy), _f32(a), _f32(b))
    _check_grad(to_host(da), ra, _is_full(sa, out), dtype, "da")
    _check_grad(to_host(db), rb, _is_full(sb, out), dtype, "db")
    # run to run
    da2, db2 = agk.mul_bcast_bwd(gyd, ad, bd)
    assert np.array_equal(to_host(da2), to_host(da)) and np.array_equal(to_host(db2), to_host(db))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_accumulation(cuda, dtype):
    sa, sb = (4, 33, 130), (4, 1, 130)
    gy, a, b = _operands(sa, sb, 12, dtype)
    ad, bd, gyd = to_dev(a, cuda), to_dev(b, cuda), to_dev(gy, cuda)
    import torch
    da0 = to_dev(_operands(sa, sa, 13, dtype)[1], cuda)            # prior gradient of a
    db0 = torch.from_numpy(np.random.default_rng(14).standard_normal(sb).astype(np.float32)).to(cuda)
    pre_a, pre_b = to_host(da0).copy(), to_host(db0).copy()
    da, db = agk.mul_bcast_bwd(gyd, ad, bd, da=da0, db=db0, accumulate=True)
    ra, rb = ro.mul_bcast_vjp(_f32(gy), _f32(a), _f32(b))
    # full operand: old + product, each rounded to storage (float32 arithmetic)
    prod = ra.astype(np.float32)
    if dtype == "bf16":
        prod = _f32(oracle.bf16_encode(prod))
        want = oracle.bf16_encode(_f32(pre_a) + prod)
    else:
        want = pre_a + prod
    assert np.array_equal(to_host(da), want)
    # broadcast operand: old + float64 sum, rounded once
    ref = pre_b.astype(np.float64) + rb
    got = to_host(db).astype(np.float64)
    assert np.all(np.abs(got - ref) <= REL * np.abs(ref) + 1e-30)
    # forward accumulation: y += a * b
    y0 = to_dev(_operands(sa, sa, 15, dtype)[1], cuda)
    pre_y = to_host(y0).copy()
    y = to_host(agk.mul_bcast_fwd(ad, bd, y=y0, accumulate=True))
    p = ro.mul_bcast_fwd(_f32(a), _f32(b))
    if dtype == "bf16":
        want = oracle.bf16_encode(_f32(pre_y) + _f32(oracle.bf16_encode(p)))
    else:
        want = pre_y + p
    assert np.array_equal(y, want)


def test_empty_output_gives_zero_gradients(cuda):
    """a [3, 0, 4] * b [3, 1, 4]: the output is empty and b's gradient is an
    empty sum, zeros.  (The reference's reduce_for_broadcast sums only axes
    whose extent is above 1, so it cannot reshape this case; the kernel gives
    the mathematical answer.)"""
    import torch
    a = torch.zeros(3, 0, 4, device=cuda)
    b = torch.ones(3, 1, 4, device=cuda)
    gy = torch.zeros(3, 0, 4, device=cuda)
    assert agk.mul_bcast_fwd(a, b).shape == (3, 0, 4)
    db0 = torch.full((3, 1, 4), 7.0, device=cuda)
    da, db = agk.mul_bcast_bwd(gy, a, b, db=db0)
    assert da.shape == (3, 0, 4) and db.dtype == torch.float32
    assert torch.count_nonzero(db).item() == 0
    db1 = torch.full((3, 1, 4), 7.0, device=cuda)
    _, db = agk.mul_bcast_bwd(gy, a, b, db=db1, want_da=False, accumulate=True)
    assert torch.all(db == 7.0).item()


def test_rejects_incompatible_shapes(cuda):
    import torch
    a = torch.zeros(3, 4, device=cuda)
    b = torch.zeros(2, 4, device=cuda)
    with pytest.raises(RuntimeError, match="AGK_EINVAL"):
        agk.mul_bcast_fwd(a, b, y=torch.zeros(3, 4, device=cuda))
    with pytest.raises(RuntimeError, match="AGK_EINVAL"):
        agk.mul_bcast_shape((2, 3, 4, 5, 6, 7, 8, 9, 10), (1,))   # more than 8 axes


def test_row_vector_cases_agree_with_the_row_kernels(cuda):
    """The row-vector broadcast has its own kernels (agk_mul_rowbcast_*); the
    general path must give the same bits for it."""
    gy, a, b = _operands((300, 257), (257,), 21, "f32")
    ad, bd, gyd = to_dev(a, cuda), to_dev(b, cuda), to_dev(gy, cuda)
    y1 = to_host(agk.mul_bcast_fwd(ad, bd))
    y2 = to_host(agk.mul_rowbcast_fwd(ad, bd))
    assert np.array_equal(y1, y2)
    da1, db1 = agk.mul_bcast_bwd(gyd, ad, bd)
    da2, db2 = agk.mul_rowbcast_bwd(gyd, ad, bd)
    assert np.array_equal(to_host(da1), to_host(da2))
    r = ro.mul_bcast_vjp(gy, a, b)[1]
    # the general kernel: two float32 ulps of the float64 sum; the row kernel
    # sums float32 partial rows first and is held to its own dgamma bar
    # (1e-5 of the largest column sum, tests/tolerances.py)
    g1, g2 = to_host(db1).astype(np.float64), to_host(db2).astype(np.float64)
    assert np.all(np.abs(g1 - r) <= REL * np.abs(r) + 1e-30)
    assert np.max(np.abs(g2 - r)) <= TOL_F32 * np.max(np.abs(r))


# rows x cols views: a vector per group of rows (one, few and many rows; one batch, a
# remainder, both), a scalar per row, and shapes just outside them
VIEW_SHAPES = [((5, 37, 61), (5, 1, 61)), ((3, 9, 8), (3, 1, 8)), ((2, 300, 129), (300, 129)),
               ((300, 17), (1, 17)), ((3, 1000, 1031), (3, 1, 1031)), ((2, 64, 4096), (2, 1, 4096)),
               ((33, 2051), (1, 2051)), ((7, 33, 5), (7, 33, 1)), ((4100, 40), (4100, 1)),
               ((2, 3, 20001), (2, 3, 1)), ((1500, 300), (1500, 1)), ((1030,), (1,)),
               ((40, 3), (40, 1)), ((2, 3, 4, 32), (2, 1, 4, 32)), ((70000, 9), (70000, 1)),
               # rows of 8 chunks and more (an odd and a whole number of them), by one vector and
               # by a scalar per row; a group of 70 rows in few tiles; tiny and large tensors,
               # where the general kernels take over and where loads pass the caches by
               ((5, 80001), (1, 80001)), ((3, 131072), (131072,)), ((3, 90003), (3, 1)),
               ((20, 70, 33), (20, 1, 33)), ((2, 70, 515), (2, 1, 515)), ((3, 5, 4096), (5, 4096)),
               ((16, 2200000), (2200000,)), ((70001, 1030), (70001, 1)), ((9, 4, 2000001), (9, 4, 1))]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shapes", VIEW_SHAPES, ids=str)
@pytest.mark.parametrize("swap", [False, True])
def test_row_views_match_torch(cuda, dtype, shapes, swap):
    """Products and full gradients: torch's element-wise product, bit for bit; sums: fp64 sums of
    exact products rounded once (2^-24 relative, plus fp64 rounding of the terms' magnitude);
    one operand's gradient alone and accumulation."""
    import torch
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    gen = torch.Generator(device=cuda)
    gen.manual_seed(sum(shapes[0]))
    a = torch.randn(*shapes[0], generator=gen, device=cuda).to(dt)
    b = torch.randn(*shapes[1], generator=gen, device=cuda).to(dt)
    if swap:
        a, b = b, a
    want = a * b
    gy = torch.randn(want.shape, generator=gen, device=cuda).to(dt)
    full, vec = (b, a) if swap else (a, b)
    y = agk.mul_bcast_fwd(a, b)
    assert torch.equal(y, want)
    da, db = agk.mul_bcast_bwd(gy, a, b)
    d_full, d_vec = (db, da) if swap else (da, db)
    assert torch.equal(d_full, gy * vec)
    axes = [i for i in range(want.dim())
            if i < want.dim() - vec.dim() or vec.shape[i - want.dim() + vec.dim()] != want.shape[i]]
    terms = gy.double() * full.double()
    ref = terms.sum(axes, keepdim=True).reshape(vec.shape)
    mag = terms.abs().sum(axes, keepdim=True).reshape(vec.shape)
    assert ((d_vec.double() - ref).abs() <= 2.0 ** -24 * ref.abs() + 1e-13 * mag).all().item()
    # each gradient alone, and added to what is there
    only_a, _ = agk.mul_bcast_bwd(gy, a, b, want_db=False)
    _, only_b = agk.mul_bcast_bwd(gy, a, b, want_da=False)
    assert torch.equal(only_a, da) and torch.equal(only_b, db)
    pre_a, pre_b = torch.full_like(da, 0.5), torch.full_like(db, 0.5)
    acc_a, acc_b = agk.mul_bcast_bwd(gy, a, b, da=pre_a.clone(), db=pre_b.clone(),
                                     accumulate=agk.AGK_ACCUM_ALL)
    torch.cuda.synchronize()
    acc_full, acc_vec = (acc_b, acc_a) if swap else (acc_a, acc_b)
    assert torch.equal(acc_full, 0.5 + d_full)
    assert ((acc_vec.double() - (0.5 + ref)).abs()
            <= 2.0 ** -24 * (0.5 + ref).abs() + 1e-13 * mag).all().item()
    # an output over an operand: the same product
    in_place = full.clone()
    args = (a, in_place) if swap else (in_place, b)
    agk.mul_bcast_fwd(*args, y=in_place)
    torch.cuda.synchronize()
    assert torch.equal(in_place, want)


@pytest.mark.parametrize("shape,vec", [((64, 1025), (1, 1025)), ((3, 40, 2051), (3, 1, 2051)),
                                       ((700, 1025), (1, 1025)), ((5, 9, 130), (5, 9, 1))], ids=str)
@pytest.mark.parametrize("accumulate", [False, True])
def test_gradient_written_over_the_broadcast_operand(cuda, shape, vec, accumulate):
    """db over b (fp32), at widths whose last 16-byte slot reaches back into the columns of the
    slot before it: da is made of the b that the call was given, bit for bit, and db is the sum
    (added to b where it accumulates), as two passes in order give them."""
    import torch
    gen = torch.Generator(device=cuda)
    gen.manual_seed(shape[-1] + len(shape))
    a, b, gy = (torch.randn(*s, generator=gen, device=cuda) for s in (shape, vec, shape))
    over = b.clone()
    da, db = agk.mul_bcast_bwd(gy, a, over, db=over, accumulate=agk.AGK_ACCUM_DGAMMA * accumulate)
    torch.cuda.synchronize()
    assert db.data_ptr() == over.data_ptr()
    assert torch.equal(da, gy * b)
    axes = [i for i in range(len(shape)) if vec[i] != shape[i]]
    terms = gy.double() * a.double()
    ref = terms.sum(axes, keepdim=True) + (b.double() if accumulate else 0.0)
    # an fp64 sum of exact products, rounded once
    mag = terms.abs().sum(axes, keepdim=True) + b.double().abs()
    assert ((db.double() - ref).abs() <= 2.0 ** -24 * ref.abs() + 1e-13 * mag).all().item()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shape,vec", [((4, 700, 96), (4, 1, 96)), ((300, 1025), (1, 1025)),
                                       ((6, 50, 77), (6, 50, 1))], ids=str)
def test_bits_do_not_depend_on_where_the_operands_lie(cuda, dtype, shape, vec):
    """The broadcast operand right below y and da in one buffer, or far from them: the same
    kernels, so the same bits in the product and both gradients."""
    import math
    import torch
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    gen = torch.Generator(device=cuda)
    gen.manual_seed(shape[-1])
    b = torch.randn(vec, generator=gen, device=cuda).to(dt)
    # terms of many magnitudes that cancel along the summed axes: what is left of an fp64 sum is
    # its rounding, which shows the order of the terms
    a = torch.randn(shape, generator=gen, device=cuda)
    a *= 2.0 ** torch.randint(-30, 31, shape, generator=gen, device=cuda)
    axis = [i for i in range(len(shape)) if vec[i] != shape[i]][0]
    a = (a - a.flip(axis)).to(dt)
    gy = torch.ones_like(a)
    n, m = math.prod(shape), math.prod(vec)
    far = torch.empty(64 * n, device=cuda, dtype=dt)  # b, then 62 tensors of room, then y

    def run(at):
        bb, out = far[:m].view(vec), far[at:at + n].view(shape)
        bb.copy_(b)
        y = agk.mul_bcast_fwd(a, bb, y=out).clone()
        da, db = agk.mul_bcast_bwd(gy, a, bb, da=out)
        torch.cuda.synchronize()
        return y, da.clone(), db.clone()

    near, apart = run(m), run(62 * n)
    for got, want in zip(near, apart):
        assert torch.equal(got, want)
    assert torch.equal(near[0], a * b) and torch.equal(near[1], gy * b)
