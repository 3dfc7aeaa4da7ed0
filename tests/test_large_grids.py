"""Calls whose kernels would need more lanes along a grid dimension than HIP launches (2^32 - 1):
tall narrow products and tall ragged rows.  They run in fewer workgroups, or on another kernel.
Values are checked at both ends of the tensors and where the rows first leave the grid."""
import pytest

import cgadimpl_amd as agk


def _windows(rows, edge):
    return [slice(0, 4096), slice(edge - 2048, edge + 2048), slice(rows - 4096, rows)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,cols", [("f32", 4), ("bf16", 8)])
def test_scalar_per_row_product_of_2_28_rows(cuda, dtype, cols):
    """16 lanes a row: 2^28 rows are 2^32 lanes."""
    import torch
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    rows = 2 ** 28 + 16
    gen = torch.Generator(device=cuda)
    gen.manual_seed(cols)
    print("mul_bcast", dtype, rows, cols, flush=True)
    a = torch.empty(rows, cols, device=cuda, dtype=dt).normal_(generator=gen)
    b = torch.empty(rows, 1, device=cuda, dtype=dt).normal_(generator=gen)
    y = agk.mul_bcast_fwd(a, b)
    da, db = agk.mul_bcast_bwd(a, a, b)
    torch.cuda.synchronize()
    for w in _windows(rows, 2 ** 28):
        assert torch.equal(y[w], a[w] * b[w])
        assert torch.equal(da[w], a[w] * b[w])
        # an fp64 sum of exact products, rounded once
        ref = (a[w].double() ** 2).sum(1, keepdim=True)
        assert ((db[w].double() - ref).abs() <= 2.0 ** -24 * ref + 1e-30).all().item()


@pytest.mark.gpu
def test_ragged_rows_by_the_million(cuda):
    """512 lanes a row of 2051 floats: 2^23 rows are 2^32 lanes (in place: one 69 GB tensor)."""
    import torch
    rows, cols = 2 ** 23 + 8, 2051
    print("softmax and rmsnorm in place", rows, cols, flush=True)
    x = torch.empty(rows, cols, device=cuda)
    x.copy_((torch.arange(rows, device=cuda) % 7 - 3.0).unsqueeze(1).expand(rows, cols))
    x[:, 0] += 1.0
    probe = [x[w].double().clone() for w in _windows(rows, 2 ** 23 - 4096)]
    agk.softmax_fwd(x, y=x, workspace=False)
    torch.cuda.synchronize()
    for w, z in zip(_windows(rows, 2 ** 23 - 4096), probe):
        ref = torch.softmax(z, -1)
        assert ((x[w].double() - ref).abs() <= 1e-5 * ref).all().item()
    probe = [x[w].double().clone() for w in _windows(rows, 2 ** 23 - 4096)]
    agk.rmsnorm_fwd(x, None, 1e-6, y=x)
    torch.cuda.synchronize()
    for w, z in zip(_windows(rows, 2 ** 23 - 4096), probe):
        ref = z * (z.square().mean(-1, keepdim=True) + 1e-6).rsqrt()
        assert ((x[w].double() - ref).abs() <= 1e-5 * ref.abs()).all().item()


@pytest.mark.gpu
def test_f32_outer_product_of_2_29_columns(cuda):
    """32 x 32 tiles of 256 lanes: 2^29 columns are 2^32 lanes."""
    import torch
    N = 2 ** 29 + 40
    gen = torch.Generator(device=cuda)
    gen.manual_seed(3)
    a = torch.randn(2, 1, generator=gen, device=cuda)
    b = torch.empty(1, N, device=cuda).normal_(generator=gen)
    print("gemm_f32", 2, N, 1, flush=True)
    c = agk.gemm_f32(a, b)
    torch.cuda.synchronize()
    for w in _windows(N, 2 ** 29):
        assert torch.equal(c[:, w], a * b[:, w])


@pytest.mark.gpu
def test_bf16_product_of_2_30_rows(cuda):
    """64 x 64 tiles of 256 lanes: 2^30 rows are 2^32 lanes."""
    import torch
    M = 2 ** 30 + 64
    gen = torch.Generator(device=cuda)
    gen.manual_seed(4)
    a = torch.empty(M, 8, device=cuda, dtype=torch.bfloat16)
    pattern = torch.randn(8184, 8, generator=gen, device=cuda).bfloat16()
    whole = M // 8184 * 8184
    a[:whole].view(-1, 8184, 8).copy_(pattern.expand(M // 8184, 8184, 8))
    a[whole:].copy_(pattern[:M - whole])
    b = torch.randn(8, 8, generator=gen, device=cuda).bfloat16()
    print("gemm_bf16", M, 8, 8, flush=True)
    c = agk.gemm_bf16(a, b)
    torch.cuda.synchronize()
    want = agk.gemm_bf16(pattern, b)  # the ordinary grid
    assert torch.equal(c[:whole].view(-1, 8184, 8), want.expand(M // 8184, 8184, 8))
    assert torch.equal(c[whole:], want[:M - whole])
    ref = pattern.float() @ b.float()
    assert ((want.float() - ref).abs().max() / ref.abs().max()).item() <= 8e-3
