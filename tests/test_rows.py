"""Rows picked by an index, with and without a norm (csrc/norm_act.hip: ops.embed_rmsnorm, rows_add_rmsnorm, gather_rows)."""
import pytest
import torch

from kafka_llm_service_amd import ops


def _check(dev, dtype):
    """The same as the separate operations, to the last bit (on the GPU the same sums and roundings)."""
    g = torch.Generator().manual_seed(2)
    for d, n in ((64, 3), (2048, 1), (4096, 7), (5120, 2), (16384, 2)):
        table = torch.randn(11, d, generator=g).to(dtype).to(dev)
        w = torch.rand(d, generator=g).to(dtype).to(dev)
        idx = torch.randint(0, 11, (n,), generator=g).to(dev)
        r, x = ops.embed_rmsnorm(table, idx, w, 1e-5)
        assert torch.equal(r, table[idx]) and torch.equal(x, ops.rmsnorm(table[idx], w, 1e-5))
        res = torch.randn(11, d, generator=g).to(dtype).to(dev)
        for delta in [torch.randn(11, d, generator=g).to(dtype)] + [torch.randn(s, 11, d, generator=g) for s in (1, 2, 3, 8)]:
            delta, keep = delta.to(dev), res.clone()
            slab = ops.is_slab(delta)
            want = ops.fused_add_rmsnorm(delta.index_select(1 if slab else 0, idx), res.index_select(0, idx), w, 1e-5)
            assert torch.equal(ops.rows_add_rmsnorm(delta, res, idx, w, 1e-5), want) and torch.equal(res, keep)
        for t in (table, table.float(), torch.randn(11, d + 8, generator=g).to(dev)[:, :d], torch.randn(11, d + 1, generator=g).to(dev)[:, 1:]):
            assert torch.equal(ops.gather_rows(t, idx), t[idx])
    for i in (idx.int(), idx.repeat_interleave(2)[::2]):     # indices that the kernels do not read
        assert torch.equal(ops.gather_rows(table, i), table[idx]) and torch.equal(ops.embed_rmsnorm(table, i, w, 1e-5)[0], table[idx])
        assert torch.equal(ops.rows_add_rmsnorm(table, res, i, w, 1e-5), ops.rows_add_rmsnorm(table, res, idx, w, 1e-5))
    none = torch.zeros(0, dtype=torch.int64, device=dev)
    assert ops.gather_rows(table, none).shape == (0, 16384) and ops.rows_add_rmsnorm(table, res, none, w, 1e-5).shape == (0, 16384)


def test_on_the_cpu():
    _check("cpu", torch.float32)


@pytest.mark.gpu
def test_on_the_gpu():
    _check("cuda", torch.bfloat16)
    table, w = torch.randn(5, 4096, device="cuda").to(torch.bfloat16), torch.ones(4096, device="cuda", dtype=torch.bfloat16)
    idx = torch.tensor([4, 5, -1, 0], device="cuda")    # rows outside the table come out as NaN, the others as they are
    r, x = ops.embed_rmsnorm(table, idx, w, 1e-5)
    f = ops.gather_rows(table.float(), idx)
    y = ops.rows_add_rmsnorm(table, table, idx, w, 1e-5)
    for t in (r, x, f, y):
        assert torch.isnan(t[1:3]).all() and torch.isfinite(t[0]).all() and torch.isfinite(t[3]).all()
    assert torch.equal(r[[0, 3]], table[[4, 0]])


@pytest.mark.parametrize("dev,dtype", [("cpu", torch.float32), pytest.param("cuda", torch.bfloat16, marks=pytest.mark.gpu)])
def test_weights_and_slabs_that_the_kernels_do_not_read(dev, dtype):
    """A norm's weight that starts between two 16-byte pieces, and slabs that are a view: the separate operations take them."""
    g = torch.Generator().manual_seed(4)
    table, w = torch.randn(11, 256, generator=g).to(dtype).to(dev), torch.rand(257, generator=g).to(dtype).to(dev)[1:]
    idx = torch.randint(0, 11, (5,), generator=g).to(dev)
    r, x = ops.embed_rmsnorm(table, idx, w, 1e-5)
    assert torch.equal(r, table[idx]) and torch.equal(x, ops.rmsnorm(table[idx], w, 1e-5))
    want = ops.fused_add_rmsnorm(table[idx], table[idx], w, 1e-5)
    assert torch.equal(ops.rows_add_rmsnorm(table, table, idx, w, 1e-5), want)
    even, wide = w.clone(), torch.randn(2, 14, 256, generator=g).to(dev)[:, 1:12]
    want = ops.fused_add_rmsnorm(wide.index_select(1, idx), table[idx], even, 1e-5)
    assert torch.equal(ops.rows_add_rmsnorm(wide, table, idx, even, 1e-5), want)


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("d", [4, 64, 4096, 4104, 5000])
def test_rows_gathered_twice(dev, d):
    """The second output in the rows' type and in bf16, whole, as a part of wider rows, and where the kernel does not write it."""
    g = torch.Generator().manual_seed(d)
    table = torch.randn(9, d, generator=g).to(dev)
    idx = torch.randint(0, 9, (5,), generator=g).to(dev)
    for also in (torch.empty(5, d, device=dev), torch.empty(5, d, device=dev, dtype=torch.bfloat16),
                 torch.empty(5, 2 * d, device=dev, dtype=torch.bfloat16)[:, d:], torch.empty(5, d + 3, device=dev)[:, 3:],
                 torch.empty(5, d, device=dev, dtype=torch.float16)):
        assert torch.equal(ops.gather_rows(table, idx, also), table[idx]) and torch.equal(also, table[idx].to(also.dtype))


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [8, 100, 1000, 4096, 5000])
def test_layer_norm_of_picked_rows(dev, dtype, d):
    """As of the rows picked before, to the last bit, for every row length's kernel and those without one."""
    from kafka_llm_service_amd.ops import hybrid as hops

    g = torch.Generator().manual_seed(d)
    x = torch.randn(40, d, generator=g).to(dev)
    w, b = (torch.randn(d, generator=g).to(dtype).to(dev) for _ in range(2))
    for idx in (torch.tensor([39]), torch.randint(0, 40, (25,), generator=g), torch.randint(0, 40, (600,), generator=g)):
        got, want = (torch.empty(len(idx), d, dtype=dtype, device=dev) for _ in range(2))
        hops.ln_rows(x, idx.to(dev), w, b, 1e-6, got)
        hops.ln_shift(x.index_select(0, idx.to(dev)), w, b, 1e-6, want)
        assert torch.equal(got, want)
