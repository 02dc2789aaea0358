"""Uploads of a step's plan by a kernel that reads the pinned arena."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 2047, 16383, 16384, 16385, 300007, (1 << 20) + 8])
def test_bytes_arrive_again_and_again(n):
    """Odd sizes, both sides of the engine's limit, and new bytes in the same memory: a cache must not hold the old ones."""
    from kafka_llm_service_amd import ops

    arena = torch.zeros(n + 512, dtype=torch.uint8, pin_memory=True)
    src, dst = arena[256:256 + n], torch.zeros(n + 64, dtype=torch.uint8, device="cuda")
    g = torch.Generator().manual_seed(n)
    for _ in range(3):
        src.random_(generator=g)
        want = src.clone()
        if n <= ops.HOST_COPY_MAX:
            assert ops.ext().host_copy(dst[:n], src)   # (the kernel itself: a copy engine's copy would pass as well)
        else:
            ops.host_copy(dst[:n], src)
        torch.cuda.synchronize()
        assert torch.equal(dst[:n].cpu(), want) and not dst[n:].any()


def test_memory_that_is_not_pinned_goes_the_other_way():
    from kafka_llm_service_amd import ops

    src, dst = torch.arange(200, dtype=torch.uint8), torch.zeros(200, dtype=torch.uint8, device="cuda")
    assert not ops.ext().host_copy(dst, src) and not dst.any()
    ops.host_copy(dst, src)
    assert torch.equal(dst.cpu(), src)


def test_arena_given_back_before_the_copy_ran():
    """A pinned block that is freed while the copy waits behind other work is not handed out again before it ran."""
    from kafka_llm_service_amd import ops

    n = 100000
    a = torch.randn(4096, 4096, device="cuda")
    src = torch.full((n,), 7, dtype=torch.uint8, pin_memory=True)
    dst = torch.zeros(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    for _ in range(20):
        a = a @ a * 1e-3
    assert ops.ext().host_copy(dst, src)
    del src
    torch.full((n,), 9, dtype=torch.uint8, pin_memory=True)
    torch.cuda.synchronize()
    assert bool((dst == 7).all())
