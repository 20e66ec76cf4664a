"""fastmax_forward_static (the entry point that allocates nothing: its workspace is a static device
array inside the library) against fastmax_forward, through the C ABI: same kernels on the same inputs,
so the results must be the same bits.  Two calls in a row, the second on a smaller problem (the buffer
still holds the first call's contents), then a problem with moment states, then the size limit."""
import ctypes as C
import math

import pytest
import torch

from reproducing_fastmax_results_amd import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    return _capi.get_lib()


def _pair(lib, bh, n, d, dtype, seed, first=False, **kw):
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(bh, n, d, generator=gen).to(dtype).to(DEV) for _ in range(3))
    o1, g1 = lib.forward(q, k, v, **kw)
    o2 = torch.full_like(o1, float("nan"))
    g2 = torch.full_like(g1, float("nan"))
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    free_before = torch.cuda.mem_get_info()[0]               # the driver's own count of free device memory
    lib.forward_static(q, k, v, o2, g2, **kw)
    torch.cuda.synchronize()
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before     # torch's allocator saw nothing
    if not first:
        # nor did the device: a hipMalloc inside the library would lower the driver's free count (the very first
        # call on a device looks the static array's address up, which is allowed to load the code object)
        assert torch.cuda.mem_get_info()[0] == free_before
    assert torch.equal(o1, o2) and torch.equal(g1, g2), f"bh={bh} n={n} d={d} {dtype}"


def test_static_scratch_forward_matches_forward(lib):
    print("case no-alloc forward", flush=True)
    kw = dict(mask=True, inv_tau=1.0 / (8.0 * math.sqrt(64)), p=2)
    _pair(lib, 8, 2048, 64, torch.bfloat16, 1, first=True, **kw)          # first call on this device: looks the buffer up
    _pair(lib, 3, 333, 64, torch.bfloat16, 2, **kw)           # smaller, straight after, on the used buffer
    _pair(lib, 2, 1100, 64, torch.float32, 3, chunk=256, **kw)                 # through moment states
    _pair(lib, 2, 300, 32, torch.bfloat16, 4, mask=False, inv_tau=0.1, p=1)
    _pair(lib, 3, 130, 64, torch.bfloat16, 5, mask=True, inv_tau=0.1, p=1)


def test_static_scratch_limit(lib):
    # a problem whose workspace exceeds the static buffer is refused before anything is launched
    q = torch.zeros(16, 65536, 64, dtype=torch.bfloat16, device=DEV)
    d = lib.make_desc(q, q, q, mask=True, inv_tau=0.1, a0=1.0, a1=1.0, a2=0.5, p=2)
    need, _ = lib.workspace_bytes(d)
    assert need > _capi.STATIC_SCRATCH_BYTES
    o, g = torch.empty_like(q), torch.empty(16, 65536, device=DEV)
    with pytest.raises(_capi.FastmaxError, match="static buffer"):
        lib.forward_static(q, q, q, o, g, mask=True, inv_tau=0.1, p=2)


def test_static_scratch_takes_a_few_queries_on_many_keys(lib):
    """Sixteen queries of each of 1024 batch*heads: the general route, the faster one there, would need 134 MB; the static
    buffer serves the call on the route for a few queries, with the same results up to one rounding to bf16 on each side
    (2^-8 of the binade's start, rms 1.7e-3 of the norm, twice) and the general route's _Float16 weights."""
    print("case no-alloc few queries", flush=True)
    gen = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn(1024, n, 64, generator=gen).to(torch.bfloat16).to(DEV) for n in (16, 300, 300))
    kw = dict(mask=False, inv_tau=1.0 / 64.0, p=2)
    d = lib.make_desc(q, k, v, a0=1.0, a1=1.0, a2=0.5, **kw)
    assert lib.workspace_bytes(d)[0] > _capi.STATIC_SCRATCH_BYTES
    o1, g1 = lib.forward(q, k, v, **kw)
    o2, g2 = torch.full_like(o1, float("nan")), torch.full_like(g1, float("nan"))
    lib.forward_static(q, k, v, o2, g2, **kw)
    assert float((o1.double() - o2.double()).norm() / o1.double().norm()) < 4e-3
    assert float((g1.double() - g2.double()).norm() / g1.double().norm()) < 1e-3


def test_static_scratch_takes_long_fp32_problems_of_few_heads(lib):
    """States of 9000 tokens do not fit the buffer; the forward alone stays on dense tiles, whose bits it gives."""
    gen = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(4, 9000, 64, generator=gen).to(DEV) for _ in range(3))
    kw = dict(mask=True, inv_tau=1.0 / 64, p=2)
    o, g = lib.forward(q, k, v, flags=_capi.FLAG_FORCE_DENSE, **kw)
    o2, g2 = torch.empty_like(o), torch.empty_like(g)
    lib.forward_static(q, k, v, o2, g2, **kw)
    assert torch.equal(o, o2) and torch.equal(g, g2)
