"""cvk_infections_noalloc (no allocation; per-block counts in the library's fixed device array)
gives exactly what cvk_infections gives, on consecutive calls of different sizes through the C ABI.
Runs last: it is the one entry point whose scratch persists between calls."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def call(entry, beta, p1, p2, lb, rt, rs, uniforms=None, legacy=0, t=0, v=0, l=0, capacity=None):
    import torch
    from covasim_amd import _lib
    E = p1.numel()
    cap = (E if legacy else 2 * E) if capacity is None else capacity
    src = torch.full((max(cap, 1),), -7, dtype=torch.int32, device='cuda')
    tgt = torch.full((max(cap, 1),), -7, dtype=torch.int32, device='cuda')
    prob = torch.full((max(cap, 1),), -1.0, dtype=torch.float32, device='cuda')
    count = C.c_int64(-1)
    rc = getattr(_lib.lib(), entry)(float(np.float32(beta)), p1.data_ptr(), p2.data_ptr(), lb.data_ptr(), E,
                                    rt.data_ptr(), rs.data_ptr(), rt.numel(),
                                    uniforms.data_ptr() if uniforms is not None else None, 77, t, v, l, legacy,
                                    src.data_ptr(), tgt.data_ptr(), prob.data_ptr(), cap, C.byref(count),
                                    _lib.stream_ptr())
    torch.cuda.synchronize()
    k = max(count.value, 0)
    return rc, count.value, src[:k].cpu().numpy(), tgt[:k].cpu().numpy(), prob[:k].cpu().numpy().view(np.uint32)


def inputs(seed, n, E):
    import torch
    rng = np.random.default_rng(seed)
    p1 = rng.integers(0, n, E).astype(np.int32)
    p2 = rng.integers(0, n, E).astype(np.int32)
    p1[:20] = p2[:20]
    lb = rng.choice([1.0, 0.0, 2.5], E, p=[0.9, 0.05, 0.05]).astype(np.float32)
    rt = np.where(rng.random(n) < 0.2, rng.random(n) * 3, 0).astype(np.float32)
    rs = np.where(rng.random(n) < 0.8, rng.random(n), 0).astype(np.float32)
    U = rng.random((2, E))
    dev = lambda a: torch.from_numpy(a).cuda()
    return dev(p1), dev(p2), dev(lb), dev(rt), dev(rs), dev(U)


def test_noalloc_equals_allocating_entry_point(gpu):
    from covasim_amd import _lib
    # the second call is smaller: block counts left in the scratch by the first must not leak into it
    for (seed, n, E) in [(1, 200_000, 3_000_000), (2, 5_000, 70_001)]:
        p1, p2, lb, rt, rs, U = inputs(seed, n, E)
        for legacy in (0, 1):
            for uni in (None, U):
                for beta in (0.3, 0.02):
                    a = call('cvk_infections', beta, p1, p2, lb, rt, rs, uni, legacy, t=3, v=1, l=2)
                    b = call('cvk_infections_noalloc', beta, p1, p2, lb, rt, rs, uni, legacy, t=3, v=1, l=2)
                    assert a[0] == b[0] == _lib.OK
                    assert a[1] == b[1] > 0, (seed, legacy, beta)
                    for x, y in zip(a[2:], b[2:]):
                        assert np.array_equal(x, y), (seed, legacy, beta)


def test_noalloc_errors(gpu):
    import torch
    from covasim_amd import _lib
    p1, p2, lb, rt, rs, U = inputs(3, 1000, 10_000)
    # output too small: the count is reported and CVK_E_CAPACITY returned, as by cvk_infections
    a = call('cvk_infections', 0.9, p1, p2, lb, rt, rs, capacity=1)
    b = call('cvk_infections_noalloc', 0.9, p1, p2, lb, rt, rs, capacity=1)
    assert a[0] == b[0] == _lib.E_CAPACITY and a[1] == b[1] > 1
    # beyond the fixed scratch: rejected before any device work, with a message naming the limit
    L = _lib.lib()
    big = _lib.INFECTIONS_NOALLOC_MAX_SLOTS // 2 + 1
    cnt = C.c_int64(-1)
    dummy = torch.zeros(4, dtype=torch.int32, device='cuda')
    rc = L.cvk_infections_noalloc(0.1, dummy.data_ptr(), dummy.data_ptr(), dummy.data_ptr(), big, dummy.data_ptr(),
                                  dummy.data_ptr(), 4, None, 1, 0, 0, 0, 0, dummy.data_ptr(), dummy.data_ptr(), None,
                                  0, C.byref(cnt), _lib.stream_ptr())
    assert rc == _lib.E_CAPACITY and cnt.value == 0
    assert b'limit' in L.cvk_last_error()
    # and it still works afterwards
    c = call('cvk_infections_noalloc', 0.9, p1, p2, lb, rt, rs)
    d = call('cvk_infections', 0.9, p1, p2, lb, rt, rs)
    assert c[1] == d[1] and all(np.array_equal(x, y) for x, y in zip(c[2:], d[2:]))


@pytest.mark.parametrize('legacy', [0, 1])
@pytest.mark.parametrize('E', [1, 31, 32, 511, 512, 513, 4096 * 512 - 1, 4096 * 512 + 1])
def test_noalloc_chunk_edges(gpu, E, legacy):
    """Edge counts at and around a word of hits, a chunk, and a chunk for every wave of the launch: the pairs of the
    writing pass that finds the hits anew are, in their order, those of the one that kept them."""
    p1, p2, lb, rt, rs, U = inputs(E, max(20, E // 50), max(E, 20))
    p1, p2, lb, U = p1[:E].clone(), p2[:E].clone(), lb[:E].clone(), U[:, :E].contiguous()
    for uni in (None, U):
        a = call('cvk_infections', 0.9, p1, p2, lb, rt, rs, uni, legacy, t=3, v=1, l=2)
        b = call('cvk_infections_noalloc', 0.9, p1, p2, lb, rt, rs, uni, legacy, t=3, v=1, l=2)
        assert a[:2] == b[:2] and all(np.array_equal(x, y) for x, y in zip(a[2:], b[2:]))
        assert a[1] > 0 or E < 512


@pytest.mark.parametrize('legacy', [0, 1])
def test_noalloc_largest_call(gpu, legacy):
    """As many slots as it takes; with legacy the last chunks are past those that the scratch has a flag for."""
    import torch
    from covasim_amd import _lib
    n, E = 100_000, _lib.INFECTIONS_NOALLOC_MAX_SLOTS // (1 if legacy else 2)
    g = torch.Generator(device='cuda').manual_seed(5)
    p1, p2 = torch.randint(0, n, (2, E), generator=g, device='cuda', dtype=torch.int32)
    rt = torch.zeros(n, device='cuda')
    rt[:100] = 0.5
    lb, rs = torch.ones(E, device='cuda'), torch.ones(n, device='cuda')
    a = call('cvk_infections', 0.5, p1, p2, lb, rt, rs, legacy=legacy)
    b = call('cvk_infections_noalloc', 0.5, p1, p2, lb, rt, rs, legacy=legacy)
    assert a[:2] == b[:2] and a[1] > 1000 and all(np.array_equal(x, y) for x, y in zip(a[2:], b[2:]))


@pytest.mark.parametrize('entry', ['cvk_infections', 'cvk_infections_noalloc', 'cvk_infections_work'])
def test_refused_calls_leave_the_outputs_alone(gpu, entry):
    """One pair too many for the outputs, or an index outside the population: an error, and nothing written."""
    import torch
    from covasim_amd import _lib
    L = _lib.lib()
    p1, p2, lb, rt, rs, _ = inputs(4, 3000, 40_000)
    E, n = p1.numel(), rt.numel()
    work = torch.empty(L.cvk_infections_work_bytes(E, n), dtype=torch.uint8, device='cuda')
    outs = [torch.full((2 * E,), -7, dtype=torch.int32, device='cuda') for _ in range(2)]
    prob = torch.full((2 * E,), -1.0, device='cuda')

    def refused(capacity):
        count = C.c_int64(-1)
        extra = (None, work.data_ptr(), work.numel()) if entry.endswith('work') else ()
        rc = getattr(L, entry)(0.9, p1.data_ptr(), p2.data_ptr(), lb.data_ptr(), E, rt.data_ptr(), rs.data_ptr(), n,
                               None, 77, 0, 0, 0, 0, outs[0].data_ptr(), outs[1].data_ptr(), prob.data_ptr(), capacity,
                               C.byref(count), *extra, _lib.stream_ptr())
        torch.cuda.synchronize()
        return rc, count.value, int((outs[0] != -7).sum() + (outs[1] != -7).sum() + (prob != -1).sum())
    total = call('cvk_infections', 0.9, p1, p2, lb, rt, rs)[1]
    assert total > 1000
    assert refused(total - 1) == (_lib.E_CAPACITY, total, 0)
    p2[E // 2] = n
    assert refused(2 * E) == (_lib.E_INVALID, 0, 0)
