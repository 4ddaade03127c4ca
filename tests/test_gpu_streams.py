"""Operators that use the library's scratch memory, on several streams and
threads at once, in captured graphs, and with changing sizes: each call's
result is the one it has alone."""
import threading

import pytest

pytestmark = pytest.mark.gpu

N = 24_000_007


@pytest.fixture(scope="module")
def joins(dev):
    """Two full joins whose scratch (a 16-bit copy of the table and its
    presence bitmap) differs in size and contents, and their results."""
    import torch
    from sycldb_amd import ops
    out = []
    for k, length in enumerate((300_000, 1_400_000)):
        g = torch.Generator("cuda").manual_seed(k)
        pairs = torch.zeros(2 * length, dtype=torch.int32, device=dev)
        pairs[0::2] = (torch.rand(length, generator=g, device=dev) < 0.3).int()
        pairs[1::2] = torch.randint(1, 1000, (length,), generator=g, device=dev, dtype=torch.int32)
        probe = torch.randint(0, length, (N,), generator=g, device=dev, dtype=torch.int32)
        flags = (torch.rand(N, generator=g, device=dev) < 0.9).to(torch.uint8)
        hit = (flags != 0) & (pairs[0::2][probe.long()] == 1)
        want = torch.where(hit, pairs[1::2][probe.long()], -7)

        def run(stream, pairs=pairs, probe=probe, flags=flags, length=length):
            vals, left = torch.full((N,), -7, dtype=torch.int32, device=dev), torch.empty_like(flags)
            ids, count = torch.empty(N, dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
            torch.cuda.current_stream().synchronize()
            with torch.cuda.stream(stream):
                ops.probe_full(probe, vals, flags, left, pairs, 0, length - 1)
                ops.compact(left, ids, count)
            return vals, left, ids, count

        def check(got, want=want, hit=hit):
            vals, left, ids, count = got
            k = int(count.item())
            assert bool((vals == want).all()) and bool((left == hit).all())
            assert k == int(hit.sum()) and bool((ids[:k] == hit.nonzero().squeeze(1)).all())
        out.append((run, check))
    return out


def test_two_streams(joins):
    import torch
    streams = [torch.cuda.Stream() for _ in joins]
    for _ in range(4):
        got = [run(s) for (run, _), s in zip(joins, streams)]
        torch.cuda.synchronize()
        for (_, check), g in zip(joins, got):
            check(g)


@pytest.mark.parametrize("shared", [False, True])
def test_two_threads(joins, shared):
    """Each thread on its own stream, and both on one."""
    import torch
    one = torch.cuda.Stream()
    streams = [one, one] if shared else [torch.cuda.Stream() for _ in joins]
    got = [[], []]

    def work(k):
        torch.cuda.set_device(0)
        for _ in range(4):
            got[k].append(joins[k][0](streams[k]))
    threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for k in (0, 1):
        assert len(got[k]) == 4
        for g in got[k]:
            joins[k][1](g)


def test_more_streams_than_buffers_are_kept(dev):
    """40 streams of the caller's, created and destroyed, sizes up and down."""
    import ctypes
    import torch
    from sycldb_amd import ops
    hip = ctypes.CDLL("libamdhip64.so")
    f = (torch.arange(5_000_000, device=dev) % 3 == 0).to(torch.uint8)
    handles = []
    for k in range(40):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(h), 1) == 0
        handles.append(h)
        n = 5_000_000 >> (k * 7 % 10)
        ids, count = torch.full((n,), -1, dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
        torch.cuda.synchronize()
        ops.compact(f[:n], ids, count, stream=h.value)
        torch.cuda.synchronize()
        c = int(count.item())
        assert c == (n + 2) // 3 and bool((ids[:c] == torch.arange(c, device=dev) * 3).all())
        if k % 3 == 0:
            assert hip.hipStreamDestroy(handles.pop()) == 0
    for h in handles:
        assert hip.hipStreamDestroy(h) == 0


def test_captured_beside_eager_calls(joins, dev):
    """A captured full join and compaction (no call of their stream before),
    replayed with the other join's eager calls, of more scratch, between."""
    import torch
    from sycldb_amd import ops
    f = (torch.arange(9_000_000, device=dev) % 7 == 0).to(torch.uint8)
    ids, count = torch.zeros(len(f), dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
    n, length = 4_500_003, 280_000
    pairs = torch.ones(2 * length, dtype=torch.int32, device=dev)
    pairs[1::2] = torch.arange(length, device=dev, dtype=torch.int32) % 1000
    probe = torch.arange(n, device=dev, dtype=torch.int32) % length
    vals, ones = torch.zeros(n, dtype=torch.int32, device=dev), torch.ones(n, dtype=torch.uint8, device=dev)
    left = torch.zeros_like(ones)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.probe_full(probe, vals, ones, left, pairs, 0, length - 1)
        ops.compact(f, ids, count)
    side = torch.cuda.Stream()
    for rep in range(3):
        vals.zero_(), left.zero_(), ids.zero_(), count.zero_()
        f[rep * 7] = 0
        torch.cuda.synchronize()
        g.replay()
        got = joins[1][0](side)
        torch.cuda.synchronize()
        joins[1][1](got)
        assert bool((vals == pairs[1::2][probe.long()]).all()) and bool((left == 1).all())
        k = int(count.item())
        assert k == int(f.sum()) and bool((ids[:k] == f.nonzero().squeeze(1)).all())
