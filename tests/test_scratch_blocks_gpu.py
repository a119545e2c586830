"""Calls without a workspace: the per-stream kept block (first use, growth,
needs beyond it, two threads on one stream, two streams, shutdown) gives the
bits of the same call with the caller's workspace."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def _case(torch, dev, m, k, n, seed):
    import ghostflow_hip as gh
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    x = torch.randn(m, k, device=dev, generator=g)
    qw, sw, _ = gh.quantize_per_channel(torch.randn(n, k, device=dev, generator=g), symmetric=True)
    rs = qw.sum(1, dtype=torch.int32)
    ws = torch.empty(gh.lib().gfh_qlinear_dynamic_i8_workspace_size(m, k), dtype=torch.uint8, device=dev)
    ref = gh.qlinear_dynamic(x, qw, sw, rs, workspace=ws)
    return (x, qw, sw, rs), ref


# 0.4 MB, 4 MB (the block grows), 80 MB (allocated for the call), 0.4 MB again
SIZES = [(100, 4096, 128), (500, 8192, 64), (4900, 16384, 64), (100, 4096, 128)]


def test_sizes_and_shutdown(torch_dev):
    import torch
    import ghostflow_hip as gh
    for _ in range(2):
        for i, (m, k, n) in enumerate(SIZES):
            args, ref = _case(torch, torch_dev, m, k, n, i)
            for _ in range(3):
                assert torch.equal(gh.qlinear_dynamic(*args), ref)
        torch.cuda.synchronize()
        assert gh.lib().gfh_shutdown() == 0


@pytest.mark.parametrize("own_streams", [False, True])
def test_threads(torch_dev, own_streams):
    import torch
    import ghostflow_hip as gh
    cases = [_case(torch, torch_dev, 100 + 60 * i, 2048 * (1 + i), 256, i) for i in range(3)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() if own_streams else torch.cuda.current_stream() for _ in cases]
    wrong = []

    def work(i):
        (args, ref), s = cases[i], streams[i]
        with torch.cuda.stream(s):
            got = [gh.qlinear_dynamic(*args) for _ in range(40)]
        s.synchronize()
        wrong.extend(i for y in got if not torch.equal(y, ref))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_idle_blocks_pass_to_other_streams(torch_dev):
    """Blocks that fill the total and then lie idle, as those of destroyed
    streams do (a block does not know), go to streams that come later."""
    import ctypes as C

    import torch
    import ghostflow_hip as gh
    lib = C.CDLL(gh.lib()._name)
    lib.gfh_internal_scratch_kept.restype = C.c_size_t
    lib.gfh_internal_scratch_kept.argtypes = [C.c_void_p]
    big, big_ref = _case(torch, torch_dev, 2100, 16384, 64, 0)  # 34 MB: a block of 64
    small, small_ref = _case(torch, torch_dev, 100, 512, 64, 1)
    torch.cuda.synchronize()
    assert gh.lib().gfh_shutdown() == 0

    def kept(s, args=big, ref=big_ref):
        with torch.cuda.stream(s):
            got = gh.qlinear_dynamic(*args)
        s.synchronize()
        assert torch.equal(got, ref)
        return lib.gfh_internal_scratch_kept(s.cuda_stream) >> 20

    streams = [torch.cuda.Stream() for _ in range(6)]
    assert [kept(s) for s in streams] == [64] * 4 + [0] * 2
    for _ in range(300):
        kept(streams[4], small, small_ref)
    # blocks from half the total on record an event to wait for: two of the four
    assert [kept(s) for s in streams[4:]] == [64] * 2
    assert sum(lib.gfh_internal_scratch_kept(s.cuda_stream) for s in streams) <= 256 << 20
    assert [kept(s) for s in streams[:2]] == [64] * 2
    for s in streams:
        kept(s)
    assert gh.lib().gfh_shutdown() == 0
