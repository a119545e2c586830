"""fp32 SwiGLU at 5-32 rows with silu * up in the gate / up launch: edges of
the 32-column groups, the 16-row blocks and the K chunks.

Inputs are small multiples of powers of two, so gate and up are exact in fp32
whatever the order of the sums, and h equals gfh_silu_mul of them bit for
bit."""
import pytest

pytestmark = pytest.mark.gpu


def _layer(torch, dev, m, hidden, inter, bias):
    g = torch.Generator(device=dev)
    g.manual_seed(m + hidden + inter)

    def ints(*shape):
        return torch.randint(-3, 4, shape, device=dev, generator=g).float()

    x, wg, wu, wd = ints(m, hidden), ints(inter, hidden) / 64, ints(inter, hidden) / 64, ints(hidden, inter) / 64
    bg, bu = (ints(inter) / 8, ints(inter) / 8) if bias else (None, None)
    return x, wg, bg, wu, bu, wd, None


def _check(torch, gh, x, wg, bg, wu, bu, h):
    gate, up = ((x.double() @ w.double().t().contiguous() + (0 if b is None else b)).float()
                for w, b in ((wg, bg), (wu, bu)))
    assert torch.equal(h, gh.silu_mul(gate, up))


# K not split: hidden < 512, or more than 128 groups of 64 columns
@pytest.mark.parametrize("m", [5, 16, 17, 32])
@pytest.mark.parametrize("hidden,inter", [(4, 1), (60, 15), (64, 33), (196, 64), (508, 100), (640, 8257)])
def test_h_exact(torch_dev, m, hidden, inter):
    import torch
    import ghostflow_hip as gh
    for bias in (True, False):
        x, wg, bg, wu, bu, wd, bd = _layer(torch, torch_dev, m, hidden, inter, bias)
        _, h = gh.swiglu(x, wg, bg, wu, bu, wd, bd, want_h=True)
        _check(torch, gh, x, wg, bg, wu, bu, h)


def test_h_over_x(torch_dev):
    """h in x's memory: gate and up are finished before h is written."""
    import torch
    import ghostflow_hip as gh
    m, hidden, inter = 16, 256, 256
    x, wg, bg, wu, bu, wd, _ = _layer(torch, torch_dev, m, hidden, inter, True)
    x0, y = x.clone(), torch.empty(m, hidden, device=torch_dev)
    rc = gh.lib().gfh_swiglu_f32(x.data_ptr(), m, hidden, inter, wg.data_ptr(), bg.data_ptr(), wu.data_ptr(),
                                 bu.data_ptr(), wd.data_ptr(), None, y.data_ptr(), x.data_ptr(), None, 0,
                                 torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    _check(torch, gh, x0, wg, bg, wu, bu, x)
