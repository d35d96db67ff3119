"""Kernels at the far ends of what their entry points accept: sequences longer than 16 bits count."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def core():
    import fractaltensor_amd._core as c
    return c


@pytest.mark.parametrize('half,H,L', [(False, 64, 2), (True, 256, 1)])
def test_ragged_stack_longer_than_65535_steps(core, half, H, L):
    """Row block 0 lives for 65540 steps, row block 1 for exactly 65536 (zero in 16 bits).  The live places are those of the
    dense call bit for bit: the same kernel, and rows never interact."""
    T, B, ends = 65540, 17, 65536
    gen = torch.Generator(device='cuda').manual_seed(3)
    dtype = torch.float16 if half else torch.float32
    xs = torch.randn((T, B, H), generator=gen, device='cuda').to(dtype)
    WU = ((torch.rand((L, 2 * H, 4 * H), generator=gen, device='cuda') * 2 - 1) * H ** -0.5).to(dtype)
    call = core.stacked_lstm_f16 if half else core.stacked_lstm
    dense_h, dense_c = call(xs, WU, check=True)
    active = [B] * ends + [2] * (T - ends)
    print(f'ragged stack of {T} steps, H {H}, fp16 {half}', flush=True)
    h, c = call(xs, WU, active_rows=active, check=True)
    for got, ref in ((h, dense_h), (c, dense_c)):
        assert torch.equal(got[:, :ends], ref[:, :ends])
        assert torch.equal(got[:, ends:, :2], ref[:, ends:, :2])
    assert float(h[:, ends - 1].abs().max()) > 0
