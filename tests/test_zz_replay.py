"""Recorded stacks.  In a file of its own at the end: after the first capture a process launches the kernels whose workgroups wait for each
other cooperatively."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def core():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from fractaltensor_amd import _core
    return _core


@pytest.mark.parametrize('half,L,T,B,H', [(False, 3, 9, 20, 64), (False, 2, 5, 70, 256), (True, 2, 7, 33, 512)])
def test_a_replayed_stack_computes_from_its_new_inputs(core, half, L, T, B, H):
    """Every replay finds the words that the one before left in the workspace, and eager launches on it lie in between."""
    dtype = torch.float16 if half else torch.float32
    fn = core.stacked_lstm_f16 if half else core.stacked_lstm
    size = core.lib.ftk_stacked_lstm_f16_workspace_bytes if half else core.stacked_lstm_workspace_bytes
    gen = torch.Generator(device='cuda').manual_seed(5)
    draw = lambda *shape: torch.randn(shape, generator=gen, device='cuda')
    xs, ws = torch.zeros(T, B, H, device='cuda', dtype=dtype), torch.empty(size(L, T, B, H), device='cuda', dtype=torch.uint8)
    WU, bias = (draw(L, 2 * H, 4 * H) * H ** -0.5).to(dtype), draw(L, 4 * H)
    out = tuple(torch.empty(L, T, B, H, device='cuda', dtype=dtype) for _ in range(2))
    inputs = [draw(T, B, H).to(dtype) for _ in range(3)]
    refs = [[r.clone() for r in fn(x, WU, bias, workspace=ws)] for x in inputs]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        fn(xs, WU, bias, out=out, workspace=ws)
    for turn in range(6):
        xs.copy_(inputs[turn % 3])
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, r) for o, r in zip(out, refs[turn % 3])), turn
        if turn % 2:
            got = fn(inputs[(turn + 1) % 3], WU, bias, workspace=ws)
            torch.cuda.synchronize()
            assert all(torch.equal(o, r) for o, r in zip(got, refs[(turn + 1) % 3])), turn
