"""CPU-side checks of the C-ABI library: it loads, exports every symbol that
include/ftk.h declares, and rejects bad arguments before touching a device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, 'include', 'ftk.h')).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(ftk_[a-z0-9_]+)\s*\(', text)))


def test_header_and_binding_agree():
    import fractaltensor_amd._core as core
    assert sorted(core.EXPORTS) == declared_symbols()


def test_library_exports_every_declared_symbol():
    import fractaltensor_amd._core as core
    lib = ctypes.CDLL(core.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(lib, name), name
    assert core.version() >= 100


def test_argument_errors_come_back_as_codes_not_crashes():
    import fractaltensor_amd._core as core
    lib = core.lib
    nul = ctypes.c_void_p(0)
    one = ctypes.c_void_p(16)   # never dereferenced: validation fails first
    ci = ctypes.c_int
    assert lib.ftk_lstm_cell_f32(nul, nul, nul, nul, nul, nul, nul, ci(1), ci(32), ci(32), nul) == -1
    assert b'non-NULL' in lib.ftk_last_error()
    assert lib.ftk_lstm_cell_f32(one, nul, nul, one, nul, one, one, ci(4), ci(30), ci(32), nul) == -2
    assert lib.ftk_lstm_cell_f32(one, one, nul, one, nul, one, one, ci(4), ci(32), ci(32), nul) == -1
    assert lib.ftk_b2b_gemm_f16(one, one, one, one, ci(1), ci(64), ci(48), ci(64), ci(64), nul) == -2
    assert lib.ftk_b2b_gemm_f16(one, one, one, one, ci(0), ci(64), ci(64), ci(64), ci(64), nul) == -1
    assert lib.ftk_b2b_gemm_f16(one, one, one, one, ci(1), ci(64), ci(64), ci(24), ci(64), nul) == -2   # K % 16
    assert lib.ftk_b2b_gemm_rowmajor_f16(one, one, one, one, ci(1), ci(64), ci(64), ci(96), ci(128), nul) == -2
    assert lib.ftk_b2b_gemm_rowmajor_f16(one, nul, one, one, ci(1), ci(64), ci(64), ci(64), ci(128), nul) == -1
    assert lib.ftk_gemm_f16(one, one, one, ci(64), ci(96), ci(64), nul) == -2
    assert lib.ftk_gemm_f16(one, ctypes.c_void_p(18), one, ci(64), ci(256), ci(64), nul) == -1 and b'aligned' in lib.ftk_last_error()
    assert lib.ftk_batched_gemm_f16(one, one, nul, ci(2), ci(64), ci(128), ci(64), nul) == -1
    assert lib.ftk_flash_attn_f16(one, one, one, one, ci(1), ci(1), ci(64), ci(64), ci(48), ctypes.c_float(1), nul) == -2
    cf = ctypes.c_float
    assert lib.ftk_flash_attn_f32(one, nul, one, one, ci(1), ci(1), ci(64), ci(64), ci(64), cf(1), one, ctypes.c_size_t(1 << 30), nul) == -1
    assert lib.ftk_flash_attn_f32(one, one, one, one, ci(1), ci(1), ci(64), ci(64), ci(48), cf(1), one, ctypes.c_size_t(1 << 30), nul) == -2
    assert lib.ftk_flash_attn_f32(ctypes.c_void_p(20), one, one, one, ci(1), ci(1), ci(64), ci(64), ci(64), cf(1), one, ctypes.c_size_t(1 << 30), nul) == -1
    assert lib.ftk_flash_attn_f32(one, one, one, one, ci(1), ci(1), ci(64), ci(64), ci(64), cf(0), one, ctypes.c_size_t(1 << 30), nul) == -1
    assert lib.ftk_flash_attn_f32(one, one, one, one, ci(1), ci(1), ci(64), ci(64), ci(64), cf(1), nul, ctypes.c_size_t(0), nul) == -3
    assert lib.ftk_flash_attn_f32_workspace_bytes(ci(2), ci(3), ci(100), ci(77), ci(64)) >= 4 * 6 * (2 * 77) * 64   # K's and V's planes
    assert lib.ftk_b2b_gemm_f16_supported(ci(48), ci(64), ci(64)) == 0          # N % 32
    assert lib.ftk_stacked_lstm_small_states(nul, nul) == -1
    assert lib.ftk_online_softmax_f32(nul, one, ci(1), ci(1), nul) == -1
    assert lib.ftk_stacked_lstm_wavefront_f32(one, one, nul, nul, one, one, ci(1), ci(1), ci(1), ci(48), nul) == -2
    assert lib.ftk_embedding_gather_f32(one, one, ci(0), one, ctypes.c_longlong(4), ci(8), ci(6), nul, nul) == -2
    assert lib.ftk_embedding_gather_f32(one, nul, ci(0), one, ctypes.c_longlong(4), ci(8), ci(8), nul, nul) == -1
    assert lib.ftk_stacked_lstm_ragged_f32(one, one, nul, nul, nul, one, one, ci(1), ci(1), ci(1), ci(32), nul, ctypes.c_size_t(0), nul) == -1
    assert lib.ftk_lstm_cell_f16(one, nul, nul, one, nul, one, one, ci(4), ci(48), ci(64), nul) == -2
    assert lib.ftk_lstm_layer_f32(one, one, nul, one, nul, one, one, ci(2), ci(4), ci(32), ci(32), nul) == -1
    assert lib.ftk_lstm_layer_f16(one, one, nul, nul, nul, one, one, ci(2), ci(4), ci(32), ci(40), nul) == -2
    assert lib.ftk_lstm_layer_f32(one, one, nul, nul, nul, one, one, ci(0), ci(4), ci(32), ci(32), nul) == -1
    assert lib.ftk_lstm_cell_f16(one, one, nul, one, nul, one, one, ci(4), ci(64), ci(64), nul) == -1
    assert lib.ftk_stacked_lstm_f16(one, one, nul, nul, nul, one, one, ci(1), ci(1), ci(4), ci(80), nul, ctypes.c_size_t(0), nul) == -2
    # a shape whose weights are streamed needs the workspace for their re-laid copy
    assert lib.ftk_stacked_lstm_f16(one, one, nul, nul, nul, one, one, ci(2), ci(3), ci(4), ci(1024), nul, ctypes.c_size_t(0), nul) == -3
    # a layer of 2^32 16-byte pieces or more cannot be re-laid, with a workspace of any size
    assert lib.ftk_stacked_lstm_f16(one, one, nul, nul, nul, one, one, ci(1), ci(1), ci(1), ci(65504), nul, ctypes.c_size_t(0), nul) == -3
    for H in (65536, 65568, 131072):
        assert lib.ftk_stacked_lstm_f16(one, one, nul, nul, nul, one, one, ci(1), ci(1), ci(1), ci(H), nul, ctypes.c_size_t(0), nul) == -2
    # the status block (256 bytes, its first int the status word) and the re-laid weights
    assert lib.ftk_stacked_lstm_f16_workspace_bytes(2, 3, 4, 1024) == 256 + 2 * 2048 * 4096 * 2
    # per-call options: an unknown products mode, a negative poll limit; the status query without a workspace
    opts = core.LstmOptions(7, 0)
    stack = lambda o: lib.ftk_stacked_lstm_opts_f32(one, one, nul, nul, nul, one, one, ci(1), ci(1), ci(1), ci(32), o, nul,
                                                    ctypes.c_size_t(0), nul)
    assert stack(ctypes.byref(opts)) == -1
    assert stack(ctypes.byref(core.LstmOptions(-1, -5))) == -1
    assert lib.ftk_stacked_lstm_status(nul, nul) == -1
    assert lib.ftk_stacked_lstm_workspace_bytes(32, 64, 256, 256) > 0
    assert lib.ftk_stacked_lstm_workspace_bytes(0, 64, 256, 256) == 0
    # grid RNN: null operands, a hidden size that is no multiple of 32, bias rows that are neither 1 nor B, one bias only
    cz, cf = ctypes.c_size_t, ctypes.c_float
    grid = lambda *p, H=32, rows=1, bx=one, by=one: lib.ftk_grid_rnn_f32(*p, bx, one, one, by, one, ci(1), ci(2), ci(2), ci(4), ci(H),
                                                                         ci(rows), ci(0), nul, cz(0), nul)
    assert grid(nul, one, one, one) == -1
    assert grid(one, one, one, one, H=48) == -2
    assert grid(one, one, one, one, rows=3) == -1
    assert grid(one, one, one, one, by=nul) == -1
    assert lib.ftk_grid_rnn_workspace_bytes(32, 256) == 2 * 32 * 3 * 256 * 256 * 4
    assert lib.ftk_grid_rnn_workspace_bytes(0, 256) == 0
    # windowed attention: even window, head size off the 16-byte pieces, a span longer than the sequence, indices without a count
    wa = lambda S=8, D=16, W=3, dl=1, R=0, idx=nul, q=one: lib.ftk_windowed_attn_f32(q, one, one, idx, one, ci(1), ci(S), ci(D), ci(W),
                                                                                       ci(dl), ci(R), cf(1.0), nul)
    assert wa(q=nul) == -1
    assert wa(W=4) == -2
    assert wa(D=6) == -2
    assert wa(W=5, dl=4) == -2
    assert wa(idx=one) == -1
    assert wa(R=2) == -1
    assert wa(q=ctypes.c_void_p(8)) == -1          # not 16-byte aligned


def test_wrappers_check_supplied_outputs_before_any_launch():
    """A caller-supplied output of the wrong shape must never reach a kernel (it would be overrun), and a workspace
    must be device memory.  The shape is looked at first, so host tensors are enough to show it."""
    import torch
    import fractaltensor_amd._core as core
    f32 = torch.float32
    with pytest.raises(ValueError, match=r'hsss must be \(2, 3, 4, 32\)'):
        core._req_out(torch.empty((2, 3, 4, 16), dtype=f32), f32, (2, 3, 4, 32), 'hsss')
    with pytest.raises(RuntimeError, match='no CPU path'):      # right shape: the next check is the device
        core._req_out(torch.empty((2, 3, 4, 32), dtype=f32), f32, (2, 3, 4, 32), 'hsss')
    with pytest.raises(ValueError, match='workspace'):
        core._req_workspace(torch.empty(16, dtype=torch.uint8))
    with pytest.raises(ValueError, match='workspace'):
        core._req_workspace(None)


def test_wrappers_refuse_cpu_tensors():
    import torch
    import fractaltensor_amd._core as core
    x = torch.zeros((4, 32))
    with pytest.raises(RuntimeError, match='no CPU path'):
        core.lstm_cell(x, None, None, torch.zeros((64, 128)))
    with pytest.raises(RuntimeError, match='no CPU path'):
        core.online_softmax(x)


def test_f16_stack_workspace_is_that_of_the_kernels_the_shape_goes_to():
    """L 32 T 64 B 256: the streamed cells at H 1024 (status block and re-laid weights), the persistent kernel at H 256 (flags
    only); neither asks for the state buffers of the exchange kernel."""
    import fractaltensor_amd._core as core
    size = core.lib.ftk_stacked_lstm_f16_workspace_bytes
    assert size(32, 64, 256, 1024) == 256 + 32 * 2048 * 4096 * 2
    assert 0 < size(32, 64, 256, 256) < 4 << 20


def test_f32_attention_workspace_is_what_the_header_says():
    """Planes, 520 bytes a head and, on a device, what the workgroups that share keys leave: 512 D + 2048 bytes each, no more of them
    than two to a compute unit."""
    import fractaltensor_amd._core as core
    up = lambda n: (n + 255) // 256 * 256
    for B, Hd, Sq, Skv, D in [(1, 1, 4096, 1024, 64), (2, 8, 1024, 1024, 32), (1, 4, 128, 65536, 128), (4, 16, 640, 640, 96), (1, 1, 1, 1, 32)]:
        n = int(core.lib.ftk_flash_attn_f32_workspace_bytes(B, Hd, Sq, Skv, D))
        without = up(8 * B * Hd) + up(512 * B * Hd) + 2 * up(4 * D * Skv * B * Hd)
        assert without <= n <= without + 512 * (512 * D + 2048) + 512 * 4 + 512
