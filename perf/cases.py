"""Workloads that stand for the use of this package, for timing one build of it against another.

`listed()` gives the fixed ones, `draw(rng)` further ones of the same ranges.  For a case, `prepare(case, seed)` makes
what a program holds before the call (inputs on the GPU, weights, and for the LSTM stacks the output and workspace
buffers such a program keeps), `run(state)` makes one pass through the public entry points and returns its outputs,
`work(case)` says what the pass cannot do without and `tolerance(case)` how far two correct implementations may differ.

The kinds of call:

  b2b           core.b2b_gemm: D = (A @ B) @ C, fp16
  attention     core.flash_attention: fp16, prompts (many queries) and decoding (few queries on a long cache)
  attention_op  the blockwise attention program on FractalTensors (programs.flash_attention), fp32
  lstm          core.stacked_lstm: fp32 stack with plain or dilated recurrences, outputs and workspace kept by the caller
  lstm_f16      core.stacked_lstm_f16: the same with fp16 storage
  lstm_op       the stacked LSTM program on FractalTensors (programs.stacked_lstm), fp32
"""
from __future__ import annotations

import torch

from fractaltensor_amd import _core as core
from fractaltensor_amd import programs
from fractaltensor_amd.kaleido import FractalTensor


def listed():
    return [
        # the reference's fused two-GEMM benchmark at its smallest shape: a single product of a few microseconds
        dict(name='b2b_single', kind='b2b', G=1, M=8192, N=256, K=64, P=64),
        # the batched product: 32 problems, each a few times the size of its weights
        dict(name='b2b_batched', kind='b2b', G=32, M=4096, N=128, K=128, P=128),
        # the reference's attention example as it is written: fp32 blocks through the operator API, a short call
        dict(name='attention_program', kind='attention_op', B=2, Hd=8, S=1024, block=128, D=32),
        # a prompt of ordinary length over a batch
        dict(name='attention_prompt', kind='attention', B=8, Hd=16, Sq=2048, Skv=2048, D=128),
        # one new token per sample over a filled key / value cache
        dict(name='attention_decode', kind='attention', B=16, Hd=16, Sq=1, Skv=4096, D=128),
        # sequence lengths as they come, queries and keys of different lengths, the smaller head size
        dict(name='attention_ragged', kind='attention', B=3, Hd=12, Sq=777, Skv=1333, D=64),
        # one layer over a short batch of sentences, as an operator program: latency
        dict(name='lstm_program', kind='lstm_op', L=1, T=16, B=64, H=256),
        # the deep stack of the reference's sweep at its first hidden size
        dict(name='lstm_deep', kind='lstm', L=32, T=64, B=256, H=256, dilated=False),
        # the dilated stack (1, 2, 4, ... 32)
        dict(name='lstm_dilated', kind='lstm', L=6, T=128, B=256, H=256, dilated=True),
        # the stack the reference's framework comparison is quoted on
        dict(name='lstm_wide', kind='lstm', L=8, T=100, B=64, H=512, dilated=False),
        # the far end of the reference's depth sweep: a small model, many short dependent steps
        dict(name='lstm_narrow', kind='lstm', L=20, T=30, B=32, H=128, dilated=False),
        # the largest stack of the reference's sweep, fp16 storage
        dict(name='lstm_f16_wide', kind='lstm_f16', L=32, T=64, B=256, H=1024),
    ]


def _log(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(['b2b', 'attention', 'attention', 'attention_op', 'lstm', 'lstm', 'lstm', 'lstm_f16', 'lstm_op'])
    if kind == 'b2b':
        G = _log(rng, 1, 32)
        return dict(kind=kind, G=G, M=_log(rng, 512, min(16384, 131072 // G)), N=rng.choice([64, 128, 256, 512]),
                    K=rng.choice([64, 128]), P=rng.choice([64, 128, 256]))
    if kind == 'attention':
        D = rng.choice([64, 64, 128, 128, 96])
        if rng.random() < 0.5:                                       # decoding: 1 to 16 queries, up to 0.5 GB of cache
            B, Hd = _log(rng, 1, 32), rng.choice([8, 12, 16, 32])
            return dict(kind=kind, B=B, Hd=Hd, Sq=rng.choice([1, 1, 1, 4, 16]),
                        Skv=_log(rng, 256, min(32768, (1 << 27) // (B * Hd * D))), D=D)
        B, Hd, Sq = _log(rng, 1, 8), rng.choice([4, 8, 12, 16]), _log(rng, 64, 4096)
        Skv = Sq if rng.random() < 0.5 else _log(rng, 64, 4096)
        while 4 * B * Hd * Sq * Skv * D > 2.75e11 and B > 1:
            B //= 2
        return dict(kind=kind, B=B, Hd=Hd, Sq=Sq, Skv=Skv, D=D)
    if kind == 'attention_op':
        block = rng.choice([32, 64, 128])
        return dict(kind=kind, B=rng.randint(1, 4), Hd=rng.choice([4, 8, 12, 16]), S=block * _log(rng, 2, 2048 // block), block=block,
                    D=rng.choice([32, 64, 128]))
    if kind == 'lstm_op':
        return dict(kind=kind, L=rng.randint(1, 4), T=_log(rng, 8, 64), B=_log(rng, 8, 128), H=rng.choice([128, 256, 256]))
    if kind == 'lstm_f16':
        H = rng.choice([256, 512, 1024])
        return dict(kind=kind, L=_log(rng, 2, 32), T=_log(rng, 16, 64), B=_log(rng, 32, 256), H=H)
    H = rng.choice([64, 128, 256, 256, 512])
    L, T, B = _log(rng, 1, 32), _log(rng, 16, 128), _log(rng, 8, 256)
    while 16.0 * L * T * B * H * H > 1.1e12:
        L = L // 2
    return dict(kind=kind, L=L, T=T, B=B, H=H, dilated=L <= 6 and rng.random() < 0.4)


def _normal(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device='cuda', dtype=dtype)


def _uniform(gen, bound, *shape, dtype=torch.float32):
    return ((torch.rand(shape, generator=gen, device='cuda') * 2 - 1) * bound).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    kind = case['kind']
    state = dict(case=case)
    if kind == 'b2b':
        G, M, N, K, P = (case[k] for k in 'GMNKP')
        f16 = torch.float16
        state.update(A=_normal(gen, G, M, K, dtype=f16), B=_normal(gen, G, N, K, dtype=f16).mul_(K ** -0.5),
                     C=_normal(gen, G, P, N, dtype=f16).mul_(N ** -0.5))
    elif kind == 'attention':
        B, Hd, Sq, Skv, D = (case[k] for k in ('B', 'Hd', 'Sq', 'Skv', 'D'))
        state.update(q=_normal(gen, B, Hd, Sq, D, dtype=torch.float16), k=_normal(gen, B, Hd, Skv, D, dtype=torch.float16),
                     v=_normal(gen, B, Hd, Skv, D, dtype=torch.float16))
    elif kind == 'attention_op':
        B, Hd, S, blk, D = (case[k] for k in ('B', 'Hd', 'S', 'block', 'D'))
        q, k, v = (FractalTensor.from_dense(_normal(gen, B, Hd, S // blk, blk, D), 3) for _ in range(3))
        state.update(q=q, k=k, v=v, scale=D ** -0.5)
    elif kind == 'lstm_op':
        L, T, B, H = (case[k] for k in 'LTBH')
        bound = H ** -0.5                                            # the usual initialisation of an LSTM
        state.update(xss=FractalTensor.from_dense(_normal(gen, T, B, 1, H), 2), Wss=FractalTensor.from_dense(_uniform(gen, bound, L, 4, H, H), 2),
                     Uss=FractalTensor.from_dense(_uniform(gen, bound, L, 4, H, H), 2), bss=FractalTensor.from_dense(_uniform(gen, bound, L, 4, 1, H), 2))
    else:
        L, T, B, H = (case[k] for k in 'LTBH')
        bound, half = H ** -0.5, kind == 'lstm_f16'
        dtype = torch.float16 if half else torch.float32
        nbytes = (core.lib.ftk_stacked_lstm_f16_workspace_bytes if half else core.stacked_lstm_workspace_bytes)(L, T, B, H)
        state.update(xs=_normal(gen, T, B, H, dtype=dtype), WU=_uniform(gen, bound, L, 2 * H, 4 * H, dtype=dtype), bias=_uniform(gen, bound, L, 4 * H),
                     dilations=[2 ** l for l in range(L)] if case.get('dilated') else None,
                     out=(torch.empty((L, T, B, H), dtype=dtype, device='cuda'), torch.empty((L, T, B, H), dtype=dtype, device='cuda')),
                     workspace=torch.empty(nbytes, dtype=torch.uint8, device='cuda'))
    return state


def run(state):
    s, kind = state, state['case']['kind']
    if kind == 'b2b':
        return core.b2b_gemm(s['A'], s['B'], s['C'])
    if kind == 'attention':
        return core.flash_attention(s['q'], s['k'], s['v'])
    if kind == 'attention_op':
        return programs.flash_attention(s['q'], s['k'], s['v'], s['scale']).data
    if kind == 'lstm_op':
        return programs.stacked_lstm(s['xss'], s['Wss'], s['Uss'], s['bss']).data
    call = core.stacked_lstm_f16 if kind == 'lstm_f16' else core.stacked_lstm
    return call(s['xs'], s['WU'], s['bias'], dilations=s['dilations'], out=s['out'], workspace=s['workspace'])


def work(case):
    kind = case['kind']
    if kind == 'b2b':
        G, M, N, K, P = (case[k] for k in 'GMNKP')
        return dict(bytes=2 * G * (M * K + K * N + N * P + M * P), flops=2 * G * M * N * (K + P))
    if kind in ('attention', 'attention_op'):
        B, Hd, D = case['B'], case['Hd'], case['D']
        Sq, Skv = (case['Sq'], case['Skv']) if kind == 'attention' else (case['S'], case['S'])
        return dict(bytes=(2 if kind == 'attention' else 4) * 2 * B * Hd * D * (Sq + Skv), flops=4 * B * Hd * D * Sq * Skv)
    L, T, B, H = (case[k] for k in 'LTBH')
    size = 2 if kind == 'lstm_f16' else 4
    outputs = T * B * H if kind == 'lstm_op' else 2 * L * T * B * H    # the program returns the last layer's h only
    return dict(bytes=size * (T * B * H + 8 * L * H * H + outputs) + 16 * L * H, flops=16 * L * T * B * H * H)


def tolerance(case):
    if case['kind'] in ('b2b', 'attention'):
        return dict(rel=2e-3)                   # fp16 operands and results, fp32 accumulation
    if case['kind'] == 'lstm_f16':
        return dict(rel=5e-3)                   # h and c rounded to fp16 at every step and layer
    return dict(rel=1e-5)                       # fp32 throughout
