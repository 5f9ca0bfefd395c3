"""The quantized-matmul operators at the sizes they are used at: single-token and batched decode, prefill, and the
quantization of weights, through the public Python operators.

A case names an operator and its sizes; `prepare` makes what a program holds before the call (activations, quantized
weights, scales) from a seed, `run` makes the one call, `draw` gives further cases over the same ranges."""
import math

import torch

from hidet_amd.graph.ops import quant
from hidet_amd.graph.ops.matmul import matmul_f8 as f8

_DTYPES = {'float32': torch.float32, 'float16': torch.float16, 'bfloat16': torch.bfloat16}


def listed():
    return [
        # one token through an MLP up-projection: the smallest and most frequent call of a decode loop
        dict(name='w8a16_decode_one_token', op='w8a16', m=1, k=4096, n=11008, layout='row_major', bias=False),
        # sixteen sequences decoded together, an attention projection, codes stored K-contiguous as a decoding model keeps them
        dict(name='w8a16_decode_16_k_contiguous', op='w8a16', m=16, k=4096, n=4096, layout='k_contiguous', bias=False),
        # a larger decode batch (an odd number of sequences) through an MLP down-projection with its bias
        dict(name='w8a16_decode_49_bias', op='w8a16', m=49, k=11008, n=4096, layout='row_major', bias=True),
        # a prompt of 2048 tokens through the MLP up-projection
        dict(name='w8a16_prefill_2048', op='w8a16', m=2048, k=4096, n=11008, layout='row_major', bias=False),
        # a short prompt through a layer whose sizes are no multiples of the kernels' tiles
        dict(name='w8a16_ragged', op='w8a16', m=203, k=4100, n=4098, layout='row_major', bias=False),
        # int4 weights in groups of 128, one token
        dict(name='w4a16_decode_one_token', op='w4a16', m=1, k=4096, n=11008, group=128, dtype='bfloat16'),
        # int4 weights, a prompt of 512 tokens
        dict(name='w4a16_prefill_512', op='w4a16', m=512, k=4096, n=11008, group=128, dtype='bfloat16'),
        # an FP8 linear layer on 4096 tokens: the activations are quantized per tensor, then multiplied
        dict(name='fp8_linear_4096', op='fp8_linear', m=4096, k=8192, n=8192, dtype='bfloat16'),
        # the same layer on one token
        dict(name='fp8_linear_one_token', op='fp8_linear', m=1, k=8192, n=8192, dtype='bfloat16'),
        # the block-scaled FP8 matmul on a large batch of tokens
        dict(name='fp8_block_scaled_16384', op='fp8_block_scaled', m=16384, k=7168, n=1536),
        # a linear layer's weight to int8 codes with one scale per output column, and back (what the unfused graph reads)
        dict(name='int8_quantize_dequantize', op='int8_round_trip', rows=4096, cols=11008, dim=0, dtype='float32'),
        # the same weight to packed int4 codes in groups of 128
        dict(name='int4_group_quantize', op='int4_quantize', rows=4096, cols=11008, group=128, dtype='bfloat16'),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    return max(step, step * int(round(_log(rng, lo, hi) / step)))


def draw(rng):
    op = rng.choice(['w8a16', 'w8a16', 'w8a16', 'w4a16', 'w4a16', 'fp8_linear', 'fp8_linear', 'fp8_block_scaled',
                     'int8_round_trip', 'int4_quantize'])
    if op == 'w8a16':
        if rng.random() < 0.25:  # sizes off the tiles: the operator wants K and N even and nothing else
            return dict(op=op, m=_log(rng, 1, 256), k=_size(rng, 256, 4096, 2), n=_size(rng, 256, 4096, 2), layout='row_major',
                        bias=rng.random() < 0.3)
        m = _log(rng, 1, 2048)
        k_contiguous = m <= 64 and rng.random() < 0.4
        return dict(op=op, m=m, k=_size(rng, 1024, 11008, 64), n=_size(rng, 1024, 11008, 4 if rng.random() < 0.3 else 64),
                    layout='k_contiguous' if k_contiguous else 'row_major', bias=rng.random() < 0.3)
    if op == 'w4a16':
        return dict(op=op, m=_log(rng, 1, 1024), k=_size(rng, 1024, 11008, 128), n=_size(rng, 1024, 11008, 8 if rng.random() < 0.3 else 64),
                    group=rng.choice([64, 128, 128]), dtype=rng.choice(['bfloat16', 'bfloat16', 'float16']))
    if op == 'fp8_linear':
        return dict(op=op, m=_log(rng, 1, 4096), k=_size(rng, 1024, 8192, 16 if rng.random() < 0.2 else 128),
                    n=_size(rng, 1024, 8192, 4 if rng.random() < 0.3 else 64), dtype=rng.choice(['bfloat16', 'float16']))
    if op == 'fp8_block_scaled':
        return dict(op=op, m=_log(rng, 1, 16384), k=_size(rng, 1024, 7168, 128), n=_size(rng, 512, 4096, 128))
    if op == 'int8_round_trip':
        cols = _log(rng, 512, 11008) if rng.random() < 0.3 else _size(rng, 512, 11008, 64)
        return dict(op=op, rows=_log(rng, 512, 4096), cols=cols, dim=rng.choice([0, 0, 1]),
                    dtype=rng.choice(['float32', 'float32', 'float16', 'bfloat16']))
    return dict(op=op, rows=_size(rng, 512, 4096, 128), cols=_size(rng, 512, 11008, 2 if rng.random() < 0.3 else 64),
                group=rng.choice([64, 128, 128]), dtype=rng.choice(['bfloat16', 'float16']))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device='cuda', dtype=torch.float32) * std


def prepare(case, seed):
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    op = case['op']
    if op == 'w8a16':
        wq, scale = quant.symmetric_quantize(_normal(g, (case['k'], case['n']), 0.02), 'int8', dims=0)
        if case['layout'] == 'k_contiguous':
            wq = quant.to_decode_layout(wq)
        bias = _normal(g, (case['n'],), 0.1).half() if case['bias'] else None
        return dict(op=op, x=_normal(g, (case['m'], case['k'])).half(), wq=wq, scale=scale.half(), bias=bias)
    if op == 'w4a16':
        dtype = _DTYPES[case['dtype']]
        packed, scales = quant.symmetric_group_quantize_int4(_normal(g, (case['k'], case['n']), 0.02), case['group'], dtype)
        return dict(op=op, x=_normal(g, (case['m'], case['k'])).to(dtype), packed=packed, scales=scales, group=case['group'])
    if op == 'fp8_linear':
        w, w_scale = f8.fp8_quantize_per_tensor(_normal(g, (case['n'], case['k']), 0.02))
        return dict(op=op, x=_normal(g, (case['m'], case['k'])).to(_DTYPES[case['dtype']]), w=w, w_scale=w_scale,
                    dtype=_DTYPES[case['dtype']])
    if op == 'fp8_block_scaled':
        # codes as block quantization leaves them (the largest of a block of normal values at 448) and its float32 scales
        m, k, n = case['m'], case['k'], case['n']
        a = (_normal(g, (m, k), 150.0)).clamp(-448, 448).to(torch.float8_e4m3fn)
        b = (_normal(g, (n, k), 110.0)).clamp(-448, 448).to(torch.float8_e4m3fn)
        scale_a = (2.5 + torch.rand((k // 128, m), generator=g, device='cuda')) / 448
        scale_b = (3.5 + torch.rand((n // 128, k // 128), generator=g, device='cuda')) * 0.02 / 448
        return dict(op=op, a=a, b=b, scale_a=scale_a, scale_b=scale_b)
    if op == 'int8_round_trip':
        return dict(op=op, w=_normal(g, (case['rows'], case['cols']), 0.02).to(_DTYPES[case['dtype']]), dim=case['dim'])
    return dict(op=op, w=_normal(g, (case['rows'], case['cols']), 0.02), group=case['group'], dtype=_DTYPES[case['dtype']])


def run(state):
    op = state['op']
    if op == 'w8a16':
        return quant.symmetric_quant_matmul(state['x'], state['wq'], state['scale'], state['bias'])
    if op == 'w4a16':
        return quant.symmetric_quant_matmul_w4a16(state['x'], state['packed'], state['scales'], state['group'])
    if op == 'fp8_linear':
        x, x_scale = f8.fp8_quantize_per_tensor(state['x'])
        return f8.matmul_f8_per_tensor(x, state['w'], x_scale, state['w_scale'], output_dtype=state['dtype'])
    if op == 'fp8_block_scaled':
        return f8.matmul_f8_scaled(state['a'], state['b'], state['scale_a'], state['scale_b'], output_dtype='bfloat16')
    if op == 'int8_round_trip':
        wq, scale = quant.symmetric_quantize(state['w'], 'int8', dims=state['dim'])
        return wq, scale, quant.symmetric_dequantize(wq, scale, dims=state['dim'])
    return quant.symmetric_group_quantize_int4(state['w'], state['group'], state['dtype'])


def work(case):
    """Each input read once and each output written once; what a call makes and reads again itself is not counted."""
    op = case['op']
    if op in ('int8_round_trip', 'int4_quantize'):
        r, c = case['rows'], case['cols']
        if op == 'int4_quantize':
            return dict(bytes=r * c * 4 + r * c // 2 + (r // case['group']) * c * 2, flops=0)
        e = 4 if case['dtype'] == 'float32' else 2
        return dict(bytes=r * c * (e + 1 + e) + (c if case['dim'] == 0 else r) * e, flops=0)
    m, k, n = case['m'], case['k'], case['n']
    if op == 'w8a16':
        moved = k * n + 2 * m * k + 2 * m * n + 2 * n + (2 * n if case['bias'] else 0)
    elif op == 'w4a16':
        moved = k * n // 2 + 2 * (k // case['group']) * n + 2 * m * k + 2 * m * n
    elif op == 'fp8_linear':
        moved = n * k + 2 * m * k + 2 * m * n + 4
    else:
        moved = m * k + n * k + 4 * (k // 128) * (m + n // 128) + 2 * m * n
    return dict(bytes=moved, flops=2 * m * k * n)


def tolerance(case):
    """Four times what the operators showed against the same sums in float64 (the rounding of the 16-bit results; for int4
    also that of the weights, which one correct implementation rounds to 16 bits and another does not)."""
    op = case['op']
    if op in ('int8_round_trip', 'int4_quantize'):
        return 'exact'
    if op == 'w8a16':
        return {'rel': 1.2e-3 if case['bias'] else 1e-3}  # a bias is added with a second rounding
    half = case.get('dtype') == 'float16'
    if op == 'w4a16':
        return {'rel': 1.2e-3 if half else 1e-2}
    return {'rel': 1e-3 if half else 7e-3}
