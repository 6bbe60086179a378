"""The work a user of this package has it do, as cases that can be timed and compared: whole stages of the pi0.5 and GR00T
policies through the module layer, and the operations that are called on their own (the rotation, the W8A8 product, the
2-bit layer stream).

  rotation   kernels.rht on token rows: the randomized Walsh rotation in front of every quantized layer
  w8a8       kernels.gemm_i8: the INT8 product of a prefill with per-token and per-channel scales (or exact int32 sums)
  stream     a stream of 2-bit layers with the FP16 table: pre_h16 once, then one gemv_f16_post over all layers
  expert     one flow-matching step of the action expert (ExpertPolicy.velocity) against a prefix cache, as a HIP graph
  decode     one token through the language model with its cache (BackbonePolicy.decode_step_cached), as a HIP graph
  prefill    the language model over the prefix (BackbonePolicy.prefill), as a HIP graph
  vision     one SigLIP encoder layer's quantized modules (q / k / v / out projections, MLP) over 1 to 3 images
  groot      one GR00T block's quantized modules (DiT, language model or vision tower) on one-sided or two-sided records
  float      one layer's projections on the W2 float path (BF16 activations, install(..., a8=False))

Whole stages run from a captured graph because a policy's serving loop runs them so (its shapes are fixed); the three
single operations are called as they stand.
"""
import math

import torch

from yanlongvla_amd import gemma, groot, kernels, modules
from yanlongvla_amd import tcq_format as F

DEV = 'cuda'
WIDTHS = (1024, 1152, 1536, 2048, 3072, 4096, 4304, 6144, 8192, 16384)      # row widths of the two policies
PRODUCTS = ((2560, 2048), (2048, 2048), (16384, 2048), (2048, 16384), (3072, 1024), (1024, 4096), (4304, 1152), (6144, 1536))
DT = dict(bf16=torch.bfloat16, f16=torch.float16, f32=torch.float32, i32=torch.int32)


def listed():
    return [
        # the rotation of one prefill's rows at the widest MLP, memory traffic first
        dict(name='rotation_800x16384', kind='rotation', M=800, n=16384, dtype='bf16'),
        # the exact product of a prefill's gate or up projection
        dict(name='w8a8_800x2048x16384', kind='w8a8', M=800, N=16384, K=2048, out='i32'),
        # decode-GEMV over more distinct layers than any cache holds, one token
        dict(name='stream_1024', kind='stream', layers=1024, m=2048, n=2048, M=1),
        # a denoising step as the reference deploys it: 10 action tokens, 968 prefix rows, 2-bit weights decoded per call
        dict(name='expert_10_fly', kind='expert', layers=18, M=10, P=968, runtime='fly'),
        # the longer action horizon on resident INT8 weights (what the hybrid operating point runs inside a chunk)
        dict(name='expert_50_resident', kind='expert', layers=4, M=50, P=800, runtime='resident'),
        # one generated token, 2-bit and INT8 weights
        dict(name='decode_fly', kind='decode', layers=4, P=800, runtime='fly'),
        dict(name='decode_resident', kind='decode', layers=4, P=800, runtime='resident'),
        # the prefix of one observation, 2-bit and INT8 weights
        dict(name='prefill_968_fly', kind='prefill', layers=2, M=968, runtime='fly'),
        dict(name='prefill_800_resident', kind='prefill', layers=2, M=800, runtime='resident'),
        # three camera images in one vision pass: widths that are not powers of two, biases, the plain MLP
        dict(name='vision_768_fly', kind='vision', M=768, runtime='fly'),
        # a self-attention DiT block of GR00T's action head: row-group tables, column scales, one-sided records
        dict(name='groot_dit_50', kind='groot', block='dit_self', M=50, runtime='fly', one_sided=True),
        # the float path over the reference's prefix
        dict(name='float_968_fly', kind='float', part='llm', M=968, runtime='fly'),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(('rotation', 'w8a8', 'stream', 'expert', 'decode', 'prefill', 'vision', 'groot', 'float'))
    runtime = rng.choice(('fly', 'resident'))
    if kind == 'rotation':
        return dict(kind=kind, M=_log_int(rng, 1, 968), n=rng.choice(WIDTHS), dtype=rng.choice(('bf16', 'bf16', 'f16', 'f32')))
    if kind == 'w8a8':
        N, K = rng.choice(PRODUCTS)
        return dict(kind=kind, M=_log_int(rng, 1, 968), N=N, K=K, out=rng.choice(('i32', 'f32', 'bf16')))
    if kind == 'stream':
        return dict(kind=kind, layers=_log_int(rng, 256, 1024), m=rng.choice((1024, 2048)), n=rng.choice((1024, 2048)),
                    M=_log_int(rng, 1, 6))
    if kind == 'expert':
        return dict(kind=kind, layers=rng.randint(2, 6), M=_log_int(rng, 4, 64), P=rng.randint(200, 968), runtime=runtime)
    if kind == 'decode':
        return dict(kind=kind, layers=rng.randint(2, 4), P=_log_int(rng, 64, 1024), runtime=runtime)
    if kind == 'prefill':
        return dict(kind=kind, layers=2, M=_log_int(rng, 100, 968), runtime=runtime)
    if kind == 'vision':
        return dict(kind=kind, M=256 * rng.randint(1, 3) + rng.choice((0, 0, 1, 17)), runtime=runtime)
    if kind == 'groot':
        block = rng.choice(('dit_self', 'dit_cross', 'lm', 'visual'))
        M = _log_int(rng, 10, 64) if block.startswith('dit') else _log_int(rng, 64, 512)
        return dict(kind=kind, block=block, M=M, runtime=runtime, one_sided=rng.random() < 0.7)
    part = rng.choice(('llm', 'expert'))
    return dict(kind=kind, part=part, M=_log_int(rng, 4, 64) if part == 'expert' else _log_int(rng, 100, 968), runtime=runtime)


# --------------------------------------------------------------------------------------------- layers of a stage, inputs
_EXPERT = 'paligemma_with_expert.gemma_expert.model.layers.'
_LLM = 'paligemma_with_expert.paligemma.language_model.layers.'
_VISION = 'vision_tower.vision_model.encoder.layers.0.'
_DIT = 'action_head.model.transformer_blocks.'
_GROOT_LM = 'backbone.model.model.language_model.layers.2.'
_GROOT_VIS = 'backbone.model.model.visual.blocks.5.'
GROOT_BLOCKS = {     # leaf -> (m, n); one input per width of a parent's family, as the policy's block passes them
    'dit_self': (_DIT + '1.', {'attn1.to_q': (1536, 1536), 'attn1.to_k': (1536, 1536), 'attn1.to_v': (1536, 1536),
                               'attn1.to_out.0': (1536, 1536), 'ff.net.0.proj': (6144, 1536), 'ff.net.2': (1536, 6144)}),
    'dit_cross': (_DIT + '4.', {'attn1.to_q': (1536, 1536), 'attn1.to_k': (1536, 2048), 'attn1.to_v': (1536, 2048),
                                'attn1.to_out.0': (1536, 1536), 'ff.net.0.proj': (6144, 1536), 'ff.net.2': (1536, 6144)}),
    'lm': (_GROOT_LM, {'self_attn.q_proj': (2048, 2048), 'self_attn.k_proj': (1024, 2048), 'self_attn.v_proj': (1024, 2048),
                       'self_attn.o_proj': (2048, 2048), 'mlp.gate_proj': (6144, 2048), 'mlp.up_proj': (6144, 2048),
                       'mlp.down_proj': (2048, 6144)}),
    'visual': (_GROOT_VIS, {'attn.qkv': (3072, 1024), 'attn.proj': (1024, 1024), 'mlp.linear_fc1': (4096, 1024),
                            'mlp.linear_fc2': (1024, 4096)}),
}


def _gemma_shapes(width, hidden):
    return {'self_attn.q_proj': (2048, width), 'self_attn.k_proj': (256, width), 'self_attn.v_proj': (256, width),
            'self_attn.o_proj': (width, 2048), 'mlp.gate_proj': (hidden, width), 'mlp.up_proj': (hidden, width),
            'mlp.down_proj': (width, hidden)}


_SIGLIP = {'self_attn.q_proj': (1152, 1152), 'self_attn.k_proj': (1152, 1152), 'self_attn.v_proj': (1152, 1152),
           'self_attn.out_proj': (1152, 1152), 'mlp.fc1': (4304, 1152), 'mlp.fc2': (1152, 4304)}


def _shapes(case):
    """{layer name: (m, n)} of the quantized layers one pass runs."""
    kind = case['kind']
    if kind == 'vision':
        return {_VISION + leaf: s for leaf, s in _SIGLIP.items()}
    if kind == 'groot':
        prefix, leaves = GROOT_BLOCKS[case['block']]
        return {prefix + leaf: s for leaf, s in leaves.items()}
    expert = kind == 'expert' or case.get('part') == 'expert'
    prefix, width, hidden = (_EXPERT, 1024, 4096) if expert else (_LLM, 2048, 16384)
    return {f'{prefix}{i}.{leaf}': s for i in range(case.get('layers', 1)) for leaf, s in _gemma_shapes(width, hidden).items()}


_FAMILIES = (('q_proj', 'k_proj', 'v_proj'), ('gate_proj', 'up_proj'), ('to_q', 'to_k', 'to_v'))


def _input_key(name, n):
    """Layers with one key read one tensor with one set of input signs."""
    parent, _, leaf = name.rpartition('.')
    family = next((i for i, f in enumerate(_FAMILIES) if leaf in f), None)
    return name if family is None else f'{parent}/{family}/{n}'


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _signs(g, n):
    return (torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1).to(torch.int8)


def _words(g, *shape):
    return torch.randint(-32768, 32768, shape, generator=g, device=DEV, dtype=torch.int32).to(torch.int16)


def _records(case, g):
    """{layer name: packed tensors}: uniform words, a normal table, scales that keep a layer's outputs near its inputs'
    size, signs shared by the layers that read one tensor, biases where the policy has them."""
    out, shared = {}, {}
    gain = 0.4 if case['kind'] in ('expert', 'decode', 'prefill') else 1.0      # a layer adds less than the residual holds
    two_sided = case['kind'] != 'groot' or not case['one_sided']
    for name, (m, n) in _shapes(case).items():
        key = f'width/{n}' if case['kind'] == 'groot' else _input_key(name, n)
        if key not in shared:
            cs = (torch.rand(n, generator=g, device=DEV) + 0.5).half() if case['kind'] == 'groot' else None
            shared[key] = _signs(g, n), cs
        su, cs = shared[key]
        tables = groot.row_groups(m, n) if case['kind'] == 'groot' else 1
        t = dict(bits=_words(g, (m // 16) * (n // 16), 32),
                 tlut=torch.randn(*((tables,) if tables > 1 else ()), 512, 2, generator=g, device=DEV).half(),
                 row_scale=((torch.rand(m, generator=g, device=DEV) + 0.5) * gain / math.sqrt(n)).half(), su=su)
        if two_sided:
            t['sv'] = _signs(g, m)
        if cs is not None:
            t['col_scale'] = cs
        biased = case['kind'] == 'vision' or (case['kind'] == 'groot' and case['block'] != 'lm')
        out[name] = t, torch.randn(m, generator=g, device=DEV) * 0.1 if biased else None
    return out


def _rows(g, M, n, dtype=torch.bfloat16):
    """Token rows as the policies' hidden states look: unit scale with a few large columns."""
    x = torch.randn(M, n, generator=g, device=DEV)
    x[:, :: max(1, n // 8)] *= 8.0
    return x.to(dtype)


def _data(case, seed):
    """Everything a pass reads, from the seed alone."""
    g, kind = _gen(seed), case['kind']
    if kind == 'rotation':
        return dict(x=_rows(g, case['M'], case['n'], DT[case['dtype']]), su=_signs(g, case['n']))
    if kind == 'w8a8':
        M, N, K = case['M'], case['N'], case['K']
        return dict(a=torch.randint(-127, 128, (M, K), generator=g, device=DEV, dtype=torch.int8),
                    w=torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8),
                    sa=torch.rand(M, generator=g, device=DEV) * 0.02 + 0.01, sw=torch.rand(N, generator=g, device=DEV) * 0.002 + 1e-4)
    if kind == 'stream':
        L, m, n = case['layers'], case['m'], case['n']
        return dict(x=_rows(g, case['M'], n, torch.float16), su=_signs(g, n), bits=_words(g, L, (m // 16) * (n // 16), 32),
                    tlut=torch.randn(L, 512, 2, generator=g, device=DEV).half(), sv=_signs(g, L * m).view(L, m),
                    row_scale=((torch.rand(L, m, generator=g, device=DEV) + 0.5) / math.sqrt(n)).half())
    d = dict(records=_records(case, g))
    if kind in ('expert', 'decode', 'prefill'):
        width = 1024 if kind == 'expert' else 2048
        d['norms'] = [(0.1 * torch.randn(width, generator=g, device=DEV)).bfloat16() for _ in range(2 * case['layers'] + 1)]
        if kind == 'expert':
            d['proj_in'] = (torch.randn(width, 32, generator=g, device=DEV) / math.sqrt(32)).bfloat16()
            d['proj_out'] = (torch.randn(32, width, generator=g, device=DEV) / math.sqrt(width)).bfloat16()
            d['x'] = torch.randn(case['M'], 32, generator=g, device=DEV).bfloat16()
        else:
            d['x'] = _rows(g, case.get('M', 1), width)
        if kind != 'prefill':
            d['k'], d['v'] = ([torch.randn(case['P'], 256, generator=g, device=DEV).bfloat16() for _ in range(case['layers'])]
                              for _ in range(2))
    else:
        d['x'] = {}
        for name, (m, n) in _shapes(case).items():
            key = _input_key(name, n)
            if key not in d['x'] and not (kind == 'vision' and name.endswith('fc2')):
                d['x'][key] = _rows(g, case['M'], n)
    return d


# ------------------------------------------------------------------------------------------------------ prepare and run
class SiglipMLP(torch.nn.Module):
    """The vision encoder's MLP under its policy name; install puts the quantized one in its place."""

    def __init__(self):
        super().__init__()
        self.fc1, self.fc2 = torch.nn.Linear(1152, 4304, device='meta'), torch.nn.Linear(4304, 1152, device='meta')


def _tree(shapes):
    """A module tree holding an nn.Linear (meta device: its weight is never read) at each of the given names."""
    root = torch.nn.Module()
    for name, (m, n) in shapes.items():
        *path, leaf = name.split('.')
        at = root
        for p in path:
            if p not in at._modules:
                at.add_module(p, SiglipMLP() if p == 'mlp' and name.startswith('vision_tower') else torch.nn.Module())
            at = at._modules[p]
        if leaf not in at._modules:
            at.add_module(leaf, torch.nn.Linear(n, m, bias=False, device='meta'))
    return root


def _install(model, case, records, a8=True):
    layers = {name: F.Layer(name, t, bias=b, device=DEV) for name, (t, b) in records.items()}
    modules.install(model, runtime=case['runtime'], layers=layers, a8=a8)
    return model


def _policy(case, d):
    cls = gemma.ExpertPolicy if case['kind'] == 'expert' else gemma.BackbonePolicy
    extra = {} if case['kind'] == 'expert' else dict(vocab=16)
    model = gemma.make_policy(cls, DEV, layers=case['layers'], **extra)
    norms = iter(d['norms'])
    for layer in model.stack.layers:
        layer.input_layernorm.weight.data.copy_(next(norms))
        layer.post_attention_layernorm.weight.data.copy_(next(norms))
    model.stack.norm.weight.data.copy_(next(norms))
    return _install(model, case, d['records'])


def _captured(call):
    """(graph, outputs) of one call, warmed up on the capturing stream first."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def prepare(case, seed):
    d, kind = _data(case, seed), case['kind']
    st = dict(case=case, d=d)
    if kind == 'rotation':
        st['y'] = torch.empty_like(d['x'])
    elif kind == 'w8a8':
        st['out'] = torch.empty(case['M'], case['N'], dtype=DT[case['out']], device=DEV)
    elif kind == 'stream':
        L, m, n, M = case['layers'], case['m'], case['n'], case['M']
        words = torch.empty(L, kernels.repack_words(m, n), dtype=torch.int32, device=DEV)
        for i in range(L):
            kernels.repack(d['bits'][i], m, n, out=words[i])
        y = torch.empty(L, M, m, dtype=torch.float16, device=DEV)
        st.update(words=words, y=y, h=torch.empty(M, n, dtype=torch.float16, device=DEV), hs=torch.empty(M, device=DEV))
        st['desc'] = kernels.gemv_post_descriptors([(words[i], d['tlut'][i], d['row_scale'][i], d['sv'][i], None, y[i]) for i in range(L)])
        d['bits'] = None
    elif kind in ('expert', 'decode', 'prefill'):
        model = st['model'] = _policy(case, d)
        with torch.inference_mode():
            if kind == 'expert':
                model.set_prefix(d['k'], d['v'])
                model.action_in_proj.weight.data.copy_(d['proj_in'])
                model.action_out_proj.weight.data.copy_(d['proj_out'])
                st['graph'], st['out'] = _captured(lambda: model.velocity(d['x']))
            elif kind == 'decode':
                cache = st['cache'] = gemma.KVCache(d['k'], d['v'], 1)

                def token():
                    cache.rewind()
                    return model.decode_step_cached(d['x'], cache)
                st['graph'], hidden = _captured(token)
                st['out'] = hidden, [t[case['P']:] for t in cache.k], [t[case['P']:] for t in cache.v]
            else:
                st['graph'], st['out'] = _captured(lambda: model.prefill(d['x']))
    else:
        model = st['model'] = _install(_tree(_shapes(case)), case, d['records'], a8=kind != 'float')
        st['calls'] = [(model.get_submodule(n), d['x'][_input_key(n, s[1])]) for n, s in _shapes(case).items()
                       if not (kind == 'vision' and '.mlp.' in n)]
        if kind == 'vision':
            st['calls'].append((model.get_submodule(_VISION + 'mlp'), d['x'][_VISION + 'mlp.fc1']))
        with torch.inference_mode():
            st['graph'], st['out'] = _captured(lambda: [mod(x) for mod, x in st['calls']])
    d.pop('records', None)
    return st


def run(st):
    case, d, kind = st['case'], st['d'], st['case']['kind']
    if 'graph' in st:
        st['graph'].replay()
        return st['out']
    if kind == 'rotation':
        return kernels.rht(d['x'], d['su'], st['y'])
    if kind == 'w8a8':
        scaled = case['out'] != 'i32'
        return kernels.gemm_i8(d['a'], d['w'], st['out'], sa=d['sa'] if scaled else None, sw=d['sw'] if scaled else None)
    kernels.pre_h16(d['x'], d['su'], st['h'], st['hs'])
    kernels.gemv_f16_post(st['desc'], st['h'], st['hs'], case['m'], case['n'], torch.float16)
    return st['y']


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    """Every input read once, every output written once, the products' multiply-adds (the rotations' butterflies in
    'rotation' only: elsewhere they are far below the products)."""
    kind, M = case['kind'], case.get('M', 1)
    if kind == 'rotation':
        size = 4 if case['dtype'] == 'f32' else 2
        return dict(bytes=2 * M * case['n'] * size + case['n'], flops=sum(M * w * (w.bit_length() - 1) for w in _blocks(case['n'])))
    if kind == 'w8a8':
        N, K = case['N'], case['K']
        return dict(bytes=M * K + N * K + M * N * (2 if case['out'] == 'bf16' else 4) + 4 * (M + N) * (case['out'] != 'i32'),
                    flops=2 * M * N * K)
    if kind == 'stream':
        L, m, n = case['layers'], case['m'], case['n']
        return dict(bytes=L * (m * n // 4 + 2048 + 3 * m + 2 * M * m) + 2 * M * n + n, flops=2 * L * M * m * n)
    weights = sum(m * n for m, n in _shapes(case).values())
    sides = sum(m * 5 + n for m, n in _shapes(case).values())                  # scales and signs
    moved = weights // (1 if case['runtime'] == 'resident' else 4) + sides
    flops = 2 * M * weights
    layers = case.get('layers', 1)
    if kind in ('expert', 'decode', 'prefill'):
        P = case.get('P', 0)
        seen = M * (M + 1) // 2 if kind == 'prefill' else M * (P + M)
        flops += layers * 4 * seen * 2048
        moved += layers * 4 * 256 * P + 4 * M * (32 if kind == 'expert' else 2048) + (0 if kind == 'expert' else layers * 4 * 256 * M)
    else:
        moved += sum(2 * M * n for n in {_input_key(k, s[1]): s[1] for k, s in _shapes(case).items()}.values())
        moved += sum(2 * M * m for m, n in _shapes(case).values())
        if kind == 'vision':
            moved -= 4 * M * 4304                                               # the MLP's middle is nobody's output
    return dict(bytes=moved, flops=flops)


def tolerance(case):
    kind = case['kind']
    if kind == 'rotation':                     # FP32 butterflies, one rounding to the output type
        return dict(rel=dict(f32=1e-6, f16=1e-3, bf16=8e-3)[case['dtype']])
    if kind == 'w8a8':                         # whole sums; their scaling in FP32
        return 'exact' if case['out'] == 'i32' else dict(rel=1e-6 if case['out'] == 'f32' else 8e-3)
    if kind == 'stream':                       # FP16 activations and tables, FP32 sums, FP16 outputs
        return dict(rel=1.2e-3)
    if kind in ('float', 'groot'):             # BF16 outputs; an activation at a rounding tie moves by one step
        return dict(rel=2e-3)
    if kind == 'vision':                       # the same through two layers
        return dict(rel=4e-3)
    return dict(rel=0.03)                      # stacks of layers: the same, through every layer that follows


# ------------------------------------------------------------------------------------------ the same results in 64 bits
def _blocks(width):
    out = []
    while width:
        out.append(1 << (width.bit_length() - 1))
        width -= out[-1]
    return out


def _walsh(x):
    """Block Walsh of the last axis, orthonormal."""
    parts, at = [], 0
    for w in _blocks(x.shape[-1]):
        y, h = x[..., at:at + w], 1
        while h < w:
            y = y.reshape(-1, w // (2 * h), 2, h)
            y = torch.stack((y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]), 2)
            h *= 2
        parts.append(y.reshape(*x.shape[:-1], w) / math.sqrt(w))
        at += w
    return torch.cat(parts, -1)


def _decoded(bits, table, m, n):
    """(m, n) table values of the trellis words: state t of a 16 x 16 tile is bits [4 t, 4 t + 16) of its 512, the end
    running into the start; hash x = (s + 1) s, entry (x >> 6) & 511, bit 15 negating the first coordinate."""
    b = bits.long() & 0xffff
    t = torch.arange(128, device=b.device)
    s = (((b[:, t // 4] << 16) | b[:, (t // 4 + 1) % 32]) >> (16 - 4 * (t % 4))) & 0xffff
    s = s.view(m // 16, n // 16, 16, 8).permute(0, 2, 1, 3).reshape(m, n // 2)
    x = (s + 1) * s
    table = table.double().view(-1, 512, 2)
    row = torch.arange(m, device=b.device)[:, None] // (m // table.shape[0])
    v = table[row, (x >> 6) & 511]
    return torch.stack((torch.where((x >> 15) & 1 == 1, -v[..., 0], v[..., 0]), v[..., 1]), -1).view(m, n)


def _snapped(t):
    """(INT8 table, row scale) of one layer's tables."""
    tables = t['tlut'].float().view(-1, 512, 2)
    gain = (1.0 / tables.abs().amax((1, 2))) * 127.0
    t8 = torch.clamp(torch.round(tables * gain[:, None, None]), -127, 127)
    return t8, t['row_scale'].double() / gain.double().repeat_interleave(t['row_scale'].numel() // gain.numel())


def _bf(x):
    return x.bfloat16().double()


def _linear(x, record, mode='a8'):
    """One quantized layer in 64 bits; the INT8 (or, on the float path, BF16) activations belong to its definition."""
    t, bias = record
    m, n = t['row_scale'].numel(), t['su'].numel()
    t8, rs = _snapped(t)
    w = _decoded(t['bits'], t8, m, n)
    h = _walsh(x.double() * t['su'].double())
    if t.get('col_scale') is not None:
        h = h * t['col_scale'].double()
    if mode == 'a8':
        s = h.abs().amax(1, keepdim=True) / 127.0
        s = torch.where(s > 0, s, torch.ones_like(s))
        z = (torch.clamp(torch.round(h / s), -127, 127) @ w.t()) * s * rs
    else:
        z = _bf(h) @ w.t()
        z = (_bf(z) if mode == 'llm' else z) * rs
    if t.get('sv') is not None:
        z = _walsh(z) * t['sv'].double()
    return _bf(z if bias is None else z + bias.double())


def _norm(x, w):
    return _bf(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1.0 + w.double()))


def _attention(q, k, v, causal):
    M, T = q.shape[0], k.shape[0]
    s = q.view(M, 8, 256).transpose(0, 1) @ k.t() / 16.0
    if causal:
        s = s.masked_fill(torch.ones(M, T, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    return _bf((torch.softmax(s, -1) @ v).transpose(0, 1).reshape(M, 2048))


def _gelu(x):
    return _bf(torch.nn.functional.gelu(x, approximate='tanh'))


def _decoder(case, d):
    expert = case['kind'] == 'expert'
    rec, norms, prefix = d['records'], iter(d['norms']), _EXPERT if expert else _LLM
    x = _bf(d['x'].double() @ d['proj_in'].double().t()) if expert else d['x'].double()
    ks, vs = [], []
    for i in range(case['layers']):
        def lin(y, leaf):
            return _linear(y, rec[f'{prefix}{i}.{leaf}'])
        h = _norm(x, next(norms))
        q, k, v = (lin(h, f'self_attn.{c}_proj') for c in 'qkv')
        ks.append(k), vs.append(v)
        if 'k' in d:
            k, v = torch.cat((d['k'][i].double(), k)), torch.cat((d['v'][i].double(), v))
        x = _bf(x + lin(_attention(q, k, v, case['kind'] == 'prefill'), 'self_attn.o_proj'))
        h = _norm(x, next(norms))
        x = _bf(x + lin(_bf(_gelu(lin(h, 'mlp.gate_proj')) * lin(h, 'mlp.up_proj')), 'mlp.down_proj'))
    x = _norm(x, next(norms))
    return _bf(x @ d['proj_out'].double().t()) if expert else (x, ks, vs)


def exact(case, seed):
    d, kind = _data(case, seed), case['kind']
    if kind == 'rotation':
        return _walsh(d['x'].double() * d['su'].double())
    if kind == 'w8a8':
        if case['out'] == 'i32':
            return None
        return (d['a'].double() @ d['w'].double().t()) * d['sa'].double()[:, None] * d['sw'].double()
    if kind == 'stream':
        h = _walsh(d['x'].double() * d['su'].double())
        y = [(h @ _decoded(d['bits'][i], d['tlut'][i], case['m'], case['n']).t()) * d['row_scale'][i].double() for i in range(case['layers'])]
        return _walsh(torch.stack(y)) * d['sv'].double()[:, None, :]
    if kind in ('expert', 'decode', 'prefill'):
        return _decoder(case, d)
    if kind == 'vision':
        fc1, fc2 = _VISION + 'mlp.fc1', _VISION + 'mlp.fc2'
        out = [_linear(d['x'][_input_key(n, s[1])], d['records'][n]) for n, s in _shapes(case).items() if '.mlp.' not in n]
        return out + [_linear(_gelu(_linear(d['x'][fc1], d['records'][fc1])), d['records'][fc2])]
    mode = 'a8' if kind == 'groot' else case['part']
    return [_linear(d['x'][_input_key(n, s[1])], d['records'][n], mode) for n, s in _shapes(case).items()]
