"""Dense weights of a layer group in one launch (tcq_decode_group, tcq_i8_to_bf16) and the float path's many-token product."""
import numpy as np
import pytest
import torch

from oracle import tcq_oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'


def layer(m, n, seed, tables=1):
    from yanlongvla_amd import tcq_format as F
    g = torch.Generator(device=DEV).manual_seed(seed)
    t = dict(bits=torch.randint(-32768, 32768, ((m // 16) * (n // 16), 32), generator=g, device=DEV, dtype=torch.int32).to(torch.int16),
             tlut=torch.randn(*((tables,) if tables > 1 else ()), 512, 2, generator=g, device=DEV).half(),
             row_scale=((torch.rand(m, generator=g, device=DEV) + 0.5) * 0.02).half(),
             su=(torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1).to(torch.int8),
             sv=(torch.randint(0, 2, (m,), generator=g, device=DEV) * 2 - 1).to(torch.int8))
    return F.Layer(f'l{seed}', t, device=DEV)


# (rows, tables) of the segments and their width: both workgroup sizes, one / two / four chunks per wave, partial chunks,
# uneven segments, row-group tables beside single ones
GROUPS = [([(16, 1)], 16), ([(2048, 1), (256, 1), (256, 1)], 2048), ([(48, 1), (32, 2), (64, 4)], 400), ([(1152, 1)] * 3, 1152),
          ([(4304, 1)], 1152), ([(4096, 16)], 2064), ([(16384, 1)] * 2, 2048), ([(16384, 8), (16400, 1)], 4304)]


@pytest.mark.parametrize('shapes,n', GROUPS)
def test_decode_group_equals_decode(shapes, n):
    from yanlongvla_amd import kernels as Kn
    layers = [layer(m, n, 10 + i, G) for i, (m, G) in enumerate(shapes)]
    want = [Kn_decode(L) for L in layers]
    total = sum(m for m, _ in shapes)
    for dt in (torch.int8, torch.bfloat16):
        out = torch.full((total + 1, n), 99, dtype=dt, device=DEV)
        c, segs = 0, []
        for L in layers:
            segs.append((L.words(), L.t8, out[c:c + L.m]))
            c += L.m
        Kn.decode_group(segs, n)
        for (_, _, got), w in zip(segs, want):
            assert torch.equal(got.float(), w.float())
        assert bool((out[total] == 99).all())
    for w in want:
        assert torch.equal(Kn.i8_to_bf16(w, torch.empty_like(w, dtype=torch.bfloat16)), w.bfloat16())


def Kn_decode(L):
    from yanlongvla_amd import kernels as Kn
    out = torch.empty(L.m, L.n, dtype=torch.int8, device=DEV)
    Kn.decode(L.bits, L.t8, out)
    return out


@pytest.mark.parametrize('part', ['llm', 'expert'])
@pytest.mark.parametrize('M', [64, 65, 130])
def test_float_group_across_the_token_bound(M, part):
    """Group.run_float on both sides of the bound between the fused products and the dense-weight GEMM, fly and resident:
    the same bits from both weight forms, and the layer definition within its 2e-3."""
    from yanlongvla_amd import modules
    shapes = [(512, 1), (256, 1)]
    layers = [layer(m, 1152, 50 + i) for i, (m, _) in enumerate(shapes)]
    layers[1].su = layers[0].su
    x = torch.randn(M, 1152, device=DEV, generator=torch.Generator(device=DEV).manual_seed(M)).bfloat16()
    outs = [modules.Group(layers, part, mode, a8=False).run(x) for mode in ('fly', 'resident')]
    for i, L in enumerate(layers):
        assert torch.equal(outs[0][i], outs[1][i])
        ol = O.Layer(L.name, dict(bits=L.bits.cpu().numpy(), tlut=L.tlut.cpu().numpy(), row_scale=L.row_scale.cpu().numpy(),
                                  su=L.su.cpu().numpy(), sv=L.sv.cpu().numpy()))
        ref = O.bf16_to_f32(O.w2_linear(x.float().cpu().numpy(), ol, small=part == 'expert'))
        got = outs[0][i].float().cpu().numpy()
        assert np.linalg.norm(got - ref) <= 2e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize('part', ['llm', 'expert'])
@pytest.mark.parametrize('widths,K,M', [((2048, 1024), 1152, 226), ((2048, 1024), 1152, 227), ((512,), 16384, 190), ((512,), 16384, 191), ((2048,), 16384, 65)])
def test_float_group_across_the_dense_line(widths, K, M, part):
    """As test_float_group_across_the_token_bound on both sides of the line between the fused products and dense weights (226 / 227
    tokens of 3072 x 1152, 190 / 191 of 512 x 16384) and where 65 tokens are past it."""
    from yanlongvla_amd import modules
    layers = [layer(m, K, 70 + i) for i, m in enumerate(widths)]
    for L in layers[1:]:
        L.su = layers[0].su
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(M)).bfloat16()
    groups = [modules.Group(layers, part, mode, a8=False) for mode in ('fly', 'resident')]
    assert all(G.dense_float(M) == (M in (227, 191, 65)) for G in groups)
    outs = [G.run(x) for G in groups]
    for i, L in enumerate(layers):
        assert torch.equal(outs[0][i], outs[1][i])
        ol = O.Layer(L.name, dict(bits=L.bits.cpu().numpy(), tlut=L.tlut.cpu().numpy(), row_scale=L.row_scale.cpu().numpy(),
                                  su=L.su.cpu().numpy(), sv=L.sv.cpu().numpy()))
        ref = O.bf16_to_f32(O.w2_linear(x.float().cpu().numpy(), ol, small=part == 'expert'))
        got = outs[0][i].float().cpu().numpy()
        assert np.linalg.norm(got - ref) <= 2e-3 * np.linalg.norm(ref)
