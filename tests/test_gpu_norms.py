"""GPU parity of the RMSNorm kernel and its fusions (norm + rotate + quantize; epilogue + residual + norm + rotate +
quantize) against the oracle and against the unfused launches, and of the fused decoder layer against the module-by-module
forward."""
import numpy as np
import pytest
import torch

from oracle import tcq_oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.fixture(scope='module', autouse=True)
def _lib():
    from yanlongvla_amd import _lib
    _lib.lib()
    torch.cuda.init()


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def bf16_dev(bits):
    return T(bits.view(np.int16)).view(torch.bfloat16)


def bits_of(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def signs(rng, n):
    return np.where(rng.integers(0, 2, n) > 0, 1, -1).astype(np.int8)


@pytest.mark.parametrize('M,K', [(1, 1024), (50, 1024), (50, 2048), (800, 2048), (3, 16384), (5, 48)])
def test_rmsnorm_bitexact(M, K):
    from yanlongvla_amd import kernels as Kn
    rng = np.random.default_rng(M + K)
    x = O.bf16_bits(rng.standard_normal((M, K)).astype(np.float32) * 2)
    w = O.bf16_bits(rng.standard_normal(K).astype(np.float32) * 0.2)
    y = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    Kn.rmsnorm(bf16_dev(x), bf16_dev(w), 1e-6, y)
    assert np.array_equal(bits_of(y), O.rmsnorm_bf16(O.bf16_to_f32(x), w, 1e-6))


@pytest.mark.parametrize('M,K', [(1, 1024), (50, 1024), (800, 2048), (2, 16384)])
def test_norm_pre_bitexact(M, K):
    from yanlongvla_amd import kernels as Kn
    rng = np.random.default_rng(M * 3 + K)
    x = O.bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    w = O.bf16_bits(rng.standard_normal(K).astype(np.float32) * 0.2)
    su = signs(rng, K)
    q = torch.empty(M, K, dtype=torch.int8, device=DEV)
    s = torch.empty(M, dtype=torch.float32, device=DEV)
    Kn.norm_pre(bf16_dev(x), bf16_dev(w), 1e-6, T(su), q=q, scale=s)
    qr, sr = O.quantize_tokens(O.fwht(O.bf16_to_f32(O.rmsnorm_bf16(O.bf16_to_f32(x), w, 1e-6)) * su.astype(np.float32)))
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr[:, 0])


@pytest.mark.parametrize('M,K', [(1, 16), (7, 1040), (968, 1024), (65, 2048), (3, 4096), (2, 8192)])
@pytest.mark.parametrize('off', [0, 1])
def test_norms_in_registers_match_lds(M, K, off):
    """Rows in registers (16-byte aligned; off = 0) and on the LDS path (off = 1 element) give the oracle's bits: rmsnorm at
    partial waves, norm_pre at each register width and beyond, with q, token blocks and words."""
    from yanlongvla_amd import kernels as Kn
    rng = np.random.default_rng(M + 2 * K)
    x = O.bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    w = O.bf16_bits(rng.standard_normal(K).astype(np.float32) * 0.2)
    su = signs(rng, K)
    xb = torch.zeros(M * K + 8, dtype=torch.bfloat16, device=DEV)[off:off + M * K].view(M, K)
    xb.copy_(bf16_dev(x))
    y = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    Kn.rmsnorm(xb, bf16_dev(w), 1e-6, y)
    n = O.rmsnorm_bf16(O.bf16_to_f32(x), w, 1e-6)
    assert np.array_equal(bits_of(y), n)
    qr, sr = O.quantize_tokens(O.fwht(O.bf16_to_f32(n) * su.astype(np.float32)))
    s = torch.empty(M, dtype=torch.float32, device=DEV)
    q = torch.empty(M, K, dtype=torch.int8, device=DEV)
    blocks, words = Kn.token_blocks(M, K, DEV), torch.empty(K // 4, M, dtype=torch.int32, device=DEV)
    Kn.norm_pre(xb, bf16_dev(w), 1e-6, T(su), q=q, q4=blocks, scale=s)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr[:, 0])
    assert torch.equal(Kn.rows_of_token_blocks(blocks, M), q)
    Kn.norm_pre(xb, bf16_dev(w), 1e-6, T(su), q4=words, scale=s)
    assert np.array_equal(words.cpu().numpy().T.copy().view(np.int8).reshape(M, K), qr)


@pytest.mark.parametrize('M,N,parts', [(1, 2048, 2), (50, 1024, 4), (3, 4096, 2), (2, 8192, 4), (1, 16384, 2)])
def test_post_add_norm_pre_k_parts(M, N, parts):
    """int32 K parts in: the same outputs as their int32 sum in one accumulator (register + transpose engine up to 4096,
    register engine beyond); a row the LDS path would take (N = 1152) is refused."""
    from yanlongvla_amd import kernels as Kn, _lib
    rng = np.random.default_rng(M + N + parts)
    lda = N + 64
    part = rng.integers(-2 ** 16, 2 ** 16, size=(parts, M, lda)).astype(np.int32)
    s = T((rng.random(M) * 1e-3 + 1e-4).astype(np.float32))
    rs = T((rng.random(N) * 1e-2).astype(np.float32))
    sv, su = T(signs(rng, N)), T(signs(rng, N))
    bias = T((rng.standard_normal(N) * 0.1).astype(np.float32))
    x = bf16_dev(O.bf16_bits(rng.standard_normal((M, N)).astype(np.float32)))
    w = bf16_dev(O.bf16_bits(rng.standard_normal(N).astype(np.float32) * 0.2))
    outs = []
    for acc in (T(part), T(part.sum(0, dtype=np.int32))):
        xo = torch.empty_like(x)
        q = torch.empty(M, N, dtype=torch.int8, device=DEV)
        sc = torch.empty(M, dtype=torch.float32, device=DEV)
        Kn.post_add_norm_pre(acc, s, rs, sv, bias, x, xo, w, 1e-6, su, q=q, scale=sc, col0=16)
        outs.append((xo, q, sc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    with pytest.raises(_lib.TcqError):
        N2 = 1152
        acc = torch.zeros(parts, M, N2, dtype=torch.int32, device=DEV)
        xx = torch.zeros(M, N2, dtype=torch.bfloat16, device=DEV)
        Kn.post_add_norm_pre(acc, s, torch.ones(N2, device=DEV), T(signs(rng, N2)), None, xx, torch.empty_like(xx))


@pytest.mark.parametrize('kind', ['f32', 'i32'])
@pytest.mark.parametrize('M,N,col0', [(1, 1024, 16), (50, 1024, 16), (300, 2048, 16), (5, 4096, 16), (2, 16384, 16),
                                      (50, 1024, 2), (3, 4096, 2)])
@pytest.mark.parametrize('with_norm', [True, False])
def test_post_add_norm_pre_bitexact(kind, M, N, col0, with_norm):
    """== post (BF16) -> BF16 residual add -> rmsnorm -> pre, the unfused chain of launches. Aligned power-of-two rows
    run the register path (rows of 4096 and 16384 exchange between waves), col0 = 2 (rows not 16-byte aligned) the LDS
    path."""
    from yanlongvla_amd import kernels as Kn
    rng = np.random.default_rng(M * 5 + N)
    lda = N + 32
    if kind == 'i32':
        acc = T(rng.integers(-2 ** 18, 2 ** 18, size=(M, lda)).astype(np.int32))
        s = T((rng.random(M) * 1e-3 + 1e-4).astype(np.float32))
        rs = T((rng.random(N) * 1e-2).astype(np.float32))
    else:
        acc, s, rs = T(rng.standard_normal((M, lda)).astype(np.float32)), None, None
    sv, su = T(signs(rng, N)), T(signs(rng, N))
    bias = T((rng.standard_normal(N) * 0.1).astype(np.float32))
    x = bf16_dev(O.bf16_bits(rng.standard_normal((M, N)).astype(np.float32)))
    w = bf16_dev(O.bf16_bits(rng.standard_normal(N).astype(np.float32) * 0.2))
    xo = torch.empty_like(x)
    q = torch.empty(M, N, dtype=torch.int8, device=DEV)
    sc = torch.empty(M, dtype=torch.float32, device=DEV)
    if with_norm:
        Kn.post_add_norm_pre(acc, s, rs, sv, bias, x, xo, w, 1e-6, su, q=q, scale=sc, col0=col0)
    else:
        Kn.post_add_norm_pre(acc, s, rs, sv, bias, x, xo, col0=col0)
    a = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    Kn.post(acc, s, rs, sv, bias, a, col0=col0)
    x2 = x + a
    assert torch.equal(xo, x2)
    if with_norm:
        n = torch.empty_like(x2)
        Kn.rmsnorm(x2, w, 1e-6, n)
        q2 = torch.empty_like(q)
        s2 = torch.empty_like(sc)
        Kn.pre(n, su, q=q2, scale=s2)
        assert torch.equal(q, q2) and torch.equal(sc, s2)


def test_decoder_layer_fusion_is_bitexact():
    """KDecoderLayer (norms and residuals fused into the TCQ kernels) == the module-by-module forward (KLinear groups,
    KGatedMLP, device RMSNorm, PyTorch residual adds), at 50 tokens (small-M products) and 200 tokens (INT8 GEMM)."""
    from yanlongvla_amd import gemma, modules
    outs = {}
    for fuse in (False, True):
        old = modules.FUSE['layer']
        modules.FUSE['layer'] = fuse
        try:
            model = gemma.make_policy(gemma.ExpertPolicy, DEV, seed=1, layers=2)
            g = torch.Generator(device=DEV).manual_seed(2)
            model.set_prefix([torch.randn(64, 256, generator=g, device=DEV).bfloat16() for _ in range(2)],
                             [torch.randn(64, 256, generator=g, device=DEV).bfloat16() for _ in range(2)])
            with torch.no_grad():
                for n, p in model.named_parameters():
                    if n.endswith('layernorm.weight') or n.endswith('norm.weight'):
                        p.copy_((torch.randn(p.shape, generator=g, device=DEV) * 0.1).bfloat16())
            info = modules.install(model, runtime='fly', layers=gemma.synthetic_layers(model, 3, DEV))
            assert info['fused_layers'] == (2 if fuse else 0)
            if fuse:
                assert type(model.stack.layers[0]).__name__ == 'KDecoderLayer'
            x = torch.randn(50, 32, generator=torch.Generator(device=DEV).manual_seed(4), device=DEV)
            h = torch.randn(200, 1024, generator=torch.Generator(device=DEV).manual_seed(6), device=DEV).bfloat16()
            with torch.inference_mode():
                outs[fuse] = (model.velocity(x), model.stack.layers[1](h, model.prefix_k[1], model.prefix_v[1])[0])
        finally:
            modules.FUSE['layer'] = old
    assert torch.equal(outs[True][0], outs[False][0])
    assert torch.equal(outs[True][1], outs[False][1])


@pytest.mark.parametrize('M,N', [(65, 2048), (419, 2048), (420, 2048), (839, 1024), (840, 1024)])
def test_epilogues_of_more_rows_match_few(M, N):
    """post_add_norm_pre, post and post_group around the row counts where their engine changes: each row as in calls of 40."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(M)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    acc, x, w = r(M, N + 512), r(M, N).bfloat16(), r(N).bfloat16()
    sv, su = (torch.where(r(N) > 0, 1, -1).to(torch.int8) for _ in range(2))

    def run(a, b):
        a_, x_, m = acc[a:b], x[a:b], b - a
        xo, q, s = torch.empty_like(x_), torch.empty(m, N, dtype=torch.int8, device=DEV), torch.empty(m, device=DEV)
        Kn.post_add_norm_pre(a_, None, None, sv, None, x_, xo, w, 1e-6, su, q=q, scale=s)
        y = torch.empty_like(x_)
        Kn.post(a_, None, None, sv, None, y)
        ys = [torch.empty(m, n, dtype=torch.bfloat16, device=DEV) for n in (N, 256, 256)]
        c = (0, N, N + 256)
        Kn.post_group([(a_, c0, None, sv[:t.shape[1]], None, t, False) for c0, t in zip(c, ys)], torch.float32, torch.bfloat16, None, m)
        one = torch.empty_like(x_)
        Kn.post_group([(a_, 0, None, sv, None, one, False)], torch.float32, torch.bfloat16, None, m)
        return [xo, q, s, y, one] + ys
    whole = run(0, M)
    parts = [run(a, min(a + 40, M)) for a in range(0, M, 40)]
    for i, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[i] for p in parts]))


@pytest.mark.parametrize('parts', [2, 4])
@pytest.mark.parametrize('M,N', [(65, 2048), (419, 2048), (420, 2048), (839, 1024), (840, 1024), (130, 4096)])
def test_k_parts_of_more_rows(M, N, parts):
    """post_add_norm_pre without a bias over the int32 K parts that a product of more than 64 tokens hands it, on both sides of the
    row counts where its engine changes: the outputs of their sum in one accumulator, and of calls of 40 rows."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(M + parts)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    acc, x, w = (r(parts, M, N) * 1e4).int(), r(M, N).bfloat16(), r(N).bfloat16()
    s, rs = (torch.rand(n, generator=g, device=DEV) * 1e-2 + 1e-4 for n in (M, N))
    sv, su = (torch.where(r(N) > 0, 1, -1).to(torch.int8) for _ in range(2))

    def run(acc, a, b):
        x_, m = x[a:b], b - a
        xo, q, sc = torch.empty_like(x_), torch.empty(m, N, dtype=torch.int8, device=DEV), torch.empty(m, device=DEV)
        Kn.post_add_norm_pre(acc[..., a:b, :].contiguous(), s[a:b], rs, sv, None, x_, xo, w, 1e-6, su, q=q, scale=sc)
        return xo, q, sc
    whole, one = run(acc, 0, M), run(acc.sum(0).int(), 0, M)
    pieces = [run(acc, a, min(a + 40, M)) for a in range(0, M, 40)]
    for i, t in enumerate(whole):
        assert torch.equal(t, one[i]) and torch.equal(t, torch.cat([p[i] for p in pieces]))


@pytest.mark.parametrize('runtime', ['fly', 'resident'])
@pytest.mark.parametrize('M', [65, 200, 450])
def test_decoder_layers_with_and_without_k_parts(M, runtime):
    """A backbone prefill whose o and down products run in K parts (more than one at these counts) gives the outputs of one part,
    bit for bit, chained prologues included."""
    from yanlongvla_amd import gemma, modules
    model = gemma.make_policy(gemma.BackbonePolicy, DEV, seed=5, layers=2, vocab=512)
    modules.install(model, runtime=runtime, layers=gemma.synthetic_layers(model, 16, DEV))
    down = [G for G in model._tcq_groups if G.K == 16384]
    assert len(down) == 2 and all(G.epilogue_parts(M) > 1 for G in down)
    x = torch.randn(M, 2048, generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).bfloat16()
    outs = {}
    for parts in (False, True):
        modules.FUSE['k_parts'] = parts
        try:
            h, ks, vs = model.prefill(x)
            outs[parts] = [h, *ks, *vs]
        finally:
            modules.FUSE['k_parts'] = True
    for a, b in zip(outs[False], outs[True]):
        assert torch.equal(a, b)
