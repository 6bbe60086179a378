"""GPU tests of the multi-query attention kernel: against FP64 attention (the BF16 output rounding is the only sizeable
difference), causal visibility, the fused o-projection prologue against attention followed by the separate prologue, and
run-to-run determinism."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.fixture(scope='module', autouse=True)
def _lib():
    from yanlongvla_amd import _lib
    _lib.lib()
    torch.cuda.init()


def reference(q, kc, vc, kn, vn, H, causal):
    """FP64 softmax(q k^T / 16) v over cache + new rows; query t sees key j iff causal is None or j <= causal + t."""
    k = torch.cat([kc, kn]) if kc is not None else kn
    v = torch.cat([vc, vn]) if vc is not None else vn
    M, D = q.shape[0], k.shape[1]
    qh = q.double().cpu().reshape(M, H, D)
    s = torch.einsum('thd,jd->thj', qh, k.double().cpu()) / 16.0
    if causal is not None:
        j = torch.arange(k.shape[0])[None, None, :]
        t = torch.arange(M)[:, None, None]
        s = s.masked_fill(j > t + causal, float('-inf'))
    p = torch.softmax(s, -1)
    return torch.einsum('thj,jd->thd', p, v.double().cpu()).reshape(M, H * D)


def inputs(M, P, H, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    return r(M, H * 256), (r(P, 256) if P else None), (r(P, 256) if P else None), r(M, 256), r(M, 256)


@pytest.mark.parametrize('M,P,H,causal', [(50, 800, 8, None), (1, 832, 8, None), (800, 0, 8, 0), (7, 0, 8, 0), (3, 63, 4, None),
                                          (1, 0, 1, None), (65, 10, 8, 10)])
def test_attend_matches_fp64(M, P, H, causal):
    from yanlongvla_amd import kernels as K
    q, kc, vc, kn, vn = inputs(M, P, H, M + P + H)
    o = torch.empty(M, H * 256, dtype=torch.bfloat16, device=DEV)
    K.attend(q, kc, vc, kn, vn, H, causal, o=o)
    ref = reference(q, kc, vc, kn, vn, H, causal)
    got = o.double().cpu()
    assert torch.isfinite(got).all()
    assert ((got - ref).norm() / ref.norm()).item() < 4e-3
    assert (got - ref).abs().max().item() < 2e-2 * ref.abs().max().item() + 1e-3


def test_causal_rows_ignore_later_keys():
    """Changing the keys / values a causal query may not see leaves its output unchanged."""
    from yanlongvla_amd import kernels as K
    q, _, _, kn, vn = inputs(200, 0, 8, 3)
    o1 = torch.empty(200, 2048, dtype=torch.bfloat16, device=DEV)
    K.attend(q, None, None, kn, vn, 8, 0, o=o1)
    kn2, vn2 = kn.clone(), vn.clone()
    kn2[100:] = torch.randn_like(kn2[100:].float()).bfloat16()
    vn2[100:] = torch.randn_like(vn2[100:].float()).bfloat16()
    o2 = torch.empty_like(o1)
    K.attend(q, None, None, kn2, vn2, 8, 0, o=o2)
    assert torch.equal(o1[:100], o2[:100]) and not torch.equal(o1[100:], o2[100:])


@pytest.mark.parametrize('H', [1, 2, 4, 8])
@pytest.mark.parametrize('M,P,causal', [(50, 800, None), (1, 800, None), (300, 0, 0), (7, 0, 0), (20, 40, 40)])
def test_fused_prologue_bitexact(M, P, causal, H):
    """The o-projection prologue fused into attention (rotate + quantize of the BF16 attention output, every engine width
    H * 256 = 256 .. 2048) equals attention followed by kernels.pre bit for bit: q8, the token-block q4 and the scales.
    Cases: a prefix without masking, a causal prefill with no prefix, and causal rows over a prefix (causal offset P)."""
    from yanlongvla_amd import kernels as K
    q, kc, vc, kn, vn = inputs(M, P, H, 7 + M + H)
    W = H * 256
    su = (torch.randint(0, 2, (W,), generator=torch.Generator(device=DEV).manual_seed(H), device=DEV) * 2 - 1).to(torch.int8)
    o = torch.empty(M, W, dtype=torch.bfloat16, device=DEV)
    K.attend(q, kc, vc, kn, vn, H, causal, o=o)
    q1, s1, tb1 = torch.empty(M, W, dtype=torch.int8, device=DEV), torch.empty(M, device=DEV), K.token_blocks(M, W, DEV)
    K.pre(o, su, q=q1, q4=tb1, scale=s1)
    q2, s2, tb2 = torch.empty_like(q1), torch.empty_like(s1), K.token_blocks(M, W, DEV)
    K.attend(q, kc, vc, kn, vn, H, causal, su=su, q8=q2, scale=s2, q4=tb2)
    assert torch.equal(q1, q2) and torch.equal(s1, s2)
    assert torch.equal(K.rows_of_token_blocks(tb1, M), K.rows_of_token_blocks(tb2, M))
    o2 = torch.empty_like(o)
    K.attend(q, kc, vc, kn, vn, H, causal, o=o2)
    assert torch.equal(o, o2)


@pytest.mark.parametrize('M,P,H,causal', [(255, 0, 8, 0), (256, 0, 8, 0), (257, 0, 3, 0), (301, 70, 8, 70), (258, 31, 1, 31), (259, 64, 8, 3),
                                          (260, 1, 8, 400)])
def test_many_causal_tokens(M, P, H, causal):
    """Around the token count where the running-maximum kernel takes over: odd counts (a half empty last group), fewer heads,
    caches that end inside a 32-key block, offsets below and past the cache. The BF16 output rounds to 2^-9 of a value and
    the probabilities, rounded to BF16 alike, add no more than that again, so the norm of the error stays below 2^-8."""
    from yanlongvla_amd import kernels as K
    q, kc, vc, kn, vn = inputs(M, P, H, 2 * M + P)
    o = torch.empty(M, H * 256, dtype=torch.bfloat16, device=DEV)
    K.attend(q, kc, vc, kn, vn, H, causal, o=o)
    ref = reference(q, kc, vc, kn, vn, H, causal)
    assert ((o.double().cpu() - ref).norm() / ref.norm()).item() < 2.0 ** -8
    su = torch.ones(H * 256, dtype=torch.int8, device=DEV)
    q1, q2 = (torch.empty(M, H * 256, dtype=torch.int8, device=DEV) for _ in range(2))
    s1, s2 = (torch.empty(M, device=DEV) for _ in range(2))
    K.attend(q, kc, vc, kn, vn, H, causal, su=su, q8=q1, scale=s1)
    K.pre(o, su, q=q2, scale=s2)
    assert torch.equal(q1, q2) and torch.equal(s1, s2)


def _near_ties(n):
    """n FP32 distances d whose exp(-d) lies within a few 1e-6 of the midpoint of two BF16 values, on the other side of it than
    2^(d log2 e) with the product rounded to FP32, and more than 2.4e-7 (two FP32 ulps) from it on both sides."""
    d = np.random.default_rng(0).uniform(45, 80, 1 << 22).astype(np.float32)
    right, coarse = np.exp(-d.astype(np.float64)), np.exp2((-d * np.float32(np.log2(np.e))).astype(np.float64))
    half = np.exp2(np.floor(np.log2(right)) - 8)                               # half a BF16 ulp
    tie = (np.floor(right / (2 * half)) + 0.5) * 2 * half
    apart = 2.4e-7 * right
    found = d[(np.abs(right - tie) > apart) & (np.abs(coarse - tie) > apart) & ((right > tie) != (coarse > tie))]
    assert len(found) >= n
    return torch.from_numpy(found[:n])


def test_many_causal_tokens_exponentials():
    """The probabilities of k_attn_rows are FP32 exponentials of at most one ulp, as everywhere else: with one key at the maximum
    (value 0) and one at distance d (value 1), an output is bf16(exp(-d)), here for distances next to a rounding boundary."""
    from yanlongvla_amd import kernels as K
    M, H = 288, 8
    d = _near_ties(512).repeat(5)[:M * H].view(M, H)
    q, rest = torch.zeros(M, H, 256), d.clone()
    for i in range(3):                                                         # the distance in three exact BF16 pieces
        piece = rest.bfloat16().float()
        q[:, :, i], rest = -16 * piece, rest - piece
    assert not rest.any()
    q[:, :, 3] = -65536                                                        # the call's own keys: 4096 below the maximum
    kc, vc, kn = torch.zeros(2, 256), torch.zeros(2, 256), torch.zeros(M, 256)
    kc[1, :3], vc[1], kn[:, 3] = 1, 1, 1
    q, kc, vc, kn = (t.bfloat16().to(DEV) for t in (q.view(M, H * 256), kc, vc, kn))
    o = torch.empty_like(q)
    K.attend(q, kc, vc, kn, torch.zeros_like(kn), H, 2, o=o)
    want = torch.exp(-d.double()).bfloat16()
    assert torch.equal(o.view(M, H, 256).cpu(), want[:, :, None].expand(M, H, 256))


@pytest.mark.parametrize('M,P,H,causal', [(287, 31, 8, 31), (289, 31, 5, 31), (290, 64, 8, 3), (291, 1, 8, 400), (288, 33, 7, 33), (511, 0, 4, 0),
                                          (513, 40, 3, 40), (967, 5, 2, 5), (969, 31, 2, 31), (970, 0, 1, 0)])
def test_many_causal_tokens_by_heads_and_cache(M, P, H, causal):
    """test_many_causal_tokens around the counts that fewer heads and a cache move the kernels' line to."""
    test_many_causal_tokens(M, P, H, causal)


@pytest.mark.parametrize('P,causal', [(0, 0), (40, 40)])
@pytest.mark.parametrize('M', [255, 290])
def test_infinite_and_nan_keys_and_values(M, P, causal):
    """On either kernel (255 tokens on the chunks, 290 on k_attn_rows): a NaN key or a key of infinite score makes every row that
    sees it NaN, an infinite value gives that infinity in its column and nothing else; rows of token pairs before it keep their
    bits (a pair shares its products, so the token just before may not)."""
    from yanlongvla_amd import kernels as K
    q, kc, vc, kn, vn = inputs(M, P, 8, 3 * M + P)

    def run(kn, vn):
        o = torch.empty(M, 2048, dtype=torch.bfloat16, device=DEV)
        K.attend(q, kc, vc, kn, vn, 8, causal, o=o)
        return o.view(M, 8, 256)
    clean = run(kn, vn)
    j = 100                                                                    # even: the first of its pair
    for bad in (float('nan'), float('inf')):
        k2 = kn.clone()
        k2[j] = bad
        o = run(k2, vn)
        assert torch.equal(o[:j], clean[:j]) and bool(o[j:].isnan().all())     # (inf x both signs of q: NaN too)
    for bad in (float('inf'), float('-inf')):
        v2 = vn.clone()
        v2[j, 7] = bad
        o = run(kn, v2)
        assert torch.equal(o[:j], clean[:j]) and bool((o[j:, :, 7] == bad).all())
        o[j:, :, 7] = clean[j:, :, 7]
        assert torch.equal(o, clean)
