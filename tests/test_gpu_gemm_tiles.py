"""The many-token GEMM (tcq_gemm_i8, tcq_gemm_bf16) at the edges of its tiles: sizes that select each tile, with remainders in
tokens, weight rows and K (whole and partial 128-byte steps, fewer steps than the rings hold)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'

# 64 x 64, 128 x 64, 128 x 128, 256 x 128 and 256 x 256 tiles (the last line of each pair with remainders)
SIZES = [(65, 64, 16), (129, 1156, 1168), (65, 12800, 128), (80, 16388, 272), (200, 16384, 384), (449, 8196, 144), (400, 16384, 256),
         (385, 16420, 400), (768, 16384, 512), (801, 16516, 656), (1, 132, 32), (66, 16640, 2048)]


def _ints(*shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8)


@pytest.mark.parametrize('M,N,K', SIZES)
def test_int8_tiles_bitexact(M, N, K):
    from yanlongvla_amd import kernels as Kn
    a, w = _ints(M, K, seed=1), _ints(N, K, seed=2)
    sa = torch.rand(M, device=DEV) + 0.01
    sw = torch.rand(N, device=DEV) + 0.01
    want = (a.double() @ w.double().t()).to(torch.int32)                       # exact: |sum| < 2^53
    pad = torch.full((M, N + 8), 7, dtype=torch.int32, device=DEV)
    acc = Kn.gemm_i8(a, w, pad[:, :N])
    assert torch.equal(acc, want) and bool((pad[:, N:] == 7).all())            # a wider row stride, nothing past the columns
    z = (want.float() * sa[:, None]) * sw[None, :]
    assert torch.equal(Kn.gemm_i8(a, w, torch.empty(M, N, device=DEV), sa=sa, sw=sw), z)
    y = torch.full((M, N + 4), 3.0, dtype=torch.bfloat16, device=DEV)
    assert torch.equal(Kn.gemm_i8(a, w, y[:, :N], sa=sa, sw=sw), z.bfloat16()) and bool((y[:, N:] == 3.0).all())


@pytest.mark.parametrize('M,N,K', SIZES)
def test_bf16_tiles_against_fp64(M, N, K):
    """Products of BF16 values are exact in FP32; every sum of K of them in FP32, in whatever order, is within K 2^-24 of the
    sum of their magnitudes."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(3)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), _ints(N, K, seed=4).bfloat16()
    want, mag = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    z = Kn.gemm_bf16(a, w, torch.empty(M, N, device=DEV))
    assert bool(((z.double() - want).abs() <= K * 2.0 ** -24 * mag).all())
    sw = torch.rand(N, device=DEV) + 0.01
    assert torch.equal(Kn.gemm_bf16(a, w, torch.empty(M, N, device=DEV), sw=sw), z * sw)
    assert torch.equal(Kn.gemm_bf16(a, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV)), z.bfloat16())


@pytest.mark.parametrize('M,N,K', [(65, 64, 2048), (129, 132, 2064), (300, 1156, 4304), (968, 2048, 16384)])
@pytest.mark.parametrize('parts', [1, 2, 4])
def test_k_parts_bitexact(M, N, K, parts):
    """The parts add to the exact product: parts with a partial last K step, uneven and equal ones."""
    from yanlongvla_amd import kernels as Kn
    a, w = _ints(M, K, seed=5), _ints(N, K, seed=6)
    acc = Kn.gemm_i8_parts(a, w, parts)
    assert acc.shape == (parts, M, N)
    assert torch.equal(acc.sum(0), (a.double() @ w.double().t()).to(torch.int64))


def test_k_parts_refused():
    from yanlongvla_amd import _lib, kernels as Kn
    for K, parts in ((2032, 2), (4096, 3)):
        with pytest.raises(_lib.TcqError):
            Kn.gemm_i8_parts(_ints(80, K, seed=7), _ints(64, K, seed=8), parts)


@pytest.mark.parametrize('M,N,K', [(65, 64, 1024), (129, 132, 1040), (300, 1156, 4304), (968, 2048, 16384)])
@pytest.mark.parametrize('parts', [2, 4])
def test_bf16_parts_against_fp64(M, N, K, parts):
    """As test_bf16_tiles_against_fp64 (any order of FP32 sums); FP32 and BF16 outputs with and without row scales agree."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(5)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), _ints(N, K, seed=6).bfloat16()
    want, mag = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    z = Kn.gemm_bf16_parts(a, w, torch.empty(M, N, device=DEV), parts)
    assert bool(((z.double() - want).abs() <= K * 2.0 ** -24 * mag).all())
    sw = torch.rand(N, device=DEV) + 0.01
    assert torch.equal(Kn.gemm_bf16_parts(a, w, torch.empty(M, N, device=DEV), parts, sw=sw), z * sw)
    assert torch.equal(Kn.gemm_bf16_parts(a, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), parts), z.bfloat16())


@pytest.mark.parametrize('parts', [1, 2, 4])
@pytest.mark.parametrize('M,N,K', [(65, 64, 128), (80, 68, 1024), (129, 132, 2048), (65, 64, 16384)])
def test_bf16_infinite_operands_and_sums(M, N, K, parts):
    """An infinite activation in each K chain's range, and products whose sums pass the largest FP32 value, give the infinities
    (of one sign each, every weight positive) that any FP32 accumulation gives; a NaN stays one, other tokens are untouched."""
    from yanlongvla_amd import kernels as Kn
    if parts > 1 and K < 1024:
        pytest.skip('K parts start at 1024 columns')
    g = torch.Generator(device=DEV).manual_seed(K)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), _ints(N, K, seed=9).abs().clamp(min=1).bfloat16()
    out = torch.empty(M, N, device=DEV)
    run = lambda: (Kn.gemm_bf16(a, w, out) if parts == 1 else Kn.gemm_bf16_parts(a, w, out, parts)).clone()
    finite = run()
    cols = [0, 63, 64, K // 3, K // 2, K - 65, K - 1]
    inf = float('inf')
    for i, c in enumerate(cols):
        a[i, c] = inf if i % 2 == 0 else -inf
    a[10], a[11] = 3e38, -3e38
    a[12, K // 3] = float('nan')
    got = run()
    for i in range(len(cols)):
        assert bool((got[i] == (inf if i % 2 == 0 else -inf)).all()), cols[i]
    assert bool((got[10] == inf).all()) and bool((got[11] == -inf).all()) and bool(got[12].isnan().all())
    others = [i for i in range(M) if not (i < len(cols) or 10 <= i <= 12)]
    assert torch.equal(got[others], finite[others])


@pytest.mark.parametrize('M,N,K', [(65, 1024, 1024), (300, 1024, 1024), (968, 4096, 1024), (130, 2048, 2048), (968, 2048, 2048), (130, 1024, 4096),
                                   (968, 1024, 4096), (130, 2048, 16384), (968, 2048, 16384)])
def test_bf16_sums_as_close_to_fp64_as_the_few_token_product(M, N, K):
    """The float path crosses from gemmf_segments to gemm_bf16 at 64 tokens and loses no precision there: on one set of operands
    the sums (one part, and the parts that the size calls for) are no further from 64 bits, in the 2-norm over at least 66 000
    outputs, than that product's. Plain second-level sums are 6 to 11 % further."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(K + M)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), _ints(N, K, seed=11)
    want = a.double() @ w.double().t()
    few, wb = torch.empty(M, N, device=DEV), w.bfloat16()
    Kn.gemmf_segments([(w, None, torch.ones(N, device=DEV), few)], a, N, resident=True)
    err = lambda z: float((z.double() - want).norm())
    bound = err(few)
    assert err(Kn.gemm_bf16(a, wb, torch.empty(M, N, device=DEV))) <= bound
    assert err(Kn.gemm_bf16_best(a, wb, torch.empty(M, N, device=DEV))) <= bound


@pytest.mark.parametrize('M,N,K', [(300, 32768, 144), (330, 32768, 272), (960, 12288, 256)])
def test_tiles_of_equal_estimates(M, N, K):
    """Sizes whose tiles lie close together: full rounds of several, and partly filled ones."""
    test_int8_tiles_bitexact(M, N, K)
    test_bf16_tiles_against_fp64(M, N, K)


@pytest.mark.parametrize('M,N,K', [(65, 68, 1024), (130, 132, 2048), (300, 2052, 2048), (129, 8200, 528)])
def test_bf16_scaled_infinities(M, N, K):
    """Scaled FP32 and BF16 outputs of every tile width around infinite sums: (z sa) sw of the unscaled FP32 output z, its BF16
    rounding, infinities where z is checked to have them."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(N)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), _ints(N, K, seed=9).abs().clamp(min=1).bfloat16()
    a[5, 3], a[M - 1, K - 1], a[40, 64] = float('inf'), float('-inf'), float('nan')
    w[N - 2, 100] = float('inf')                                               # both signs of activations: infinities of both
    sa, sw = torch.rand(M, generator=g, device=DEV) + 0.1, torch.rand(N, generator=g, device=DEV) + 0.1
    z = Kn.gemm_bf16(a, w, torch.empty(M, N, device=DEV))
    col = torch.sign(a[:, 100].float()) * float('inf')
    rows = [m for m in range(M) if m not in (5, 40, M - 1)]
    assert torch.equal(z[rows, N - 2], col[rows]) and bool(z[40].isnan().all())
    rest = [n for n in range(N) if n != N - 2]
    assert bool((z[5, rest] == float('inf')).all()) and bool((z[M - 1, rest] == float('-inf')).all())
    want = (z * sa[:, None]) * sw
    got = Kn.gemm_bf16(a, w, torch.empty(M, N, device=DEV), sa=sa, sw=sw)
    assert torch.equal(got.nan_to_num(nan=7.0, posinf=8.0, neginf=9.0), want.nan_to_num(nan=7.0, posinf=8.0, neginf=9.0))
    b = Kn.gemm_bf16(a, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), sa=sa, sw=sw)
    assert torch.equal(b.nan_to_num(nan=7.0, posinf=8.0, neginf=9.0), want.bfloat16().nan_to_num(nan=7.0, posinf=8.0, neginf=9.0))
