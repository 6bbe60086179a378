"""Row kernels that hold a row in the registers of one wave or four (csrc/tcq_blocks.hip): widths at the edges of their block
decomposition and of the kernel variants, few and many rows, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from oracle import tcq_oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'
# last-group blocks alone, whole groups only, both, quarters with and without remainders; one wave below 2048, four up to
# 7164 (and from 1024 on for few rows), the LDS engine beyond
WIDTHS = [64, 68, 80, 208, 252, 256, 260, 512, 768, 1020, 1024, 1028, 1152, 1280, 1536, 2044, 2300, 2304, 3072, 4304, 4348, 4352,
          6144, 7164, 7168, 8444, 8448, 12304, 15868, 16380]


def bits16(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def draw(M, K, seed):
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).bfloat16()
    return x, (rng.integers(0, 2, K) * 2 - 1).astype(np.int8), rng


@pytest.mark.parametrize('K', WIDTHS)
@pytest.mark.parametrize('M', [2, 259])
def test_rotation_and_quantizer(K, M):
    from yanlongvla_amd import kernels as Kn
    x, su, rng = draw(M, K, K + M)
    want = O.fwht(x.float().numpy() * su.astype(np.float32))
    xd, sd = x.to(DEV), torch.from_numpy(su).to(DEV)
    y = Kn.rht(xd, sd, torch.empty(M, K, device=DEV))
    assert np.array_equal(y.cpu().numpy(), want)
    assert np.array_equal(bits16(Kn.rht(xd, sd, torch.empty_like(xd))), O.bf16_bits(want))
    pad = torch.zeros(M, K + 4, dtype=torch.float16, device=DEV)
    pad[:, :K] = xd.half()
    got = torch.full((M, K + 8), 7.0, dtype=torch.float16, device=DEV)
    Kn.rht(pad[:, :K], None, got[:, :K])
    assert np.array_equal(got[:, :K].cpu().numpy(), O.fwht(pad[:, :K].float().cpu().numpy()).astype(np.float16))
    assert bool((got[:, K:] == 7.0).all())
    cs = (rng.random(K) + 0.5).astype(np.float16)
    for scaled in (False, True):
        q = torch.empty(M, K, dtype=torch.int8, device=DEV)
        q4 = torch.empty(K // 4, M, dtype=torch.int32, device=DEV)
        s = torch.empty(M, device=DEV)
        Kn.pre(xd, sd, q=q, q4=q4, scale=s, col_scale=torch.from_numpy(cs).to(DEV) if scaled else None)
        wq, ws = O.quantize_tokens(want * cs.astype(np.float32) if scaled else want)
        assert np.array_equal(s.cpu().numpy(), ws[:, 0]) and np.array_equal(q.cpu().numpy(), wq)
        assert np.array_equal(q4.cpu().numpy(), O.q4_layout(wq))
        if K % 16 == 0:
            tb = Kn.token_blocks(M, K, DEV)
            Kn.pre(xd, sd, q4=tb, scale=s, col_scale=torch.from_numpy(cs).to(DEV) if scaled else None)
            assert np.array_equal(Kn.rows_of_token_blocks(tb, M).cpu().numpy(), wq)


@pytest.mark.parametrize('N', [80, 256, 1152, 1536, 4304, 6144, 8192, 8448, 16368, 16384])
@pytest.mark.parametrize('M', [3, 270])
@pytest.mark.parametrize('adt', ['i32', 'f32', 'bf16'])
def test_epilogue_and_plain_middle(N, M, adt):
    from yanlongvla_amd import kernels as Kn
    rng = np.random.default_rng(N + M)
    f32 = np.float32
    rs, sv, bias = (rng.random(N) * 0.01 + 1e-3).astype(f32), (rng.integers(0, 2, N) * 2 - 1).astype(np.int8), rng.standard_normal(N).astype(f32)
    su, s = (rng.integers(0, 2, N) * 2 - 1).astype(np.int8), (rng.random(M) * 0.02 + 0.01).astype(f32)
    a = rng.integers(-20000, 20000, (M, N))
    if adt == 'i32':
        acc, z = torch.from_numpy(a.astype(np.int32)), (a.astype(f32) * s[:, None]) * rs
    elif adt == 'f32':
        acc = torch.from_numpy((a * 1e-3).astype(f32))
        z = acc.numpy()
    else:
        acc = torch.from_numpy((a * 0.1).astype(f32)).bfloat16()
        z = acc.float().numpy() * rs
    T = [torch.from_numpy(v).to(DEV) for v in (s, rs, sv, bias, su)]
    ds, drs = (T[0] if adt == 'i32' else None), (None if adt == 'f32' else T[1])
    want = O.fwht(z) * sv.astype(f32) + bias
    y = torch.empty(M, N, device=DEV)
    Kn.post(acc.to(DEV), ds, drs, T[2], T[3], y)
    assert np.array_equal(y.cpu().numpy(), want)
    y2 = [torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2)]          # the group form: equal segments
    both = torch.cat([acc, acc], 1).contiguous().to(DEV)
    Kn.post_group([(both, 0, drs, T[2], T[3], y2[0], False), (both, N, drs, T[2], T[3], y2[1], False)], both.dtype, torch.bfloat16, ds, M)
    assert np.array_equal(bits16(y2[0]), O.bf16_bits(want)) and torch.equal(y2[0], y2[1])
    # the group form: two segments of different widths on one accumulator, GELU on the first
    wide = torch.cat([acc, acc[:, :64]], 1).contiguous().to(DEV)
    ys = [torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for n in (N, 64)]
    lut = Kn.gelu_table(torch.device(DEV))
    Kn.post_group([(wide, 0, drs, T[2], T[3], ys[0], True), (wide, N, None if drs is None else drs[:64].contiguous(), T[2][:64].contiguous(), None, ys[1], False)],
                  wide.dtype, torch.bfloat16, ds, M, gelu_lut=lut)
    act = bits16(lut)[O.bf16_bits(want)]
    assert np.array_equal(bits16(ys[0]), act)
    z64 = z[:, :64] if adt == 'f32' else (a[:, :64].astype(f32) * s[:, None]) * rs[:64] if adt == 'i32' else acc[:, :64].float().numpy() * rs[:64]
    assert np.array_equal(bits16(ys[1]), O.bf16_bits(O.fwht(np.ascontiguousarray(z64)) * sv[:64].astype(f32)))
    q, sc = torch.empty(M, N, dtype=torch.int8, device=DEV), torch.empty(M, device=DEV)
    Kn.mid1(acc.to(DEV), ds, drs, T[2], T[3], T[4], q=q, scale=sc)
    wq, ws = O.quantize_tokens(O.fwht(O.bf16_to_f32(act) * su.astype(f32)))
    assert np.array_equal(sc.cpu().numpy(), ws[:, 0]) and np.array_equal(q.cpu().numpy(), wq)


@pytest.mark.parametrize('adt', [torch.int32, torch.float32, torch.bfloat16])
@pytest.mark.parametrize('N,M', [(4096, 256), (4096, 257), (4096, 513), (6144, 256), (6144, 257), (4608, 256), (4608, 257), (2048, 256), (2048, 257)])
def test_rows_around_the_lines_between_engines(N, M, adt):
    """Widths and row counts where calls change between the wave rows and the LDS engine: each row as in calls of 40, whole
    vectors and (columns 8 bytes off) not; epilogues alone and in a group, the plain middle, column scales."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(N + M)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    sign = lambda n: torch.where(r(n) > 0, 1, -1).to(torch.int8)
    acc, x, cs = (r(M, N + 8) * 1000).to(adt), r(M, N).bfloat16(), (torch.rand(N, generator=g, device=DEV) + 0.5).half()
    sv, su, bias, rs, s = sign(N), sign(N), r(N), torch.rand(N, generator=g, device=DEV) + 0.1, torch.rand(M, generator=g, device=DEV) + 0.1
    rs = None if adt == torch.float32 else rs

    def run(a, b):
        m, st, out = b - a, s[a:b] if adt == torch.int32 else None, []
        for col0 in (0, 8 // acc.element_size()):
            y = torch.empty(m, N, dtype=torch.bfloat16, device=DEV)
            Kn.post(acc[a:b], st, rs, sv, bias, y, col0=col0)
            ys = [torch.empty(m, N, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
            Kn.post_group([(acc[a:b], col0, rs, sv, None, t, False) for t in ys], adt, torch.bfloat16, st, m)
            out += [y] + ys
        q, sc = torch.empty(m, N, dtype=torch.int8, device=DEV), torch.empty(m, device=DEV)
        Kn.mid1(acc[a:b, :N].contiguous(), st, rs, sv, bias, su, q=q, scale=sc)
        q2, sc2 = torch.empty_like(q), torch.empty_like(sc)
        Kn.pre(x[a:b], su, q=q2, scale=sc2, col_scale=cs)
        return out + [q, sc, q2, sc2]
    whole, parts = run(0, M), [run(a, min(a + 40, M)) for a in range(0, M, 40)]
    for i, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[i] for p in parts]))


@pytest.mark.parametrize('widths', [(2048, 1024, 1024), (2048, 256, 256), (2048, 2048), (2048,), (8192, 8192), (16384,)])
@pytest.mark.parametrize('M', [64, 65, 256, 257, 384, 385, 512, 513])
def test_group_epilogues_around_the_lines(widths, M):
    """Epilogue groups where row counts, widths and types change the engine, segments in the launch and in device memory: the
    rows of tcq_post in calls of 40."""
    from yanlongvla_amd import kernels as Kn
    g = torch.Generator(device=DEV).manual_seed(M + sum(widths))
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    s = torch.rand(M, generator=g, device=DEV) + 0.1
    for adt in (torch.int32, torch.float32, torch.bfloat16):
        acc = (r(M, sum(widths)) * 1000).to(adt)
        st = s if adt == torch.int32 else None
        for ydt in (torch.bfloat16, torch.float32):
            segs, want, c = [], [], 0
            for n in widths:
                sv, rs = torch.where(r(n) > 0, 1, -1).to(torch.int8), None if adt == torch.float32 else torch.rand(n, generator=g, device=DEV)
                segs.append((acc, c, rs, sv, None, torch.empty(M, n, dtype=ydt, device=DEV), False))
                want.append(torch.empty(M, n, dtype=ydt, device=DEV))
                for a in range(0, M, 40):
                    Kn.post(acc[a:a + 40], None if st is None else st[a:a + 40], rs, sv, None, want[-1][a:a + 40], col0=c)
                c += n
            Kn.post_group(segs, adt, ydt, st, M)
            assert all(torch.equal(t[5], w) for t, w in zip(segs, want))
            for t in segs:
                t[5].zero_()
            Kn.post_batched(Kn.post_segments(segs, DEV), len(segs), adt, ydt, st, M, max(widths))
            assert all(torch.equal(t[5], w) for t, w in zip(segs, want))
