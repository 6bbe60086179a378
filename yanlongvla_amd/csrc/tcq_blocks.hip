// Row kernels for widths of several Walsh blocks (1152 = 1024 + 128, 1536, 3072, 4304 = 4096 + 128 + 64 + 16, 6144, ...) and
// for column scales: a row lives in the registers of one wave, or of four.
//
// A row is cut into groups of 256 elements, lane l of a wave holding elements 4 l .. 4 l + 3 of each of its groups, so every
// load and store instruction covers consecutive memory. Index bits 0, 1 are then inside a lane, bits 2 .. 7 across the lanes
// and the rest across a wave's groups: the butterflies run in the ascending stage order of the definition, each the FP32
// (a + b, a - b), so the results equal the LDS engine's bit for bit. Blocks of 256 and more are whole groups; since block
// widths descend, the blocks below 256 (128, 64, 32, 16, ...) lie side by side in the row's last group, each on an aligned
// power of two of lanes, and run together: a lane takes part in the lane stages its block has.
// One wave needs no LDS and no barrier. Four waves share a row of which each block of 1024 and more is split into quarters:
// a wave runs its quarter, then the block's last two stages go across the waves through LDS (one barrier); smaller blocks
// and the last group stay with wave 0.
// What bounds it: a few rows are bound by latency, many by VALU issue (about 17 instructions per element and transform). The
// LDS engine, which these widths took before, moves every element through the LDS once per four or five stages with most
// threads idle in the small blocks: rotate + quantize of 50 x 1536 13.1 us, 768 x 1152 9.2 us, the plain MLP middle of
// 768 x 4304 25.4 us.
#include "tcq_blocks.h"

#include "tcq_launch.h"

namespace {

// a lane's place in the row. NW waves per row; local full groups l < nf of this wave: for NW = 1 groups 0 .. K / 256 - 1;
// for NW = 4 its quarters of the blocks >= 1024 (l < S), then (wave 0) the other full groups.
template <int NW>
struct Place {
    int K, wave, lane, S, nf, n4;                    // n4: lanes of the last group (wave 0)
    __device__ Place(int K_) : K(K_) {
        wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lane = threadIdx.x & 63;
        S = NW == 1 ? K >> 8 : K >> 10;
        nf = NW == 1 ? S : S + (wave == 0 ? (K & 1023) >> 8 : 0);
        n4 = wave == 0 ? (K & 255) >> 2 : 0;
    }
    // log2 of the local groups of the block that holds local group l: blocks are the set bits of the group count from the top
    __device__ __forceinline__ int block(int l) const {
        return l < S ? 31 - __clz(S ^ l) : 31 - __clz(((K & 1023) >> 8) ^ (l - S));
    }
    __device__ __forceinline__ int local(int l) const { return l < S ? l : l - S; }
    // first row index of the lane in local group l / in the last group
    __device__ __forceinline__ int at(int l) const {
        if (NW == 1) return 256 * l + 4 * lane;
        if (l >= S) return 1024 * S + 256 * (l - S) + 4 * lane;
        const int j = block(l), b0 = S & ~((2 << j) - 1);
        return 1024 * b0 + (wave << (8 + j)) + 256 * (l - b0) + 4 * lane;
    }
    __device__ __forceinline__ int tail() const { return (K & ~255) + 4 * lane; }
    // float(1 / sqrt(2^L)): a power of two, or one times float(1 / sqrt(2))
    static __device__ __forceinline__ float norm(int L) {
        return __uint_as_float((u32)(127 - (L >> 1)) << 23) * ((L & 1) ? (float)(1.0 / __builtin_sqrt(2.0)) : 1.f);
    }
    __device__ __forceinline__ float c(int l) const { return norm((NW == 1 || l >= S ? 8 : 10) + block(l)); }
    __device__ __forceinline__ int tail_bits() const { return 31 - __clz(n4 ^ lane); }      // lane stages of the lane's block
    __device__ __forceinline__ bool in_tail() const { return lane < n4; }
};

// one lane stage (partner lane ^ 2^s) of 4 values; every lane gets a + b of the pair's lower and upper value, or a - b
template <int s>
__device__ __forceinline__ void lane_stage(float (&v)[4], int lane) {
    if constexpr (s < 4) {
        const u32 neg = (lane >> s & 1) << 31;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            // partner: quad permutes, row_ror:8, and for 4 the reversed quad mirrored in its half row (^ 3, then ^ 7)
            const float p = s == 0 ? dpp<0xB1>(v[e]) : s == 1 ? dpp<0x4E>(v[e]) : s == 2 ? dpp<0x141>(dpp<0x1B>(v[e])) : dpp<0x128>(v[e]);
            v[e] = __uint_as_float(__float_as_uint(v[e]) ^ neg) + p;
        }
    } else {
        // two values a, b at a time: the swap gathers the lower lanes' halves of both in one register and the upper lanes'
        // in the other; after the butterfly the same swap takes them back
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            const u32 a = __float_as_uint(v[e]), b = __float_as_uint(v[e + 1]);
            const auto r = s == 4 ? __builtin_amdgcn_permlane16_swap(a, b, false, false) : __builtin_amdgcn_permlane32_swap(a, b, false, false);
            const float lo = __uint_as_float(r[0]), hi = __uint_as_float(r[1]);
            const u32 x = __float_as_uint(lo + hi), y = __float_as_uint(lo - hi);
            const auto t = s == 4 ? __builtin_amdgcn_permlane16_swap(x, y, false, false) : __builtin_amdgcn_permlane32_swap(x, y, false, false);
            v[e] = __uint_as_float(t[0]);
            v[e + 1] = __uint_as_float(t[1]);
        }
    }
}

// a row's values in a wave (FM >= nf: 9 for quarters of up to 6 x 1024 and three more groups, 7 below 2048)
template <int FM>
struct Row {
    float v[FM][4], t[4];
};

// use(values, first row index, normalisation constant, loaded) over the lane's values, four groups at a time: load(index) is
// issued for all four before the first use (a group outside the row loads at NONE, past every buffer's end)
constexpr int NONE = 0x10000000;
template <int NW, int FM, class L, class U>
__device__ __forceinline__ void each(const Place<NW>& P, Row<FM>& R, L&& load, U&& use) {
    const int it = P.in_tail() ? P.tail() : NONE;
    const auto rt = load(it);
#pragma unroll
    for (int l0 = 0; l0 < FM; l0 += 4) {
        decltype(load(0)) r[4];
        int i[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (l0 + k < FM) r[k] = load(i[k] = l0 + k < P.nf ? P.at(l0 + k) : NONE);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (l0 + k < FM && l0 + k < P.nf) use(R.v[l0 + k], i[k], P.c(l0 + k), r[k]);
    }
    if (P.in_tail()) use(R.t, it, Place<NW>::norm(2 + P.tail_bits()), rt);
}
template <int NW, int FM, class U>
__device__ __forceinline__ void each(const Place<NW>& P, Row<FM>& R, U&& use) {
    each(P, R, [](int) { return 0; }, [&](float(&v)[4], int i, float c, int) { use(v, i, c); });
}

// unnormalised block Walsh; NW = 4: ex holds K floats, one barrier inside (ex may be written again after a later barrier)
template <int NW, int FM>
__device__ __forceinline__ void rows_walsh(const Place<NW>& P, Row<FM>& R, float* ex) {
    const int lane = P.lane;
#pragma unroll
    for (int l = 0; l < FM; ++l) {
        if (l < P.nf) {
            butterflies<2>(R.v[l]);
            lane_stage<0>(R.v[l], lane);
            lane_stage<1>(R.v[l], lane);
            lane_stage<2>(R.v[l], lane);
            lane_stage<3>(R.v[l], lane);
            lane_stage<4>(R.v[l], lane);
            lane_stage<5>(R.v[l], lane);
        }
    }
    if (P.n4) {                                      // uniform
        butterflies<2>(R.t);
        const int bits = P.in_tail() ? P.tail_bits() : 0;
        auto stage = [&](auto s) {
            constexpr int S = decltype(s)::value;
            float u[4] = {R.t[0], R.t[1], R.t[2], R.t[3]};
            lane_stage<S>(u, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) R.t[e] = S < bits ? u[e] : R.t[e];
        };
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 3>{});
        stage(std::integral_constant<int, 4>{});     // a block of the last group has at most 32 lanes
    }
#pragma unroll
    for (int s = 0; (1 << s) < FM; ++s) {            // across the wave's groups
        const int h = 1 << s;
#pragma unroll
        for (int l = 0; l + h < FM; ++l)
            if (l + h < P.nf && s < P.block(l) && !(P.local(l) & h)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = R.v[l][e], b = R.v[l + h][e];
                    R.v[l][e] = a + b;
                    R.v[l + h][e] = a - b;
                }
            }
    }
    if constexpr (NW == 4) {                         // the blocks' last two stages, across the waves
        float4_t* x4 = (float4_t*)ex;
#pragma unroll
        for (int l = 0; l < FM; ++l)
            if (l < P.S) x4[(l * 4 + P.wave) * 64 + lane] = float4_t{R.v[l][0], R.v[l][1], R.v[l][2], R.v[l][3]};
        __syncthreads();
#pragma unroll
        for (int l = 0; l < FM; ++l)
            if (l < P.S) {
                float4_t w[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) w[k] = x4[(l * 4 + k) * 64 + lane];
                const int o = P.wave & 1;            // value of position o of each pair, then of the wave's half
                const float4_t a = o ? w[0] - w[1] : w[0] + w[1], b = o ? w[2] - w[3] : w[2] + w[3];
                const float4_t r = (P.wave & 2) ? a - b : a + b;
#pragma unroll
                for (int e = 0; e < 4; ++e) R.v[l][e] = r[e];
            }
    }
}

// 4 consecutive elements at index i of a row of type DT behind a buffer resource (zeros at NONE), raw and as FP32
template <int DT>
__device__ __forceinline__ auto raw4(rsrc_t r, int i) {
    if constexpr (DT == TCQ_F32 || DT == TCQ_I32) return __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(r, i * 4, 0, 0));
    else if constexpr (DT == TCQ_I8) return (u32)__builtin_amdgcn_raw_buffer_load_b32(r, i, 0, 0);
    else return __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(r, i * 2, 0, 0));
}
template <int DT, class R4>
__device__ __forceinline__ float elem4(const R4& a, int e) {
    if constexpr (DT == TCQ_F32) return __uint_as_float(a[e]);
    else if constexpr (DT == TCQ_I32) return (float)(int)a[e];
    else if constexpr (DT == TCQ_I8) return i8_f32(a, e);
    else {
        const u16 h = (u16)(a[e >> 1] >> (16 * (e & 1)));
        return DT == TCQ_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
    }
}
__device__ __forceinline__ void st4(void* p, size_t i, int dt, const float (&v)[4]) {
    if (dt == TCQ_F32) *gptr((float4_t*)((float*)p + i)) = float4_t{v[0], v[1], v[2], v[3]};
    else if (dt == TCQ_BF16) *gptr((uint2_t*)((u16*)p + i)) = uint2_t{bf16x2(v[0], v[1]), bf16x2(v[2], v[3])};
    else *gptr((uint2_t*)((u16*)p + i)) = uint2_t{(u32)f32_to_f16(v[0]) | ((u32)f32_to_f16(v[1]) << 16), (u32)f32_to_f16(v[2]) | ((u32)f32_to_f16(v[3]) << 16)};
}

// the row of type DT into R: every load issued before the first use
template <int DT, int NW, int FM>
__device__ __forceinline__ void load_row4(const Place<NW>& P, Row<FM>& R, const void* row) {
    constexpr int SZ = DT == TCQ_F32 || DT == TCQ_I32 ? 4 : 2;
    const rsrc_t rx = make_rsrc(row, (u32)P.K * SZ);
    decltype(raw4<DT>(rx, 0)) raw[FM + 1];
#pragma unroll
    for (int l = 0; l < FM; ++l) raw[l] = raw4<DT>(rx, l < P.nf ? P.at(l) : NONE);
    raw[FM] = raw4<DT>(rx, P.in_tail() ? P.tail() : NONE);
#pragma unroll
    for (int l = 0; l <= FM; ++l)
#pragma unroll
        for (int e = 0; e < 4; ++e) (l < FM ? R.v[l < FM ? l : 0][e] : R.t[e]) = elem4<DT>(raw[l], e);
}
// x * su of a row into R
template <int NW, int FM>
__device__ __forceinline__ void load_x(const Place<NW>& P, Row<FM>& R, const void* x, int dt, size_t base, const i8* su) {
    if (dt == TCQ_F32) load_row4<TCQ_F32>(P, R, (const float*)x + base);
    else if (dt == TCQ_BF16) load_row4<TCQ_BF16>(P, R, (const u16*)x + base);
    else load_row4<TCQ_F16>(P, R, (const u16*)x + base);
    if (!su) return;
    const rsrc_t rs = make_rsrc(su, P.K);
    each(P, R, [&](int i) { return raw4<TCQ_I8>(rs, i); }, [&](float(&v)[4], int, float, u32 w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * elem4<TCQ_I8>(w, e);
    });
}
// SCALE(acc) of a row (tcq_post) into R
template <int NW, int FM>
__device__ __forceinline__ void load_acc(const Place<NW>& P, Row<FM>& R, const void* acc, int dt, size_t base, float s, const float* rs) {
    if (dt == TCQ_F32) {
        load_row4<TCQ_F32>(P, R, (const float*)acc + base);
        return;
    }
    if (dt == TCQ_I32) load_row4<TCQ_I32>(P, R, (const int*)acc + base);
    else load_row4<TCQ_BF16>(P, R, (const u16*)acc + base);
    const rsrc_t rr = make_rsrc(rs, P.K * 4);
    each(P, R, [&](int i) { return raw4<TCQ_F32>(rr, i); }, [&](float(&v)[4], int, float, const uint4_t& r) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (dt == TCQ_I32 ? v[e] * s : v[e]) * elem4<TCQ_F32>(r, e);
    });
}
// the values of walsh(acc) -> * c -> * sv (+ bias) (-> GELU(BF16)) of a row epilogue, in place
template <int NW, int FM>
__device__ __forceinline__ void finish(const Place<NW>& P, Row<FM>& R, const i8* sv, const float* bias, const u16* lut) {
    const rsrc_t rv = make_rsrc(sv, P.K);
    each(P, R, [&](int i) { return raw4<TCQ_I8>(rv, i); }, [&](float(&v)[4], int, float c, u32 w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (v[e] * c) * elem4<TCQ_I8>(w, e);
    });
    if (bias) {
        const rsrc_t rb = make_rsrc(bias, P.K * 4);
        each(P, R, [&](int i) { return raw4<TCQ_F32>(rb, i); }, [&](float(&v)[4], int, float, const uint4_t& b) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] + elem4<TCQ_F32>(b, e);
        });
    }
    if (lut) {                                       // 16 lookups in flight
        struct G { u16 g[4]; };
        const rsrc_t rl = make_rsrc(lut, 131072);
        auto look = [&](const float(&v)[4]) {
            G o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.g[e] = __builtin_amdgcn_raw_buffer_load_b16(rl, (int)f32_to_bf16(v[e]) * 2, 0, 0);
            return o;
        };
        const G gt = look(R.t);
#pragma unroll
        for (int l0 = 0; l0 < FM; l0 += 4) {
            G g[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (l0 + k < FM) g[k] = look(R.v[l0 + k]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (l0 + k < FM)
#pragma unroll
                    for (int e = 0; e < 4; ++e) R.v[l0 + k][e] = bf16_to_f32(g[k].g[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) R.t[e] = bf16_to_f32(gt.g[e]);
    }
}

// walsh, * c (* cs), per-token absmax, INT8 (the operations of k_pre)
template <int NW, int FM>
__device__ __forceinline__ void rotate_quantize_row(const Place<NW>& P, Row<FM>& R, float* ex, float* red, const u16* cs, i8* q, int* q4,
                                                    int ldq, float* scale, int tok) {
    rows_walsh<NW, FM>(P, R, ex);
    float mx = 0.f;
    if (cs) {
        const rsrc_t rc = make_rsrc(cs, P.K * 2);
        each(P, R, [&](int i) { return raw4<TCQ_F16>(rc, i); }, [&](float(&v)[4], int, float c, const uint2_t& k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = (v[e] * c) * elem4<TCQ_F16>(k, e);
                mx = fmaxf(mx, fabsf(v[e]));
            }
        });
    } else {
        each(P, R, [&](float(&v)[4], int, float c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = v[e] * c;
                mx = fmaxf(mx, fabsf(v[e]));
            }
        });
    }
    mx = NW == 1 ? wave_max(mx) : block_max(mx, red);
    const float sc = token_scale(mx);
    if (threadIdx.x == 0) scale[tok] = sc;
    const QScale S = qscale(sc);
    each(P, R, [&](float(&v)[4], int i, float) {
        u32 w;
        q8_words<1>(v, S, &w);
        if (q) *gptr((u32*)(q + (size_t)tok * P.K + i)) = w;
        if (q4) {
            if (ldq == TCQ_LDQ_TOKEN_BLOCKS) *gptr((u32*)((i8*)q4 + tb_offset(tok, i, P.K))) = w;
            else gptr(q4)[(size_t)(i >> 2) * ldq + tok] = (int)w;
        }
    });
}

template <int NW, int FM>
__global__ __launch_bounds__(64 * NW) void k_rht_rows(const void* x, int xdt, int ldx, const i8* su, void* y, int ydt, int ldy, int K) {
    extern __shared__ float ex[];
    const Place<NW> P(K);
    Row<FM> R;
    load_x<NW, FM>(P, R, x, xdt, (size_t)blockIdx.x * ldx, su);
    rows_walsh<NW, FM>(P, R, ex);
    const size_t base = (size_t)blockIdx.x * ldy;
    each(P, R, [&](float(&v)[4], int i, float c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * c;
        st4(y, base + i, ydt, v);
    });
}

template <int NW, int FM>
__global__ __launch_bounds__(64 * NW) void k_pre_rows(const void* x, int xdt, const i8* su, const u16* cs, i8* q, int* q4, int ldq, float* scale, int K) {
    extern __shared__ float ex[];
    __shared__ float red[16];
    const Place<NW> P(K);
    Row<FM> R;
    load_x<NW, FM>(P, R, x, xdt, (size_t)blockIdx.x * K, su);
    rotate_quantize_row<NW, FM>(P, R, ex, red, cs, q, q4, ldq, scale, blockIdx.x);
}

struct PostRows {
    tcq_post_seg s[TCQ_MAX_SEGS];
};

template <int NW, int FM>
__global__ __launch_bounds__(64 * NW) void k_post_rows(const PostRows A, const float* s, const u16* gelu_lut, int adt, int ydt) {
    extern __shared__ float ex[];
    const tcq_post_seg S = A.s[blockIdx.y];
    const int tok = blockIdx.x;
    const Place<NW> P(S.N);
    Row<FM> R;
    load_acc<NW, FM>(P, R, S.acc, adt, (size_t)tok * S.lda + S.col0, adt == TCQ_I32 ? gptr(s)[tok] : 1.f, S.rs);
    rows_walsh<NW, FM>(P, R, ex);
    finish(P, R, S.sv, S.bias, S.gelu ? gelu_lut : nullptr);
    const size_t base = (size_t)tok * S.N;
    each(P, R, [&](float(&v)[4], int i, float) { st4(S.y, base + i, ydt, v); });
}

// x = GELU(BF16(walsh(acc) * sv + bias)) * su -> walsh -> per-token INT8 (k_mid1)
template <int NW, int FM>
__global__ __launch_bounds__(64 * NW) void k_mid1_rows(const void* acc, int adt, int lda, const float* s, const float* rs, const i8* sv,
                                                       const float* bias, const u16* lut, const i8* su, i8* q, int* q4, int ldq, float* scale, int N) {
    extern __shared__ float ex[];
    __shared__ float red[16];
    const int tok = blockIdx.x;
    const Place<NW> P(N);
    Row<FM> R;
    load_acc<NW, FM>(P, R, acc, adt, (size_t)tok * lda, adt == TCQ_I32 ? gptr(s)[tok] : 1.f, rs);
    rows_walsh<NW, FM>(P, R, ex);
    finish(P, R, sv, bias, lut);
    const rsrc_t ru = make_rsrc(su, N);
    each(P, R, [&](int i) { return raw4<TCQ_I8>(ru, i); }, [&](float(&v)[4], int, float, u32 w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * elem4<TCQ_I8>(w, e);
    });
    if (NW > 1) __syncthreads();                     // every wave has read ex
    rotate_quantize_row<NW, FM>(P, R, ex, red, nullptr, q, q4, ldq, scale, tok);
}

bool al(const void* p, int n) { return ((uintptr_t)p & (n - 1)) == 0; }
int bytes_of(int dt) { return dt == TCQ_F32 || dt == TCQ_I32 ? 4 : 2; }
bool input_type(int dt) { return dt == TCQ_F32 || dt == TCQ_BF16 || dt == TCQ_F16; }
// Widths up to 7164: beyond, a wave's quarter no longer fits its registers well (two rows of 16384: 102 us against 59 through
// the LDS engine).
bool takes(int K) { return K % 4 == 0 && K >= 64 && K < 7 * 1024; }
// Four waves per row from 2048 on (one wave of 17 groups runs 28 us through the plain middle of 768 x 4304), and from 1024 on
// while the rows leave SIMDs idle
bool four_waves(int M, int K) { return K >= 2048 || (M <= 256 && K >= 1024); }
// Wide rows of one block, or of two, that the LDS engine's vectors move faster: few passes with every thread busy, against side
// vectors read in series here. MI355X, us, LDS engine / wave rows. Epilogues: 64 x 4096 from int32 5.1 / 6.6, from FP32 5.0 / 5.9, 400:
// 8.6 / 7.9, 968: 9.7 / 10.5; 64 x 6144 with bias from BF16 7.4 / 8.5, from FP32 7.3 / 7.7, 968 from BF16 13.6 / 14.2, from FP32 14.1 /
// 13.4; 64 x 4608 from BF16 7.3 / 7.8, 400: 9.5 / 9.2. Plain middle: 64 x 4096 9.9 / 11.8, 64 x 2048 8.5 / 9.1, 257 x 4096 16.0 / 13.1.
// Rotate + quantize with column scales: 64 x 4096 6.2 / 7.1, 257: 10.2 / 7.7. (Its threads per row fall from 257 rows on.)
bool lds_post(int rows, int N, int acc_dtype) {
    const bool scaled = acc_dtype != TCQ_F32, two = __builtin_popcount(N) == 2;
    if (rows <= 256) return N == 4096 || N == 6144 || (N > 4096 && two && scaled);
    return scaled && (N == 6144 || (N == 4096 && rows > 512));
}
bool lds_mid1(int M, int N) { return M <= 256 && (N == 2048 || N == 4096); }
bool lds_pre(int M, int K, bool cs) { return M <= 256 && cs && K == 4096; }

}  // namespace

#define ROWS_LAUNCH(KER, GRID, M, K, ...)                                                                                  \
    do {                                                                                                                   \
        if (four_waves(M, K)) {                                                                                            \
            const size_t sh = (size_t)(K >> 10) * 4096;                                                                    \
            launch_k(KER<4, 9>, GRID, dim3(256), sh, st, __VA_ARGS__);                                                     \
        } else launch_k(KER<1, 7>, GRID, dim3(64), 0, st, __VA_ARGS__);                                                    \
    } while (0)

bool blocks_rht(const void* x, int x_dtype, int ldx, const i8* su, void* y, int y_dtype, int ldy, int M, int K, hipStream_t st) {
    const int xs = bytes_of(x_dtype), ys = bytes_of(y_dtype);
    if (!takes(K) || !input_type(x_dtype) || !input_type(y_dtype) || !al(x, 4 * xs) || !al(y, 4 * ys) || ldx % 4 || ldy % 4 || (su && !al(su, 4)))
        return false;
    ROWS_LAUNCH(k_rht_rows, dim3(M), M, K, x, x_dtype, ldx, su, y, y_dtype, ldy, K);
    return true;
}

bool blocks_pre(const void* x, int x_dtype, const i8* su, const u16* cs, i8* q, int* q4, int ldq, float* scale, int M, int K, bool lds,
                hipStream_t st) {
    if (!takes(K) || (lds && lds_pre(M, K, cs)) || !input_type(x_dtype) || !al(x, 4 * bytes_of(x_dtype)) || (su && !al(su, 4)) || (cs && !al(cs, 8)) || (q && !al(q, 4)) ||
        (q4 && !al(q4, 4)))
        return false;
    ROWS_LAUNCH(k_pre_rows, dim3(M), M, K, x, x_dtype, su, cs, q, q4, ldq, scale, K);
    return true;
}

bool blocks_post(const tcq_post_seg* segs, int nseg, int acc_dtype, const float* s, const u16* gelu_lut, int y_dtype, int M,
                 bool lds, hipStream_t st) {
    if ((acc_dtype != TCQ_F32 && acc_dtype != TCQ_I32 && acc_dtype != TCQ_BF16) || !input_type(y_dtype)) return false;
    PostRows A = {};
    int most = 0;
    for (int i = 0; i < nseg; ++i) {
        const tcq_post_seg& g = segs[i];
        if (!takes(g.N) || (lds && lds_post(M * nseg, g.N, acc_dtype)) || !al(g.acc, 4 * bytes_of(acc_dtype)) || g.lda % 4 || g.col0 % 4 || !al(g.y, 4 * bytes_of(y_dtype)) || !al(g.sv, 4) ||
            (acc_dtype != TCQ_F32 && !al(g.rs, 16)) || (g.bias && !al(g.bias, 16)))
            return false;
        A.s[i] = g;
        most = g.N > most ? g.N : most;
    }
    const dim3 grid(M, nseg);
    const int K = most;                              // the variant of the widest segment holds the others
    ROWS_LAUNCH(k_post_rows, grid, M * nseg, K, A, s, gelu_lut, acc_dtype, y_dtype);
    return true;
}

bool blocks_mid1(const void* acc, int acc_dtype, int lda, const float* s, const float* rs, const i8* sv, const float* bias,
                 const u16* lut, const i8* su, i8* q, int* q4, int ldq, float* scale, int M, int N, bool lds, hipStream_t st) {
    if ((acc_dtype != TCQ_F32 && acc_dtype != TCQ_I32 && acc_dtype != TCQ_BF16) || !takes(N) || (lds && lds_mid1(M, N)) || !al(acc, 4 * bytes_of(acc_dtype)) || lda % 4 ||
        !al(sv, 4) || !al(su, 4) || (acc_dtype != TCQ_F32 && !al(rs, 16)) || (bias && !al(bias, 16)) || (q && !al(q, 4)) || (q4 && !al(q4, 4)))
        return false;
    ROWS_LAUNCH(k_mid1_rows, dim3(M), M, N, acc, acc_dtype, lda, s, rs, sv, bias, lut, su, q, q4, ldq, scale, N);
    return true;
}
