// Trellis decode kernels: load-time table snap and word repack, dense INT8 / FP16 decode.
#include "tcq_device.h"
#include "tcq_launch.h"

// 48-bit window of tile row r: hi = (word[2r] << 16) | word[2r + 1], lo = word[(2r + 2) & 31]. State p (0..7) =
// bits [4p, 4p + 16) of hi:lo from the top (reference tcq_format.py:58-63; kernels.py:186-205).
__device__ __forceinline__ u32 row_state(u32 hi, u32 lo16, int p) {
    const u64 win = ((u64)hi << 16) | lo16;
    return (u32)(win >> (32 - 4 * p)) & 0xffffu;
}

// ------------------------------------------------------------------------------------------------------------------ snap
// Workgroup g snaps table g of G (row-group tables: rows [g rpt, (g + 1) rpt) read table g, rpt = m / G).
__global__ void k_snap(const u16* tlut_all, const u16* row_scale, int rpt, i8* t8_all, float* rs, float* gain) {
    __shared__ float red[16];
    const int gi = blockIdx.x;
    const u16* tlut = tlut_all + 1024 * gi;
    i8* t8 = t8_all + 1024 * gi;
    float mx = 0.f;
    for (int i = threadIdx.x; i < 1024; i += blockDim.x) mx = fmaxf(mx, fabsf(f16_to_f32(tlut[i])));
    mx = block_max(mx, red);
    // 127.0 / tensor is Tensor.__rdiv__ = reciprocal() * 127 (torch/_tensor.py), so g = float(1 / amax) * 127
    const float g = (1.0f / mx) * 127.0f;
    for (int i = threadIdx.x; i < 1024; i += blockDim.x) {
        float v = __builtin_rintf(f16_to_f32(tlut[i]) * g);
        v = fminf(fmaxf(v, -127.f), 127.f);
        t8[i] = (i8)(int)v;
    }
    for (int i = threadIdx.x; i < rpt; i += blockDim.x) rs[gi * rpt + i] = f16_to_f32(row_scale[gi * rpt + i]) / g;
    if (threadIdx.x == 0 && gain) gain[gi] = g;
}

// ---------------------------------------------------------------------------------------------------------------- repack
__global__ void k_repack(const u16* bits, u32* wdev, int m, int n, long long total) {
    const long long d = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int tiles = n >> 4, nch = (n + 255) >> 8;
    const int j = (int)(d & 3), lane = (int)((d >> 2) & 63);
    const long long blk = d >> 8;                          // (I, c) chunk index
    const int c = (int)(blk % nch), I = (int)(blk / nch);
    const int r = lane & 15, g = lane >> 4, tile = 16 * c + 4 * j + g;
    u32 v = 0;
    if (tile < tiles) {
        const u16* t = bits + ((size_t)I * tiles + tile) * 32;
        v = ((u32)t[2 * r] << 16) | (u32)t[2 * r + 1];
    }
    wdev[d] = v;
}

// --------------------------------------------------------------------------------------------------------- dense decode
// One thread per (row, tile column): the 16 weights of one tile row. Sign-folded tables in LDS. grid (blocks per row group,
// row groups): the workgroups of group g (rows [g rpt, (g + 1) rpt)) load table g.
__global__ void k_decode_i8(const u16* bits, const i8* t8_all, i8* out, int rpt, int n) {
    __shared__ u16 tab[1024];
    const i8* t8 = t8_all + 1024 * blockIdx.y;
    for (int e = threadIdx.x; e < 1024; e += blockDim.x) {
        const int h = e & 511;
        int v0 = t8[2 * h];
        const int v1 = t8[2 * h + 1];
        if (e >> 9) v0 = -v0;
        tab[e] = (u16)((v0 & 0xff) | ((v1 & 0xff) << 8));
    }
    __syncthreads();
    const int tiles = n >> 4;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)rpt * tiles) return;
    const int row = blockIdx.y * rpt + (int)(idx / tiles), J = (int)(idx % tiles), r = row & 15;
    const u16* t = bits + ((size_t)(row >> 4) * tiles + J) * 32;
    const u32 hi = ((u32)t[2 * r] << 16) | t[2 * r + 1], lo = t[(2 * r + 2) & 31];
    uint4_t w;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const u32 s0 = row_state(hi, lo, 2 * d), s1 = row_state(hi, lo, 2 * d + 1);
        w[d] = (u32)tab[code_index((s0 + 1) * s0)] | ((u32)tab[code_index((s1 + 1) * s1)] << 16);
    }
    *(uint4_t*)(out + (size_t)row * n + 16 * J) = w;
}

// Dense decode from the tcq_repack words of up to TCQ_MAX_SEGS layers in one launch, INT8 or BF16 out. A wave takes 1 KiB
// chunks (one tile row, 256 columns); lane (g, r) holds the windows of row r for tiles 16 c + 4 j + g (j = 0..3) in one
// dwordx4 and writes their 16 weights, so a store covers 64 (INT8) or, in two, 128 contiguous bytes of each of the 16 rows.
// The lookups are those of the fused products (pk_code states, a sign-folded table with C copies, lane l reading copy
// l mod C), whose results per lane and j are the row's weights in column order, so the INT8 output equals k_decode_i8's byte
// for byte; BF16 entries are the table values' BF16 images (exact, |t8| <= 127), the sign folded into bit 15.
// grid (blocks of NW * CPW chunks, layers, row-group tables); a workgroup reads one table.
// What bounds it: the writes, once the launch and the table fill (global round trip, 4 C KiB of LDS) are paid for: one
// launch for a layer group pays them once, and CPW chunks per wave keep one round of workgroups. Backbone gate | up (2 x
// 16384 x 2048, 67 MB out): 20.9 us as two launches of one chunk per wave.
struct DecSegs {
    tcq_gemm_seg s[TCQ_MAX_SEGS];
};

template <int ODT, int NW, int C, int CPW>
__global__ __launch_bounds__(64 * NW) void k_decode_words(const DecSegs P, int n) {
    __shared__ __attribute__((aligned(16))) u32 tab[1024 * C];
    const tcq_gemm_seg S = P.s[blockIdx.y];
    const int rpt = S.rows_per_table > 0 ? S.rows_per_table : S.m;
    const int nch = (n + 255) >> 8, tiles = n >> 4;
    const int first = blockIdx.z * rpt;                                  // first row of this table's group
    const int nchunks = (rpt >> 4) * nch, c0 = blockIdx.x * (NW * CPW) + (threadIdx.x >> 6);
    if (first >= S.m || (int)blockIdx.x * (NW * CPW) >= nchunks) return; // uniform
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    uint4_t wa[CPW];
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
        wa[i] = uint4_t{0u, 0u, 0u, 0u};
        if (c0 + i * NW < nchunks) wa[i] = gptr((const uint4_t*)((const u32*)S.w + ((size_t)(first >> 4) * nch + c0 + i * NW) * 256))[lane];
    }
    const i8* t8 = S.t8 + 1024 * blockIdx.z;
    for (int e = threadIdx.x; e < 1024; e += 64 * NW) {
        const int h = e & 511, v0 = t8[2 * h], v1 = t8[2 * h + 1];
        u32 v;
        if (ODT == TCQ_I8) {
            v = (u32)((e >> 9 ? -v0 : v0) & 0xff) | ((u32)(v1 & 0xff) << 8);
            v |= v << 16;
        } else {
            v = ((__float_as_uint((float)v0) >> 16) ^ ((u32)(e >> 9) << 15)) | (__float_as_uint((float)v1) & 0xffff0000u);
        }
#pragma unroll
        for (int c = 0; c < C; c += 4) *(uint4_t*)(tab + e * C + c) = uint4_t{v, v, v, v};
    }
    __syncthreads();
    const u32 cp4 = (u32)(lane & (C - 1)) << 2;
    constexpr int SH = C == 16 ? 6 : 4;                                  // log2 of an entry's bytes
    static_assert(4 * C == 1 << SH, "copies");
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
        const int chunk = c0 + i * NW;
        if (chunk >= nchunks) break;                                     // uniform per wave
        const int I = chunk / nch, c = chunk - I * nch;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32 hi = wa[i][j];
            const u32 hn = (u32)__builtin_amdgcn_mov_dpp((int)hi, 0x12F, 0xf, 0xf, false);
            u32 e0[4], e1[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const u32 x = pk_code(p == 0 ? hi : __builtin_amdgcn_alignbit(hi, hn, 32 - 4 * p));
                const char* a0 = (const char*)tab + (((x >> 22) << SH) | cp4);               // pair p
                const char* a1 = (const char*)tab + ((((x >> 6) & 1023u) << SH) | cp4);      // pair p + 4
                if (ODT == TCQ_I8) { e0[p] = *(const u16*)a0; e1[p] = *(const u16*)a1; }
                else { e0[p] = *(const u32*)a0; e1[p] = *(const u32*)a1; }
            }
            const int tile = 16 * c + 4 * j + g;
            if (tile >= tiles) continue;
            const size_t at = (size_t)(first + 16 * I + r) * n + 16 * tile;
            if (ODT == TCQ_I8) {
                *gptr((uint4_t*)((i8*)S.out + at)) =
                    uint4_t{e0[0] | (e0[1] << 16), e0[2] | (e0[3] << 16), e1[0] | (e1[1] << 16), e1[2] | (e1[3] << 16)};
            } else {
                gptr((uint4_t*)((u16*)S.out + at))[0] = uint4_t{e0[0], e0[1], e0[2], e0[3]};
                gptr((uint4_t*)((u16*)S.out + at))[1] = uint4_t{e1[0], e1[1], e1[2], e1[3]};
            }
        }
    }
}

// INT8 -> BF16 (exact), 16 values per thread
__global__ void k_i8_to_bf16(const i8* in, u16* out, size_t n16) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n16) return;
    const uint4_t w = gptr((const uint4_t*)in)[i];
    u32 v[8];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float a = (float)(i8)(w[d] >> (16 * h)), b = (float)(i8)(w[d] >> (16 * h + 8));
            v[2 * d + h] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
        }
    gptr((uint4_t*)out)[2 * i] = uint4_t{v[0], v[1], v[2], v[3]};
    gptr((uint4_t*)out)[2 * i + 1] = uint4_t{v[4], v[5], v[6], v[7]};
}

__global__ void k_decode_f16(const u16* bits, const u16* tlut_all, u16* out, int rpt, int n) {
    __shared__ u32 tab[1024];
    const u16* tlut = tlut_all + 1024 * blockIdx.y;
    for (int e = threadIdx.x; e < 1024; e += blockDim.x) {
        const int h = e & 511;
        tab[e] = ((u32)tlut[2 * h] ^ ((u32)(e >> 9) << 15)) | ((u32)tlut[2 * h + 1] << 16);
    }
    __syncthreads();
    const int tiles = n >> 4;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)rpt * tiles) return;
    const int row = blockIdx.y * rpt + (int)(idx / tiles), J = (int)(idx % tiles), r = row & 15;
    const u16* t = bits + ((size_t)(row >> 4) * tiles + J) * 32;
    const u32 hi = ((u32)t[2 * r] << 16) | t[2 * r + 1], lo = t[(2 * r + 2) & 31];
    uint4_t w0, w1;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const u32 s = row_state(hi, lo, p);
        const u32 v = tab[code_index((s + 1) * s)];
        if (p < 4) w0[p] = v; else w1[p - 4] = v;
    }
    uint4_t* o = (uint4_t*)(out + (size_t)row * n + 16 * J);
    o[0] = w0;
    o[1] = w1;
}

// =========================================================================================================== C ABI
extern "C" const char* tcq_version(void) { return "tcq-mi355x 0.1 (gfx950)"; }
extern "C" int tcq_max_width(void) { return TCQ_MAX_WIDTH; }

// Row groups: m rows split evenly into G contiguous groups of rpt = m / G rows, each a whole number of 16-row tiles.
static bool groups_ok(int m, int G) { return G >= 1 && G <= 65535 && m % G == 0 && (m / G) % 16 == 0; }

extern "C" int tcq_snap_groups(const void* tlut, int G, const void* row_scale, int m, int8_t* t8, float* rs, float* gain,
                               tcq_stream_t stream) {
    if (!tlut || !row_scale || !t8 || !rs || m <= 0 || G <= 0) return TCQ_ERR_ARG;
    if (m % G) return TCQ_ERR_SHAPE;
    launch_k(k_snap, dim3(G), dim3(256), 0, (hipStream_t)stream, (const u16*)tlut, (const u16*)row_scale, m / G, (i8*)t8, rs, gain);
    return launch_status();
}

extern "C" int tcq_snap(const void* tlut, const void* row_scale, int m, int8_t* t8, float* rs, float* gain, tcq_stream_t stream) {
    return tcq_snap_groups(tlut, 1, row_scale, m, t8, rs, gain, stream);
}

extern "C" int64_t tcq_repack_words(int m, int n) {
    if (m <= 0 || n <= 0 || m % 16 || n % 16) return TCQ_ERR_SHAPE;
    return (int64_t)(m / 16) * ((n + 255) / 256) * 256;
}

extern "C" int tcq_repack(const void* bits, void* wdev, int m, int n, tcq_stream_t stream) {
    if (!bits || !wdev || m <= 0 || n <= 0) return TCQ_ERR_ARG;
    if (m % 16 || n % 16) return TCQ_ERR_SHAPE;
    const long long total = tcq_repack_words(m, n);
    launch_k(k_repack, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const u16*)bits, (u32*)wdev,
             m, n, total);
    return launch_status();
}

extern "C" int tcq_decode_i8_groups(const void* bits, const int8_t* t8, int G, int8_t* out, int m, int n, tcq_stream_t stream) {
    if (!bits || !t8 || !out || m <= 0 || n <= 0 || G <= 0) return TCQ_ERR_ARG;
    if (m % 16 || n % 16 || !groups_ok(m, G)) return TCQ_ERR_SHAPE;
    if ((uintptr_t)out % 16) return TCQ_ERR_ALIGN;
    const size_t per = (size_t)(m / G) * (n / 16);
    launch_k(k_decode_i8, dim3((unsigned)((per + 255) / 256), G), dim3(256), 0, (hipStream_t)stream, (const u16*)bits,
             (const i8*)t8, (i8*)out, m / G, n);
    return launch_status();
}

template <int ODT>
static void launch_words(const DecSegs& P, int nseg, int tables, long long total, long long most, int n, hipStream_t st) {
    auto grid = [&](int per) { return dim3((unsigned)((most + per - 1) / per), nseg, tables); };
    // 512 workgroups of 16 waves fill the chip (64 KiB of table, two per CU); below a quarter of that, smaller workgroups
    // with a smaller table spread over more CUs
    if (total < 2048) launch_k(k_decode_words<ODT, 4, 4, 1>, grid(4), dim3(256), 0, st, P, n);
    else if (total <= 8192) launch_k(k_decode_words<ODT, 16, 16, 1>, grid(16), dim3(1024), 0, st, P, n);
    else if (total <= 16384) launch_k(k_decode_words<ODT, 16, 16, 2>, grid(32), dim3(1024), 0, st, P, n);
    else launch_k(k_decode_words<ODT, 16, 16, 4>, grid(64), dim3(1024), 0, st, P, n);
}

extern "C" int tcq_decode_group(const tcq_gemm_seg* segs, int nseg, int n, int out_dtype, tcq_stream_t stream) {
    if (!segs || nseg <= 0 || n <= 0) return TCQ_ERR_ARG;
    if (out_dtype != TCQ_I8 && out_dtype != TCQ_BF16) return TCQ_ERR_DTYPE;
    if (nseg > TCQ_MAX_SEGS) return TCQ_ERR_UNSUPPORTED;
    if (n % 16) return TCQ_ERR_SHAPE;
    DecSegs P = {};
    const long long nch = (n + 255) / 256;
    long long total = 0, most = 0;
    int tables = 1;
    for (int i = 0; i < nseg; ++i) {
        const tcq_gemm_seg& g = segs[i];
        if (!g.w || !g.t8 || !g.out || g.m <= 0) return TCQ_ERR_ARG;
        if (g.m % 16 || g.rows_per_table < 0 || (g.rows_per_table > 0 && !groups_ok(g.m, g.m / g.rows_per_table))) return TCQ_ERR_SHAPE;
        if (g.rows_per_table > 0 && g.m % g.rows_per_table) return TCQ_ERR_SHAPE;
        if ((g.m / 16) * nch >= ((long long)1 << 31)) return TCQ_ERR_SHAPE;
        if ((uintptr_t)g.out % 16 || (uintptr_t)g.w % 16) return TCQ_ERR_ALIGN;
        const int rpt = g.rows_per_table > 0 ? g.rows_per_table : g.m;
        const long long chunks = (rpt / 16) * nch;
        if (g.m / rpt > tables) tables = g.m / rpt;
        if (chunks > most) most = chunks;
        total += chunks * (g.m / rpt);
        P.s[i] = g;
    }
    if (out_dtype == TCQ_I8) launch_words<TCQ_I8>(P, nseg, tables, total, most, n, (hipStream_t)stream);
    else launch_words<TCQ_BF16>(P, nseg, tables, total, most, n, (hipStream_t)stream);
    return launch_status();
}

extern "C" int tcq_decode_i8_words(const void* words, const int8_t* t8, int8_t* out, int m, int n, tcq_stream_t stream) {
    if (m <= 0) return TCQ_ERR_ARG;
    const tcq_gemm_seg seg = {words, t8, nullptr, out, m, 0};
    return tcq_decode_group(&seg, 1, n, TCQ_I8, stream);
}

extern "C" int tcq_i8_to_bf16(const int8_t* in, void* out, int64_t count, tcq_stream_t stream) {
    if (!in || !out || count <= 0) return TCQ_ERR_ARG;
    if (count % 16 || count / 16 > ((int64_t)1 << 31) * 64) return TCQ_ERR_SHAPE;
    if ((uintptr_t)in % 16 || (uintptr_t)out % 16) return TCQ_ERR_ALIGN;
    const size_t n16 = (size_t)count / 16;
    launch_k(k_i8_to_bf16, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const i8*)in, (u16*)out, n16);
    return launch_status();
}

extern "C" int tcq_decode_i8(const void* bits, const int8_t* t8, int8_t* out, int m, int n, tcq_stream_t stream) {
    return tcq_decode_i8_groups(bits, t8, 1, out, m, n, stream);
}

extern "C" int tcq_decode_f16_groups(const void* bits, const void* tlut, int G, void* out, int m, int n, tcq_stream_t stream) {
    if (!bits || !tlut || !out || m <= 0 || n <= 0 || G <= 0) return TCQ_ERR_ARG;
    if (m % 16 || n % 16 || !groups_ok(m, G)) return TCQ_ERR_SHAPE;
    if ((uintptr_t)out % 16) return TCQ_ERR_ALIGN;
    const size_t per = (size_t)(m / G) * (n / 16);
    launch_k(k_decode_f16, dim3((unsigned)((per + 255) / 256), G), dim3(256), 0, (hipStream_t)stream, (const u16*)bits,
             (const u16*)tlut, (u16*)out, m / G, n);
    return launch_status();
}

extern "C" int tcq_decode_f16(const void* bits, const void* tlut, void* out, int m, int n, tcq_stream_t stream) {
    return tcq_decode_f16_groups(bits, tlut, 1, out, m, n, stream);
}
