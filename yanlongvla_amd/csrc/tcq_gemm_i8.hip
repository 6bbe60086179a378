// GEMM for many tokens, acc[m, n] = sum_k x[m, k] w[n, k], x (M, K) and w (N, K) both row-major with K contiguous, so every
// MFMA operand is 16 consecutive bytes of one row:
//   INT8 (W8A8) on v_mfma_i32_16x16x64_i8: exact int32 acc, written as int32 (optionally in K parts), as FP32
//   (float(acc) * sa[m]) * sw[n], or as BF16 of that;
//   BF16 (the W2 float path: BF16 rotated activations times the INT8 table values as BF16) on v_mfma_f32_16x16x32_bf16 with
//   FP32 accumulation, written as FP32 (acc * sa[m]) * sw[n] (either scale may be absent) or as BF16 of that.
// 16 x 16 blocks although 32 x 32 ones issue at a higher peak: on random operands the part holds 2.23 GHz through
// 16x16x64 (3.95 POP/s) but drops to 1.78 GHz through 32x32x32 (3.53 POP/s), and the rest of the loop runs at that clock
// too (BF16: 1.92 against 1.85 PFLOP/s).
//
// Workgroup tile TN weights x TM tokens, WN x WM waves. MFMA A = 16 weight rows, B = 16 token rows, 64 bytes of K each; D:
// register e of lane (g, c) holds weight 4 g + e of token c, so a lane stores 4 consecutive columns (16 bytes of FP32 /
// int32) straight from its registers; for BF16 outputs the weight rows of two blocks are interleaved so that it is 8.
//
// K goes by in steps of 128 bytes, whole cache lines of both operands (64-byte steps fetch every line twice: 42.3 against
// 37.1 us at 800 x 2048 x 16384), HBM -> LDS by buffer_load_dwordx4 ... lds without registers, into two rings: NSX steps of
// activations, NSW of weights. Weights come from HBM and activations from the caches, so the 160 KiB of a 256 x 256 tile
// hold three steps of weights and two of activations. A load fills 8 rows x 128 bytes; lane p writes position p, which holds
// row p / 8 and 16-byte granule (p % 8) ^ turn(row). A fragment read takes 256 bytes of LDS a cycle, 16 lanes: two rows' width,
// so the 8 even rows of a fragment, and its 8 odd ones, need 8 turns: 16 rows in a row bits 1 .. 3, the interleaved rows of BF16
// outputs bits 1, 3 and 4, served together by bits 1, 3 and 2 ^ 4. Turns from the low three bits cost every read 4 extra
// cycles of 8: without them a BF16 layer of 968 tokens takes 424 us against 432, INT8 at 800 x 2048 x 16384 the same 32.5.
// A step runs in four quarters (k half x half of the wave's weight blocks); the fragment reads of the next quarter and the
// loads of later steps are scheduled between the MFMAs of this one. The one barrier of a step stands before its last
// quarter, whose fragments are in registers by then: it publishes the next step and frees this one, with MFMAs on both sides.
// Rows past M / N and columns past K read zeros; waves whose tokens are all padding only load.
// What bounds it (256 x 256, INT8, K long enough): 1.5 us per step, 2.8 POP/s; the MFMAs alone take 1.05 us, the loads and
// fragment reads alone 0.7 (in cache) to 1.2 us (streaming), and power: the matrix cores are busy 47 % of the cycles, at about
// 1.8 GHz. Not the LDS: its reads are 18 % of the cycles and halving them changed nothing. One wave per SIMD with 128 x 128
// each (a third fewer fragment reads) measured the same.
#include "tcq_device.h"
#include "tcq_launch.h"

namespace {

typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// s_waitcnt vmcnt(vm) lgkmcnt(lgkm), expcnt left alone (gfx9 encoding: vmcnt bits 3:0 and 15:14; lgkm 15 = no wait)
template <int vm, int lgkm>
__device__ __forceinline__ void wait_cnt() {
    static_assert(vm <= 63 && lgkm <= 15, "counter range");
    __builtin_amdgcn_s_waitcnt((vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8));
}

// Workgroup barrier without the memory fence of __syncthreads (which waits for every outstanding load, including the LDS
// loads of later steps): the LDS writes a barrier must publish are the loads waited for just before it (wait_cnt), and the
// empty asm statements keep the compiler from moving memory accesses across it.
__device__ __forceinline__ void barrier_nofence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int ESZ> struct MfmaOf;
template <> struct MfmaOf<1> {                 // INT8
    typedef int4v acc_t;
    static __device__ __forceinline__ acc_t mma(int4v a, int4v b, acc_t c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
};
template <> struct MfmaOf<2> {                 // BF16
    typedef float4v acc_t;
    static __device__ __forceinline__ acc_t mma(int4v a, int4v b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};

template <int n> struct Num { static constexpr int value = n; };
struct Full { static constexpr bool value = true; };
struct Tail { static constexpr bool value = false; };

}  // namespace

// ESZ: element size (1 INT8, 2 BF16); K in elements. parts: K parts (grid.z, int32 outputs): part z sums the steps
// [z ceil(nk / parts), ...) into out + z M ldo. flush: steps per first-level sum (BF16).
template <int ESZ, int TN, int TM, int WN, int WM, int NSW, int NSX, int ODT>
__global__ __launch_bounds__(64 * WN * WM) void k_gemm_i8(const void* x_, const void* w_, const float* sa, const float* sw, void* out,
                                                       int ldo, int M, int N, int K_, int parts, int flush) {
    typedef typename MfmaOf<ESZ>::acc_t acc_t;
    constexpr int NWAVE = WN * WM;
    constexpr int WL = TN / 8 / NWAVE, XL = TM / 8 / NWAVE;              // 1 KiB loads (8 rows x 128 bytes) per wave and step
    constexpr int NB = TN / WN / 16, MB = TM / WM / 16, HB = NB / 2;     // 16 x 16 blocks per wave; weight blocks per quarter
    static_assert(WL * 8 * NWAVE == TN && XL * 8 * NWAVE == TM && HB * 2 == NB && MB * 16 * WM == TM, "tile shape");
    const int K = K_ * ESZ;                                              // row length in bytes
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    char* ldsw = lds;
    char* ldsx = lds + NSW * TN * 128;
    const int n0 = blockIdx.x * TN, m0 = blockIdx.y * TM;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wn = wave % WN, wm = wave / WN;
    const int lr = lane & 15, lg = lane >> 4;
    const rsrc_t RX = make_rsrc(x_, (u32)M * (u32)K), RW = make_rsrc(w_, (u32)N * (u32)K);
    const int nkall = (K + 127) >> 7, per = (nkall + parts - 1) / parts, kb = blockIdx.z * per;
    const int nk = min(per, nkall - kb), kend = min(K, 128 * (kb + nk));

    // granule g of a row lies at position g ^ turn (of its row in the tile)
    auto turn_x = [](int r) { return (r >> 1) & 7; };
    auto turn_w = [](int r) { return ((r >> 1) & 1) | ((r >> 2) & 2) | (((r ^ (r >> 2)) & 4)); };
    // load u of a wave fills block (wave * L + u) of 8 rows: lane p writes position p, which holds row p / 8, slot p % 8
    const int prow = lane >> 3;
    u32 offw[WL], offx[XL];
#pragma unroll
    for (int u = 0; u < WL; ++u) {
        const int blk = wave * WL + u, row = n0 + 8 * blk + prow, g = (lane & 7) ^ turn_w(8 * blk + prow);
        offw[u] = row < N ? (u32)row * (u32)K + 16u * g : RSRC_OOB;
    }
#pragma unroll
    for (int u = 0; u < XL; ++u) {
        const int blk = wave * XL + u, row = m0 + 8 * blk + prow, g = (lane & 7) ^ turn_x(8 * blk + prow);
        offx[u] = row < M ? (u32)row * (u32)K + 16u * g : RSRC_OOB;
    }
    // loads of K step kt: the row offsets stay in registers, the step is the scalar offset; only the last, partial step of K (and
    // the loads past the end, which read zeros) select per lane
    const int nfull = (kend - 128 * kb) >> 7;
    auto issue_w = [&](int kt, auto full) {
        char* st = ldsw + (kt % NSW) * (TN * 128) + wave * WL * 1024;
        const int k = 128 * (kb + kt);
        if constexpr (decltype(full)::value) {
#pragma unroll
            for (int u = 0; u < WL; ++u) {
                char* dst = st + u * 1024;
                const u32 off = offw[u];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(RW, (__attribute__((address_space(3))) void*)dst, 16, off, k, 0, 0);
            }
        } else {
#pragma unroll
            for (int u = 0; u < WL; ++u) {
                char* dst = st + u * 1024;
                const int g = (lane & 7) ^ turn_w(8 * (wave * WL + u) + prow);
                const u32 off = (k + 16 * g < kend) ? offw[u] + (u32)k : RSRC_OOB;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(RW, (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
            }
        }
    };
    auto issue_x = [&](int kt, auto full) {
        char* st = ldsx + (kt % NSX) * (TM * 128) + wave * XL * 1024;
        const int k = 128 * (kb + kt);
        if constexpr (decltype(full)::value) {
#pragma unroll
            for (int u = 0; u < XL; ++u) {
                char* dst = st + u * 1024;
                const u32 off = offx[u];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(RX, (__attribute__((address_space(3))) void*)dst, 16, off, k, 0, 0);
            }
        } else {
#pragma unroll
            for (int u = 0; u < XL; ++u) {
                char* dst = st + u * 1024;
                const int g = (lane & 7) ^ turn_x(8 * (wave * XL + u) + prow);
                const u32 off = (k + 16 * g < kend) ? offx[u] + (u32)k : RSRC_OOB;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(RX, (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
            }
        }
    };
    constexpr int FLY0 = WL * (NSW - 2) + XL * (NSX - 1), FLY = WL * (NSW - 2) + XL * (NSX - 2);
    // stages 0 .. NSX - 1 of the activations and 0 .. NSW - 2 of the weights, in the order of the loop's own loads: the waits
    // count the loads issued after the stage they wait for
    constexpr int NS = NSX > NSW ? NSX : NSW;
#pragma unroll
    for (int t = 1 - NS; t <= 0; ++t) {
        if (t - 1 + NSX >= 0) issue_x(t - 1 + NSX, Tail{});
        if (t - 1 + NSW >= 0 && t < 0) issue_w(t - 1 + NSW, Tail{});
    }

    if (m0 + wm * (TM / WM) >= M) {                 // this wave's tokens are padding: only its share of the loads
        wait_cnt<FLY0, 15>();
        barrier_nofence();
        for (int kt = 0; kt < nk; ++kt) {
            issue_w(kt + NSW - 1, Tail{});
            wait_cnt<FLY, 15>();
            barrier_nofence();
            issue_x(kt + NSX, Tail{});
        }
        wait_cnt<0, 15>();                          // no load into the LDS outlives the workgroup
        return;
    }

    // weight row of A row r of block i: BF16 outputs pair the blocks so that a lane ends with 8 consecutive columns
    constexpr bool PAIR = ODT == TCQ_BF16;
    auto wrow = [&](int i) { return PAIR ? 32 * (i >> 1) + 8 * (lr >> 2) + 4 * (i & 1) + (lr & 3) : 16 * i + lr; };
    // rows 32 apart share their slot pattern: two (PAIR) or one base offsets per k half, the rest constants
    int fw[2][2], fx[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        fw[h][0] = wrow(0) * 128 + 16 * ((4 * h + lg) ^ turn_w(wrow(0)));
        fw[h][1] = wrow(1) * 128 + 16 * ((4 * h + lg) ^ turn_w(wrow(1)));
        fx[h] = lr * 128 + 16 * ((4 * h + lg) ^ turn_x(lr));
    }
    acc_t acc[NB][MB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = 0;
    int4v A[2][HB], B[2][MB];
    auto read_a = [&](int kt, int h, int half, int s) {                  // weight blocks half * HB .. of k half h
        const char* p = ldsw + (kt % NSW) * (TN * 128) + wn * NB * 2048;
#pragma unroll
        for (int i = 0; i < HB; ++i) {
            const int b = half * HB + i;
            A[s][i] = *(const int4v*)(p + (b >> 1) * 4096 + fw[h][b & 1]);
        }
    };
    auto read_b = [&](int kt, int h, int s) {
        const char* p = ldsx + (kt % NSX) * (TM * 128) + wm * MB * 2048 + fx[h];
#pragma unroll
        for (int j = 0; j < MB; ++j) B[s][j] = *(const int4v*)(p + j * 2048);
    };
    auto mm = [&](int half, int s, int sb) {
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j) acc[half * HB + i][j] = MfmaOf<ESZ>::mma(A[s][i], B[sb][j], acc[half * HB + i][j]);
    };
    // the fragment reads and the loads of a quarter step between its MFMAs
    auto spread = [&](auto reads, auto loads) {
        constexpr int R = decltype(reads)::value, L = decltype(loads)::value, NM = HB * MB, G = NM / (R + L) > 0 ? NM / (R + L) : 1;
#pragma unroll
        for (int q = 0; q < R + L; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, G, 0);
            if (q < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    wait_cnt<FLY0, 15>();
    barrier_nofence();
    read_b(0, 0, 0);
    read_a(0, 0, 0, 0);
    auto step = [&](int kt, auto full) {
        issue_w(kt + NSW - 1, full);
        read_a(kt, 0, 1, 1);
        mm(0, 0, 0);
        spread(Num<HB>{}, Num<WL>{});
        read_b(kt, 1, 1);
        read_a(kt, 1, 0, 0);
        mm(1, 1, 0);
        spread(Num<HB + MB>{}, Num<0>{});
        read_a(kt, 1, 1, 1);
        mm(0, 0, 1);
        spread(Num<HB>{}, Num<0>{});
        wait_cnt<FLY, 0>();
        barrier_nofence();
        issue_x(kt + NSX, full);
        read_b(kt + 1, 0, 0);
        read_a(kt + 1, 0, 0, 0);
        mm(1, 1, 1);
        spread(Num<HB + MB>{}, Num<XL>{});
    };
    if constexpr (ESZ == 1) {
        int kt = 0;
        for (; kt + NS < nfull; ++kt) step(kt, Full{});
        for (; kt < nk; ++kt) step(kt, Tail{});
    } else {
        // FP32 sums in two levels, `flush` steps (two MFMAs each) in a row, then the sums of those, each with what its addition
        // rounded away (exact - sum, by two subtractions: exact while the running sum is the larger of the two, close to it
        // otherwise) carried into the next chain; what the last one rounded away is less than half an ulp. Most of the second level's
        // error goes, and that of a chain grows with its length only. Relative error against 64 bits, K = 1024 / 2048 / 4096 / 16384:
        // 4.9e-8, 5.6e-8, 6.4e-8, 8.9e-8; without the carry 6.3e-8, 7.3e-8, 8.7e-8, 1.24e-7; the few-token product's partial sums
        // (three levels) 5.7e-8, 6.9e-8, 7.8e-8, 1.18e-7.
        acc_t sum[NB][MB];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j) sum[i][j] = acc[i][j];
        for (int kt = 0; kt < nk;) {
            const int end = min(nk, kt + flush);
            for (; kt < end && kt + NS < nfull; ++kt) step(kt, Full{});
            for (; kt < end; ++kt) step(kt, Tail{});
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < MB; ++j) {
                    const acc_t t = sum[i][j] + acc[i][j];
                    acc[i][j] = acc[i][j] - (t - sum[i][j]);
                    sum[i][j] = t;
                }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j) acc[i][j] = sum[i][j];
    }
    // BF16: an infinite sum's carry is inf - inf, so a NaN here may stand for an infinity. Such outputs are summed again in one
    // plain chain at the end (a test of every carry, so that none becomes a NaN, cost 2 to 7 %: 968 x 32768 x 2048 147.2 us, 152.7 with it
    // and 148.9 so, 800 x 8192 x 1024 23.5, 25.1, 23.6, 65 x 1152 x 1152 9.6, 9.9, 9.6)
    u64 nans = 0;                                   // bit 4 (i MB + j) + e
    if constexpr (ESZ == 2) {
        static_assert(4 * NB * MB <= 64, "a bit per value");
        bool any = false;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j)
                any |= __builtin_isunordered(acc[i][j][0], acc[i][j][1]) | __builtin_isunordered(acc[i][j][2], acc[i][j][3]);
        if (__builtin_amdgcn_ballot_w64(any))
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < MB; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) nans |= (u64)__builtin_isnan(acc[i][j][e]) << (4 * (i * MB + j) + e);
    }
    wait_cnt<0, 0>();                               // no load into the LDS outlives the workgroup
    // D: register e of lane (g, c) = weight row 4 g + e of the A block, token c of the B block
    const int z = blockIdx.z;
#pragma unroll
    for (int j = 0; j < MB; ++j) {
        const int m = m0 + (wm * MB + j) * 16 + lr;
        if (m >= M) continue;
        const float s = (ODT != TCQ_I32 && sa) ? gptr(sa)[m] : 1.f;
        if constexpr (PAIR) {
#pragma unroll
            for (int i = 0; i < NB; i += 2) {
                const int n = n0 + wn * NB * 16 + 16 * i + 8 * lg;
                if (n >= N) continue;
                float v[8];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    float4v r = {1.f, 1.f, 1.f, 1.f};
                    if (sw && n + 4 * b < N) r = gptr((const float4v*)(sw + n))[b];      // N is a multiple of 4
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float a = (float)acc[i + b][j][e];
                        if (sa) a = a * s;
                        v[4 * b + e] = sw ? a * r[e] : a;
                    }
                }
                const uint4_t o = {bf16x2(v[0], v[1]), bf16x2(v[2], v[3]), bf16x2(v[4], v[5]), bf16x2(v[6], v[7])};
                u16* p = (u16*)out + (size_t)m * ldo + n;
                if (n + 8 <= N && ldo % 8 == 0) *gptr((uint4_t*)p) = o;
                else {                                                    // N, ldo multiples of 4: 8-byte pieces
                    *gptr((uint2_t*)p) = uint2_t{o[0], o[1]};
                    if (n + 8 <= N) *gptr((uint2_t*)(p + 4)) = uint2_t{o[2], o[3]};
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int n = n0 + wn * NB * 16 + 16 * i + 4 * lg;
                if (n >= N) continue;
                if constexpr (ODT == TCQ_I32) {
                    *gptr((acc_t*)((int*)out + ((size_t)z * M + m) * ldo + n)) = acc[i][j];
                } else {
                    float4v v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = (float)acc[i][j][e];
                        if (sa) v[e] = v[e] * s;
                    }
                    if (sw) {
                        const float4v r = gptr((const float4v*)(sw + n))[0];
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = v[e] * r[e];
                    }
                    *gptr((float4v*)((float*)out + ((size_t)z * M + m) * ldo + n)) = v;
                }
            }
        }
    }
    if constexpr (ESZ == 2) {
        while (nans) {
            const int b = __builtin_ctzll(nans), e = b & 3, j = (b >> 2) % MB, i = (b >> 2) / MB;
            nans &= nans - 1;
            const int m = m0 + (wm * MB + j) * 16 + lr, n = n0 + wn * NB * 16 + (PAIR ? 32 * (i >> 1) + 8 * lg + 4 * (i & 1) : 16 * i + 4 * lg) + e;
            if (m >= M || n >= N) continue;
            const u16 *xr = (const u16*)x_ + (size_t)m * K_, *wr = (const u16*)w_ + (size_t)n * K_;
            float v = 0.f;
            for (int k = 64 * kb; k < kend / 2 && !__builtin_isnan(v); k += 8) {
                const uint4_t a = *gptr((const uint4_t*)(xr + k)), c = *gptr((const uint4_t*)(wr + k));
#pragma unroll
                for (int h = 0; h < 8; ++h)
                    v = __builtin_fmaf(bf16_to_f32((u16)(a[h >> 1] >> (16 * (h & 1)))), bf16_to_f32((u16)(c[h >> 1] >> (16 * (h & 1)))), v);
            }
            if (sa) v = v * gptr(sa)[m];
            if (sw) v = v * gptr(sw)[n];
            const size_t o = ((size_t)z * M + m) * ldo + n;
            if (PAIR) gptr((u16*)out)[o] = f32_to_bf16(v);
            else gptr((float*)out)[o] = v;
        }
    }
}

// =========================================================================================================== C ABI
template <int ESZ, int TN, int TM, int WN, int WM, int NSW, int NSX>
static void launch_gemm(int odt, hipStream_t st, const void* x, const void* w, const float* sa, const float* sw, void* out, int ldo,
                        int M, int N, int K, int parts) {
    const dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM, parts), block(64 * WN * WM);
    const size_t lds = (size_t)(NSW * TN + NSX * TM) * 128;
    int flush = 1;                                      // sqrt(steps / 2): chains of 2 flush and steps / flush are equally long
    while (2 * flush * flush < (K * ESZ + 127) / 128) ++flush;
    if (ESZ == 1 && odt == TCQ_I32) launch_k(k_gemm_i8<ESZ, TN, TM, WN, WM, NSW, NSX, ESZ == 1 ? TCQ_I32 : TCQ_F32>, grid, block, lds, st, x, w, sa, sw, out, ldo, M, N, K, parts, flush);
    else if (odt == TCQ_F32) launch_k(k_gemm_i8<ESZ, TN, TM, WN, WM, NSW, NSX, TCQ_F32>, grid, block, lds, st, x, w, sa, sw, out, ldo, M, N, K, parts, flush);
    else launch_k(k_gemm_i8<ESZ, TN, TM, WN, WM, NSW, NSX, TCQ_BF16>, grid, block, lds, st, x, w, sa, sw, out, ldo, M, N, K, parts, flush);
}

// The tile with the least estimated time. Workgroups run in rounds of 256 (one per CU; the tiles up to 128 x 128 fit two on a CU, so
// several rounds overlap): a single round takes ramp + one x its 128-byte steps, each of several ramp + more x steps, in ns. The
// constants are fitted to which tile was the fastest, and to the times, in 1304 INT8 and 1574 BF16 runs of every tile on MI355X (M = 65 ..
// 2400, N = 256 .. 32768, K = 1024 .. 16384; int32 and FP32 out; BF16 in 1, 2 and 4 K parts). Over 954 and 1215 runs of other random
// sizes the chosen tile was 0.6 % (INT8) and 0.9 % (BF16) above the best on average and more than 8 % above it in 23 and 51; one cost
// per step whatever the K, from INT8 runs alone, was 2.6 % and 2.0 % above, more than 8 % in 65 and 88. us, that rule's tile / this one:
// INT8 to FP32 400 x 2560 x 2048 11.1 / 9.4, 900 x 4608 x 1536 21.2 / 15.8, 700 x 12288 x 2048 37.2 / 32.0; BF16 600 x 16384 x 2048 60.0 / 52.3,
// 1300 x 32768 x 2048 248 / 210. Most of what is left is a partly filled last round: BF16 800 x 32768 x 2048 takes 128 x 128 at 147 where
// 256 x 128 in three rounds and a half needs 133. A short K pays the longer ramp of 128-byte steps: with int32 out 700 .. 968 tokens x 2560 or
// 3072 x 1024 take 9.2 us, 8.1 .. 8.8 with 64-byte steps and 32 x 32 blocks; from K = 1536 on that form is slower nearly everywhere, by up
// to a third. BF16 of 16384 columns and more pays its second level: one chain on 256 x 256 tiles took 968 x 32768 x 2048 in 136 us
// where this takes 150, at 1.54e-7 from 64 bits instead of 5.6e-8.
struct Tile { int tn, tm; double one, more, ramp; };
constexpr Tile TILES_I8[] = {{64, 64, 389, 247, 1386}, {128, 64, 455, 409, 3420}, {128, 128, 623, 447, 2469}, {256, 128, 820, 722, 6128},
                             {256, 256, 1113, 717, 12191}};
constexpr Tile TILES_BF16[] = {{64, 64, 359, 223, 3642}, {128, 64, 402, 369, 5058}, {128, 128, 538, 489, 4597}, {256, 128, 591, 666, 15412}};
template <int ESZ>
static int choose_tile(int M, int N, int K, int parts, double* ns = nullptr) {
    const Tile* T = ESZ == 1 ? TILES_I8 : TILES_BF16;           // BF16 keeps two levels of sums: no registers for 256 x 256
    const int nk = (int)(((long)K * ESZ + 127) / 128), steps = (nk + parts - 1) / parts;
    int best = 0;
    double bt = 0;
    for (int i = 0; i < (ESZ == 1 ? 5 : 4); ++i) {
        const long w = (long)((N + T[i].tn - 1) / T[i].tn) * ((M + T[i].tm - 1) / T[i].tm) * parts, r = (w + 255) / 256;
        const double t = r == 1 ? T[i].ramp + T[i].one * steps : r * (T[i].ramp + T[i].more * steps);
        if (i == 0 || t < bt) { best = i; bt = t; }
    }
    if (ns) *ns = bt;
    return best;
}

template <int ESZ>
static void launch_by_size(int odt, hipStream_t st, const void* x, const void* w, const float* sa, const float* sw, void* out, int ldo,
                           int M, int N, int K, int parts) {
    switch (choose_tile<ESZ>(M, N, K, parts)) {
        case 0: launch_gemm<ESZ, 64, 64, 2, 2, 4, 4>(odt, st, x, w, sa, sw, out, ldo, M, N, K, parts); break;
        case 1: launch_gemm<ESZ, 128, 64, 4, 2, 3, 3>(odt, st, x, w, sa, sw, out, ldo, M, N, K, parts); break;
        case 2: launch_gemm<ESZ, 128, 128, 2, 4, 3, 2>(odt, st, x, w, sa, sw, out, ldo, M, N, K, parts); break;
        case 3: launch_gemm<ESZ, 256, 128, 4, 2, 3, 3>(odt, st, x, w, sa, sw, out, ldo, M, N, K, parts); break;
        default:
            if constexpr (ESZ == 1) launch_gemm<ESZ, 256, 256, 2, 4, 3, 2>(odt, st, x, w, sa, sw, out, ldo, M, N, K, parts);
    }
}

extern "C" int tcq_gemm_i8(const int8_t* a, const int8_t* w, const float* sa, const float* sw, void* out, int out_dtype, int ldo,
                           int M, int N, int K, tcq_stream_t stream) {
    if (!a || !w || !out || M <= 0 || N <= 0 || K <= 0 || ldo < N) return TCQ_ERR_ARG;
    if (out_dtype != TCQ_I32 && (!sa || !sw)) return TCQ_ERR_ARG;
    if (K % 16 || N % 4) return TCQ_ERR_SHAPE;
    if ((size_t)M * K >= ((size_t)1 << 31) || (size_t)N * K >= ((size_t)1 << 31)) return TCQ_ERR_SHAPE;
    if ((uintptr_t)a % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 16 || (sw && (uintptr_t)sw % 16) || ldo % 4)
        return TCQ_ERR_ALIGN;
    if (M <= 16 || (M <= 64 && N <= 8192)) {            // few tokens: the small-M product (one K chunk per wave)
        const tcq_gemm_seg seg = {w, nullptr, sw, out, N};
        if (N % 16 == 0) return tcq_gemm_w8(&seg, 1, a, sa, M, K, out_dtype, ldo, stream);
    }
    if (out_dtype != TCQ_I32 && out_dtype != TCQ_F32 && out_dtype != TCQ_BF16) return TCQ_ERR_DTYPE;
    launch_by_size<1>(out_dtype, (hipStream_t)stream, a, w, sa, sw, out, ldo, M, N, K, 1);
    return launch_status();
}

extern "C" int tcq_gemm_i8_parts(const int8_t* a, const int8_t* w, int32_t* out, int ldo, int M, int N, int K, int parts,
                                 tcq_stream_t stream) {
    if (!a || !w || !out || M <= 0 || N <= 0 || K <= 0 || ldo < N || (parts != 1 && parts != 2 && parts != 4)) return TCQ_ERR_ARG;
    if (K % 16 || N % 4 || (parts > 1 && K < 128 * 16)) return TCQ_ERR_SHAPE;            // every part has steps of its own
    if ((size_t)M * K >= ((size_t)1 << 31) || (size_t)N * K >= ((size_t)1 << 31)) return TCQ_ERR_SHAPE;
    if ((uintptr_t)a % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 16 || ldo % 4) return TCQ_ERR_ALIGN;
    launch_by_size<1>(TCQ_I32, (hipStream_t)stream, a, w, nullptr, nullptr, out, ldo, M, N, K, parts);
    return launch_status();
}

// The K parts with the least estimated time: choose_tile's, and for each part past the first its write and the epilogue's read
// at 3 TB/s. A long K over few tiles leaves the large tiles too few workgroups and the small ones bound by their loads into
// LDS; parts give the larger tiles the whole chip. MI355X, us with the epilogue in 1 / 2 / 4 parts: 968 x 2048 x 16384 65.4 / 53.1 /
// 53.0 (2 taken), 200: 37.3 / 25.9 / 23.3 (4); 400 x 1024 x 4096 16.4 / 13.7 / 14.7 (2), 968: 19.6 / 19.4 / 21.3 (2); 968 x 2048 x 2048 23.4 /
// 25.8 / 27.8 (1). Over 160 sizes (N = 1024 .. 8192, M = 65 .. 2000) the parts taken are 0.2 % above the best on average, 5 % at most.
extern "C" int tcq_gemm_i8_best_parts(int M, int N, int K) {
    if (M <= 64 || N <= 0 || K < 128 * 16) return 1;
    int best = 1;
    double bt = 0;
    for (int parts = 1; parts <= 4; parts *= 2) {
        double t = 0;
        choose_tile<1>(M, N, K, parts, &t);
        t += (parts - 1) * (8.0 * M * N) / 3e3;
        if (parts == 1 || (t < bt && (size_t)parts * M * N < ((size_t)1 << 31))) { best = parts; bt = t; }
    }
    return best;
}

extern "C" int tcq_gemm_bf16(const void* a, const void* w, const float* sa, const float* sw, void* out, int out_dtype, int ldo, int M,
                             int N, int K, tcq_stream_t stream) {
    if (!a || !w || !out || M <= 0 || N <= 0 || K <= 0 || ldo < N) return TCQ_ERR_ARG;
    if (out_dtype != TCQ_F32 && out_dtype != TCQ_BF16) return TCQ_ERR_DTYPE;
    if (K % 16 || N % 4) return TCQ_ERR_SHAPE;
    if ((size_t)M * K * 2 >= ((size_t)1 << 31) || (size_t)N * K * 2 >= ((size_t)1 << 31)) return TCQ_ERR_SHAPE;
    if ((uintptr_t)a % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 16 || (sw && (uintptr_t)sw % 16) || ldo % 4) return TCQ_ERR_ALIGN;
    launch_by_size<2>(out_dtype, (hipStream_t)stream, a, w, sa, sw, out, ldo, M, N, K, 1);
    return launch_status();
}

// FP32 K parts added in order, * sw, to FP32 or BF16: four columns per thread. What the additions round away is added at the end,
// unless the sum is infinite (the launch is bound by memory): each part is rounded once more than a single sum, and with plain
// additions four parts of K = 1024 were 3 % further from 64 bits than the few-token product's sums.
template <int ODT>
__global__ __launch_bounds__(256) void k_sum_parts(const float* part, const float* sw, void* out, size_t n, int N, int parts) {
    const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= n) return;
    float4v v = *gptr((const float4v*)(part + i)), c = {0.f, 0.f, 0.f, 0.f};
    for (int p = 1; p < parts; ++p) {
        const float4v u = *gptr((const float4v*)(part + p * n + i));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float t = v[e] + u[e], b = t - v[e];
            c[e] = c[e] + ((v[e] - (t - b)) + (u[e] - b));
            v[e] = t;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fabsf(v[e]) < __builtin_inff() ? v[e] + c[e] : v[e];
    if (sw) {
        const float4v r = *gptr((const float4v*)(sw + i % N));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * r[e];
    }
    if (ODT == TCQ_F32) *gptr((float4v*)((float*)out + i)) = v;
    else *gptr((uint2_t*)((u16*)out + i)) = uint2_t{bf16x2(v[0], v[1]), bf16x2(v[2], v[3])};
}

extern "C" int tcq_gemm_bf16_parts(const void* a, const void* w, const float* sw, float* part, void* out, int out_dtype, int M, int N,
                                   int K, int parts, tcq_stream_t stream) {
    if (!a || !w || !part || !out || M <= 0 || N <= 0 || K <= 0 || (parts != 2 && parts != 4)) return TCQ_ERR_ARG;
    if (out_dtype != TCQ_F32 && out_dtype != TCQ_BF16) return TCQ_ERR_DTYPE;
    if (K % 16 || N % 4 || K < 64 * 16) return TCQ_ERR_SHAPE;                            // every part has steps of its own
    if ((size_t)M * K * 2 >= ((size_t)1 << 31) || (size_t)N * K * 2 >= ((size_t)1 << 31) || (size_t)parts * M * N >= ((size_t)1 << 31))
        return TCQ_ERR_SHAPE;
    if ((uintptr_t)a % 16 || (uintptr_t)w % 16 || (uintptr_t)part % 16 || (uintptr_t)out % 16 || (sw && (uintptr_t)sw % 16)) return TCQ_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    launch_by_size<2>(TCQ_F32, st, a, w, nullptr, nullptr, part, N, M, N, K, parts);
    const int e = launch_status();
    if (e) return e;
    const size_t n = (size_t)M * N;
    const dim3 grid((unsigned)((n / 4 + 255) / 256));
    if (out_dtype == TCQ_F32) launch_k(k_sum_parts<TCQ_F32>, grid, dim3(256), 0, st, (const float*)part, sw, out, n, N, parts);
    else launch_k(k_sum_parts<TCQ_BF16>, grid, dim3(256), 0, st, (const float*)part, sw, out, n, N, parts);
    return launch_status();
}

// As tcq_gemm_i8_best_parts, with 2 us for the launch that adds the parts, and their write and read at 4 TB/s (1.0 % above the best
// parts and tile on average over 471 sizes). MI355X, us in 1 / 2 / 4 parts: 968 x 2048 x 16384 105 / 81 / 76, 256: 77 / 45 / 33; 128 x 1024 x 4096 23 / 16 / 12; 400 x 2048 x 2048 14.3 / 15.0 / 17.5.
// Relative error against 64 bits, 968 x 2048 x 16384: 8.9e-8, 9.3e-8, 9.2e-8 (the few-token product's partial sums: 1.18e-7); 65 x 1024 x
// 1024: 4.9e-8, 5.5e-8, 5.0e-8 (5.7e-8).
extern "C" int tcq_gemm_bf16_best_parts(int M, int N, int K) {
    if (M <= 64 || N <= 0 || K < 64 * 16) return 1;
    int best = 1;
    double bt = 0;
    for (int parts = 1; parts <= 4; parts *= 2) {
        double t = 0;
        choose_tile<2>(M, N, K, parts, &t);
        t += parts > 1 ? 2e3 + parts * 8.0 * M * N / 4e3 : 0;
        if (parts == 1 || (t < bt && (size_t)parts * M * N < ((size_t)1 << 31))) { best = parts; bt = t; }
    }
    return best;
}
