// Prefill projections (gfx950): activations quantized to Q8_0, then
// y = W x for m tokens at once with Q1_0 weights. Same results as
// src/shaders/quantize_q8_0.wgsl and src/shaders/matmul_q1_0_q8_0.wgsl
// (reference repository), bit for bit:
//
//  * quantize: per 32 elements of a row, d = amax / 127 (f32), q =
//    clamp(rne(v * (1 / d)), -127, 127) (0 when d = 0); d (f32) at d_offset +
//    4 (row * k/32 + block), qs at qs_offset + row * k + 32 block (bytes).
//  * matmul: for each (token, weight row), over 128-blocks b and then their
//    four 32-blocks s, acc = acc + (a_d * w_d) * f32(sumi) in f32, with sumi
//    the exact integer sum of +-q over the 32 elements (bit e of the row's
//    block selects +q[e]); then f16(acc), or f16(f32(y) + acc) to accumulate.
//
// Matmul on the i8 matrix cores, one v_mfma_i32_16x16x32_i8 per 16 x 16 tile of
// tokens and weight rows and 32-block. What bounds it is issue: per (output,
// 32-block) the order of the sums leaves one conversion (or subtraction, see below),
// one or two products and one addition in f32, and a wave alone on its SIMD issues one
// instruction per six cycles (two waves: three cycles; four: 2.4), while the MFMAs
// add their own time. The kernels differ in how much of the machine a shape fills:
//  * matmul_split_kernel, few tiles: the 128-blocks of one tile spread over 8
//    waves, the terms handed over in LDS and added in order;
//  * matmul_kernel<16 or 32 tokens>: a wave runs whole sums of 16 rows, weight rows as
//    A and tokens as B, so that a lane holds four consecutive rows of one token, the
//    scale a_d * w_d from the matrix core and sumi without a conversion, two or four
//    128-blocks staged ahead;
//  * matmul_block_kernel<32 or 64 tokens>: tokens as A, one 128-block staged ahead: the
//    least start-up, and with 64 tokens the most work per weight, on large grids.
// Measured (us per call, 8 weights in turn; one 64- or 32-token block kernel alone in
// parentheses): n x k at 16 / 33 / 128 / 512 tokens
//   1024 x 2560:  4.9 /  5.0 /  6.4 / 10.5   (24.1 / 14.1 / 14.2 / 14.3)
//   4096 x 2560:  5.0 /  8.8 / 10.5 / 24.8   (24.3 / 14.2 / 14.3 / 24.8)
//   2560 x 4096:  5.8 /  8.0 / 15.1 / 29.0   (37.0 / 24.1 / 24.2 / 29.7)
//   2560 x 9728: 10.7 / 15.6 / 31.7 / 63.1   (83.9 / 48.7 / 49.4 / 67.1)
//   9728 x 2560:  8.9 / 10.7 / 20.2 / 51.6   (24.5 / 15.7 / 20.0 / 51.7)
#include "bp_device.hpp"
#include "bp_kernels.hpp"

namespace bp {
namespace {

typedef int i4v __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- quantize
// Four lanes per 32-element block: 16 bytes in, the block max by two lane
// exchanges, 8 quantized bytes out (one thread per block read and wrote with a
// 64-byte stride and left the chip emptier). Per element the operations are the
// reference's (|x| max, one IEEE divide for d, one for 1/d, rne(x * inv),
// clamp), so the bytes are identical.
__global__ __launch_bounds__(256) void quantize_act_q8_0_kernel(QuantArgs a) {
    const uint32_t nb = a.k / 32;
    const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
    const uint32_t blk = gid >> 2, part = gid & 3;   // blk = row * nb + b
    if (blk >= a.m * nb) return;
    const uint64_t at = 32 * static_cast<uint64_t>(blk) + 8 * part;   // row * k + 32 b + 8 part
    const uint16_t* src = a.act + a.input_offset + at;
    uint32_t w[4];
    if ((reinterpret_cast<uintptr_t>(src) & 15u) == 0) {
        const uint4 q = *reinterpret_cast<const uint4*>(src);
        w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
    } else {   // input_offset not a multiple of 8 elements: element loads
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = static_cast<uint32_t>(src[2 * i]) | (static_cast<uint32_t>(src[2 * i + 1]) << 16);
    }
    float v[8];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[2 * i] = h2f(static_cast<uint16_t>(w[i] & 0xFFFFu));
        v[2 * i + 1] = h2f(static_cast<uint16_t>(w[i] >> 16));
        amax = fmaxf(amax, fmaxf(fabsf(v[2 * i]), fabsf(v[2 * i + 1])));
    }
    amax = fmaxf(amax, lane_xor<1>(amax));
    amax = fmaxf(amax, lane_xor<2>(amax));
    const float d = amax / 127.0f;
    const float inv = d > 0.0f ? 1.0f / d : 0.0f;
    uint32_t out[2] = {0, 0};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float r = fminf(fmaxf(rintf(v[e] * inv), -127.0f), 127.0f);
        out[e / 4] |= (static_cast<uint32_t>(static_cast<int32_t>(r)) & 0xFFu) << (8 * (e % 4));
    }
    uint32_t* qs = reinterpret_cast<uint32_t*>(a.out + a.qs_offset + at);
    if ((reinterpret_cast<uintptr_t>(qs) & 7u) == 0) {
        *reinterpret_cast<uint2*>(qs) = make_uint2(out[0], out[1]);
    } else {   // qs_offset a multiple of 4 only
        qs[0] = out[0];
        qs[1] = out[1];
    }
    if (part == 0) *reinterpret_cast<float*>(a.out + a.d_offset + 4 * static_cast<uint64_t>(blk)) = d;
}

// ---------------------------------------------------------------- matmul
typedef float f16v __attribute__((ext_vector_type(16)));

// sumi without a conversion: the products are summed onto the bits of 1/(2 pi)
// = 0.15915494. |sumi| <= 4096 stays within that binade, where one unit in the
// last place is 2^-26, so the result read as f32 is exactly 1/(2 pi) + sumi
// 2^-26 and one exact subtraction, from that inline constant, leaves -sumi
// 2^-26. The staged w_d carries the -2^26, which changes no rounding.
constexpr int kMagicBits = 0x3E22F983;
constexpr float kMagic = 0.15915494f, kScaleUp = -67108864.0f;

// Sign byte -> 8 bytes of +-1 (bit j set: +1).
__device__ __forceinline__ void fill_sign_table(uint2* lut, uint32_t t, uint32_t n_thr) {
    for (uint32_t v = t; v < 256; v += n_thr) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo |= (((v >> j) & 1) ? 0x01u : 0xFFu) << (8 * j);
            hi |= (((v >> (j + 4)) & 1) ? 0x01u : 0xFFu) << (8 * j);
        }
        lut[v] = make_uint2(lo, hi);
    }
}

// y[out + tok * n + row + r] for four rows; vec: 8-byte aligned and n a multiple of 4.
__device__ __forceinline__ void store4(uint16_t* y, uint32_t row, uint32_t n, bool vec, uint32_t accumulate, const float* v) {
    if (vec) {
        if (row >= n) return;
        ushort4 o;
        if (accumulate) {
            o = *reinterpret_cast<const ushort4*>(y);
            o = {f2h(h2f(o.x) + v[0]), f2h(h2f(o.y) + v[1]), f2h(h2f(o.z) + v[2]), f2h(h2f(o.w) + v[3])};
        } else {
            o = {f2h(v[0]), f2h(v[1]), f2h(v[2]), f2h(v[3])};
        }
        *reinterpret_cast<ushort4*>(y) = o;
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (row + r < n) y[r] = f2h(accumulate ? h2f(y[r]) + v[r] : v[r]);
    }
}

constexpr int kMmRows = 64, kMmThreads = 256;

template <int kTok, int kStep> struct MmStage {   // kStep 128-blocks of the token tile
    uint8_t qs[kTok][128 * kStep + 16];           // + 16: the rows one read touches start in different banks
    float d[kTok][4 * kStep + 4];
};
struct WaveWeights {   // a wave's 16 weight rows, four 128-blocks
    uint4 q[4][16];
    float d[4][16];    // scales * kScaleUp
};

// 64 weight rows (16 a wave) x kTok tokens per workgroup. The tokens' qs and d
// of kStep 128-blocks are staged in LDS, double-buffered, one barrier per
// stage: with one block a stage the loop waited out the load latency (0.7 us a
// block at one or two waves per SIMD; 0.32 with four).
template <int kTok, int kStep>
__global__ __launch_bounds__(kMmThreads) void matmul_kernel(MatmulArgs a) {
    constexpr int kTiles = kTok / 16;                    // MFMA token tiles per wave
    constexpr int kThr = 8 * kStep;                      // staging threads per token
    constexpr int kRows = kMmThreads / kThr;             // tokens per staging round
    constexpr int kPer = (kTok + kRows - 1) / kRows;     // rounds
    __shared__ __attribute__((aligned(16))) MmStage<kTok, kStep> st[2];
    __shared__ __attribute__((aligned(16))) WaveWeights wsh[kMmThreads / 64];
    __shared__ uint2 lut[256];
    const uint32_t t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t nb1 = a.k / 128, nb8 = a.k / 32;
    const uint32_t n0 = blockIdx.x * kMmRows + 16 * wave, m0 = blockIdx.y * kTok;
    const uint32_t g = lane >> 4, c = lane & 15;
    fill_sign_table(lut, t, kMmThreads);

    // Consecutive threads copy consecutive 16 bytes of a token's stage. Rows past
    // the last token repeat it and blocks past the last one its end (unused).
    const uint8_t* src[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++)
        src[i] = a.acts + a.a_qs_offset + static_cast<uint64_t>(min(m0 + kRows * i + t / kThr, a.m - 1)) * a.k;
    const uint8_t* src_d = a.acts + a.a_d_offset + 4 * static_cast<uint64_t>(min(m0 + (t / kStep) % kTok, a.m - 1)) * nb8;
    struct Staged { uint4 q[kPer]; float4 d; };
    auto load_tok = [&](uint32_t b) __attribute__((always_inline)) {
        Staged r;
        const uint32_t at = min(128 * b + 16 * (t % kThr), a.k - 16);
#pragma unroll
        for (int i = 0; i < kPer; i++) r.q[i] = *reinterpret_cast<const uint4*>(src[i] + at);
        r.d = *reinterpret_cast<const float4*>(src_d + 16 * min(b + t % kStep, nb1 - 1));
        return r;
    };
    auto store_tok = [&](int buf, const Staged& r) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kPer; i++)
            if (kTok % kRows == 0 || kRows * i + t / kThr < kTok)
                *reinterpret_cast<uint4*>(&st[buf].qs[kRows * i + t / kThr][16 * (t % kThr)]) = r.q[i];
        if (t < kStep * kTok) *reinterpret_cast<float4*>(&st[buf].d[t / kStep][4 * (t % kStep)]) = r.d;
    };
    // Weights of four blocks at a time: four consecutive lanes read four consecutive
    // blocks of a row (one row per lane takes 64 cache accesses a load instead of 16).
    WaveWeights& ws = wsh[wave];
    const uint64_t wrow = static_cast<uint64_t>(min(n0 + (lane >> 2), a.n - 1)) * nb1;
    const uint8_t* wq_src = a.weights + a.w_qs_offset + 16 * wrow;
    const uint8_t* wd_src = a.weights + a.w_d_offset + 2 * wrow;
    struct Weights { uint4 q; uint16_t d; };
    auto load_w = [&](uint32_t b) __attribute__((always_inline)) {
        Weights w;
        b = min(b + (lane & 3), nb1 - 1);
        w.q = *reinterpret_cast<const uint4*>(wq_src + 16 * b);
        w.d = *reinterpret_cast<const uint16_t*>(wd_src + 2 * b);
        return w;
    };

    Weights w = load_w(0);
    Staged ns = load_tok(0);
    store_tok(0, ns);
    ns = load_tok(kStep);
    float acc[kTiles][4] = {};   // [token tile][r]: weight row 4 g + r, token 16 i + c
    const i4v magic = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    const uint32_t rot = (8 * g - 3) & 31;
    int cur = 0;
    for (uint32_t b0 = 0; b0 < nb1; b0 += kStep) {
        if (kStep == 4 || (b0 & 3) == 0) {
            ws.q[lane & 3][lane >> 2] = w.q;
            ws.d[lane & 3][lane >> 2] = h2f(w.d) * kScaleUp;
            w = load_w(b0 + 4);
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < kStep; j++) {
            if (b0 + j >= nb1) break;
            const uint32_t jw = (b0 + j) & 3;
            const uint4 w4 = ws.q[jw][c];
            const uint32_t wbits[4] = {w4.x, w4.y, w4.z, w4.w};
            const float wd = ws.d[jw][c];
            long av[4];   // elements 32 s + 8 g .. + 7 of row c, as +-1 bytes
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint2 bw = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(lut) +
                                                                 (__builtin_amdgcn_alignbit(wbits[s], wbits[s], rot) & 0x7F8u));
                av[s] = static_cast<long>((static_cast<uint64_t>(bw.y) << 32) | bw.x);
            }
#pragma unroll
            for (int i = 0; i < kTiles; i++) {
                // a_d * w_d of the four 32-blocks: four rank-1 products (K = 1: one rounding
                // each); register 4 s + r: row 4 g + r, token c
                const f16v scale = __builtin_amdgcn_mfma_f32_16x16x1f32(wd, st[cur].d[16 * i + c][4 * j + g], f16v{}, 0, 0, 0);
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const uint2 bq = *reinterpret_cast<const uint2*>(&st[cur].qs[16 * i + c][128 * j + 32 * s + 8 * g]);
                    const long bv = static_cast<long>((static_cast<uint64_t>(bq.y) << 32) | bq.x);
                    const i4v sumi = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[s], bv, magic, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int x = sumi[r];
                        const float v = scale[4 * s + r] * (kMagic - __builtin_bit_cast(float, x));
                        acc[i][r] = acc[i][r] + v;
                    }
                }
            }
        }
        cur ^= 1;
        store_tok(cur, ns);
        ns = load_tok(b0 + 2 * kStep);
    }

    const bool vec = ((a.n | a.out_offset) & 3u) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 7u) == 0;
#pragma unroll
    for (int i = 0; i < kTiles; i++) {
        const uint32_t tok = m0 + 16 * i + c, row = n0 + 4 * g;
        if (tok < a.m)
            store4(a.y + a.out_offset + static_cast<uint64_t>(tok) * a.n + row, row, a.n, vec, a.accumulate, acc[i]);
    }
}

// One tile of 16 rows x 16 tokens per workgroup, its 128-blocks spread over the
// waves, 8 blocks a chunk: each wave computes the four terms (a_d w_d) f32(sumi)
// of every output for one block and puts them in LDS; 256 threads then add the
// chunk's 32 terms to their output in the reference's order. The chain of one
// wave per output (0.3 us a block) becomes about 1.2 us a chunk, so this serves
// shapes whose tiles do not fill the chip.
constexpr int kSpWaves = 8;
constexpr int kTermStride = 4 * kSpWaves + 4;    // floats per output, + 4 against bank conflicts
constexpr int kTokenStride = 17 * kTermStride;   // 16 rows, + 1 likewise

struct SpStage {   // a chunk of 8 blocks
    uint8_t qs[16][128 * kSpWaves + 16];
    uint8_t w[16][16 * kSpWaves + 16];
    float wd[kSpWaves][16];                      // scales * kScaleUp
    float d[16][4 * kSpWaves + 4];
};

__global__ __launch_bounds__(64 * kSpWaves) void matmul_split_kernel(MatmulArgs a) {
    __shared__ __attribute__((aligned(16))) float terms[16 * kTokenStride];
    __shared__ __attribute__((aligned(16))) SpStage st;
    __shared__ uint2 lut[256];
    const uint32_t t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t nb1 = a.k / 128, nb8 = a.k / 32;
    const uint32_t n0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
    const uint32_t c = lane & 15, g = lane >> 4;
    fill_sign_table(lut, t, 64 * kSpWaves);

    // Staging: wave w copies tokens 2 w and 2 w + 1 (1 KB each), waves 0 and 1 the
    // weights and 6 and 7 the tokens' scales (8 lanes a row). Rows past the last
    // repeat it, blocks past the last one its end (unused).
    const uint8_t* acts_q = a.acts + a.a_qs_offset;
    const uint32_t row = 8 * (wave & 1) + (lane >> 3), piece = lane & 7;
    const uint64_t wat = static_cast<uint64_t>(min(n0 + row, a.n - 1)) * nb1;
    const uint64_t dat = static_cast<uint64_t>(min(m0 + row, a.m - 1)) * nb8;
    const uint64_t tok0 = static_cast<uint64_t>(min(m0 + 2 * wave, a.m - 1)) * a.k;
    const uint64_t tok1 = static_cast<uint64_t>(min(m0 + 2 * wave + 1, a.m - 1)) * a.k;
    struct Staged { uint4 q[2]; uint4 w; float4 d; uint16_t wd; };
    auto load = [&](uint32_t b0) __attribute__((always_inline)) {
        Staged r{};
        const uint32_t b = min(b0 + piece, nb1 - 1);
        const uint32_t at = min(128 * b0 + 16 * lane, a.k - 16);
        r.q[0] = *reinterpret_cast<const uint4*>(acts_q + tok0 + at);
        r.q[1] = *reinterpret_cast<const uint4*>(acts_q + tok1 + at);
        if (wave < 2) {
            r.w = *reinterpret_cast<const uint4*>(a.weights + a.w_qs_offset + 16 * (wat + b));
            r.wd = *reinterpret_cast<const uint16_t*>(a.weights + a.w_d_offset + 2 * (wat + b));
        }
        if (wave >= 6) r.d = *reinterpret_cast<const float4*>(a.acts + a.a_d_offset + 4 * (dat + 4 * b));
        return r;
    };
    auto store = [&](const Staged& r) __attribute__((always_inline)) {
        *reinterpret_cast<uint4*>(&st.qs[2 * wave][16 * lane]) = r.q[0];
        *reinterpret_cast<uint4*>(&st.qs[2 * wave + 1][16 * lane]) = r.q[1];
        if (wave < 2) {
            *reinterpret_cast<uint4*>(&st.w[row][16 * piece]) = r.w;
            st.wd[piece][row] = h2f(r.wd) * kScaleUp;
        }
        if (wave >= 6) *reinterpret_cast<float4*>(&st.d[row][4 * piece]) = r.d;
    };
    store(load(0));
    Staged nxt = load(kSpWaves);
    lds_barrier();

    const i4v magic = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    const int lo_mask = g < 2 ? -1 : 0;
    // adder: thread t < 256 owns token t / 16, row t % 16
    const float4* my_terms = reinterpret_cast<const float4*>(&terms[((t >> 4) & 15) * kTokenStride + (t & 15) * kTermStride]);
    float acc = 0.0f;
    for (uint32_t b0 = 0; b0 < nb1; b0 += kSpWaves) {
        if (b0 + wave < nb1) {
            const f16v scale = __builtin_amdgcn_mfma_f32_16x16x1f32(st.wd[wave][c], st.d[c][4 * wave + g], f16v{}, 0, 0, 0);
            i4v sumi[4];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                // 64 elements per MFMA: lane group g holds 16 of them, groups 0 and 1 the
                // 32-block 2 p, groups 2 and 3 the next; the other one's weights are zeroed
                const uint32_t bits = *reinterpret_cast<const uint16_t*>(&st.w[c][16 * wave + 8 * p + 2 * g]);
                const uint2 lo = lut[bits & 0xFFu], hi = lut[bits >> 8];
                const i4v x = {static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(hi.x), static_cast<int>(hi.y)};
                const i4v q = *reinterpret_cast<const i4v*>(&st.qs[c][128 * wave + 64 * p + 16 * g]);
                sumi[2 * p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x & lo_mask, q, magic, 0, 0, 0);
                sumi[2 * p + 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x & ~lo_mask, q, magic, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v[4];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const int x = sumi[s][r];
                    v[s] = scale[4 * s + r] * (kMagic - __builtin_bit_cast(float, x));
                }
                *reinterpret_cast<float4*>(&terms[c * kTokenStride + (4 * g + r) * kTermStride + 4 * wave]) =
                    make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        lds_barrier();
        store(nxt);
        nxt = load(b0 + 2 * kSpWaves);
        if (t < 256) {
            if (b0 + kSpWaves <= nb1) {
                float4 v[kSpWaves];
#pragma unroll
                for (int j = 0; j < kSpWaves; j++) v[j] = my_terms[j];
#pragma unroll
                for (int j = 0; j < kSpWaves; j++) acc = (((acc + v[j].x) + v[j].y) + v[j].z) + v[j].w;
            } else {
                for (uint32_t j = 0; j < nb1 - b0; j++) {
                    const float4 v = my_terms[j];
                    acc = (((acc + v.x) + v.y) + v.z) + v.w;
                }
            }
        }
        lds_barrier();
    }
    const uint32_t out_row = n0 + (t & 15), tok = m0 + ((t >> 4) & 15);
    if (t < 256 && out_row < a.n && tok < a.m) {
        uint16_t* y = a.y + a.out_offset + static_cast<uint64_t>(tok) * a.n + out_row;
        *y = f2h(a.accumulate ? h2f(*y) + acc : acc);
    }
}

constexpr int kRowStride = 136;   // bytes per token row of the staged qs (128 + 8)

template <int kTok> struct BlockStage {   // LDS image of one 128-block of the token tile
    uint8_t qs[kTok * kRowStride];
    float d[kTok * 4];   // [token][s]
};

// kTok tokens (A) x 64 weight rows (B) per workgroup, one 128-block a stage, scales
// and conversions in f32. A wave owns 16 weight rows for all the tokens; a lane
// holds four tokens of one row and reads their a_d of all four 32-blocks as 16-byte
// LDS loads. Rows of the staged qs are padded to 136 bytes: the 16 rows that one
// read touches start in different banks. Nothing past the last block is loaded.
template <int kTok>
__global__ __launch_bounds__(kMmThreads) void matmul_block_kernel(MatmulArgs a) {
    constexpr int kTiles = kTok / 16;          // MFMA token tiles per wave
    constexpr int kTpt = kMmThreads / kTok;    // staging threads per token
    constexpr int kQpt = kTok / 32;            // 16-byte pieces per staging thread
    __shared__ __attribute__((aligned(16))) BlockStage<kTok> st[2];
    __shared__ uint2 lut[256];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t nb1 = a.k / 128, nb8 = a.k / 32;
    const uint32_t n0 = blockIdx.x * kMmRows, m0 = blockIdx.y * kTok;
    const uint32_t g = lane >> 4, c = lane & 15;

    fill_sign_table(lut, t, kMmThreads);

    // token tile loads: thread t -> token t / kTpt, kQpt 16-byte pieces at
    // 16 kQpt (t % kTpt); threads with t % kTpt < 4 also load d of s = t % kTpt
    const uint32_t lt = t / kTpt, lq = t % kTpt;
    const bool tok_ok = m0 + lt < a.m;
    auto load_tok = [&](uint32_t b, uint4 (&q)[kQpt], float& dv) {
#pragma unroll
        for (int i = 0; i < kQpt; i++) q[i] = make_uint4(0u, 0u, 0u, 0u);
        dv = 0.0f;
        if (tok_ok && b < nb1) {
            const uint8_t* src = a.acts + a.a_qs_offset + static_cast<uint64_t>(m0 + lt) * a.k + 128 * b + 16 * kQpt * lq;
#pragma unroll
            for (int i = 0; i < kQpt; i++) q[i] = *reinterpret_cast<const uint4*>(src + 16 * i);
            if (lq < 4)
                dv = *reinterpret_cast<const float*>(a.acts + a.a_d_offset +
                                                     4 * (static_cast<uint64_t>(m0 + lt) * nb8 + 4 * b + lq));
        }
    };
    auto store_tok = [&](int buf, const uint4 (&q)[kQpt], float dv) {
        uint8_t* dst = st[buf].qs + lt * kRowStride + 16 * kQpt * lq;
#pragma unroll
        for (int i = 0; i < kQpt; i++) {
            *reinterpret_cast<uint2*>(dst + 16 * i) = make_uint2(q[i].x, q[i].y);   // 8-byte aligned rows
            *reinterpret_cast<uint2*>(dst + 16 * i + 8) = make_uint2(q[i].z, q[i].w);
        }
        if (lq < 4) st[buf].d[lt * 4 + lq] = dv;
    };
    // this lane's weight row (B column c of the wave's 16)
    const uint32_t wn = n0 + 16 * wave + c;
    const bool w_ok = wn < a.n;
    auto load_w = [&](uint32_t b, uint4& q, uint16_t& d) {
        q = make_uint4(0u, 0u, 0u, 0u);
        d = 0;
        if (w_ok && b < nb1) {
            const uint64_t rb = static_cast<uint64_t>(wn) * nb1 + b;
            q = *reinterpret_cast<const uint4*>(a.weights + a.w_qs_offset + 16 * rb);
            d = *reinterpret_cast<const uint16_t*>(a.weights + a.w_d_offset + 2 * rb);
        }
    };

    uint4 tq[kQpt], wq;
    float tdv;
    uint16_t wd16;
    load_tok(0, tq, tdv);
    load_w(0, wq, wd16);
    store_tok(0, tq, tdv);
    __syncthreads();

    float acc[kTiles][4] = {};   // [token tile][j]: token 16 i + 4g + j, weight row wn
    for (uint32_t b = 0; b < nb1; b++) {
        const int cur = b & 1;
        // next 128-block in flight
        uint4 nq[kQpt], nwq;
        float ndv;
        uint16_t nwd;
        load_tok(b + 1, nq, ndv);
        load_w(b + 1, nwq, nwd);

        const float wd = h2f(wd16);
        const uint32_t wbits[4] = {wq.x, wq.y, wq.z, wq.w};
        long bv[4];   // B for the four 32-blocks: elements 32 s + 8 g .. + 7 of the row, as +-1 bytes
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            const uint2 bw = lut[(wbits[s4] >> (8 * g)) & 0xFFu];
            bv[s4] = static_cast<long>((static_cast<uint64_t>(bw.y) << 32) | bw.x);
        }
#pragma unroll
        for (int i = 0; i < kTiles; i++) {
            // a_d of this lane's 4 tokens, all four 32-blocks at once
            float4 ad[4];
#pragma unroll
            for (int j = 0; j < 4; j++) ad[j] = *reinterpret_cast<const float4*>(&st[cur].d[(16 * i + 4 * g + j) * 4]);
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                // A: tokens 16 i + c, the same 8 elements
                const uint2 av2 = *reinterpret_cast<const uint2*>(st[cur].qs + (16 * i + c) * kRowStride + 32 * s4 + 8 * g);
                const long av = static_cast<long>((static_cast<uint64_t>(av2.y) << 32) | av2.x);
                const i4v z = {0, 0, 0, 0};
                const i4v sumi = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv[s4], z, 0, 0, 0);
                // D[token 16 i + 4g + j][row c]; acc = acc + (a_d * w_d) * f32(sumi), blocks in order
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float adv = s4 == 0 ? ad[j].x : s4 == 1 ? ad[j].y : s4 == 2 ? ad[j].z : ad[j].w;
                    const float scale = adv * wd;
                    const float v = scale * static_cast<float>(sumi[j]);
                    acc[i][j] = acc[i][j] + v;
                }
            }
        }
        store_tok(cur ^ 1, nq, ndv);
        wq = nwq;
        wd16 = nwd;
        __syncthreads();
    }

    // output: y[out + token * n + row]
    if (w_ok) {
#pragma unroll
        for (int i = 0; i < kTiles; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t tok = m0 + 16 * i + 4 * g + j;
                if (tok < a.m) {
                    uint16_t* y = a.y + a.out_offset + static_cast<uint64_t>(tok) * a.n + wn;
                    if (a.accumulate) *y = f2h(h2f(*y) + acc[i][j]);
                    else *y = f2h(acc[i][j]);
                }
            }
    }
}

template <int kTok, int kStep>
void launch_tiles(const MatmulArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((matmul_kernel<kTok, kStep>), dim3((a.n + kMmRows - 1) / kMmRows, (a.m + kTok - 1) / kTok),
                       dim3(kMmThreads), 0, s, a);
}

template <int kTok>
void launch_blocks(const MatmulArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(matmul_block_kernel<kTok>, dim3((a.n + kMmRows - 1) / kMmRows, (a.m + kTok - 1) / kTok),
                       dim3(kMmThreads), 0, s, a);
}

}  // namespace

hipError_t launch_quantize_act_q8_0(const QuantArgs& a, hipStream_t s) {
    const uint32_t blocks = a.m * (a.k / 32);
    hipLaunchKernelGGL(quantize_act_q8_0_kernel, dim3((blocks + 63) / 64), dim3(256), 0, s, a);
    return hipGetLastError();
}

// By how many workgroups a shape gives and by its 128-blocks; us per call, weights
// of 8 tensors in turn, at n x k and tokens:
//  * 64 tokens a workgroup where that still gives three per CU: with the most sums per
//    staged weight (16384 x 2560 at 512 77.5, 32 tokens in two-block stages 86.9) and
//    the least start-up (16384 x 128 at 512 10.2 and 20.5). Not where its last tile is
//    padding for more than the 1/8 (at long k 1/16) that it gains (16384 x 9728 at 200
//    156 and 140), nor past 80 blocks (6144 x 12288 at 512 161 and 155);
//  * 16 x 16 tiles split by blocks up to three per CU (4096 x 2560 at 33: 768 tiles 9.6,
//    whole sums 9.5; 2560 x 4096 at 33: 480, 8.7 and 13.1), fewer where the 8 waves
//    have less than two blocks each (2560 x 640 at 64: 640 tiles, 5.5 and 4.7) or hardly
//    one (512 tiles, 256 x 128 at 512: 3.8 and 3.5);
//  * else 16 tokens while those workgroups fit three per CU (2560 x 4096 at 256 20.3,
//    with 32 tokens 23.1); a single block has nothing to stage ahead (9728 x 128 at 64
//    4.4, one-block stages 3.8);
//  * else 32 tokens. Four-block stages while their LDS holds all workgroups (2560 x 4096
//    at 512 29.4, two-block 31.2), two beyond (4096 x 2560 at 512 26.2, four-block
//    30.2); one where the stages are few (3072 x 640 at 512 7.5, four-block 9.6; 6144 x
//    1280 at 448 19.9, two-block 23.1), but, from two workgroups per CU, not with rows
//    of a multiple of 1024 (2048 past three) elements, whose weight loads, a row per
//    lane, then meet in few cache sets (4096 x 1024: 8.3 and 8.6 at 256 tokens, 10.5
//    and 10.0 at 384; 2560 x 4096 at 1000 65.3, two-block 51.8).
hipError_t launch_matmul_q1_0_q8_0(const MatmulArgs& a, hipStream_t s) {
    const uint64_t cus = a.cu_count, three = 3 * cus;
    const uint64_t t16 = (a.m + 15) / 16, t32 = (a.m + 31) / 32, t64 = (a.m + 63) / 64;
    const uint64_t nx = (a.n + kMmRows - 1) / kMmRows, tiles = (a.n + 15) / 16 * t16;
    const uint32_t nb = a.k / 128;
    const uint64_t pad = 64 * t64 * 24, full = 32 * t32;   // padded tokens, in 24ths of the 32-token tiles'
    if (nx * t64 >= three && nb <= 80 && pad <= full * (nb <= 6 ? 32 : nb <= 20 ? 27 : 25))
        launch_blocks<64>(a, s);
    else if (tiles <= cus * (nb <= 2 ? 1 : nb < 16 ? 2 : 3))
        hipLaunchKernelGGL(matmul_split_kernel, dim3((a.n + 15) / 16, t16), dim3(64 * kSpWaves), 0, s, a);
    else if (nx * t16 <= three && nb > 1)
        launch_tiles<16, 4>(a, s);
    else if (nx * t32 <= three ? nb <= 12 && (nb % 8 != 0 || nx * t32 <= 2 * cus) : nb <= 20 && nb % 16 != 0)
        launch_blocks<32>(a, s);
    else if (nx * t32 <= three)
        launch_tiles<32, 4>(a, s);
    else
        launch_tiles<32, 2>(a, s);
    return hipGetLastError();
}

}  // namespace bp
