// Q1_0 decode matvecs (gfx950): y = W x with 1-bit weights, one f16 scale per
// 128-weight block. Same results as src/shaders/matvec_q1_0.wgsl,
// matvec_q1_0_silu.wgsl and matvec_q1_0_fused_normed.wgsl (reference
// repository), bit for bit wherever the reference fixes the arithmetic:
//
//  * Weight tensor layout (byte offsets into the weight buffer): d[n][nb] f16
//    at d_offset, qs[n][nb][16] at qs_offset (4-byte aligned); bit e of a
//    block's 128-bit little-endian qs selects +x[e] (1) or -x[e] (0).
//  * Per (row, block): four f16 accumulators (component c = e mod 4, elements
//    in increasing order), block sum ((c0 + c1) + c2) + c3 in f16, then in f32
//    acc_t = acc_t + d * sum for the row's lane t = block mod 8 (blocks in
//    increasing order), and the 8 lane sums combined by the xor 1, 2, 4
//    butterfly (matvec_q1_0.wgsl:93-123).
//
// x (the staged activation: plain, silu(gate) * up, or RMS-normed) sits in LDS
// as f16, each 128-element block split into two half-blocks: half 0 holds the
// pairs (x[4i], x[4i+1]) and half 1 the pairs (x[4i+2], x[4i+3]), i = 0..31, so
// that one lane runs the accumulators of components 0, 1 and its neighbour
// those of 2, 3 (two independent packed f16 chains; the order of every chain
// is unchanged). Half-blocks are 144 bytes apart, so the 8 half-blocks that a
// wave reads at once fall in 8 different bank groups.
//
// Inner loop: a sign bit becomes the f16 multiplier +-1 with one v_perm_b32
// per two elements, from pre-shifted copies of the inverted qs word whose
// bytes are 0x3C | (sign << 7); then one v_pk_fma_f16 adds +-x to the lane's
// two accumulators. (fma(+-1, x, c) rounds once, exactly as c + (+-x) does.)
#include <algorithm>

#include "bp_device.hpp"
#include "bp_kernels.hpp"

namespace bp {
namespace {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int kMvMaxThreads = 1024;
constexpr int kQ1Block = 128;
constexpr int kHalfStride = 72;               // halves from one half-block to the next (64 + 8 pad)
constexpr int kBlockHalves = 2 * kHalfStride; // one 128-element block in LDS

// One lane's half of kRows (row, block)s of the same block: components 2h and
// 2h + 1, i.e. the elements 4i + 2h and 4i + 2h + 1 for i = 0..31 in order, as
// one packed pair of f16 accumulators per row. xh: the half-block of x, read
// once for the rows.
template <int kRows>
__device__ __forceinline__ void q1_half(const uint4 (&q)[kRows], const uint16_t* xh, uint32_t h, h2v (&c)[kRows]) {
    const uint32_t sh = 2 - 2 * h;
#pragma unroll
    for (int j = 0; j < kRows; j++) c[j] = h2v{static_cast<_Float16>(0.0f), static_cast<_Float16>(0.0f)};
#pragma unroll
    for (int w = 0; w < 4; w++) {
        uint32_t s[kRows][4];
#pragma unroll
        for (int j = 0; j < kRows; j++) {
            // byte k of s[j][..] = 0x3C | (inverted bit 8k + p << 7), p = 2h + {0, 1, 4, 5};
            // doublings by an add, which issues at twice the rate of a shift
            const uint32_t b5 = (w == 0 ? q[j].x : w == 1 ? q[j].y : w == 2 ? q[j].z : q[j].w) << sh;
            const uint32_t b4 = b5 + b5, b1 = b5 << 4, b0 = b1 + b1;
            s[j][0] = __builtin_amdgcn_bitop3_b32(b0, 0x80808080u, 0x3C3C3C3Cu, 0xAE);   // (~a & b) | c
            s[j][1] = __builtin_amdgcn_bitop3_b32(b1, 0x80808080u, 0x3C3C3C3Cu, 0xAE);
            s[j][2] = __builtin_amdgcn_bitop3_b32(b4, 0x80808080u, 0x3C3C3C3Cu, 0xAE);
            s[j][3] = __builtin_amdgcn_bitop3_b32(b5, 0x80808080u, 0x3C3C3C3Cu, 0xAE);
        }
        const h8v xa = *reinterpret_cast<const h8v*>(xh + 16 * w);       // pairs i = 8w .. 8w + 3
        const h8v xb = *reinterpret_cast<const h8v*>(xh + 16 * w + 8);   // pairs i = 8w + 4 .. 8w + 7
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // bytes: 0x00, byte k of the low word, 0x00, byte k of the high word
            const uint32_t sel = 0x000C000Cu | (static_cast<uint32_t>(4 + k) << 24) | (static_cast<uint32_t>(k) << 8);
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {   // pair m = 2k + hh of the word: bits 8k + 4hh + 2h + {0, 1}
                const int m = 2 * k + hh;
                const h2v xp = m < 4 ? h2v{xa[2 * m], xa[2 * m + 1]} : h2v{xb[2 * m - 8], xb[2 * m - 7]};
#pragma unroll
                for (int j = 0; j < kRows; j++) {
                    const h2v sg = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(s[j][2 * hh + 1], s[j][2 * hh], sel));
                    c[j] = __builtin_elementwise_fma(sg, xp, c[j]);
                }
            }
        }
    }
}

// Weights of one lane in a tile: 16 qs bytes and the f16 scale of kRows rows.
template <int kRows>
struct WTile {
    uint4 q[kRows];
    uint16_t d[kRows];
};

// Tile t of a workgroup: kTR rows (slots) by 32 / kTR blocks by 2 halves, rows
// kTR kRows (t / tcols) .. + kTR kRows - 1, blocks from 32 / kTR (t % tcols) on; a
// lane's kRows rows are kTR apart. A wave walks tiles wave, wave + n_wave, ...; it keeps the tile's
// (row group, block group) in scalar registers and steps them without a division.
struct TilePos {
    uint32_t tile, rq, col;   // wave-uniform
};
template <int kTR>
__device__ __forceinline__ uint32_t tile_row(int lane) { return static_cast<uint32_t>(lane) / (64 / kTR); }
template <int kTR>
__device__ __forceinline__ uint32_t tile_block(int lane) { return (lane >> 1) & (32 / kTR - 1); }
__device__ __forceinline__ void tile_step(TilePos& p, uint32_t n_wave, uint32_t tcols) {
    p.tile += n_wave;
    p.col += n_wave;
    while (p.col >= tcols) {
        p.col -= tcols;
        ++p.rq;
    }
}

// Weights of one lane in a tile. Loads are unconditional (rows and block
// clamped into range), so no lane branches around them.
template <int kTR, int kRows>
__device__ __forceinline__ WTile<kRows> load_tile(const MatvecArgs& a, const TilePos& p, uint32_t nb, uint32_t n_here,
                                                  uint32_t rbase, uint32_t d_off, uint32_t qs_off, int lane) {
    WTile<kRows> w;
    const uint32_t b = min(p.col * (32 / kTR) + tile_block<kTR>(lane), nb - 1);
#pragma unroll
    for (int j = 0; j < kRows; j++) {
        const uint32_t r = min((p.rq * kRows + j) * kTR + tile_row<kTR>(lane), n_here - 1);
        const uint32_t rb = (rbase + r) * nb + b;
        w.q[j] = *reinterpret_cast<const uint4*>(a.weights + qs_off + 16 * rb);
        w.d[j] = *reinterpret_cast<const uint16_t*>(a.weights + d_off + 2 * rb);
    }
    return w;
}

// Stores 8 consecutive x values (elements e .. e + 7, e a multiple of 8) into
// the two half-blocks.
__device__ __forceinline__ void stage8(uint16_t* x_sh, uint32_t e, h8v r) {
    uint16_t* blk = x_sh + (e / kQ1Block) * kBlockHalves + (e % kQ1Block) / 2;
    typedef _Float16 h4v __attribute__((ext_vector_type(4)));
    *reinterpret_cast<h4v*>(blk) = h4v{r[0], r[1], r[4], r[5]};
    *reinterpret_cast<h4v*>(blk + kHalfStride) = h4v{r[2], r[3], r[6], r[7]};
}

// kMode: 0 plain (x = act), 1 silu (x = f16(silu(gate)) * up), 2 normed
// (x = act * w_norm, scale d * inv_rms, up to 3 row ranges).
//
// A workgroup owns rows_per_wg rows, a multiple of kTR kRows (its first weight
// loads are issued before anything else). Pass 1 stages x. Pass 2: its waves share
// the tiles of those rows (kTR kRows rows x 32 / kTR blocks x 2 halves each) and put each block's f32 term
// d * sum in LDS. Pass 3: thread (row, t) adds its terms t, t + 8, ... in order
// and the 8 row lanes combine by the xor 1, 2, 4 butterfly.
template <int kMode, int kTR, int kRows>
__global__ __launch_bounds__(kRows == 1 ? kMvMaxThreads : 512) void matvec_q1_0_kernel(MatvecArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t x_sh[];
    __shared__ float red_sh[4];
    const int t = threadIdx.x, n_thr = blockDim.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), n_wave = n_thr >> 6;
    const uint32_t k = a.k, nb = k / kQ1Block;
    const uint32_t rows = a.rows_per_wg;
    float* terms = reinterpret_cast<float*>(x_sh + nb * kBlockHalves);   // [rows][nb]

    // This workgroup's rows lie in one range (rows_per_wg divides all but the last).
    const uint32_t row0 = blockIdx.x * rows;
    uint32_t d_off = a.range[0].d_offset, qs_off = a.range[0].qs_offset, out_off = a.range[0].output_offset;
    uint32_t rbase = row0;                       // first row of the workgroup within its range
    if constexpr (kMode == 2) {
        if (rbase >= a.range[0].n) {
            rbase -= a.range[0].n;
            d_off = a.range[1].d_offset; qs_off = a.range[1].qs_offset; out_off = a.range[1].output_offset;
            if (rbase >= a.range[1].n) {
                rbase -= a.range[1].n;
                d_off = a.range[2].d_offset; qs_off = a.range[2].qs_offset; out_off = a.range[2].output_offset;
            }
        }
    }
    const uint32_t n_here = min(rows, a.n_total - row0);   // rows of this workgroup that exist

    const uint32_t tcols = (nb + 32 / kTR - 1) / (32 / kTR);
    const uint32_t n_tiles = rows / (kTR * kRows) * tcols;
    TilePos pos = {static_cast<uint32_t>(wave), 0u, static_cast<uint32_t>(wave)};   // (rq, col) = divmod(wave, tcols)
    while (pos.col >= tcols) {   // no division: wave < 16, usually < tcols
        pos.col -= tcols;
        ++pos.rq;
    }
    WTile<kRows> cur = load_tile<kTR, kRows>(a, pos, nb, n_here, rbase, d_off, qs_off, lane);   // in flight during pass 1

    // ---- pass 1: stage x (f16) into LDS, 8 elements at a time --------------------
    float ssq = 0.0f;
    if constexpr (kMode == 0) {
        for (uint32_t v = t; v < k / 8; v += n_thr)
            stage8(x_sh, 8 * v, *reinterpret_cast<const h8v*>(a.act + a.input_offset + 8 * v));
    } else if constexpr (kMode == 1) {
        // matvec_q1_0_silu.wgsl:86-102: silu in f32, then f16(silu) * up in f16.
        for (uint32_t v = t; v < k / 8; v += n_thr) {
            const h8v g = *reinterpret_cast<const h8v*>(a.act + a.gate_offset + 8 * v);
            const h8v u = *reinterpret_cast<const h8v*>(a.act + a.up_offset + 8 * v);
            h8v r;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float gf = static_cast<float>(g[i]);
                const float sl = gf / (1.0f + expf(-gf));
                r[i] = static_cast<_Float16>(sl) * u[i];
            }
            stage8(x_sh, 8 * v, r);
        }
    } else {
        // matvec_q1_0_fused_normed.wgsl:102-121: x * w_norm in f16; the sum of
        // x^2 in f32 by 256 threads (element groups v = t, t + 256, ... in order).
        if (t < 256) {
            for (uint32_t v = t; v < k / 8; v += 256) {
                const h8v x = *reinterpret_cast<const h8v*>(a.act + a.input_offset + 8 * v);
                const h8v w = *reinterpret_cast<const h8v*>(a.w_norms + a.w_norm_off + 8 * v);
                h8v r;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float xf = static_cast<float>(x[i]);
                    ssq = ssq + xf * xf;
                    r[i] = x[i] * w[i];
                }
                stage8(x_sh, 8 * v, r);
            }
        }
    }
    float inv_rms = 1.0f;
    if constexpr (kMode == 2) {
        // Sum over the 256 threads: xor butterfly in each wave, then waves 0..3 in order.
        if (wave < 4) {
            ssq = wave_sum(ssq);
            if (lane == 0) red_sh[wave] = ssq;
        }
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) total += red_sh[w];
        inv_rms = 1.0f / sqrtf(total / static_cast<float>(k) + a.eps);
    } else {
        __syncthreads();
    }

    // ---- pass 2: block terms (weights of the next tile loaded ahead) --------------
    const uint32_t h = lane & 1;
    while (pos.tile < n_tiles) {
        TilePos nxt_pos = pos;
        tile_step(nxt_pos, n_wave, tcols);
        const WTile<kRows> nxt = load_tile<kTR, kRows>(a, nxt_pos, nb, n_here, rbase, d_off, qs_off, lane);
        const uint32_t b0 = pos.col * (32 / kTR) + tile_block<kTR>(lane), b = min(b0, nb - 1);
        // the lane exchange is executed by all lanes
        h2v c[kRows];
        q1_half<kRows>(cur.q, x_sh + b * kBlockHalves + h * kHalfStride, h, c);
        // The pair's lane h keeps row j = h of two rows (one row: lane 0 keeps it).
        h2v c23[kRows];
#pragma unroll
        for (int j = 0; j < kRows; j++) c23[j] = __builtin_bit_cast(h2v, lane_xor<1>(__builtin_bit_cast(uint32_t, c[j])));
        if (b0 < nb && (kRows == 2 || h == 0)) {
            h2v lo = c[0], hi = c23[0];   // components 0, 1 and 2, 3
            uint16_t dj = cur.d[0];
            if (kRows == 2 && h == 1) {
                lo = c23[kRows - 1];
                hi = c[kRows - 1];
                dj = cur.d[kRows - 1];
            }
            const uint32_t r = (pos.rq * kRows + (kRows == 2 ? h : 0u)) * kTR + tile_row<kTR>(lane);
            const _Float16 sum = ((lo.x + lo.y) + hi.x) + hi.y;   // f16 adds, in this order
            float d = static_cast<float>(__builtin_bit_cast(_Float16, dj));
            if constexpr (kMode == 2) d = d * inv_rms;
            if (r < n_here) terms[r * nb + b] = d * static_cast<float>(sum);
        }
        cur = nxt;
        pos = nxt_pos;
    }
    __syncthreads();

    // ---- pass 3: the 8 ordered lane sums of each row, then the butterfly ----------
    for (uint32_t i = t; i < rows * 8; i += n_thr) {   // (a row's 8 lanes stay together)
        const uint32_t r = i >> 3, bt = i & 7;
        float acc = 0.0f;
        if (r < n_here)
            for (uint32_t b = bt; b < nb; b += 8) acc = acc + terms[r * nb + b];
        acc = acc + lane_xor<1>(acc);
        acc = acc + lane_xor<2>(acc);
        acc = acc + lane_xor<4>(acc);
        if (bt == 0 && r < n_here) {
            uint16_t* y = a.act + out_off + rbase + r;
            if (kMode != 2 && a.accumulate) *y = f2h(h2f(*y) + acc);
            else *y = f2h(acc);
        }
    }
}

}  // namespace

hipError_t launch_matvec_q1_0(const MatvecArgs& args, int mode, hipStream_t s) {
    MatvecArgs a = args;
    const uint32_t nb = a.k / kQ1Block, cus = a.cu_count;
    auto lds_bytes = [&](uint32_t rows) { return static_cast<size_t>(nb) * kBlockHalves * 2 + static_cast<size_t>(rows) * nb * 4; };
    auto div_up = [](uint64_t x, uint64_t y) { return static_cast<uint32_t>((x + y - 1) / y); };
    auto launch = [&](auto kernel, uint32_t rows, uint32_t waves) {
        a.rows_per_wg = rows;
        hipLaunchKernelGGL(kernel, dim3(div_up(a.n_total, rows)), dim3(64 * waves), lds_bytes(rows), s, a);
        return hipGetLastError();
    };

    // Rows and waves per workgroup; us measured with all weights in turn.
    if (mode == 1) {
        // The silu matvec stages an expensive x: one workgroup per CU (or as few
        // as keep it to 32 rows), so that no CU stages twice or idles, in tiles of
        // 2 rows: 2560 x 9728 10 rows 6.52 (16 rows on 160 CUs 7.11, 8 rows 8.82),
        // 2048 x 6144 5.26 -> 4.78, 1024 x 6144 5.07 -> 4.40; 4096 x 12288 (16 rows
        // either way) 8.19 and 8.24. 16 waves where staging takes more than 12
        // (2560 x 9728: 8 waves 6.79; 2048 x 6144: 16 waves 4.87).
        // Below k = 3072 the staging is cheap and 16 blocks fill badly: 16 rows there
        // (1024 x 2048 3.07, 4096 x 1024 2.87, tiles of 2 rows 3.20 and 3.18). Nor do
        // they help where 16 rows come out anyway: two tiles of 8 rows use each x read
        // from LDS for more rows (4096 x 6144 5.79, tiles of 2 rows 6.00).
        const uint32_t rows = nb < 24 ? 16 : 2 * div_up(a.n_total, 2ull * cus * div_up(a.n_total, 32ull * cus));
        if (rows == 16) return launch(matvec_q1_0_kernel<1, 8, 1>, rows, std::min(2 * div_up(nb, 4), 16u));
        return launch(matvec_q1_0_kernel<1, 2, 1>, rows, a.k > 6144 ? 16 : 8);
    }
    if (mode == 0 && nb >= 32 && nb % 8 == 0 && a.n_total <= 24 * cus) {
        // Long rows, few of them: one workgroup per CU here too, tiles of 4 rows
        // (2560 x 4096 4.23 -> 3.97, 4096 x 4096 4.40 -> 4.31, 1024 x 4096 3.24 ->
        // 3.14; with k = 2048 the smaller workgroups below are as fast). Whole tiles of 8
        // blocks only: past one the gain is gone on most sizes (k = 4224: 1024 / 2560 /
        // 4096 / 6144 rows 3.8 / 4.3 / 4.5 / 5.4, below 3.7 / 4.5 / 4.6 / 5.2).
        const uint32_t rows = 4 * div_up(a.n_total, 4 * cus), tiles = rows / 4 * (nb / 8);
        return launch(matvec_q1_0_kernel<0, 4, 1>, rows, std::min(tiles, 16u));
    }
    // Up to 3 workgroups of 8 rows per CU: one tile per wave. Larger grids: each
    // workgroup stages x again, about the work of 4 rows, and the busiest CU gets
    // ceil(workgroups / CUs) of them, so the rows with the least of that times
    // (rows + 4). Several ranges: rows have to divide them (16 always does), and x
    // and the terms fit 64 KB of LDS. By 16 / 32 / 64 rows: 12288 x 2048 4.68 /
    // 5.11 / 5.04 (8 rows 5.18), 19456 x 2560 6.9 / 6.9 / 7.2, 16384 x 2560 5.94 /
    // 5.68 / 5.51, 24576 x 4096 9.95 / 9.31 / 10.3, 151936 x 2560 37 / 27.5 / 26.8.
    // 8 rows still where a plain x of up to 32 blocks is staged and that cost is no
    // higher (9728 x 2560 4.93, 16 rows 5.19; with 33 blocks 6.71 and 6.79, with 40
    // 7.09 and 6.86, and the normed staging costs more: 5.55 and 5.29); a few of these
    // small workgroups (1/16 per CU) run beside the others (6160 x 2560 4.23, 32 rows
    // 4.40; from 6400 the two are equal).
    const uint32_t tcols = (nb + 3) / 4;
    uint32_t rows = 8;
    if (a.n_total > 24 * cus) {
        const bool one_range = a.range[0].n == a.n_total;
        uint64_t best = ~0ull;
        if (mode == 0 && tcols <= 8) best = 12ull * div_up(div_up(a.n_total, 8) - cus / 16, cus);
        for (uint32_t r : {16u, 32u, 64u}) {
            if (r > 16 && ((!one_range && (a.range[0].n % r || a.range[1].n % r)) || lds_bytes(r) > 65536)) continue;
            const uint64_t cost = static_cast<uint64_t>(div_up(a.n_total, static_cast<uint64_t>(r) * cus)) * (r + 4);
            if (cost < best || (cost == best && rows > 8)) best = cost, rows = r;
        }
    }
    // Waves. 8 rows: one tile each (with k = 2560's 5 on 4 SIMDs every workgroup adds
    // to the first one, yet 8 waves of which 3 only stage took 5.34 at 9728 x 2560),
    // but 8 where there are two or more workgroups of 10 to 16 per CU (6144 x 8192
    // normed 7.14, 16 waves 8.78). 16 rows: 8 waves (12288 x 4224 6.84, 4 waves 7.11;
    // 19456 x 16384 23.9 and 27.6), 4 where x is small (under 20 blocks both the same)
    // or the normed sum, over 256 threads (4 waves at least), holds the others up
    // (9728 x 4096 6.37, 8 waves 6.45; past k = 8192 again 8).
    if (rows == 8) {
        const bool two = a.n_total > 16 * cus && tcols >= 10;
        const uint32_t waves = two ? 8u : std::max(std::min(tcols, 16u), mode == 2 ? 4u : 1u);
        return mode == 0 ? launch(matvec_q1_0_kernel<0, 8, 1>, rows, waves) : launch(matvec_q1_0_kernel<2, 8, 1>, rows, waves);
    }
    if (rows == 16) {
        const uint32_t waves = (mode == 0 && nb >= 20) || a.k > 8192 ? 8u : 4u;
        return mode == 0 ? launch(matvec_q1_0_kernel<0, 8, 1>, rows, waves) : launch(matvec_q1_0_kernel<2, 8, 1>, rows, waves);
    }
    // Two rows per lane (x read from LDS once for both, two independent chains:
    // 151936 x 2560 28.6 -> 26.8, 24576 x 4096 9.65 -> 9.31) unless 32 rows then
    // keep the waves busy for longer (k = 2560: 20 tiles on 8 waves 5.68, 10 double
    // ones 5.98). 4 waves for grids of many workgroups, 8 otherwise (151936 x 2560
    // 26.8 and 27.4; 32000 x 2048 7.50 and 7.21); the normed staging is done by 4
    // waves, so there from 2 workgroups per CU (24576 x 4096 9.31 and 9.64).
    const uint32_t doubles = rows / 16 * tcols, n_wg = div_up(a.n_total, rows);
    if (rows == 64 || 2 * ((doubles + 7) / 8) <= (2 * doubles + 7) / 8) {
        const uint32_t waves = n_wg >= 4 * cus || (mode == 2 && rows == 32 && n_wg >= 2 * cus) ? 4 : 8;
        return mode == 0 ? launch(matvec_q1_0_kernel<0, 8, 2>, rows, waves) : launch(matvec_q1_0_kernel<2, 8, 2>, rows, waves);
    }
    return mode == 0 ? launch(matvec_q1_0_kernel<0, 8, 1>, rows, 8) : launch(matvec_q1_0_kernel<2, 8, 1>, rows, 8);
}

uint32_t matvec_max_k() { return 16384; }

}  // namespace bp
