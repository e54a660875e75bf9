// Matrix products of few rows (more than a GEMV's, fewer than fill the tiled
// GEMM): weights streamed from HBM straight into MFMA operand registers.
#pragma once

#include "kernels.hpp"

namespace hm {

// Block = NWV waves over CT 16-column weight tiles (plain: CT adjacent tiles;
// SwiGLU: a gate tile and the up tile 32 packed columns on) and 16 RT rows. The
// waves split K: wave w takes units w, w + NWV, ... of four weight planes (64 k
// of W8, 128 k of W4), so a lane's 16 loaded bytes are its share of
// v_mfma_i32_16x16x64_i8's B operand as they lie (column lane % 16, plane
// lane / 16; the two nibbles of a W4 entry give one operand each) and a block
// reads 512-byte runs of its tiles. The rows' codes are loaded the same way
// ([plane][row][16]: one 16-byte entry per lane). WW units of weights and AD
// steps of codes are in flight per wave. The waves' int32 sums meet in LDS by
// integer atomics (exact in any order), then every thread dequantizes and
// stores 4 neighbouring columns of a row.
//
// What it is for: the tiled GEMM walks K with one block per output tile and a
// barrier per 64 k, so with few rows its time is K / 64 times a stage's latency
// on the few CUs that have a tile, whatever the bytes. Here K is NWV chains per
// column tile, on 4 to 8 times as many blocks. Measured per call in a graph, the
// rows' quantization launch included (a kernel of 3.4 us at 16 rows, 4.1 to 4.7 at
// 64, in a kernel trace), distinct weights from HBM, us, tiled GEMM -> this kernel:
//                              16 rows        64 rows        128 rows
//   o       4096x2560   W4  19.4 ->  7.5   19.1 ->  9.6   19.7 -> 13.0
//   o       4096x2560   W8  18.6 ->  8.5   19.6 -> 11.4   20.7 -> 14.6
//   qkv     2560x6144   W4  14.7 ->  7.5   14.8 ->  9.3   15.4 -> 12.2
//   gate_up 2560x19456  W4  22.6 -> 12.0   28.6 -> 16.5   28.8 -> 26.6
//   down    9728x2560   W4  39.3 -> 11.3   21.4 -> 18.1   23.4 -> 25.4
//   up      2560x9728   W8  16.5 -> 11.2   17.8 -> 16.9   18.1 -> 22.4
// At 16 rows what is left is the two launches (about 2.3 us each) and the
// weight stream (gate_up's 25 MB at 3.2 TB/s with its launch); from 64 rows on
// it is the codes: a block reads 16 RT rows of all of K, at 35 bytes per clock
// and CU, so calls come here where few blocks a CU read them (skinny_gains,
// hip_matmul.hip) and the rest stays with the tiled GEMM, which stages them in
// LDS for 128 columns. Row maxima leave as one partial per row and block: met by
// atomics on the rows' few cache lines, they took gate_up of 16 rows from 12.0
// to 15.8 us and of 64 rows from 16.5 to 23.4.
//
// Four waves of W4 and eight of W8 give every wave the same bytes; eight and
// sixteen of W4 took gate_up of 64 rows to 20.9 and 52.8 us.
struct SkinnyParams {
    GemmParams g;
    float* part;  // SwiGLU row maxima [row][gridDim.x], or nullptr: none wanted
    int staged;   // 16-byte aligned output base and row pitch: vector stores
};

template <int BITS, int RT, int CT, int EPI, int NWV, int WW>
__global__ __launch_bounds__(64 * NWV) void skinny_kernel(SkinnyParams S) {
    static_assert(EPI == EPI_PLAIN || CT == 2, "SwiGLU: one gate and one up tile");
    constexpr int HN = BITS == 4 ? 2 : 1;  // MFMA steps per unit
    constexpr int AD = RT == 8 ? 2 : (RT == 4 ? 4 : (WW * HN < 8 ? WW * HN : 8));  // code steps in flight
    constexpr int NT = 64 * NWV;
    // Only the widest window is reloaded (a narrower one holds all of a wave's
    // units): its steps are a whole number of code slots, so every slot index
    // is a constant.
    constexpr bool REFILL = WW >= 8;
    static_assert(!REFILL || WW * HN % AD == 0, "static register slots");
    const GemmParams& P = S.g;
    __shared__ __attribute__((aligned(16))) int sums[RT * CT * 256];  // [row tile][col tile][row % 4][lane]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lo = lane & 15, hi = lane >> 4;
    // packed columns of the block's tiles
    const int b = blockIdx.x;
    const int col0 = EPI == EPI_PLAIN ? b * 16 * CT : (b >> 1) * 64 + (b & 1) * 16;
    constexpr int CSTEP = EPI == EPI_PLAIN ? 16 : 32;
    if (col0 >= P.N) return;  // (tiles of padding columns only; none of SwiGLU's)
    const int row0 = blockIdx.y * (16 * RT);

    const int planes = P.K_pad / (BITS == 8 ? 16 : 32);
    const int U = (planes + 3) >> 2;
    const int nu = U > wave ? (U - wave + NWV - 1) / NWV : 0;  // this wave's units

    const uint8_t* wsrc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
        wsrc[c] = P.b + ((size_t)((col0 + c * CSTEP) / 8 + (lo >> 3)) * planes) * 128 + (lo & 7) * 16;
    const int8_t* asrc = P.a + (size_t)(row0 + lo) * 16;
    const size_t aplane = (size_t)P.M_alloc * 16;
    // lane's weight plane in unit i of this wave (past the end: a valid one)
    auto plane_of = [&](int i) { return min(4 * (wave + NWV * min(i, nu - 1)) + hi, planes - 1); };
    auto load_w = [&](int i, v4u (&w)[CT]) {
        const size_t off = (size_t)plane_of(i) * 128;
#pragma unroll
        for (int c = 0; c < CT; ++c) w[c] = gload_nt<v4u>(wsrc[c] + off);
    };
    // codes of step s = i * HN + h: W8 plane = the weights' own; W4 plane j
    // holds k = 64 (j / 2) + 16 (j % 2) .. +15 in its low nibbles, 32 on in its
    // high ones
    auto load_a = [&](int s, v4i (&a)[RT]) {
        const int p = plane_of(s / HN);
        const int k16 = BITS == 8 ? p : 4 * (p >> 1) + (p & 1) + 2 * (s % HN);
        const int8_t* src = asrc + (size_t)k16 * aplane;
#pragma unroll
        for (int t = 0; t < RT; ++t) a[t] = gload<v4i>(src + t * 256);
    };

    v4i acc[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = v4i{0, 0, 0, 0};
    v4i a[AD][RT];
    v4u w[WW][CT];
    if (nu > 0) {
#pragma unroll
        for (int j = 0; j < AD; ++j) load_a(j, a[j]);
#pragma unroll
        for (int i = 0; i < WW; ++i) load_w(i, w[i]);
    }

    // the epilogue's operands, requested under the weight stream; quad q =
    // columns 4 (q % 4)..+3 of row (q / 4) % (16 RT) in column tile q / (64 RT)
    constexpr int OT = EPI == EPI_PLAIN ? CT : 1;  // output column tiles
    constexpr int QUADS = OT * 64 * RT, QPT = (QUADS + NT - 1) / NT;
    float rs[QPT];
    int rc[QPT];
    float4 cs[QPT], cu[QPT];
#pragma unroll
    for (int e = 0; e < QPT; ++e) {
        const int q = tid + e * NT;
        const int row = row0 + (q >> 2) % (16 * RT), src = row < P.M ? row : 0;
        const int c = min(q / (64 * RT), OT - 1);
        rs[e] = P.rowscale[src];
        rc[e] = BITS == 4 ? 8 * P.rowsum[src] : 0;
        cs[e] = *reinterpret_cast<const float4*>(P.colscale + col0 + c * CSTEP + 4 * (q & 3));
        if constexpr (EPI != EPI_PLAIN) cu[e] = *reinterpret_cast<const float4*>(P.colscale + col0 + CSTEP + 4 * (q & 3));
    }
#pragma unroll
    for (int i = tid; i < RT * CT * 64; i += NT) reinterpret_cast<v4i*>(sums)[i] = v4i{0, 0, 0, 0};

    const bool refill = REFILL && U > NWV * WW;  // (uniform over the block)
    const bool ragged = BITS == 4 && (planes & 3) != 0;
    for (int base = 0; base < nu; base += WW) {
#pragma unroll
        for (int i = 0; i < WW; ++i) {
            if (base + i >= nu) break;
            // (planes past the end, in the last unit of an odd count: no weight)
            if (ragged && wave + NWV * (base + i) == U - 1 && 4 * (U - 1) + hi >= planes) {
#pragma unroll
                for (int c = 0; c < CT; ++c) w[i][c] = v4u{0u, 0u, 0u, 0u};
            }
#pragma unroll
            for (int h = 0; h < HN; ++h) {
                const int slot = (i * HN + h) % AD;
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const v4i wv = __builtin_bit_cast(
                        v4i, BITS == 8 ? w[i][c] : (h == 0 ? (w[i][c] & 0x0F0F0F0Fu) : ((w[i][c] >> 4) & 0x0F0F0F0Fu)));
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        acc[t][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[slot][t], wv, acc[t][c], 0, 0, 0);
                }
                load_a((base + i) * HN + h + AD, a[slot]);
            }
            if (refill) load_w(base + i + WW, w[i]);
        }
    }
    __syncthreads();  // (the sums are cleared)
    if (nu > 0) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) atomicAdd(&sums[((t * CT + c) * 4 + r) * 64 + lane], acc[t][c][r]);
    }
    __syncthreads();

#pragma unroll
    for (int e = 0; e < QPT; ++e) {
        const int q = tid + e * NT;
        if (q >= QUADS) break;
        const int local = (q >> 2) % (16 * RT), row = row0 + local, quad = q & 3, c = q / (64 * RT);
        // accumulator layout: row 4 (lane / 16) + r of the tile, column lane % 16
        const int at = ((local >> 4) * CT * 4 + (local & 3)) * 64 + ((local >> 2) & 3) * 16 + 4 * quad;
        const v4i s0 = *reinterpret_cast<const v4i*>(&sums[at + c * 256]);
        const float csv[4] = {cs[e].x, cs[e].y, cs[e].z, cs[e].w};
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = ((float)(s0[j] - rc[e]) * rs[e]) * csv[j];
        const int p = col0 + c * CSTEP + 4 * quad;  // packed column
        const int col = EPI == EPI_PLAIN ? orig_col(p, P.half) : ((p >> 6) << 5) + (p & 31);
        const int valid = row < P.M ? (EPI == EPI_PLAIN ? min(4, P.N - p) : 4) : 0;
        if constexpr (EPI != EPI_PLAIN) {
            const v4i s1 = *reinterpret_cast<const v4i*>(&sums[at + 256]);
            const float cuv[4] = {cu[e].x, cu[e].y, cu[e].z, cu[e].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = hm_swiglu(y[j], ((float)(s1[j] - rc[e]) * rs[e]) * cuv[j]);
            float mx = fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3])));
            mx = fmaxf(mx, dpp_move<DPP_QUAD_XOR1>(mx));
            mx = fmaxf(mx, dpp_move<DPP_QUAD_XOR2>(mx));
            if (S.part && quad == 0 && row < P.M) S.part[(size_t)row * gridDim.x + b] = mx;
        }
        const size_t o = (size_t)row * P.ldc + col;
        if (S.staged && valid == 4) {
            if (P.c_type == DT_F32) {
                *reinterpret_cast<float4*>(static_cast<float*>(P.c) + o) = float4{y[0], y[1], y[2], y[3]};
            } else {
                const unsigned w0 = (unsigned)__half_as_ushort(f32_to_f16(y[0])) |
                                    ((unsigned)__half_as_ushort(f32_to_f16(y[1])) << 16);
                const unsigned w1 = (unsigned)__half_as_ushort(f32_to_f16(y[2])) |
                                    ((unsigned)__half_as_ushort(f32_to_f16(y[3])) << 16);
                *reinterpret_cast<uint2*>(static_cast<__half*>(P.c) + o) = uint2{w0, w1};
            }
        } else {
            for (int j = 0; j < valid; ++j) store_out(P.c, P.c_type, o + j, y[j]);
        }
    }
}

}  // namespace hm
