// Routed-expert products of few rows per expert: each expert's weights are
// streamed from HBM straight into matrix-core operands, as skinny_kernel does
// for one matrix.
#pragma once

#include "moe_kernels.hpp"

namespace hm {

typedef float v4f __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Routing and token quantization in one launch: block 0 sorts the assignments
// (moe_route_block), the others quantize the token rows, one wave per row, in
// row-major order [row][K_pad], which a gathered matrix-core operand load reads
// in 64-byte runs. Values and rounding are quant_rows_kernel's.
// ---------------------------------------------------------------------------
struct TokenQuant {
    const float* x;
    int rows, K, K_pad;
    int vec;  // 1: rows are 16-byte aligned and K % 16 == 0
    int8_t* codes;
    float* rowscale;
    int* rowsum;
};

constexpr int FRONT_THREADS = 1024;
constexpr int FRONT_CHUNKS = 3;  // 16-element chunks per lane kept in registers

__device__ __forceinline__ void moe_quant_token(const TokenQuant& Q, int r, int lane) {
    const float* xr = Q.x + (size_t)r * Q.K;
    const int KG = Q.K_pad >> 4;
    auto chunk = [&](int kg, float (&v)[16]) {
        if (Q.vec && kg * 16 < Q.K) {
            v4u raw[4];
            load16_raw(xr + kg * 16, raw);
            cvt16_raw(raw, v, float());
        } else {
#pragma unroll
            for (int b = 0; b < 16; ++b) v[b] = kg * 16 + b < Q.K ? xr[kg * 16 + b] : 0.0f;
        }
    };
    float held[FRONT_CHUNKS][16];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < FRONT_CHUNKS; ++j)
        if (lane + 64 * j < KG) chunk(lane + 64 * j, held[j]);
#pragma unroll
    for (int j = 0; j < FRONT_CHUNKS; ++j)
        if (lane + 64 * j < KG)
#pragma unroll
            for (int b = 0; b < 16; ++b) m = fmaxf(m, fabsf(held[j][b]));
    for (int kg = lane + 64 * FRONT_CHUNKS; kg < KG; kg += 64) {
        float v[16];
        chunk(kg, v);
#pragma unroll
        for (int b = 0; b < 16; ++b) m = fmaxf(m, fabsf(v[b]));
    }
    m = wave_max(m);
    const float sc = quant_scale<QUANT_MOE>(m);
    const float inv = 1.0f / sc;
    int8_t* dst = Q.codes + (size_t)r * Q.K_pad;
    int sum = 0;
#pragma unroll
    for (int j = 0; j < FRONT_CHUNKS; ++j) {
        const int kg = lane + 64 * j;
        if (kg < KG) *reinterpret_cast<v4u*>(dst + kg * 16) = quant_chunk<QUANT_MOE>(held[j], inv, sum);
    }
    for (int kg = lane + 64 * FRONT_CHUNKS; kg < KG; kg += 64) {
        float v[16];
        chunk(kg, v);
        *reinterpret_cast<v4u*>(dst + kg * 16) = quant_chunk<QUANT_MOE>(v, inv, sum);
    }
    sum = wave_sum(sum);
    if (lane == 0) {
        Q.rowscale[r] = sc;
        Q.rowsum[r] = sum;
    }
}

template <int BM>
__global__ __launch_bounds__(FRONT_THREADS) void moe_front_kernel(RouteParams R, TokenQuant Q) {
    if (blockIdx.x == 0) {
        moe_route_block<BM>(R);
        return;
    }
    const int r = (blockIdx.x - 1) * (FRONT_THREADS / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r < Q.rows) moe_quant_token(Q, r, threadIdx.x & 63);
}

// ---------------------------------------------------------------------------
// Grouped product. Block = one routing tile (up to 16 RTM slots of one expert)
// x 64 packed columns, 4 waves. The waves split K: wave w takes units w, w + 4,
// ... of four weight planes (64 k of W8, 128 k of W4), a lane's 16 loaded bytes
// being its share of v_mfma_i32_16x16x64_i8's B operand as they lie; the waves'
// int32 sums meet in LDS by integer atomics (exact in any order). WW units of
// weights are in flight per wave: 16 KB at WW = 4, all of a wave's share of K
// for the usual sizes (K = 2048 of W4, 1024 of W8), so a block asks for its
// whole weight tile at once. The body is instantiated per number of 16-row
// tiles, so a run of 20 slots loads and multiplies 32 rows, not 48.
//
// Rows: codes at a + row * a_row + (k / 16) * a_plane (row-major token codes, or
// the k16 planes of a quantized middle), row = perm[slot] / top, or the slot
// itself without perm. With AQ (one row tile) the block quantizes its rows of
// the f32 middle itself, from the maxima that the gate/up blocks left.
//
// Bound: the expert weights' bytes. The tiled GEMM pads every run to 64 rows
// and walks K with a barrier per 64 k. Measured at hidden 2048, intermediate
// 768, 128 experts, top 8, us, tiled -> streamed:
//                        25 tokens (161 MB each)    512 tokens (201 MB each)
//   route + token codes     9.8 -> 4.6                 17.7 -> 6.2
//   gate/up W4             44.7 -> 29.4 (5.5 TB/s)     62.4 -> 59.2 (3.4 TB/s)
//   down W8                33.9 -> 28.0 (5.8 TB/s)     52.4 -> 44.2 (4.6 TB/s, and 34 MB written)
//   middle's codes          5.0 -> in down              7.3 -> 5.7
//   whole call             89.0 -> 64.0               135.3 -> 117.2
// 48 rows and two code steps in flight let three blocks share a CU; 64 rows
// and four steps (two blocks) took gate/up of 512 tokens to 63.6 and down to
// 51. There, the gathered code rows (adjacent lanes read different lines) are
// 10 us of gate/up; codes copied into slot order first cost 7.7 us more.
// ---------------------------------------------------------------------------
struct MoeStreamParams {
    const int8_t* a;
    size_t a_row, a_plane;
    const int* perm;
    int top;
    const float* rowscale;
    const int* rowsum;
    const float* mid;       // AQ: f32 middle [slot][K]
    const float* part_in;   // AQ: its row maxima [slot][part_count]
    int part_count;
    const uint8_t* const* b_tab;
    const float* const* s_tab;
    const int4* tiles;
    const int* counts;
    float* c;  // [slot][ldc]
    long ldc;
    float* part;  // SwiGLU: row maxima [slot][tiles_n]
    int N, K, K_pad, half, tiles_n;
    int max_tiles;  // >= 1 entries of tiles that may be read
    int staged;  // 16-byte aligned output base and row pitch: vector stores
};

constexpr int STREAM_CT = 4;   // 16-column tiles per block: one 32 gate + 32 up group
constexpr int STREAM_NWV = 4;  // waves per block
constexpr int STREAM_NT = 64 * STREAM_NWV;

template <int BITS, int EPI, int RT, int WW, bool REFILL, bool AQ>
__device__ __forceinline__ void moe_stream_body(const MoeStreamParams& P, int e, int begin, int nrows, int tn,
                                                int* sums, float* s_rs, int* s_rc, int8_t* s_codes) {
    constexpr int CT = STREAM_CT, NWV = STREAM_NWV, NT = STREAM_NT;
    constexpr int HN = BITS == 4 ? 2 : 1;  // MFMA steps per unit
    constexpr int STEPS = WW * HN;
    constexpr int AD = AQ ? 1 : (STEPS < 4 ? STEPS : (RT == 3 ? 2 : 4));  // code steps in flight
    static_assert(!REFILL || STEPS % AD == 0, "static register slots");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lo = lane & 15, hi = lane >> 4;
    const int col0 = tn * 64;
    const int planes = P.K_pad / (BITS == 8 ? 16 : 32);
    const int U = (planes + 3) >> 2;
    const int nu = U > wave ? (U - wave + NWV - 1) / NWV : 0;  // this wave's units
    const int KG = P.K_pad >> 4;

    // the rows of this lane's operands (past the run: its first row, not stored)
    auto row_of = [&](int local) {
        const int slot = begin + (local < nrows ? local : 0);
        return P.perm ? P.perm[slot] / P.top : slot;
    };
    const int8_t* asrc[RT];
    if constexpr (!AQ) {
#pragma unroll
        for (int t = 0; t < RT; ++t) asrc[t] = P.a + (size_t)row_of(16 * t + lo) * P.a_row;
    }
    // AQ: the first NT chunks of the middle, and (below) the row maxima
    v4u raw[4];
    const int tasks = nrows * KG;
    const float* mid = P.mid + (size_t)begin * P.K;
    float pm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (AQ) {
        const int r = tid / KG, kg = tid - r * KG;
        const bool ok = tid < tasks && kg * 16 < P.K;
        load16_raw(ok ? mid + (size_t)r * P.K + kg * 16 : mid, raw);
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // row maxima of rows wave, wave + 4, ...
            const int row = wave + 4 * i;
            if (row < nrows)
                for (int j = lane; j < P.part_count; j += 64)
                    pm[i] = fmaxf(pm[i], P.part_in[(size_t)(begin + row) * P.part_count + j]);
        }
        asm volatile("" ::: "memory");
    }

    const uint8_t* bw = P.b_tab[e];
    const float* colscale = P.s_tab[e];
    const uint8_t* wsrc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
        wsrc[c] = bw + ((size_t)(col0 / 8 + 2 * c + (lo >> 3)) * planes) * 128 + (lo & 7) * 16;
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
    auto k16_of = [&](int s) {
        const int p = plane_of(s / HN);
        return BITS == 8 ? p : 4 * (p >> 1) + (p & 1) + 2 * (s % HN);
    };
    auto load_a = [&](int s, v4i (&a)[RT]) {
        const int k16 = k16_of(s);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            if constexpr (AQ)
                a[t] = *reinterpret_cast<const v4i*>(s_codes + (k16 * 16 + lo) * 16);
            else
                a[t] = gload<v4i>(asrc[t] + (size_t)k16 * P.a_plane);
        }
    };

    v4i acc[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = v4i{0, 0, 0, 0};
    v4u w[WW][CT];
    v4i a[AD][RT];
    if (nu > 0) {
        // (codes first: they come from the L2, and loads complete in order)
        if constexpr (!AQ) {
#pragma unroll
            for (int j = 0; j < AD; ++j) load_a(j, a[j]);
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int i = 0; i < WW; ++i) load_w(i, w[i]);
    }

    // the epilogue's operands, requested under the weight stream; quad q =
    // columns 4 (q % 4)..+3 of column tile (q / 4) % OT of row q / (4 OT)
    constexpr int OT = EPI == EPI_PLAIN ? CT : CT / 2;  // output column tiles
    constexpr int QUADS = OT * 64 * RT, QPT = (QUADS + NT - 1) / NT;
    const int quad = tid & 3, qc = (tid >> 2) % OT;  // (NT is a multiple of 4 OT: the same for all of a thread's)
    const v4f cs = gload<v4f>(colscale + col0 + 16 * qc + 4 * quad);
    v4f cu;
    if constexpr (EPI != EPI_PLAIN) cu = gload<v4f>(colscale + col0 + 32 + 16 * qc + 4 * quad);
    if constexpr (!AQ) {
        if (tid < 16 * RT) {
            const int src = row_of(tid);
            s_rs[tid] = P.rowscale[src];
            s_rc[tid] = BITS == 4 ? 8 * P.rowsum[src] : 0;
        }
    }
#pragma unroll
    for (int i = tid; i < RT * CT * 64; i += NT) reinterpret_cast<v4i*>(sums)[i] = v4i{0, 0, 0, 0};

    if constexpr (AQ) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = wave + 4 * i;
            if (row < nrows) {
                const float m = wave_max(pm[i]);
                if (lane == 0) {
                    s_rs[row] = quant_scale<QUANT_MOE>(m);
                    s_rc[row] = 0;
                }
            }
        }
        __syncthreads();
        for (int task = tid; task < tasks; task += NT) {
            const int r = task / KG, kg = task - r * KG;
            const bool in = kg * 16 < P.K;
            if (task != tid) load16_raw(in ? mid + (size_t)r * P.K + kg * 16 : mid, raw);
            float v[16];
            cvt16_raw(raw, v, float());
#pragma unroll
            for (int b = 0; b < 16; ++b) v[b] = in ? v[b] : 0.0f;
            int sum = 0;
            *reinterpret_cast<v4u*>(s_codes + (kg * 16 + r) * 16) = quant_chunk<QUANT_MOE>(v, 1.0f / s_rs[r], sum);
            if constexpr (BITS == 4) atomicAdd(&s_rc[r], 8 * sum);
        }
        __syncthreads();
        if (nu > 0) {
#pragma unroll
            for (int j = 0; j < AD; ++j) load_a(j, a[j]);
        }
    }

    const bool ragged = BITS == 4 && (planes & 3) != 0;
    auto window = [&](int base) {
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
                const int s = i * HN + h, slot = s % AD;
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const v4i wv = __builtin_bit_cast(
                        v4i, BITS == 8 ? w[i][c] : (h == 0 ? (w[i][c] & 0x0F0F0F0Fu) : ((w[i][c] >> 4) & 0x0F0F0F0Fu)));
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        acc[t][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[slot][t], wv, acc[t][c], 0, 0, 0);
                }
                if (REFILL || s + AD < STEPS) load_a(base * HN + s + AD, a[slot]);
            }
            if constexpr (REFILL) load_w(base + i + WW, w[i]);
        }
    };
    if constexpr (REFILL) {
        for (int base = 0; base < nu; base += WW) window(base);
    } else {
        window(0);
    }
    __syncthreads();  // (the sums are cleared, the rows' scales are there)
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
    for (int i = 0; i < QPT; ++i) {
        const int q = tid + i * NT;
        if (q >= QUADS) break;
        const int local = q / (4 * OT);
        // accumulator layout: row 4 (lane / 16) + r of the tile, column lane % 16
        const int at = ((local >> 4) * CT * 4 + (local & 3)) * 64 + ((local >> 2) & 3) * 16 + 4 * quad;
        const v4i s0 = *reinterpret_cast<const v4i*>(&sums[at + qc * 256]);
        const float rs = s_rs[local];
        const int rc = BITS == 4 ? s_rc[local] : 0;
                float y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = ((float)(s0[j] - rc) * rs) * cs[j];
        const int slot = begin + local;
        if constexpr (EPI != EPI_PLAIN) {
            const v4i s1 = *reinterpret_cast<const v4i*>(&sums[at + (qc + 2) * 256]);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = hm_swiglu(y[j], ((float)(s1[j] - rc) * rs) * cu[j]);
            // the row's 32 outputs sit in 8 neighbouring lanes
            const float mx = max8(fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3]))));
            if (local < nrows) {
                if ((tid & 7) == 0) P.part[(size_t)slot * P.tiles_n + tn] = mx;
                *reinterpret_cast<float4*>(P.c + (size_t)slot * P.ldc + tn * 32 + 16 * qc + 4 * quad) =
                    float4{y[0], y[1], y[2], y[3]};
            }
        } else if (local < nrows) {
            const int p = col0 + 16 * qc + 4 * quad;  // packed column
            const size_t o = (size_t)slot * P.ldc + orig_col(p, P.half);
            const int valid = min(4, P.N - p);
            if (P.staged && valid == 4) {
                *reinterpret_cast<float4*>(P.c + o) = float4{y[0], y[1], y[2], y[3]};
            } else {
                for (int j = 0; j < valid; ++j) P.c[o + j] = y[j];
            }
        }
    }
}

template <int BITS, int EPI, int RTM, int WW, bool REFILL, bool AQ>
__global__ __launch_bounds__(STREAM_NT, (RTM == 1 ? 4 : 3) - REFILL) void moe_stream_kernel(MoeStreamParams P) {
    static_assert(!AQ || RTM == 1, "a block quantizes one row tile");
    __shared__ __attribute__((aligned(16))) int sums[RTM * STREAM_CT * 256];  // [row tile][col tile][row % 4][lane]
    __shared__ float s_rs[16 * RTM];
    __shared__ int s_rc[16 * RTM];
    extern __shared__ __attribute__((aligned(16))) int8_t s_codes[];  // AQ: [K_pad / 16][16 rows][16]
    // XCD x (block % 8) takes the row tiles x, x + 8, ..., all column tiles of
    // one row tile in a row (as moe_gemm_kernel): its rows come from one L2.
    const int i = blockIdx.x >> 3;
    const int t = (blockIdx.x & 7) + 8 * (i / P.tiles_n), tn = i % P.tiles_n;
    const int4 tile = P.tiles[min(t, P.max_tiles - 1)];  // (requested along with the count)
    if (t >= P.counts[1]) return;
    const int e = tile.x, begin = tile.y, nrows = tile.z - tile.y;
    if (RTM == 1 || nrows <= 16)
        moe_stream_body<BITS, EPI, 1, WW, REFILL, AQ>(P, e, begin, nrows, tn, sums, s_rs, s_rc, s_codes);
    else if constexpr (RTM == 3) {
        if (nrows <= 32)
            moe_stream_body<BITS, EPI, 2, WW, REFILL, AQ>(P, e, begin, nrows, tn, sums, s_rs, s_rc, s_codes);
        else
            moe_stream_body<BITS, EPI, 3, WW, REFILL, AQ>(P, e, begin, nrows, tn, sums, s_rs, s_rc, s_codes);
    }
}

// Whether a wave's share of K stays in its weight window (no reloads).
inline bool stream_holds(int bits, int K_pad) {
    const int units = (K_pad / (bits == 8 ? 16 : 32) + 3) / 4;
    return units <= 4 * STREAM_NWV;
}

// Launchers (launch_moe_stream.hip). bm: 16 or 48, the routing tile.
void launch_moe_front(int bm, const RouteParams& R, const TokenQuant& Q, hipStream_t s);
void launch_moe_stream(int bits, int epi, int bm, bool aq, const MoeStreamParams& P, int tiles, hipStream_t s);

}  // namespace hm
