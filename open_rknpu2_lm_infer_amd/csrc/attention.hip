// FP16 grouped-query attention over a device KV cache: the rk_npu_attention_f16
// C ABI (include/rk_npu_attention_f16.h) and its kernels.
//
// Layout in HBM: a cache holds K and V as [kv_heads][capacity][head_dim] fp16
// (one contiguous head_dim row per key). A run takes Q as
// [query_heads][rows][head_dim] fp16 and writes [query_heads][rows][head_dim]
// f32 or fp16. Math is f32: q is scaled by softmax_scale on load, scores are
// f32 dot products, the softmax is online (running max and sum, the
// accumulators rescaled when the max grows), and the output is the
// accumulated sum of p * v divided by the sum of p.
//
// Work split: block = (key split, tile of RT query rows, KV head). The query
// rows of one KV head are its (query head of the group, query row) pairs, so
// the group's heads share every K/V tile read. A block streams 64-key tiles
// of K and V through LDS; where the rows give fewer blocks than CUs, the keys
// are spread over splits whose partial (max, sum, accumulators) a second
// launch combines. Three kernels (plan_attention): attn_tile_kernel, the
// general one; attn_wide_kernel, many rows over many keys; attn_split_kernel,
// a row or four of head_dim 256 over few keys.

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>

#include "../../include/rk_npu_attention_f16.h"
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wunused-function"  // (the header's other kernels)
#include "kernels.hpp"
#pragma clang diagnostic pop
#include "launch.hpp"
#include "runtime.hpp"

namespace hm {

constexpr uint32_t MAGIC_ATTN_CACHE = 0x43414841u;
constexpr uint32_t MAGIC_ATTN_WORK = 0x57414841u;
constexpr int ATTN_KT = 64;              // keys per tile
constexpr int ATTN_MAX_SPLITS = 256;     // key splits per (KV head, row tile)
// Partial rows a workspace holds: when it splits the keys, plan_attention
// launches fewer than 512 blocks of 64 or 128 query rows, or 1024 of 32 or 4
// (head_dim 256: 64 rows at most).
static inline size_t attn_partial_rows(int head_dim) { return (size_t)2048 * (head_dim <= 128 ? 64 : 16); }

struct AttnParams {
    const __half* q;  // [qh][m][D]
    const __half* k;  // [kh][cap][D]
    const __half* v;
    void* out;        // [qh][m][D], f32 or fp16
    int out_f16;
    float* part;      // [kh][row_tiles*RT][splits][D + 2]: max, sum, accumulators
    int qh, kh, m, cap, len, pos, causal;
    float scale;
    int splits, keys_per_split, row_tiles, key_end;
    int rows_pad;     // row_tiles * RT: partial rows per KV head
    float max_unit;   // the partials' maxima in powers of 2: 1 (base 2) or log2(e) (natural)
};

// max / sum over a wave
__device__ __forceinline__ float lanes_max(float v) {
    v = fmaxf(v, dpp_move<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp_move<DPP_QUAD_XOR2>(v));
    v = fmaxf(v, dpp_move<DPP_ROW_HALF_MIRROR>(v));
    v = fmaxf(v, dpp_move<DPP_ROW_MIRROR>(v));
    v = fmaxf(v, dpp_move<DPP_ROW_BCAST15, 0xa>(v));
    v = fmaxf(v, dpp_move<DPP_ROW_BCAST31, 0xc>(v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float lanes_sum(float v) {
    v = v + dpp_move<DPP_QUAD_XOR1>(v);
    v = v + dpp_move<DPP_QUAD_XOR2>(v);
    v = v + dpp_move<DPP_ROW_HALF_MIRROR>(v);
    v = v + dpp_move<DPP_ROW_MIRROR>(v);
    v = v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), DPP_ROW_BCAST15, 0xa,
                                                                  0xf, false));
    v = v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), DPP_ROW_BCAST31, 0xc,
                                                                  0xf, false));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// An output that came out NaN, of query row qrow (within its head) of KV head g
// with weights' sum l. An infinity among the values it sees makes it that
// infinity; the kernels' sums hold NaN then wherever a weight of 0 met it: the
// remainder of a weight split in two, a key past the split, a split's weight.
// NaN stays where a weight or a value is NaN or the infinities have both signs.
__device__ __forceinline__ float nan_output(const AttnParams& P, int g, int qrow, int D, int dim, float l) {
    const __half* v = P.v + (size_t)g * P.cap * D + dim;
    const int keys = l == l ? (P.causal ? min(P.len, P.pos + qrow + 1) : P.len) : 0;
    bool up = false, down = false, nan = false;
    for (int j = 0; j < keys && !nan; j += 16) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {  // (one memory round trip for 16 keys)
            const unsigned b = reinterpret_cast<const unsigned short*>(v)[(size_t)min(j + u, keys - 1) * D];
            up |= b == 0x7C00u;
            down |= b == 0xFC00u;
            nan |= (b & 0x7FFFu) > 0x7C00u;
        }
    }
    return nan || up == down ? NAN : up ? INFINITY : -INFINITY;
}

// At most 4 rows of head_dim 256 over few keys. Block: 4 query rows, a wave
// each. Lane sub scores key sub of each tile of 32 and owns output dims 4 sub..+3
// of its row. K/V tiles go through LDS; the next tile's loads are in flight
// (registers) while the current tile is computed. What is left here is launch and
// latency: one row of 4-head groups over 1000 keys of 8 KV heads 8.7 us, on
// attn_tile_kernel 9.2; over 300 7.2 and 8.3. Scores are v_dot2_f32_f16 sums over
// the fp16 q and k pairs (exact products, f32 accumulation) times the scale; p * v
// folds the fp16 conversion into the multiply-add.
__global__ __launch_bounds__(256) void attn_split_kernel(AttnParams P) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    constexpr int D = 256, RT = 4;
    constexpr int KT = 32;                   // keys per tile
    constexpr int DPT = D / 64;              // output dims per lane
    constexpr int KP = D + 8;                // LDS row pitch of a K/V tile (halves)
    constexpr int PER = KT * (D / 8) / 256;  // 16-byte K (and V) pieces per thread per tile
    constexpr int QPT = RT * D / 256;        // q halves per thread
    constexpr int QW = QPT / 2;              // q words per thread
    __shared__ __attribute__((aligned(16))) __half qs[RT][D];
    __shared__ __attribute__((aligned(16))) __half ks[KT][KP];
    __shared__ __attribute__((aligned(16))) __half vs[KT][KP];
    __shared__ float ps[RT][KT];
    const int split = blockIdx.x, rt = blockIdx.y, g = blockIdx.z;
    const int G = P.qh / P.kh, R = G * P.m;
    const int tid = threadIdx.x, row = tid / 64, sub = tid % 64;
    const int rr = rt * RT + row;
    const bool row_ok = rr < R;
    const int gi = row_ok ? rr / P.m : 0, qr = row_ok ? rr % P.m : 0;
    int klimit = P.len;  // keys [0, klimit) are visible to this row
    if (P.causal) klimit = min(klimit, P.pos + qr + 1);
    const int k0 = split * P.keys_per_split;
    const int k1 = min(k0 + P.keys_per_split, P.key_end);
    const __half* kbase = P.k + (size_t)g * P.cap * D;
    const __half* vbase = P.v + (size_t)g * P.cap * D;
    // q: thread's QPT halves of the [RT][D] tile, one load (rows past R: 0)
    const int qe = tid * QPT, qrow = qe / D, qcol = qe % D, qrr = rt * RT + qrow;
    const bool q_ok = qrr < R;
    const __half* qsrc = P.q + ((size_t)(g * G + (q_ok ? qrr / P.m : 0)) * P.m + (q_ok ? qrr % P.m : 0)) * D + qcol;
    unsigned qv[QW];
#pragma unroll
    for (int i = 0; i < QW; ++i) qv[i] = reinterpret_cast<const unsigned*>(qsrc)[i];
    v4u kr[PER], vr[PER];
    auto issue = [&](int kb) {
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int i = tid + 256 * t, j = i / (D / 8), c = i % (D / 8), key = kb + j;
            const bool ok = key < k1;
            const size_t off = ok ? (size_t)key * D + c * 8 : 0;  // (masked: a valid row, zeroed at the store)
            kr[t] = *reinterpret_cast<const v4u*>(kbase + off);
            vr[t] = *reinterpret_cast<const v4u*>(vbase + off);
        }
    };
    auto store = [&](int kb) {
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int i = tid + 256 * t, j = i / (D / 8), c = i % (D / 8), key = kb + j;
            const bool ok = key < k1;
            *reinterpret_cast<v4u*>(&ks[j][c * 8]) = ok ? kr[t] : v4u{0u, 0u, 0u, 0u};
            *reinterpret_cast<v4u*>(&vs[j][c * 8]) = ok ? vr[t] : v4u{0u, 0u, 0u, 0u};
        }
    };
    if (k0 < k1) issue(k0);
#pragma unroll
    for (int i = 0; i < QW; ++i) reinterpret_cast<unsigned*>(&qs[qrow][qcol])[i] = q_ok ? qv[i] : 0u;
    float mrun = -INFINITY, lrun = 0.0f;
    float acc[DPT];
#pragma unroll
    for (int e = 0; e < DPT; ++e) acc[e] = 0.0f;
    for (int kb = k0; kb < k1; kb += KT) {
        __syncthreads();  // (the previous tile's reads are done)
        store(kb);
        __syncthreads();
        if (kb + KT < k1) issue(kb + KT);  // next tile in flight during this one
        float a = 0.0f;
        if (sub < KT) {
#pragma unroll 4
            for (int c = 0; c < D; c += 8) {
                const v4u kw = *reinterpret_cast<const v4u*>(&ks[sub][c]);
                const v4u qw = *reinterpret_cast<const v4u*>(&qs[row][c]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const unsigned qu = qw[e], ku = kw[e];  // (copied out before the bit casts)
                    a = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, qu), __builtin_bit_cast(h2, ku), a, false);
                }
            }
        }
        const int key = kb + sub;
        const float s = (row_ok && sub < KT && key < klimit && key < k1) ? a * P.scale : -INFINITY;
        const float mnew = fmaxf(mrun, lanes_max(s));
        // (a row with no visible key yet keeps max -inf, sum 0, scale 1)
        const float alpha = (mnew == -INFINITY) ? 1.0f : __expf(mrun - mnew);
        const float p = (s == -INFINITY) ? 0.0f : __expf(s - mnew);
        if (sub < KT) ps[row][sub] = p;
        lrun = lrun * alpha + lanes_sum(p);
        mrun = mnew;
#pragma unroll
        for (int e = 0; e < DPT; ++e) acc[e] *= alpha;
        __syncthreads();  // (p written)
#pragma unroll 4
        for (int j = 0; j < KT; ++j) {
            const float p = ps[row][j];
#pragma unroll
            for (int e = 0; e < DPT; ++e) acc[e] = __builtin_fmaf(p, __half2float(vs[j][sub * DPT + e]), acc[e]);
        }
    }
    if (!row_ok) return;
    const int h = g * G + gi;
    if (P.splits == 1) {
        const float inv = 1.0f / lrun;
        const size_t o = ((size_t)h * P.m + qr) * D + sub * DPT;
#pragma unroll
        for (int e = 0; e < DPT; ++e) {
            const float y = acc[e] * inv;
            if (P.out_f16)
                static_cast<__half*>(P.out)[o + e] = __float2half_rn(y);
            else
                static_cast<float*>(P.out)[o + e] = y;
        }
        return;
    }
    float* part = P.part + (((size_t)g * P.rows_pad + rr) * P.splits + split) * (D + 2);
    if (sub == 0) {
        part[0] = mrun;
        part[1] = lrun;
    }
#pragma unroll
    for (int e = 0; e < DPT; ++e) part[2 + sub * DPT + e] = acc[e];
}

// Many rows over many keys (head_dim 64 or 128). Block = 8 waves, each owning
// 16 query rows of one KV head, over 64-key tiles of its key split; the K/V
// tile is shared by the block. Per tile, with v_mfma_f32_16x16x32_f16 (fp16
// operands, f32 accumulation):
//   S^T = K Q^T   A = K rows from LDS, B = Q fragments held in registers;
//                 the accumulator gives lane l the raw scores of query row
//                 l%16 for keys 4(l/16)..+3 of each 16-key block,
//   softmax       weights p = 2^(s c - m) with c = scale * log2(e) and m the
//                 row's running max in those units, rounded to fp16 in place;
//                 m moves only when a row's max grows by more than ATTN_LAZY
//                 (so p <= 2^ATTN_LAZY, which fp16 holds), and only then are
//                 the accumulators and sums rescaled: each lane compares the
//                 max of its own 16 scores with that bound, and the row max
//                 over the row's 4 lanes is formed only when one passes it,
//   O^T += V^T P^T  A = V^T fragments, B = the weights as they lie (the
//                 accumulator layout of S^T is the B layout of P^T once each
//                 lane's 8 k-slots name keys {4(l/16)..+3, 16+4(l/16)..+3} of
//                 a 32-key step, which the A fragments are read to match),
// so a lane's O^T accumulators all belong to its own query row and every
// rescale is lane-local; each lane keeps a partial sum of its own weights
// (v_dot2 against ones: the fp16 weights summed exactly in f32), added over
// the row's 4 lanes at the end. Masks (causal, keys past the split) apply
// only on tiles that cross them.
// Tiles reach LDS by direct global->LDS loads into three buffers, K and V
// row-major (key, dim) in 16-byte slots permuted within each row against bank
// conflicts; tile t + 2 is requested after tile t's last LDS reads, into the
// buffer of tile t - 1 (every wave has passed tile t's barrier, so it is
// free), one barrier per tile; V^T fragments come from transposing LDS reads
// (ds_read_b64_tr_b16).
// Against attn_tile_kernel, whose waves share a row group's keys: half the LDS
// writes and barriers per row and key, but 128 rows per block and twice the
// partial rows. 512 rows per KV head (8 heads of 128) over 4096 keys 25.0 us
// here, 26.9 there; 1024 over 16128 94 and 128; 512 over 2028 20.6 and 19.0.
// Operand layouts (16x16x32, wave64): A lane l = row l%16, k-slots
// 8(l/16)..+7; B lane l = column l%16, same k-slots; C lane l = rows
// 4(l/16)..+3 of column l%16.
constexpr float ATTN_LAZY = 8.0f;

// Max / sum over the 4 lanes l % 16 + 16 j (a query row's lanes in the
// accumulator layout), in each of them: v_permlane16_swap exchanges odd with
// even 16-lane rows and v_permlane32_swap the upper with the lower half, so
// each swap's two results are a lane pair 16 (then 32) apart, without an LDS
// round trip.
__device__ __forceinline__ float max_rows4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_rows4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

constexpr int ATTN_WIDE_WAVES = 8;
template <int D>
__global__ __launch_bounds__(64 * ATTN_WIDE_WAVES) void attn_wide_kernel(AttnParams P) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    typedef _Float16 hh2 __attribute__((ext_vector_type(2)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    constexpr int KT = ATTN_KT, KS = D / 32, NB = D / 16;
    constexpr int NW = ATTN_WIDE_WAVES, NT = 64 * NW;
    // 16-byte slots per row, bytes of one matrix of a tile, slots per thread
    // per matrix, tile buffers
    constexpr int SPR = D / 8, MAT = KT * D * 2, DPT = KT * SPR / NT, NBUF = 3;
    static_assert(D == 64 || D == 128, "head_dim 64 or 128");
    static_assert(KT == 64 && KT * SPR % NT == 0, "tile shape");
    __shared__ __attribute__((aligned(16))) uint8_t smem[NBUF * 2 * MAT];

    const int split = blockIdx.x, rt = blockIdx.y, g = blockIdx.z;
    const int G = P.qh / P.kh, R = G * P.m;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lo = lane & 15, hi = lane >> 4;
    const int k0 = split * P.keys_per_split;
    const int k1 = min(k0 + P.keys_per_split, P.key_end);
    const float c = P.scale * 1.4426950408889634f;
    const __half* kbase = P.k + (size_t)g * P.cap * D;
    const __half* vbase = P.v + (size_t)g * P.cap * D;
    // this lane's query row, its key limit and Q fragments
    const int rr = rt * (16 * NW) + wave * 16 + lo;
    const bool row_ok = rr < R;
    int lim = 0;
    if (row_ok) {
        lim = P.len;
        if (P.causal) lim = min(lim, P.pos + rr % P.m + 1);
    }
    // keys below `open` are visible to every row of this wave (rows past R
    // are discarded, so they do not count)
    int open = row_ok ? lim : 0x7fffffff;
    open = min(open, __shfl_xor(open, 1));
    open = min(open, __shfl_xor(open, 2));
    open = min(open, __shfl_xor(open, 4));
    open = min(open, __shfl_xor(open, 8));
    open = __builtin_amdgcn_readfirstlane(min(open, k1));  // (uniform: a scalar branch below)
    h8 qf[KS];
    {
        const __half* qp = P.q + ((size_t)(g * G + (row_ok ? rr / P.m : 0)) * P.m + (row_ok ? rr % P.m : 0)) * D;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const v4u x = row_ok ? *reinterpret_cast<const v4u*>(qp + 32 * k + 8 * hi) : v4u{0u, 0u, 0u, 0u};
            qf[k] = __builtin_bit_cast(h8, x);
        }
    }

    // Direct loads: slot c of row r lies at c ^ swk(r) (K: 16 consecutive
    // rows take 16 distinct slots of one logical column, which the score
    // fragments read per 16 lanes) or c ^ swv(r) (V: 8 consecutive rows take
    // distinct slot pairs 2c, 2c + 1, the 32 bytes of each of 8 rows a half
    // wave's transposing reads take).
    auto swk = [](int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); };
    auto swv = [](int r) { return D == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); };
    // this thread's slots: physical slot t * NT + tid of each matrix -> row,
    // and the logical slot (16-byte column) it holds
    int drow[DPT], dkc[DPT], dvc[DPT];
#pragma unroll
    for (int t = 0; t < DPT; ++t) {
        const int pslot = t * NT + tid, r = pslot / SPR, ps = pslot % SPR;
        drow[t] = r;
        dkc[t] = ps ^ swk(r);
        dvc[t] = ps ^ swv(r);
    }
    // keys past the split read the split's last key (finite data; masked)
    auto issue_dma = [&](int kb, int buf) {
        const char* kt = reinterpret_cast<const char*>(kbase + (size_t)kb * D);
        const char* vtp = reinterpret_cast<const char*>(vbase + (size_t)kb * D);
        const int last = k1 - 1 - kb;
        uint8_t* dst = smem + buf * 2 * MAT + (wave * 64) * 16;
#pragma unroll
        for (int t = 0; t < DPT; ++t) {
            const int r = min(drow[t], last);
            lds_dma16(kt + (r * D + dkc[t] * 8) * 2, dst + t * NT * 16);
            lds_dma16(vtp + (r * D + dvc[t] * 8) * 2, dst + MAT + t * NT * 16);
        }
    };

    f4 o[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) o[n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float mrun = -INFINITY, lpart = 0.0f;
    const hh2 ones = {(_Float16)1.0f, (_Float16)1.0f};
    if (k0 < k1) issue_dma(k0, 0);
    if (k0 + KT < k1) issue_dma(k0 + KT, 1);
    int buf = 0;
    for (int kb = k0; kb < k1; kb += KT) {
        const uint8_t* kst = smem + buf * 2 * MAT;
        const uint8_t* vst = kst + MAT;
        if (kb + KT < k1)
            wait_vmcnt<2 * DPT>();  // (this thread's loads of the tile have landed; the next tile's may not)
        else
            wait_vmcnt<0>();
        __syncthreads();  // (every thread's have)
        // (k outermost: the 4 key blocks' products are independent, so they
        // issue back to back instead of waiting on each other)
        f4 sacc[4];
        h8 ka[4][KS];
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                const void* src = kst + (cb * 16 + lo) * (D * 2) + ((4 * k + hi) ^ swk(lo)) * 16;
                ka[cb][k] = __builtin_bit_cast(h8, *reinterpret_cast<const v4u*>(src));
            }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) sacc[cb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
                sacc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[cb][k], qf[k], sacc[cb], 0, 0, 0);
        if (__builtin_expect(kb + KT > open, 0)) {  // (uniform) the tile crosses a mask
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = kb + cb * 16 + 4 * hi + r;
                    if (!(key < lim && key < k1)) sacc[cb][r] = -INFINITY;
                }
        }
        // the lane's max of its 16 scores (3-input maxima); the row max only
        // when some lane's max passes its row's bound
        float lmax = -INFINITY;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
            lmax = __builtin_elementwise_maximum(
                __builtin_elementwise_maximum(lmax, __builtin_elementwise_maximum(sacc[cb][0], sacc[cb][1])),
                __builtin_elementwise_maximum(sacc[cb][2], sacc[cb][3]));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(lmax * c > mrun + ATTN_LAZY) != 0, 0)) {  // (uniform)
            const float tm = max_rows4(lmax) * c;
            float alpha = 1.0f;
            if (tm > mrun + ATTN_LAZY) {
                alpha = __builtin_amdgcn_exp2f(mrun - tm);  // (0 from -inf)
                mrun = tm;
            }
            lpart *= alpha;
#pragma unroll
            for (int n = 0; n < NB; ++n) o[n] *= alpha;
        }
        const float msub = (mrun == -INFINITY) ? 0.0f : mrun;  // (no visible key yet: all scores -inf)
        h8 pb[2];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[cb][r], c, -msub));
                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[cb][r + 1], c, -msub));
                const hh2 ph = {(_Float16)p0, (_Float16)p1};
                pb[cb >> 1][(cb & 1) * 4 + r] = ph[0];
                pb[cb >> 1][(cb & 1) * 4 + r + 1] = ph[1];
                lpart = __builtin_amdgcn_fdot2(ph, ones, lpart, false);
            }
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {  // (k outermost: the NB products are independent)
            h8 va[NB];
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                // transposing reads: lane j of a 16-lane group names dims
                // 4 (j % 4)..+3 of key row 4 (j / 4) of the group's 16
                // keys; lane i receives dim i of the rows named by lanes
                // i / 4, 4 + i / 4, 8 + i / 4, 12 + i / 4: its dim of keys
                // 4 hi..+3 (then of keys 16 + 4 hi..+3) of the step
                const int vr0 = 32 * k + 4 * hi + (lo >> 2);
                const uint8_t* p =
                    vst + vr0 * (D * 2) + (((2 * n + ((lo & 3) >> 1)) ^ swv(vr0)) * 16) + (lo & 1) * 8;
                const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
                const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + 16 * (D * 2)));
                const u2 ua = __builtin_bit_cast(u2, a), ub = __builtin_bit_cast(u2, b);
                va[n] = __builtin_bit_cast(h8, v4u{ua[0], ua[1], ub[0], ub[1]});
            }
#pragma unroll
            for (int n = 0; n < NB; ++n) o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[n], pb[k], o[n], 0, 0, 0);
        }
        // (the compiler waits for every direct load in flight before a
        // transposing read, so the request comes after this tile's)
        if (kb + 2 * KT < k1) issue_dma(kb + 2 * KT, buf == 0 ? NBUF - 1 : buf - 1);
        buf = buf == NBUF - 1 ? 0 : buf + 1;
    }
    float l = lpart;
    l = sum_rows4(l);
    if (!row_ok) return;
    const int h = g * G + rr / P.m, qr = rr % P.m;
    if (P.splits == 1) {
        const float inv = 1.0f / l;
        const size_t o0 = ((size_t)h * P.m + qr) * D + 4 * hi;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const f4 y = o[n] * inv;
            if (P.out_f16) {
                const unsigned short b0 = __half_as_ushort(__float2half_rn(y[0]));
                const unsigned short b1 = __half_as_ushort(__float2half_rn(y[1]));
                const unsigned short b2 = __half_as_ushort(__float2half_rn(y[2]));
                const unsigned short b3 = __half_as_ushort(__float2half_rn(y[3]));
                *reinterpret_cast<u2*>(static_cast<__half*>(P.out) + o0 + 16 * n) =
                    u2{b0 | ((unsigned)b1 << 16), b2 | ((unsigned)b3 << 16)};
            } else {
                *reinterpret_cast<f4*>(static_cast<float*>(P.out) + o0 + 16 * n) = y;
            }
        }
    } else {
        float* part = P.part + (((size_t)g * P.rows_pad + rr) * P.splits + split) * (D + 2);
        if (hi == 0) {
            part[0] = mrun;
            part[1] = l;
        }
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[2 + 16 * n + 4 * hi + r] = o[n][r];
    }
}

// The general kernel: block = WR x WK waves; wave (wr, wk) owns 16 query rows
// of one KV head and, of every stage of 32 WK keys, the 32 keys 32 wk..+31, so
// WK waves share a row group's keys and their partial (max, sum, accumulators)
// meet in LDS at the end; waves whose rows or keys are all masked skip their
// products. Operands and lane layouts are attn_wide_kernel's: S^T = K Q^T,
// softmax in place, O^T += V^T P^T with transposing V reads. Stages go global ->
// registers -> one of two LDS buffers: stage t + 1 is in registers while stage t
// is computed, then stored to the buffer stage t - 1 left (every wave passed the
// barrier after it), one barrier per stage.
//
// SPLIT: the softmax weights keep f32's precision on the fp16 matrix cores as
// a sum of two fp16 (p = ph + pl, pl = the rounded remainder: 22 bits of p),
// two products per V fragment into the same accumulator, and the weights' sum
// is taken in f32 before the split. They are scaled by 2^ATTN_SHIFT (which
// leaves in the division), so that with the lazy maximum p stays below 2^15
// and what the remainder loses below fp16's smallest value is 2^-32 of the
// row's largest weight. Against 64 bits the outputs are nearer than the VALU
// kernels' whose place this took (f32 weights, v_dot2 scores): 128 rows of 8-head
// groups of 256 over 2048 keys 3.0e-7 (5.8e-7), one row of 128 over 16000
// 2.9e-7 (4.4e-7). Over 147 shapes of one to 800 rows per KV head, 65 to 16000
// keys and every head_dim, each at three spreads of the scores, the error is
// 0.59 times theirs (geometric mean; largest at normal q and k 4.6e-7, theirs
// 1.4e-6). An infinite value leaves NaN with a remainder of 0 or below;
// nan_output puts that right.
//
// Calls that had fp16 weights keep them (SPLIT = false). There the maximum is not
// lazy over a wave's first two stages, 64 keys: the largest weight among them is
// then exactly 1, as in the 64-key tiles of the 4-wave blocks these calls had.
// With a lazy one its rounding showed: 1.13 times those blocks' error against 64
// bits on 64 rows of 8 heads over 4000 keys, 3.9 times with 4 times wider scores.
// Now at most the same over 78 shapes of 16 to 800 rows per KV head at normal q and k
// (0.94 times, geometric mean), in the same time (those 64 rows with their append
// 16.6 and 16.5 us, 512 rows over 2000 keys 20.3 and 20.4); exact to the end of
// longer chains they take up to 5% longer.
//
// Measured per run with its combine, us, the kernels before -> this (one row =
// one query row, so 4 or 8 rows per KV head):
//   head_dim 256, 16 heads / 2 KV, 128 rows x 2048 keys       112.5 -> 25.7
//                 64 / 8, 128 rows x 8128                      1633 -> 138
//                 16 / 2, 1 row x 16000                        26.0 -> 14.8
//   head_dim 128, 32 / 8, 1 row x 3968                          9.1 ->  8.4
//                 16 / 8, 1 row x 16000                        20.6 -> 16.6
//                 32 / 8, 3 rows x 3970                        14.1 ->  9.3
//                 32 / 8, 16 rows x 4016                       17.6 -> 14.4
//                 32 / 8, 32 rows x 2032                       17.9 -> 13.5
//   head_dim 64,  16 / 8, 1 row x 16000                        14.4 ->  9.7
// At few rows it is launches and one or two memory round trips; at many, the
// LDS reads of a fragment per 16 rows, the exponentials and the products,
// which the two waves of a SIMD overlap only in part (head_dim 256: about 2 us
// per 64 keys of a 64-row block, the 138 us above being 64 such stages). RW = 2 (a
// fragment read serves 32 rows) and 4-wave blocks of 64 or 128 rows were slower at
// every size tried.
constexpr float ATTN_SHIFT = 7.0f;

template <int D, int WR, int WK, bool SPLIT>
__global__ __launch_bounds__(64 * WR * WK) void attn_tile_kernel(AttnParams P) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    // (q and out of any element alignment)
    typedef unsigned q16 __attribute__((ext_vector_type(4), aligned(2)));
    typedef unsigned o8 __attribute__((ext_vector_type(2), aligned(2)));
    typedef float o16 __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int KS = D / 32, NB = D / 16, NT = 64 * WR * WK, RT = 16 * WR;
    constexpr int KT = 32 * WK;                     // keys per stage
    constexpr int SPR = D / 8, MAT = KT * D * 2;    // 16-byte slots per row, bytes of K (V) per stage
    constexpr int PT = KT * SPR / NT;               // slots per thread and matrix
    // two stage buffers, and the merge's maxima and sums (its accumulators lie
    // in the stage buffer that the last stage does not use)
    constexpr int WAVES1 = (WK - 1) * WR, SMEM = 4 * MAT + WAVES1 * 512;
    constexpr float SHIFT = SPLIT ? ATTN_SHIFT : 0.0f;
    static_assert(KT * SPR % NT == 0 && SMEM <= 160 * 1024 && WAVES1 * NB * 1024 <= 2 * MAT, "stage shape");
    __shared__ __attribute__((aligned(16))) uint8_t smem[SMEM];

    const int split = blockIdx.x, rt = blockIdx.y, g = blockIdx.z;
    const int G = P.qh / P.kh, R = G * P.m;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave % WR, wk = wave / WR;
    const int lo = lane & 15, hi = lane >> 4;
    const int k0 = split * P.keys_per_split;
    const int k1 = min(k0 + P.keys_per_split, P.key_end);
    const float c = P.scale * 1.4426950408889634f;
    const __half* kbase = P.k + (size_t)g * P.cap * D;
    const __half* vbase = P.v + (size_t)g * P.cap * D;
    // slot of (row, 16-byte column) in a K / V tile: permuted within the row
    // as in attn_wide_kernel's tiles
    auto swk = [](int r) { return D >= 128 ? (r & 15) : ((r >> 1) & 7); };
    auto swv = [](int r) { return D >= 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); };

    auto issue = [&](int kb, v4u (&kr)[PT], v4u (&vr)[PT]) {
        const int last = k1 - 1 - kb;  // (keys past the split read its last key, masked)
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            const int i = t * NT + tid;
            const size_t off = (size_t)(kb + min(i / SPR, last)) * D + (i % SPR) * 8;
            kr[t] = *reinterpret_cast<const v4u*>(kbase + off);
            vr[t] = *reinterpret_cast<const v4u*>(vbase + off);
        }
    };
    auto store = [&](int buf, const v4u (&kr)[PT], const v4u (&vr)[PT]) {
        uint8_t* dst = smem + buf * 2 * MAT;
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            const int i = t * NT + tid, r = i / SPR, col = i % SPR;
            *reinterpret_cast<v4u*>(dst + r * (D * 2) + (col ^ swk(r)) * 16) = kr[t];
            *reinterpret_cast<v4u*>(dst + MAT + r * (D * 2) + (col ^ swv(r)) * 16) = vr[t];
        }
    };

    v4u kr[PT], vr[PT], k0r[PT], v0r[PT];
    if (k0 < k1) issue(k0, k0r, v0r);
    // this lane's query row, its key limit and Q fragments
    const int rr = rt * RT + wr * 16 + lo;
    const bool ok = rr < R;
    int lim = 0;
    if (ok) lim = P.causal ? min(P.len, P.pos + rr % P.m + 1) : P.len;
    // keys below `open` are visible to every row of the wave (rows past R are
    // discarded and do not count), keys from `seen` on to none. (causal: the
    // rows' places in their heads run from `first` to `last`)
    const int r0 = rt * RT + wr * 16, rows = min(16, R - r0);
    int open = min(P.len, k1), seen = rows > 0 ? open : 0;
    if (P.causal && rows > 0) {
        const int at = r0 % P.m;
        const bool one = at + rows <= P.m;  // (all of one head)
        const int first = one ? at : 0, last = one ? at + rows - 1 : P.m - 1;
        open = min(open, P.pos + first + 1);
        seen = min(seen, P.pos + last + 1);
    }
    h8 qf[KS];
    const __half* qp = P.q + ((size_t)(g * G + (ok ? rr / P.m : 0)) * P.m + (ok ? rr % P.m : 0)) * D;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const v4u x = ok ? v4u(*reinterpret_cast<const q16*>(qp + 32 * k + 8 * hi)) : v4u{0u, 0u, 0u, 0u};
        qf[k] = __builtin_bit_cast(h8, x);
    }
    if (k0 + KT < k1) issue(k0 + KT, kr, vr);
    if (k0 < k1) store(0, k0r, v0r);

    f4 o[NB];
    float mrun = -INFINITY, lpart = 0.0f;  // (mrun: the row's maximum less SHIFT)
#pragma unroll
    for (int n = 0; n < NB; ++n) o[n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    int buf = 0;
    for (int kb = k0; kb < k1; kb += KT) {
        const uint8_t* kst = smem + buf * 2 * MAT + wk * (32 * D * 2);
        const uint8_t* vst = kst + MAT;
        const int key0 = kb + 32 * wk;
        if (key0 < seen) {  // (wave-uniform)
            f4 sacc[2] = {f4{0.0f, 0.0f, 0.0f, 0.0f}, f4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) {
                    const h8 ka = __builtin_bit_cast(
                        h8, *reinterpret_cast<const v4u*>(kst + (cb * 16 + lo) * (D * 2) + ((4 * k + hi) ^ swk(lo)) * 16));
                    sacc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qf[k], sacc[cb], 0, 0, 0);
                }
            h8 ph, pl;
            if (__builtin_expect(key0 + 32 > open, 0)) {  // (uniform) the tile crosses a mask
#pragma unroll
                for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = key0 + cb * 16 + 4 * hi + r;
                        if (!(key < lim && key < k1)) sacc[cb][r] = -INFINITY;
                    }
            }
            // (the maximum follows the scores from this rise on)
            const float lazy = SPLIT || kb >= k0 + 2 * KT ? ATTN_LAZY : 0.0f;
            float lmax = -INFINITY;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
                lmax = __builtin_elementwise_maximum(
                    __builtin_elementwise_maximum(lmax, __builtin_elementwise_maximum(sacc[cb][0], sacc[cb][1])),
                    __builtin_elementwise_maximum(sacc[cb][2], sacc[cb][3]));
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(lmax * c > mrun + (lazy + SHIFT)) != 0, 0)) {
                const float tm = max_rows4(lmax) * c - SHIFT;
                float alpha = 1.0f;
                if (tm > mrun + lazy) {
                    alpha = __builtin_amdgcn_exp2f(mrun - tm);  // (0 from -inf)
                    mrun = tm;
                }
                lpart *= alpha;
#pragma unroll
                for (int n = 0; n < NB; ++n) o[n] *= alpha;
            }
            const float msub = (mrun == -INFINITY) ? 0.0f : mrun;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[cb][r], c, -msub));
                    const _Float16 h = (_Float16)p;
                    ph[cb * 4 + r] = h;
                    if constexpr (SPLIT) {
                        pl[cb * 4 + r] = (_Float16)(p - (float)h);
                        lpart += p;
                    } else {
                        lpart += (float)h;
                    }
                }
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                // transposing reads (as attn_wide_kernel's)
                const int r0 = 4 * hi + (lo >> 2);
                const uint8_t* p = vst + r0 * (D * 2) + (((2 * n + ((lo & 3) >> 1)) ^ swv(r0)) * 16) + (lo & 1) * 8;
                const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
                const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + 16 * (D * 2)));
                const u2 ua = __builtin_bit_cast(u2, a), ub = __builtin_bit_cast(u2, b);
                const h8 va = __builtin_bit_cast(h8, v4u{ua[0], ua[1], ub[0], ub[1]});
                o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph, o[n], 0, 0, 0);
                if constexpr (SPLIT) o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl, o[n], 0, 0, 0);
            }
        }
        if (kb + KT < k1) {
            store(buf ^ 1, kr, vr);
            if (kb + 2 * KT < k1) issue(kb + 2 * KT, kr, vr);
            __syncthreads();
        }
        buf ^= 1;
    }

    if constexpr (WK > 1) {
        // the key groups' partials: waves wk > 0 leave theirs in LDS, wave
        // (wr, 0) adds them
        // (the stage buffer `buf` is free: the last stage uses the other one)
        uint8_t* acc1 = smem + buf * 2 * MAT;
        float* ml1 = reinterpret_cast<float*>(smem + 4 * MAT) + lane;
        if (wk > 0) {
            const int w = (wk - 1) * WR + wr;
#pragma unroll
            for (int n = 0; n < NB; ++n) *reinterpret_cast<f4*>(acc1 + ((w * NB + n) * 64 + lane) * 16) = o[n];
            ml1[w * 128] = mrun;
            ml1[w * 128 + 64] = lpart;
        }
        __syncthreads();
        if (wk > 0) return;
#pragma unroll
        for (int g1 = 1; g1 < WK; ++g1) {
            const int w = (g1 - 1) * WR + wr;
            const float m1 = ml1[w * 128], l1 = ml1[w * 128 + 64], m = fmaxf(mrun, m1);
            const float a0 = mrun == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrun - m);
            const float a1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - m);
            mrun = m;
            lpart = lpart * a0 + l1 * a1;
#pragma unroll
            for (int n = 0; n < NB; ++n)
                o[n] = o[n] * a0 + *reinterpret_cast<const f4*>(acc1 + ((w * NB + n) * 64 + lane) * 16) * a1;
        }
    }
    const float l = sum_rows4(lpart);
    if (rr >= R) return;
    if (P.splits == 1) {
        const float inv = 1.0f / l;
        const size_t o0 = ((size_t)(g * G + rr / P.m) * P.m + rr % P.m) * D + 4 * hi;
        float sum = 0.0f;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            o[n] *= inv;
            sum += (o[n][0] + o[n][1]) + (o[n][2] + o[n][3]);
        }
        if (__builtin_expect(sum != sum, 0)) {
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (o[n][r] != o[n][r]) o[n][r] = nan_output(P, g, rr % P.m, D, 16 * n + 4 * hi + r, l);
        }
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const f4 y = o[n];
            if (P.out_f16) {
                const unsigned short b0 = __half_as_ushort(__float2half_rn(y[0]));
                const unsigned short b1 = __half_as_ushort(__float2half_rn(y[1]));
                const unsigned short b2 = __half_as_ushort(__float2half_rn(y[2]));
                const unsigned short b3 = __half_as_ushort(__float2half_rn(y[3]));
                *reinterpret_cast<o8*>(static_cast<__half*>(P.out) + o0 + 16 * n) =
                    o8{b0 | ((unsigned)b1 << 16), b2 | ((unsigned)b3 << 16)};
            } else {
                *reinterpret_cast<o16*>(static_cast<float*>(P.out) + o0 + 16 * n) = y;
            }
        }
    } else {
        float* part = P.part + (((size_t)g * P.rows_pad + rr) * P.splits + split) * (D + 2);
        if (hi == 0) {
            part[0] = mrun;
            part[1] = l;
        }
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[2 + 16 * n + 4 * hi + r] = o[n][r];
    }
}

// Combine the key splits of one (KV head, row): block = (row, KV head).
// Thread t takes split t for the max M and the weight w_t = e^(m_t - M) (or
// 2^, as the maxima are kept: max_unit; 0 for a split that saw no key) and the
// denominator sum_t w_t l_t; then wave w
// takes splits w, w + 4, ... for all head dims (lane + 64 j), loading up to 16
// splits at once so their latencies overlap; the 4 waves' sums meet in LDS:
// out = sum_s w_s acc_s / sum_s w_s l_s.
template <int D>
__global__ __launch_bounds__(256) void attn_combine_kernel(AttnParams P) {
    constexpr int ND = D / 64;  // dims per lane
    constexpr int B = 16;       // splits loaded at once per wave
    constexpr size_t STRIDE = D + 2;
    static_assert(ATTN_MAX_SPLITS <= 256, "one thread per split");
    __shared__ float w_s[256];
    __shared__ float red[2][4];
    __shared__ float sums[4][D];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rr = blockIdx.x, g = blockIdx.y;
    const int G = P.qh / P.kh, R = G * P.m;
    if (rr >= R) return;  // (block-uniform)
    const int h = g * G + rr / P.m, qr = rr % P.m;
    const int S = P.splits;
    const float* p0 = P.part + ((size_t)g * P.rows_pad + rr) * S * STRIDE;
    // the first batch of accumulators is requested with the maxima and sums
    // (its addresses do not depend on them: one memory round trip)
    float v[B][ND];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int sp = min(wave + 4 * u, S - 1);
#pragma unroll
        for (int d = 0; d < ND; ++d) v[u][d] = p0[sp * STRIDE + 2 + lane + 64 * d];
    }
    const float m = tid < S ? p0[tid * STRIDE] : -INFINITY;
    const float l = tid < S ? p0[tid * STRIDE + 1] : 0.0f;
    float mx = lanes_max(m);
    if (lane == 0) red[0][wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    const float w = (m == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m - mx) * P.max_unit);
    w_s[tid] = w;
    const float den = lanes_sum(w * l);
    if (lane == 0) red[1][wave] = den;
    __syncthreads();
    float num[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) num[d] = 0.0f;
    for (int s0 = wave; s0 < S; s0 += 4 * B) {
        if (s0 != wave) {
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int sp = min(s0 + 4 * u, S - 1);
#pragma unroll
                for (int d = 0; d < ND; ++d) v[u][d] = p0[sp * STRIDE + 2 + lane + 64 * d];
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int sp = s0 + 4 * u;
            const float wi = sp < S ? w_s[sp] : 0.0f;
#pragma unroll
            for (int d = 0; d < ND; ++d) num[d] = __builtin_fmaf(wi, v[u][d], num[d]);
        }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) sums[wave][lane + 64 * d] = num[d];
    __syncthreads();
    if (wave == 0) {
        const float inv = 1.0f / ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
        const size_t o = ((size_t)h * P.m + qr) * D + lane;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const int dd = lane + 64 * d;
            float y = ((sums[0][dd] + sums[1][dd]) + (sums[2][dd] + sums[3][dd])) * inv;
            if (__builtin_expect(y != y, 0)) y = nan_output(P, g, qr, D, dd, inv);
            if (P.out_f16)
                static_cast<__half*>(P.out)[o + 64 * d] = __float2half_rn(y);
            else
                static_cast<float*>(P.out)[o + 64 * d] = y;
        }
    }
}

// The same combine for few splits (at most 64) over many rows: one wave per
// row, lane s holds split s's weight; the splits' accumulators are loaded B
// (8 or 16) at a time (dims lane + 64 j) and each weight is broadcast from
// its lane.
template <int D, int B>
__global__ __launch_bounds__(256) void attn_combine_rows_kernel(AttnParams P) {
    constexpr int ND = D / 64;
    constexpr size_t STRIDE = D + 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rr = blockIdx.x * 4 + wave, g = blockIdx.y;
    const int G = P.qh / P.kh, R = G * P.m;
    if (rr >= R) return;  // (wave-uniform; no barrier below)
    const int h = g * G + rr / P.m, qr = rr % P.m;
    const int S = P.splits;
    const float* p0 = P.part + ((size_t)g * P.rows_pad + rr) * S * STRIDE;
    // the first 16 splits' accumulators are loaded together with the maxima
    // and sums (one memory round trip for up to 16 splits)
    float v[B][ND];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int sp = min(u, S - 1);
#pragma unroll
        for (int d = 0; d < ND; ++d) v[u][d] = p0[sp * STRIDE + 2 + lane + 64 * d];
    }
    const float m = lane < S ? p0[lane * STRIDE] : -INFINITY;
    const float l = lane < S ? p0[lane * STRIDE + 1] : 0.0f;
    const float mx = lanes_max(m);
    const float w = (m == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m - mx) * P.max_unit);
    const float den = lanes_sum(w * l);
    float num[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) num[d] = 0.0f;
    for (int s0 = 0; s0 < S; s0 += B) {
        if (s0 > 0) {
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int sp = min(s0 + u, S - 1);
#pragma unroll
                for (int d = 0; d < ND; ++d) v[u][d] = p0[sp * STRIDE + 2 + lane + 64 * d];
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            // (lanes past S hold weight 0)
            const float wi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), s0 + u));
#pragma unroll
            for (int d = 0; d < ND; ++d) num[d] = __builtin_fmaf(wi, v[u][d], num[d]);
        }
    }
    const float inv = 1.0f / den;
    const size_t o = ((size_t)h * P.m + qr) * D + lane;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        float y = num[d] * inv;
        if (__builtin_expect(y != y, 0)) y = nan_output(P, g, qr, D, lane + 64 * d, den);
        if (P.out_f16)
            static_cast<__half*>(P.out)[o + 64 * d] = __float2half_rn(y);
        else
            static_cast<float*>(P.out)[o + 64 * d] = y;
    }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
// Device-path work (rk_npu_hip_attention_cache_append / _run, enqueued on the
// caller's streams) that a later host call on the same cache or workspace must
// wait for. The host call waits for events after that work, not for the whole
// device:
// - work on the null stream: the event is recorded by the first wait after it.
//   An event costs 4.3 us of the stream's time (its cache flush and signal), a
//   decode step noted three, 25.8 -> 13.6 us without them, and the null stream
//   exists until the process ends and is never captured, so it can be recorded
//   on at any later time;
// - work on another stream, which its owner may destroy or capture afterwards:
//   recorded at once. Work from a second such stream while the first's is still
//   pending, or work under graph capture (whose replays the host cannot see),
//   makes the next wait a device-wide synchronize instead.
struct DevFence {
    std::mutex mu;
    hipEvent_t ev = nullptr;
    hipEvent_t null_ev = nullptr;
    hipStream_t last = nullptr;
    bool used = false;       // ev holds the last work of a stream other than the null stream
    bool null_used = false;  // null_ev holds the null stream's work up to the last wait
    bool null_new = false;   // there is null-stream work since
    bool broad = false;      // wait for the whole device next time

    static bool create(hipEvent_t& e) {
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            e = nullptr;
        }
        return e != nullptr;
    }
    static bool record(hipEvent_t e, hipStream_t s) {
        if (hipEventRecord(e, s) == hipSuccess) return true;
        (void)hipGetLastError();
        return false;
    }
    // Note device-path work just enqueued on stream s.
    void note(hipStream_t s) {
        std::lock_guard<std::mutex> lock(mu);
        if (!s) {
            null_new = true;
            return;
        }
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            broad = true;
            return;
        }
        if (used && s != last) {
            const hipError_t q = hipEventQuery(ev);
            (void)hipGetLastError();  // (not-ready is an answer, not an error)
            if (q != hipSuccess) broad = true;
        }
        if (!create(ev) || !record(ev, s)) {
            broad = true;
            return;
        }
        used = true;
        last = s;
    }
    // Order stream s after the noted work (s == nullptr: the host waits).
    hipError_t wait(hipStream_t s) {
        std::lock_guard<std::mutex> lock(mu);
        if (null_new && !broad) {
            if (create(null_ev) && record(null_ev, nullptr)) {
                null_used = true;
                null_new = false;
            } else {
                broad = true;
            }
        }
        if (broad) {
            const hipError_t e = hipDeviceSynchronize();
            if (e == hipSuccess) broad = used = null_used = null_new = false;
            return e;
        }
        hipError_t e = hipSuccess;
        if (used) e = s ? hipStreamWaitEvent(s, ev, 0) : hipEventSynchronize(ev);
        if (e == hipSuccess && null_used) e = s ? hipStreamWaitEvent(s, null_ev, 0) : hipEventSynchronize(null_ev);
        return e;
    }
    void destroy() {
        if (ev) (void)hipEventDestroy(ev);
        if (null_ev) (void)hipEventDestroy(null_ev);
        ev = null_ev = nullptr;
    }
};

struct AttnCache {
    uint32_t magic;
    Domain* domain;
    rk_npu_attention_f16_config cfg;
    __half* k;
    __half* v;
    int length, capacity;
    size_t bytes_each;  // of k and of v
    uint64_t generation;  // bumped whenever the K/V storage is replaced or reloaded
    DevFence fence;       // device-path appends (writes) and runs (reads) of the rows
    hipStream_t stream = nullptr;  // host-buffer appends (created on the first)
    HostStage hs;                  // their pinned staging
};

struct AttnWork {
    uint32_t magic;
    Domain* domain;
    rk_npu_attention_f16_config cfg;
    __half* q;     // host-call staging [qh][max_query_rows][D]
    float* out;    // host-call staging (f32; fp16 output uses the first half)
    float* part;   // split partials
    size_t q_bytes, out_bytes, part_bytes;
    hipStream_t stream;
    std::atomic<bool> busy;
    DevFence fence;  // device-path runs writing this workspace's partials
    HostStage hs;    // pinned staging of host-buffer runs
};

// The reference's checks (src/npu.rs:714-728) plus this library's limits.
static bool valid_config(const rk_npu_attention_f16_config* c) {
    if (!c) return false;
    const int d = c->head_dim;
    return c->kv_heads >= 1 && c->kv_heads <= 32 && c->query_heads >= c->kv_heads &&
           c->query_heads % c->kv_heads == 0 && c->query_heads <= 256 && d > 0 && d % 32 == 0 && d <= 256 &&
           std::isfinite(c->softmax_scale) && c->softmax_scale > 0.0f && c->max_query_rows >= 1 &&
           c->max_query_rows <= 256 && c->max_capacity >= 1 && c->initial_capacity >= 0 &&
           c->initial_capacity <= c->max_capacity &&
           (c->mask_mode == RK_NPU_ATTENTION_F16_CAUSAL || c->mask_mode == RK_NPU_ATTENTION_F16_NO_MASK);
}

// Head dims with a kernel instantiation.
static bool supported_dim(int d) { return d == 64 || d == 128 || d == 256; }

static size_t kv_bytes(const rk_npu_attention_f16_config* c, int capacity) {
    return (size_t)c->kv_heads * (size_t)capacity * c->head_dim * sizeof(__half);
}

static size_t part_bytes(const rk_npu_attention_f16_config* c) {
    return attn_partial_rows(c->head_dim) * (size_t)(c->head_dim + 2) * sizeof(float);
}

static AttnCache* as_cache(void* p) {
    AttnCache* c = static_cast<AttnCache*>(p);
    return (c && c->magic == MAGIC_ATTN_CACHE) ? c : nullptr;
}
static AttnWork* as_attn_work(void* p) {
    AttnWork* w = static_cast<AttnWork*>(p);
    return (w && w->magic == MAGIC_ATTN_WORK) ? w : nullptr;
}

// Grow to `capacity` rows (multiple of 32), keeping the rows held.
static int cache_grow(AttnCache* c, int capacity) {
    capacity = round_up(capacity, 32);
    if (capacity <= c->capacity) return RK_NPU_OK;
    if (capacity > round_up(c->cfg.max_capacity, 32)) return RK_NPU_ERR_PARAM;
    const size_t nb = kv_bytes(&c->cfg, capacity);
    __half* nk = static_cast<__half*>(domain_alloc(c->domain, nb));
    __half* nv = nk ? static_cast<__half*>(domain_alloc(c->domain, nb)) : nullptr;
    if (!nk || !nv) {
        domain_free(c->domain, nk, nb);
        return RK_NPU_ERR_NOMEM;
    }
    const size_t row = (size_t)c->cfg.head_dim * sizeof(__half);
    bool ok = true;
    if (c->length > 0) {
        ok = hipMemcpy2D(nk, capacity * row, c->k, (size_t)c->capacity * row, (size_t)c->length * row,
                         c->cfg.kv_heads, hipMemcpyDeviceToDevice) == hipSuccess &&
             hipMemcpy2D(nv, capacity * row, c->v, (size_t)c->capacity * row, (size_t)c->length * row,
                         c->cfg.kv_heads, hipMemcpyDeviceToDevice) == hipSuccess;
    }
    if (!ok) {
        domain_free(c->domain, nk, nb);
        domain_free(c->domain, nv, nb);
        return RK_NPU_ERR_DEVICE;
    }
    domain_free(c->domain, c->k, c->bytes_each);
    domain_free(c->domain, c->v, c->bytes_each);
    c->k = nk;
    c->v = nv;
    c->capacity = capacity;
    c->generation += 1;
    c->bytes_each = nb;
    return RK_NPU_OK;
}

// Copy `rows` rows per KV head ([kv_heads][rows][D]) after the rows held.
static int cache_put(AttnCache* c, const void* k, const void* v, int rows, hipMemcpyKind kind, hipStream_t s,
                     bool async) {
    const size_t row = (size_t)c->cfg.head_dim * sizeof(__half);
    const size_t dpitch = (size_t)c->capacity * row, spitch = (size_t)rows * row;
    __half* dk = c->k + (size_t)c->length * c->cfg.head_dim;
    __half* dv = c->v + (size_t)c->length * c->cfg.head_dim;
    hipError_t e1, e2;
    if (async) {
        e1 = hipMemcpy2DAsync(dk, dpitch, k, spitch, spitch, c->cfg.kv_heads, kind, s);
        e2 = hipMemcpy2DAsync(dv, dpitch, v, spitch, spitch, c->cfg.kv_heads, kind, s);
    } else {
        e1 = hipMemcpy2D(dk, dpitch, k, spitch, spitch, c->cfg.kv_heads, kind);
        e2 = hipMemcpy2D(dv, dpitch, v, spitch, spitch, c->cfg.kv_heads, kind);
    }
    if (e1 != hipSuccess || e2 != hipSuccess) return RK_NPU_ERR_DEVICE;
    c->length += rows;
    return RK_NPU_OK;
}

// Append: rows of K (blockIdx.z 0) and V (1), [kv_heads][rows][D] each, into
// the rows [length, length + rows) of every head (blockIdx.y), 16 bytes per
// thread and step. One launch where two 2-D copies took one each (a decode
// step's two copies 4.5 us apiece on the stream).
__global__ __launch_bounds__(256) void attn_append_kernel(const v4u* __restrict__ ksrc, const v4u* __restrict__ vsrc,
                                                          v4u* __restrict__ k, v4u* __restrict__ v, int pieces,
                                                          size_t head_pieces, size_t first) {
    const v4u* src = (blockIdx.z ? vsrc : ksrc) + (size_t)blockIdx.y * pieces;
    v4u* dst = (blockIdx.z ? v : k) + (size_t)blockIdx.y * head_pieces + first;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) dst[i] = src[i];
}

// Whether a kernel on `device` may read caller memory at p: that GPU's own.
// Another GPU's (readable only where peer access is on), managed and host
// memory (pageable memory faults a kernel) keep the copies, which the runtime
// checks and stages.
static bool kernel_readable(const void* p, int device) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeDevice && a.device == device;
}

// Launches it for `rows` rows whose K and V lie at 16-byte aligned device (or
// mapped host) addresses; the caller advances the length.
static void enqueue_append(AttnCache* c, const void* k, const void* v, int rows, hipStream_t s) {
    const int row_pieces = c->cfg.head_dim / 8, pieces = rows * row_pieces;
    hipLaunchKernelGGL(attn_append_kernel, dim3(std::min(1024, (pieces + 255) / 256), c->cfg.kv_heads, 2), dim3(256), 0,
                       s, static_cast<const v4u*>(k), static_cast<const v4u*>(v), reinterpret_cast<v4u*>(c->k),
                       reinterpret_cast<v4u*>(c->v), pieces, (size_t)c->capacity * row_pieces,
                       (size_t)c->length * row_pieces);
}

// Appends host rows through the cache's pinned stage and stream, returning
// once they are in the cache (the stage's completion word); false when the
// stage path is not available (the caller copies directly).
static bool cache_put_staged(AttnCache* c, const void* k, const void* v, int rows, int& rc) {
    const int kh = c->cfg.kv_heads, D = c->cfg.head_dim;
    const size_t each = (size_t)kh * rows * D * sizeof(__half), voff = round_up_z(each, 256);
    if (!host_kernels_enabled()) return false;
    if (!c->stream && hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        (void)hipGetLastError();
        c->stream = nullptr;
        return false;
    }
    void* st = stage_reserve(c->hs, voff + each);
    if (!st) return false;
    std::memcpy(st, k, each);
    std::memcpy(static_cast<uint8_t*>(st) + voff, v, each);
    enqueue_append(c, c->hs.dev, static_cast<const uint8_t*>(c->hs.dev) + voff, rows, c->stream);
    if (hipGetLastError() != hipSuccess || !stage_download(c->hs, true, st, nullptr, nullptr, 0, c->stream)) {
        (void)hipStreamSynchronize(c->stream);
        rc = RK_NPU_ERR_DEVICE;
        return true;
    }
    c->length += rows;
    rc = RK_NPU_OK;
    return true;
}

enum AttnKernel { ATTN_VALU, ATTN_TILE, ATTN_WIDE };
struct AttnPlan {
    AttnKernel kernel;
    int rt, row_tiles, splits, keys_per_split, key_end;
};

// Kernel and rows per tile, for the R = (heads of a group) x rows query rows
// of a KV head (measured per run, us):
// - head_dim 256: attn_tile_kernel of 64 rows; at most 4 rows over few keys
//   (10240 or less over all KV heads, 40 a CU) attn_split_kernel (8 heads of
//   1000 keys 8.7 against 9.2; 4 of 3000 10.5 against 9.7, 8 of 16000 34.3
//   against 28.3).
// - head_dim 64 and 128, R < 16: attn_tile_kernel of 32 rows, weights in 32
//   bits, 4 waves so that two blocks share a CU (one row of 4-head groups over
//   3968 keys 8.4; blocks of 16 rows 8.5, of 64 and 8 waves 9.3).
// - R >= 16: attn_tile_kernel of 64 rows, fp16 weights; more than 64 rows
//   attn_wide_kernel once a CU's share of the work passes 640 keys of a
//   64-row tile (8 heads: 512 rows x 2028 keys, 507 keys a CU, 20.6 wide and
//   19.0 tiles; 512 x 4096, 1024 keys, 25.0 and 26.9; 96 rows, two thirds of a
//   wide block, x 16000, 1000 keys, 23.8 and 26.3).
// Keys: enough splits that about 512 of the 4-wave blocks run, 256 of the
// 8-wave ones (one per CU), each split a whole number of tiles; with more than
// one split the blocks write partials (enqueue_attention checks that the
// workspace holds them).
// Overrides for measurement: HM_ATTN_BLOCKS, HM_ATTN_WIDE_BLOCKS (the block
// counts the key splits aim at).
static int attn_env(const char* name, int fallback) {
    const char* v = std::getenv(name);
    return v ? std::atoi(v) : fallback;
}

static AttnPlan plan_attention(const rk_npu_attention_f16_config& c, int rows, int len, int pos) {
    AttnPlan p;
    const int G = c.query_heads / c.kv_heads, R = G * rows;
    static const int env_blocks = attn_env("HM_ATTN_BLOCKS", 512);
    static const int env_wide = attn_env("HM_ATTN_WIDE_BLOCKS", 256);
    p.key_end = (c.mask_mode == RK_NPU_ATTENTION_F16_CAUSAL) ? std::min(len, pos + rows) : len;
    p.kernel = ATTN_TILE;
    if (c.head_dim == 256) {
        p.rt = 64;
        if (R <= 4 && (long long)c.kv_heads * p.key_end <= 40LL * device_cus()) {
            p.kernel = ATTN_VALU;
            p.rt = 4;
        }
    } else {
        p.rt = R < 16 ? 32 : 64;
        const long long tile_keys = (long long)((R + 63) / 64) * c.kv_heads * p.key_end;
        if (R > 64 && tile_keys > 640LL * device_cus()) {
            p.kernel = ATTN_WIDE;
            p.rt = 128;
        }
    }
    p.row_tiles = (R + p.rt - 1) / p.rt;
    const int kt = p.kernel == ATTN_VALU ? 32 : ATTN_KT;  // keys per tile of the kernel
    const int tiles = (p.key_end + kt - 1) / kt;
    const int base = p.row_tiles * c.kv_heads;
    // (head_dim 256: its partial rows hold 64-row tiles of 256 + base blocks)
    const int target = std::min(std::max(p.rt >= 64 ? env_wide : env_blocks, 64), c.head_dim == 256 && p.rt == 64 ? 256 : 1024);
    int want = base >= target ? 1 : (target + base - 1) / base;
    want = std::max(1, std::min(std::min(want, tiles), ATTN_MAX_SPLITS));
    const int tiles_per_split = (tiles + want - 1) / want;
    p.keys_per_split = tiles_per_split * kt;
    p.splits = (p.key_end + p.keys_per_split - 1) / p.keys_per_split;
    if (p.splits < 1) p.splits = 1;
    return p;
}

template <int D>
static void launch_attn(const AttnParams& P, const AttnPlan& pl, const dim3& grid, hipStream_t s) {
    if constexpr (D == 256) {
        if (pl.kernel == ATTN_VALU)
            hipLaunchKernelGGL(attn_split_kernel, grid, dim3(256), 0, s, P);
        else
            hipLaunchKernelGGL((attn_tile_kernel<256, 4, 2, true>), grid, dim3(512), 0, s, P);
    } else {
        if (pl.kernel == ATTN_WIDE)
            hipLaunchKernelGGL(attn_wide_kernel<D>, grid, dim3(64 * ATTN_WIDE_WAVES), 0, s, P);
        else if (pl.rt == 32)
            hipLaunchKernelGGL((attn_tile_kernel<D, 2, 2, true>), grid, dim3(256), 0, s, P);
        else
            hipLaunchKernelGGL((attn_tile_kernel<D, 4, 2, false>), grid, dim3(512), 0, s, P);
    }
}

static int enqueue_attention(AttnWork* w, AttnCache* c, const __half* q, int rows, int pos, void* out, int out_f16,
                             hipStream_t s) {
    const rk_npu_attention_f16_config& cfg = c->cfg;
    const bool causal = cfg.mask_mode == RK_NPU_ATTENTION_F16_CAUSAL;
    if (rows < 1 || rows > w->cfg.max_query_rows || pos < 0 || c->length < 1) return RK_NPU_ERR_PARAM;
    if (causal && (long)pos + rows > c->length) return RK_NPU_ERR_PARAM;
    const AttnPlan pl = plan_attention(cfg, rows, c->length, pos);
    if (pl.splits > 1 && (size_t)pl.row_tiles * pl.rt * cfg.kv_heads * pl.splits > attn_partial_rows(cfg.head_dim))
        return RK_NPU_ERR_UNSUPPORTED;
    AttnParams P;
    P.q = q;
    P.k = c->k;
    P.v = c->v;
    P.out = out;
    P.out_f16 = out_f16;
    P.part = w->part;
    P.qh = cfg.query_heads;
    P.kh = cfg.kv_heads;
    P.m = rows;
    P.cap = c->capacity;
    P.len = c->length;
    P.pos = pos;
    P.causal = causal ? 1 : 0;
    P.scale = cfg.softmax_scale;
    P.splits = pl.splits;
    P.keys_per_split = pl.keys_per_split;
    P.row_tiles = pl.row_tiles;
    P.key_end = pl.key_end;
    P.rows_pad = pl.row_tiles * pl.rt;
    P.max_unit = pl.kernel == ATTN_VALU ? 1.4426950408889634f : 1.0f;
    const int D = cfg.head_dim;
    const dim3 grid(pl.splits, pl.row_tiles, cfg.kv_heads);
    if (D == 64)
        launch_attn<64>(P, pl, grid, s);
    else if (D == 128)
        launch_attn<128>(P, pl, grid, s);
    else
        launch_attn<256>(P, pl, grid, s);
    if (pl.splits > 1) {
        const int G = cfg.query_heads / cfg.kv_heads;
        // few splits: a wave per row; many: a block per row (measured: 8
        // splits over 4096 rows 2 us faster by wave, 64 splits over 32 rows
        // 14 us faster by block)
        const bool by_wave = pl.splits <= 16;
        const dim3 cgrid(by_wave ? (G * rows + 3) / 4 : G * rows, cfg.kv_heads);
        if (by_wave) {
            // (splits loaded per batch: 8 when there are at most 8, else 16)
#define HM_COMB_ROWS(DD)                                                                            \
    if (pl.splits <= 8)                                                                             \
        hipLaunchKernelGGL((attn_combine_rows_kernel<DD, 8>), cgrid, dim3(256), 0, s, P);           \
    else                                                                                            \
        hipLaunchKernelGGL((attn_combine_rows_kernel<DD, 16>), cgrid, dim3(256), 0, s, P);
            if (D == 64) {
                HM_COMB_ROWS(64)
            } else if (D == 128) {
                HM_COMB_ROWS(128)
            } else {
                HM_COMB_ROWS(256)
            }
#undef HM_COMB_ROWS
        } else if (D == 64) {
            hipLaunchKernelGGL(attn_combine_kernel<64>, cgrid, dim3(256), 0, s, P);
        } else if (D == 128) {
            hipLaunchKernelGGL(attn_combine_kernel<128>, cgrid, dim3(256), 0, s, P);
        } else {
            hipLaunchKernelGGL(attn_combine_kernel<256>, cgrid, dim3(256), 0, s, P);
        }
    }
    return hipGetLastError() == hipSuccess ? RK_NPU_OK : RK_NPU_ERR_DEVICE;
}

static int run_host(rk_npu_attention_f16_workspace* workspace, rk_npu_attention_f16_cache* cache, const uint16_t* q,
                    int rows, int pos, void* out, int out_f16, rk_npu_attention_f16_timings* t, const void* reserved) {
    AttnWork* w = as_attn_work(workspace);
    AttnCache* c = as_cache(cache);
    if (!w || !c || !q || !out || reserved) return RK_NPU_ERR_PARAM;
    if (w->cfg.query_heads != c->cfg.query_heads || w->cfg.kv_heads != c->cfg.kv_heads ||
        w->cfg.head_dim != c->cfg.head_dim || w->cfg.mask_mode != c->cfg.mask_mode ||
        w->cfg.softmax_scale != c->cfg.softmax_scale)
        return RK_NPU_ERR_PARAM;
    if (rows < 1 || rows > w->cfg.max_query_rows) return RK_NPU_ERR_PARAM;
    bool expected = false;
    if (!w->busy.compare_exchange_strong(expected, true)) return RK_NPU_ERR_BUSY;
    const double t0 = now_us();
    const size_t n = (size_t)c->cfg.query_heads * rows * c->cfg.head_dim;
    int rc = RK_NPU_OK;
    // Device-path appends and runs (rk_npu_hip_attention_cache_append / _run)
    // are enqueued on the caller's streams and may still be writing the
    // cache's rows or this workspace's partials: this call's stream waits for
    // them first. q comes in and the output goes out through the workspace's
    // pinned stage (the kernel path of small calls, else copies and a wait).
    const size_t qb = n * sizeof(__half), ob = n * (out_f16 ? sizeof(__half) : sizeof(float));
    void* st = nullptr;
    bool small = false;
    if (hipSetDevice(device_of(w->domain)) != hipSuccess || c->fence.wait(w->stream) != hipSuccess ||
        w->fence.wait(w->stream) != hipSuccess) {
        rc = RK_NPU_ERR_DEVICE;
    } else {
        st = stage_reserve(w->hs, std::max(qb, ob));
        small = stage_small(w->hs, st, qb, ob);
        const HostSeg seg{q, w->q, qb, 0};
        if (!stage_upload(w->hs, small, st, &seg, 1, w->stream) ||
            (t && hipStreamSynchronize(w->stream) != hipSuccess))
            rc = RK_NPU_ERR_DEVICE;
    }
    const double t1 = now_us();
    if (rc == RK_NPU_OK) rc = enqueue_attention(w, c, w->q, rows, pos, w->out, out_f16, w->stream);
    if (rc == RK_NPU_OK && t && hipStreamSynchronize(w->stream) != hipSuccess) rc = RK_NPU_ERR_DEVICE;
    const double t2 = now_us();
    if (rc == RK_NPU_OK && !stage_download(w->hs, small, st, out, w->out, ob, w->stream)) rc = RK_NPU_ERR_DEVICE;
    if (rc != RK_NPU_OK) (void)hipStreamSynchronize(w->stream);
    const double t3 = now_us();
    if (t) {
        t->upload_us = t1 - t0;
        t->device_us = t2 - t1;
        t->download_us = t3 - t2;
        t->total_us = t3 - t0;
    }
    w->busy.store(false);
    return rc;
}

}  // namespace hm

using namespace hm;

extern "C" {

void rk_npu_attention_f16_config_init(rk_npu_attention_f16_config* c) {
    if (!c) return;
    std::memset(c, 0, sizeof(*c));
    c->query_heads = 32;
    c->kv_heads = 8;
    c->head_dim = 128;
    c->softmax_scale = 1.0f / std::sqrt(128.0f);
    c->max_query_rows = 128;
    c->max_capacity = 4096;
    c->initial_capacity = 128;
    c->kv_tile = 512;
    c->flags = RK_NPU_ATTENTION_F16_STABLE_SOFTMAX;
    c->mask_mode = RK_NPU_ATTENTION_F16_CAUSAL;
}

int rk_npu_attention_f16_query(const rk_npu_attention_f16_config* c, int32_t capacity, int32_t query_rows,
                               int32_t kv_capacity, rk_npu_attention_f16_sizes* sizes) {
    if (!valid_config(c) || !sizes || capacity < 0 || query_rows < 1 || query_rows > 256 || kv_capacity < 0)
        return RK_NPU_ERR_PARAM;
    const int cap = round_up(capacity, 32);
    sizes->key_bytes = kv_bytes(c, cap);
    sizes->value_bytes = kv_bytes(c, cap);
    sizes->tail_bytes = 0;
    sizes->workspace_bytes = (uint64_t)c->query_heads * query_rows * c->head_dim * (sizeof(__half) + sizeof(float)) +
                             part_bytes(c);
    sizes->active_core_mask = 1u;
    return RK_NPU_OK;
}

int rk_npu_attention_f16_prepare(rk_npu_iommu_domain* domain, const rk_npu_attention_f16_config* config,
                                 rk_npu_attention_f16_workspace** out) {
    if (out) *out = nullptr;
    Domain* d = static_cast<Domain*>(domain);
    if (!d || !out || !valid_config(config)) return RK_NPU_ERR_PARAM;
    if (!supported_dim(config->head_dim)) return RK_NPU_ERR_UNSUPPORTED;
    if (hipSetDevice(device_of(d)) != hipSuccess) return RK_NPU_ERR_DEVICE;
    AttnWork* w = new (std::nothrow) AttnWork();
    if (!w) return RK_NPU_ERR_NOMEM;
    w->magic = MAGIC_ATTN_WORK;
    w->domain = d;
    w->cfg = *config;
    w->busy.store(false);
    w->stream = nullptr;
    const size_t n = (size_t)config->query_heads * config->max_query_rows * config->head_dim;
    w->q_bytes = n * sizeof(__half);
    w->out_bytes = n * sizeof(float);
    w->part_bytes = part_bytes(config);
    w->q = static_cast<__half*>(domain_alloc(d, w->q_bytes));
    w->out = static_cast<float*>(domain_alloc(d, w->out_bytes));
    w->part = static_cast<float*>(domain_alloc(d, w->part_bytes));
    if (!w->q || !w->out || !w->part || hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking) != hipSuccess) {
        rk_npu_attention_f16_workspace_free(reinterpret_cast<rk_npu_attention_f16_workspace*>(w));
        return RK_NPU_ERR_NOMEM;
    }
    *out = reinterpret_cast<rk_npu_attention_f16_workspace*>(w);
    return RK_NPU_OK;
}

void rk_npu_attention_f16_workspace_free(rk_npu_attention_f16_workspace* workspace) {
    AttnWork* w = as_attn_work(workspace);
    if (!w) return;
    (void)hipSetDevice(device_of(w->domain));
    if (w->stream) {
        (void)hipStreamSynchronize(w->stream);
        (void)hipStreamDestroy(w->stream);
    }
    (void)w->fence.wait(nullptr);
    w->fence.destroy();
    stage_release(w->hs);
    domain_free(w->domain, w->q, w->q_bytes);
    domain_free(w->domain, w->out, w->out_bytes);
    domain_free(w->domain, w->part, w->part_bytes);
    w->magic = 0;
    delete w;
}

int rk_npu_attention_f16_cache_create(rk_npu_iommu_domain* domain, const rk_npu_attention_f16_config* config,
                                      rk_npu_attention_f16_cache** out) {
    if (out) *out = nullptr;
    Domain* d = static_cast<Domain*>(domain);
    if (!d || !out || !valid_config(config)) return RK_NPU_ERR_PARAM;
    if (!supported_dim(config->head_dim)) return RK_NPU_ERR_UNSUPPORTED;
    if (hipSetDevice(device_of(d)) != hipSuccess) return RK_NPU_ERR_DEVICE;
    AttnCache* c = new (std::nothrow) AttnCache();
    if (!c) return RK_NPU_ERR_NOMEM;
    c->magic = MAGIC_ATTN_CACHE;
    c->domain = d;
    c->cfg = *config;
    c->length = 0;
    c->generation = 0;
    c->capacity = std::max(32, round_up(config->initial_capacity, 32));
    c->bytes_each = kv_bytes(config, c->capacity);
    c->k = static_cast<__half*>(domain_alloc(d, c->bytes_each));
    c->v = c->k ? static_cast<__half*>(domain_alloc(d, c->bytes_each)) : nullptr;
    if (!c->k || !c->v) {
        rk_npu_attention_f16_cache_free(reinterpret_cast<rk_npu_attention_f16_cache*>(c));
        return RK_NPU_ERR_NOMEM;
    }
    *out = reinterpret_cast<rk_npu_attention_f16_cache*>(c);
    return RK_NPU_OK;
}

void rk_npu_attention_f16_cache_free(rk_npu_attention_f16_cache* cache) {
    AttnCache* c = as_cache(cache);
    if (!c) return;
    (void)hipSetDevice(device_of(c->domain));
    (void)c->fence.wait(nullptr);
    c->fence.destroy();
    if (c->stream) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamDestroy(c->stream);
    }
    stage_release(c->hs);
    domain_free(c->domain, c->k, c->bytes_each);
    domain_free(c->domain, c->v, c->bytes_each);
    c->magic = 0;
    delete c;
}

int rk_npu_attention_f16_cache_reserve(rk_npu_ctx* ctx, rk_npu_attention_f16_cache* cache, int32_t capacity) {
    AttnCache* c = as_cache(cache);
    if (!ctx || !c || capacity < 0) return RK_NPU_ERR_PARAM;
    if (hipSetDevice(device_of(c->domain)) != hipSuccess || c->fence.wait(nullptr) != hipSuccess)
        return RK_NPU_ERR_DEVICE;
    return cache_grow(c, capacity);
}

int rk_npu_attention_f16_cache_load(rk_npu_ctx* ctx, rk_npu_attention_f16_cache* cache, const uint16_t* k,
                                    const uint16_t* v, int32_t rows) {
    AttnCache* c = as_cache(cache);
    if (!ctx || !c || rows < 0 || (rows > 0 && (!k || !v))) return RK_NPU_ERR_PARAM;
    if (hipSetDevice(device_of(c->domain)) != hipSuccess || c->fence.wait(nullptr) != hipSuccess)
        return RK_NPU_ERR_DEVICE;
    c->length = 0;
    c->generation += 1;  // the contents are replaced (a reset when rows == 0)
    if (rows == 0) return RK_NPU_OK;
    int rc = cache_grow(c, rows);
    if (rc != RK_NPU_OK) return rc;
    return cache_put(c, k, v, rows, hipMemcpyHostToDevice, nullptr, false);
}

int rk_npu_attention_f16_cache_append(rk_npu_ctx* ctx, rk_npu_attention_f16_cache* cache, const uint16_t* k,
                                      const uint16_t* v, int32_t rows) {
    AttnCache* c = as_cache(cache);
    if (!ctx || !c || rows < 1 || !k || !v) return RK_NPU_ERR_PARAM;
    if ((long)c->length + rows > round_up(c->cfg.max_capacity, 32)) return RK_NPU_ERR_PARAM;
    if (hipSetDevice(device_of(c->domain)) != hipSuccess || c->fence.wait(nullptr) != hipSuccess)
        return RK_NPU_ERR_DEVICE;
    if (c->length + rows > c->capacity) {
        const int grown = std::min(round_up(c->cfg.max_capacity, 32), std::max(c->length + rows, 2 * c->capacity));
        int rc = cache_grow(c, grown);
        if (rc != RK_NPU_OK) return rc;
    }
    int rc = RK_NPU_OK;
    if (cache_put_staged(c, k, v, rows, rc)) return rc;
    return cache_put(c, k, v, rows, hipMemcpyHostToDevice, nullptr, false);
}

int rk_npu_attention_f16_cache_truncate(rk_npu_attention_f16_cache* cache, int32_t length) {
    AttnCache* c = as_cache(cache);
    if (!c || length < 0 || length > c->length) return RK_NPU_ERR_PARAM;
    c->length = length;
    return RK_NPU_OK;
}

int rk_npu_attention_f16_cache_get_info(const rk_npu_attention_f16_cache* cache,
                                        rk_npu_attention_f16_cache_info* info) {
    AttnCache* c = as_cache(const_cast<rk_npu_attention_f16_cache*>(cache));
    if (!c || !info) return RK_NPU_ERR_PARAM;
    info->length = c->length;
    info->capacity = c->capacity;
    info->max_capacity = round_up(c->cfg.max_capacity, 32);
    info->generation = c->generation;
    info->key_bytes = c->bytes_each;
    info->value_bytes = c->bytes_each;
    info->tail_bytes = 0;
    return RK_NPU_OK;
}

int rk_npu_attention_f16_run(rk_npu_ctx* ctx, rk_npu_attention_f16_workspace* workspace,
                             rk_npu_attention_f16_cache* cache, const uint16_t* q, int32_t rows, int32_t position,
                             float* output, rk_npu_attention_f16_timings* timings, const void* reserved) {
    if (!ctx) return RK_NPU_ERR_PARAM;
    return run_host(workspace, cache, q, rows, position, output, 0, timings, reserved);
}

int rk_npu_attention_f16_run_half(rk_npu_ctx* ctx, rk_npu_attention_f16_workspace* workspace,
                                  rk_npu_attention_f16_cache* cache, const uint16_t* q, int32_t rows,
                                  int32_t position, uint16_t* output, rk_npu_attention_f16_timings* timings,
                                  const void* reserved) {
    if (!ctx) return RK_NPU_ERR_PARAM;
    return run_host(workspace, cache, q, rows, position, output, 1, timings, reserved);
}

int rk_npu_hip_attention_cache_append(rk_npu_attention_f16_cache* cache, const void* k_dev, const void* v_dev,
                                      int32_t rows, void* stream) {
    AttnCache* c = as_cache(cache);
    if (!c || rows < 1 || !k_dev || !v_dev) return RK_NPU_ERR_PARAM;
    if ((long)c->length + rows > c->capacity) return RK_NPU_ERR_PARAM;  // (reserve first: no allocation here)
    if (hipSetDevice(device_of(c->domain)) != hipSuccess) return RK_NPU_ERR_DEVICE;
    int rc;
    if (((reinterpret_cast<uintptr_t>(k_dev) | reinterpret_cast<uintptr_t>(v_dev)) & 15) == 0 &&
        kernel_readable(k_dev, device_of(c->domain)) && kernel_readable(v_dev, device_of(c->domain))) {
        enqueue_append(c, k_dev, v_dev, rows, static_cast<hipStream_t>(stream));
        rc = hipGetLastError() == hipSuccess ? RK_NPU_OK : RK_NPU_ERR_DEVICE;
        if (rc == RK_NPU_OK) c->length += rows;
    } else {
        rc = cache_put(c, k_dev, v_dev, rows, hipMemcpyDeviceToDevice, static_cast<hipStream_t>(stream), true);
    }
    if (rc == RK_NPU_OK) c->fence.note(static_cast<hipStream_t>(stream));
    return rc;
}

int rk_npu_hip_attention_run(rk_npu_attention_f16_workspace* workspace, rk_npu_attention_f16_cache* cache,
                             const void* q_dev, int32_t rows, int32_t position, void* out_dev, int32_t out_f16,
                             void* stream) {
    AttnWork* w = as_attn_work(workspace);
    AttnCache* c = as_cache(cache);
    if (!w || !c || !q_dev || !out_dev) return RK_NPU_ERR_PARAM;
    if (w->cfg.query_heads != c->cfg.query_heads || w->cfg.kv_heads != c->cfg.kv_heads ||
        w->cfg.head_dim != c->cfg.head_dim || w->cfg.mask_mode != c->cfg.mask_mode ||
        w->cfg.softmax_scale != c->cfg.softmax_scale)
        return RK_NPU_ERR_PARAM;
    if (hipSetDevice(device_of(w->domain)) != hipSuccess) return RK_NPU_ERR_DEVICE;
    const int rc = enqueue_attention(w, c, static_cast<const __half*>(q_dev), rows, position, out_dev,
                                     out_f16 ? 1 : 0, static_cast<hipStream_t>(stream));
    if (rc == RK_NPU_OK) {
        c->fence.note(static_cast<hipStream_t>(stream));
        w->fence.note(static_cast<hipStream_t>(stream));
    }
    return rc;
}

}  // extern "C"
