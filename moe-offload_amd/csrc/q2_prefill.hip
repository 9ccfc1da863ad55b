// Grouped Q2 SwitchGLU for chunked prefill on gfx950 (MFMA).
//
// Reference semantics: mlx-qwen38/loader.py:566-699 (CachedSwitchGLU prefill: the (token, k)
// rows sorted by expert, chunk-local slot = rank of the expert in the chunk),
// prefill_qproj.py:18-40 (gather_qmm over the sorted rows), cpp/src/layers.cpp:364-600.
// For the sorted rows r of segment u (one expert, weights = blob seg_slot[u] of the pool):
//     h_r = silu(G_u x_r) * (U_u x_r)        (fp16 out)
//     y_r = D_u h_r                          (fp16 out, row row_out[r])
// with W = scale * q + bias per group of 64 inputs (2-bit codes, 16 per u32, LSB first).
//
// Tiling.  The rows of a segment form M tiles of 16 (v_mfma_f32_16x16x32_f16).  k_q2g_mm takes up to
// 64 rows of a segment per pass over its weights, with their activations staged in LDS for the whole
// K and, for all but short calls, a fixed grid whose blocks split the work evenly.  With few rows per
// expert the whole-K forms run: gate/up at K = 2048 in k_q2g_gu_wk (per M tile, each wave's weight
// subtiles requested over the whole K at once, the tile's activations staged once), both products at
// K = 512 and up to K = 256 in k_q2g_wk (each wave's 4 subtiles loaded once and kept in registers while
// the segment's M tiles pass through LDS).  All but the last with K <= 256 for down have a grid that
// holds every (segment, slice) item twice: segments of several passes run in the first half, so their
// blocks, the longest, are dispatched before the rest.
//
// Dequantisation.  A 2-bit code in the low bits of a nibble is the fp4 (e2m1) value q/2, so
// w & 0x33333333 (even codes) and (w >> 2) & 0x33333333 (odd codes) are 8 fp4 values each;
// v_cvt_scalef32_pk_f16_fp4 with scale 2 turns a byte into two exact halves q, and one v_pk_fma_f16
// with (scale, bias) gives the fp16 weight scale*q + bias rounded once (MLX's dequantised weight).
//
// K order.  Inside an MFMA the K positions are permuted identically for A and B: the even codes
// of a 32-bit word pair with activations [x0 x2 .. x14] of its 16 inputs and the odd codes with
// [x1 x3 .. x15]; the activation halves are regrouped in registers with v_perm_b32.
//
// Weight sources (SBF): 0 = the blob pool, (scale, bias) interleaved as fp16 words; 1 / 2 = the
// reference's 9 tensors (loader.py:332-406: codes, scales, biases in pools of their own), scales and
// biases fp16 / bf16, turned into the same (scale, bias) fp16 words as they are loaded (bf16 ->
// fp16 is exact for the normal range of fp16).
#include <hip/hip_fp16.h>

#include <type_traits>

#include "moe_common.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMT = 16;          // rows per M tile
constexpr int kMaxChunks = 10;   // K <= 2560
constexpr int kGateUp = 0, kDown = 1;

// Block index -> work item, keeping consecutive work items on one XCD (blocks are dealt to the
// 8 XCDs round robin), so the blocks of one segment share that XCD's L2 for the activations.
__device__ __forceinline__ int xcd_order(int b, int nb) {
    const int per = nb / 8, rem = nb % 8, x = b % 8, i = b / 8;
    return x < rem ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// Codes of one 32-bit word (8 of them: bits already masked to the low two bits of every nibble) ->
// 8 fp16 weights scale * q + bias.  sb = (scale, bias) as one fp16 pair.
__device__ __forceinline__ f16x8 dequant8(uint32_t bits, uint32_t sb) {
    const f16x2 p = __builtin_bit_cast(f16x2, sb);
    const f16x2 s2 = {p.x, p.x}, b2 = {p.y, p.y};
    f16x2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(bits, 2.0f, 0);
    f16x2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(bits, 2.0f, 1);
    f16x2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(bits, 2.0f, 2);
    f16x2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(bits, 2.0f, 3);
    a = __builtin_elementwise_fma(a, s2, b2);
    b = __builtin_elementwise_fma(b, s2, b2);
    c = __builtin_elementwise_fma(c, s2, b2);
    d = __builtin_elementwise_fma(d, s2, b2);
    return (f16x8){a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// 16 activations x[0..15] (two 16-byte words, natural order) -> (even, odd) MFMA fragments.
__device__ __forceinline__ void split_even_odd(uint4 lo, uint4 hi, f16x8& ev, f16x8& od) {
    const uint32_t r[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t e[4], o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        e[i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x05040100u);
        o[i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x07060302u);
    }
    ev = __builtin_bit_cast(f16x8, make_uint4(e[0], e[1], e[2], e[3]));
    od = __builtin_bit_cast(f16x8, make_uint4(o[0], o[1], o[2], o[3]));
}

// Block barrier ordering LDS only (the loop shares nothing else between waves): the fences
// are limited to the local address space, so a wait at the barrier covers LDS accesses and
// not the global loads in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One (scale, bias) fp16 word from two 16-bit values of the 9-tensor form.
template <int SBF>
__device__ __forceinline__ uint32_t sb_word(uint32_t sc, uint32_t bi) {
    if constexpr (SBF == 2) {
        sc = __half_as_ushort(__float2half_rn(__uint_as_float(sc << 16)));
        bi = __half_as_ushort(__float2half_rn(__uint_as_float(bi << 16)));
    }
    return (sc & 0xFFFFu) | (bi << 16);
}

// Four words of each of a wave's four 16-lane groups, transposed between the groups: afterwards
// word p of group q is what word q of group p was.
__device__ __forceinline__ void transpose4(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    auto swap32 = [](uint32_t& x, uint32_t& y) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
        x = r[0];
        y = r[1];
    };
    auto swap16 = [](uint32_t& x, uint32_t& y) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        x = r[0];
        y = r[1];
    };
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
}

// Gate/up of one M tile (at most 16 rows r0 .. r0 + rows - 1 of a segment) and one 128-row slice,
// the weight rows streamed whole: each wave owns two (gate, up) pairs of 16-row subtiles and
// requests a pair's whole K at once (lane (n, kq) loads groups 8p + 2kq and 8p + 2kq + 1, p < 4, of
// row n: 16 rows x 64 * GPL contiguous bytes per subtile), the second pair's loads issued before the
// first pair is multiplied.  The tile's activation rows are staged in LDS once for the whole K,
// already split into the MFMA's even / odd input fragments: one barrier per tile, after which the
// waves run independently.  A K position of an MFMA pairs lane group kq's group 8p + 2kq + h with
// the same inputs on the A side; the even/odd code split inside a word is the one described above.
// These are k_q2g_mm's positions in k_q2g_mm's order, so a row's h has the same bits whichever of
// the two kernels a call's size selects.  (The other way round, a quarter of K per lane group in
// both, costs k_q2g_mm 25% at this K: each of its steps would touch every line of a weight row.)
// The scales and biases still come in 16-byte loads, a quarter of a row per lane group, and are dealt
// out between the groups in registers: gate/up + down + combine of 512 tokens, top-10 of 512, 2048 x
// 512: 176 us (bf16) against 190 with a 4-byte load per pair of groups; gate/up of one to four
// blob segments 13.1 us against 13.9 with 8-byte loads.
template <int GPL, int SBF>
__device__ __forceinline__ void gu_whole_k(const __half* __restrict__ src, int n_src_rows,
                                           const int32_t* __restrict__ row_map, int r0, int rows, int slot,
                                           int tile, const Q2Experts& E, int inter, __half* __restrict__ out,
                                           uint4* __restrict__ a_lds) {
    static_assert(GPL == 8, "four steps of 8 groups");
    constexpr int K = 256 * GPL;
    constexpr int kg = 4 * GPL;                       // groups per weight row
    constexpr int UPR = K / 8;                        // 16-byte units per activation row
    constexpr int kPairsPerThread = UPR / 32;         // unit pairs a thread stages
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));                       // per call: no address is kept across calls
    const int lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int n = lane & 15, kq = lane >> 4;

    // thread t stages unit pairs (2 pv, 2 pv + 1), pv = (t & 15) + 16 c, of row t >> 4; rows past
    // the segment and out-of-range source rows are staged as zeros (a_lds: unit v of row m at
    // m * UPR + (v ^ m), so the 16 lanes reading one unit column hit distinct banks)
    const int sm = t >> 4, sv0 = t & 15;
    int srow = -1;
    if (sm < rows) {
        srow = row_map ? row_map[r0 + sm] : r0 + sm;
        if (srow < 0 || srow >= n_src_rows) srow = -1;
    }
    uint4 xv[2 * kPairsPerThread];
    {
        const uint4* xr = reinterpret_cast<const uint4*>(src + (size_t)(srow < 0 ? 0 : srow) * K);
#pragma unroll
        for (int c = 0; c < kPairsPerThread; ++c) {
            xv[2 * c] = xr[2 * (sv0 + 16 * c)];
            xv[2 * c + 1] = xr[2 * (sv0 + 16 * c) + 1];
        }
    }

    // pair pp: gate and up rows base .. base + 15 (inter is a multiple of 64: a subtile is wholly
    // in range or wholly out; one that is out re-reads the last subtile and is not written)
    const Q2Proj& Pg = E.p[0];
    const Q2Proj& Pu = E.p[1];
    const size_t code_row = (size_t)K / 4;
    auto pair_base = [&](int pp) { return tile * 128 + (wv * 2 + pp) * 16; };
    auto load_pair = [&](int pp, uint4 (&c)[2][GPL], uint32_t (&wd)[2][GPL]) {
        int base = pair_base(pp);
        base = base < inter ? base : inter - 16;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Q2Proj& P = h ? Pu : Pg;
            const uint8_t* cr = P.w + (size_t)slot * P.w_stride + (size_t)(base + n) * code_row + (size_t)kq * 32;
#pragma unroll
            for (int i = 0; i < GPL; ++i) c[h][i] = *reinterpret_cast<const uint4*>(cr + (i >> 1) * 128 + (i & 1) * 16);
            if constexpr (SBF == 0) {
                const uint32_t* sr = reinterpret_cast<const uint32_t*>(P.s + (size_t)slot * P.s_stride) +
                                     (size_t)(base + n) * kg + GPL * kq;
#pragma unroll
                for (int i = 0; i < GPL / 4; ++i) {
                    const uint4 v = reinterpret_cast<const uint4*>(sr)[i];
                    wd[h][4 * i] = v.x;
                    wd[h][4 * i + 1] = v.y;
                    wd[h][4 * i + 2] = v.z;
                    wd[h][4 * i + 3] = v.w;
                }
            } else {
                // groups 8kq .. 8kq + 7, two to a word: scales in the even elements, biases in the odd
                const size_t o = (size_t)(base + n) * (2 * kg) + 16 * kq;
                const uint4 sc = *reinterpret_cast<const uint4*>(P.s + (size_t)slot * P.s_stride + o);
                const uint4 bi = *reinterpret_cast<const uint4*>(P.b + (size_t)slot * P.b_stride + o);
                wd[h][0] = sc.x, wd[h][2] = sc.y, wd[h][4] = sc.z, wd[h][6] = sc.w;
                wd[h][1] = bi.x, wd[h][3] = bi.y, wd[h][5] = bi.z, wd[h][7] = bi.w;
            }
        }
    };
    auto multiply = [&](int pp, const uint4 (&c)[2][GPL], const uint32_t (&wd)[2][GPL]) {
        f32x4 accg = (f32x4){0.f, 0.f, 0.f, 0.f}, accu = (f32x4){0.f, 0.f, 0.f, 0.f};
        const uint4* arow = a_lds + n * UPR;
        uint32_t w[2][GPL];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < GPL; ++i) w[h][i] = wd[h][i];
            transpose4(w[h][0], w[h][2], w[h][4], w[h][6]);
            transpose4(w[h][1], w[h][3], w[h][5], w[h][7]);
        }
#pragma unroll
        for (int i = 0; i < GPL; ++i) {
            const int u0 = 8 * (8 * (i >> 1) + 2 * kq + (i & 1));
            uint32_t sb[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t sc = w[h][i & ~1], bi = w[h][i | 1];
                if constexpr (SBF == 0) sb[h] = w[h][i];
                else sb[h] = i & 1 ? sb_word<SBF>(sc >> 16, bi >> 16) : sb_word<SBF>(sc & 0xFFFFu, bi & 0xFFFFu);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int v = u0 + 2 * q;
                const f16x8 a_ev = __builtin_bit_cast(f16x8, arow[v ^ n]);
                const f16x8 a_od = __builtin_bit_cast(f16x8, arow[(v + 1) ^ n]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint4 cv = c[h][i];
                    const uint32_t wq = q == 0 ? cv.x : q == 1 ? cv.y : q == 2 ? cv.z : cv.w;
                    const f16x8 b_ev = dequant8(wq & 0x33333333u, sb[h]);
                    const f16x8 b_od = dequant8((wq >> 2) & 0x33333333u, sb[h]);
                    f32x4& acc = h ? accu : accg;
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_ev, b_ev, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_od, b_od, acc, 0, 0, 0);
                }
            }
        }
        // lane holds rows 4 kq + i of column n
        const int base = pair_base(pp);
        if (base < inter) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 4 * kq + i;
                if (m < rows) {
                    const float g = accg[i], u = accu[i];
                    out[(size_t)(r0 + m) * inter + base + n] = __float2half_rn(g / (1.0f + __expf(-g)) * u);
                }
            }
        }
    };

    uint4 cw0[2][GPL], cw1[2][GPL];
    uint32_t sw0[2][GPL], sw1[2][GPL];
    load_pair(0, cw0, sw0);                           // after the activations: those retire first
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kPairsPerThread; ++c) {
        const int v = 2 * (sv0 + 16 * c);
        f16x8 ev, od;
        split_even_odd(xv[2 * c], xv[2 * c + 1], ev, od);
        const uint4 e4 = __builtin_bit_cast(uint4, ev), o4 = __builtin_bit_cast(uint4, od);
        a_lds[sm * UPR + (v ^ sm)] = srow >= 0 ? e4 : make_uint4(0, 0, 0, 0);
        a_lds[sm * UPR + ((v + 1) ^ sm)] = srow >= 0 ? o4 : make_uint4(0, 0, 0, 0);
    }
    lds_barrier();
    load_pair(1, cw1, sw1);
    __builtin_amdgcn_sched_barrier(0);                // pair 1's loads go out before pair 0's multiply
    multiply(0, cw0, sw0);
    // both pairs read the same activation fragments; without this fence the compiler keeps pair
    // 0's 256 fragment registers for pair 1 and spills
    asm volatile("" ::: "memory");
    multiply(1, cw1, sw1);
}

template <int GPL, int SBF>
__global__ __launch_bounds__(256, 2) void k_q2g_gu_wk(
    const __half* __restrict__ src, int n_src_rows, const int32_t* __restrict__ row_map,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot, int n_seg, int n_rows,
    Q2Experts E, int n_slots, int inter, int tiles_per_seg, __half* __restrict__ out) {
    __shared__ uint4 a_lds[16 * 32 * GPL];
    // two passes over the (segment, slice) items: segments of more than one M tile first (their
    // blocks run longest); a block takes its segment's tiles one after the other, each tile's
    // weights loaded again (from L2 while they are still there), since both pairs' weights held
    // across tiles would not fit beside a tile's staging
    const int items = n_seg * tiles_per_seg;
    const int pass = (int)blockIdx.x >= items ? 1 : 0;
    const int work = xcd_order((int)blockIdx.x - pass * items, items);
    const int seg = work / tiles_per_seg, tile = work % tiles_per_seg;
    if (seg >= n_seg) return;
    int r0 = seg_start[seg], r1 = seg_start[seg + 1];
    r0 = r0 < 0 ? 0 : (r0 > n_rows ? n_rows : r0);
    r1 = r1 < r0 ? r0 : (r1 > n_rows ? n_rows : r1);
    const int slot = seg_slot ? seg_slot[seg] : seg;
    if (r1 == r0 || slot < 0 || slot >= n_slots) return;
    if ((pass == 0) != (r1 - r0 > kMT)) return;
#pragma unroll 1
    for (int m0 = r0; m0 < r1; m0 += kMT) {          // block-uniform
        if (m0 > r0) __syncthreads();                // every wave is done with the previous tile
        int slot_i = slot;                           // opaque: the weights are loaded again per tile
        asm volatile("" : "+s"(slot_i) : : "memory");
        gu_whole_k<GPL, SBF>(src, n_src_rows, row_map, m0, (r1 - m0) < kMT ? (r1 - m0) : kMT, slot_i, tile, E, inter,
                             out, a_lds);
    }
}

// ---- every K and any number of rows --------------------------------------------------------------
//
// Work.  A batch is up to TM M tiles of one segment (fewer where their activations would not fit in
// LDS: 2 of 4 at K 2048 and 2560); an item is a batch times one column tile (WV waves, each one
// (gate, up) pair of 16-row subtiles or two down subtiles: 16 intermediate or 32 output columns per
// wave).  With span 0 a fixed grid (one block per CU at TM 4, two at TM 1) sums the items' costs
// over the segments, and each block takes its own equal part of them in the order (segment, batch,
// column tile), so neither a long segment nor the last round of blocks leaves CUs idle (777 tokens
// over 100 experts of 1152 x 320: 118 -> 54 us, where one block used to take a 140-row segment in
// five passes of dependent round trips).  With span > 0 a block is one segment and `span` column tiles.
//
// A block stages a batch's activations once, for the whole K (split into even / odd fragments), and
// then runs its column tiles without a barrier: the queue of outstanding loads holds weights only, so
// they can be requested one or two steps (512 inputs each) ahead.  With activations staged chunk by chunk, each
// wait for a chunk's activations also waited for the weights requested before them (loads retire in
// order), which held the requests in flight to one chunk: 16-36 KB per CU, 3 TB/s.
//
// What bounds it: the dequantisation (19 VALU operations per 16 weights and lane, about 83 cycles
// against 33 of matrix unit per M tile).  Every weight is dequantised once per batch, so 64-row
// batches where they fit.  Timed passes of 2560 x 640 bf16, top-10 of 512 experts (gate/up + down +
// combine, back to back), the chunk-by-chunk kernel this replaced (32 rows per pass) -> this: 37 tokens
// 126 -> 115 us, 512 tokens 287 -> 242, 2048 tokens 590 -> 427.  Per launch under the profiler, which slows
// both sides: 512 tokens gate/up 218 -> 168 us (524 MB of weights; VALU issuing 56% of the time), down 107
// -> 109 (no gain, nor at 37 tokens); 2048 tokens 411 -> 306 and 225 -> 170.  Tried and not kept, 512
// tokens, gate/up and down, in one session where this ran 161 and 102: two subtile pairs per wave
// (256-column tiles, 2.5 of them at 640) 211 and 136; 12 waves per block 188 and 111; phase 0 of a half
// built under the half before 157 and 106.
constexpr int kMaxTiles = 4;                             // M tiles per batch, at most
constexpr int kMmSubs = 2;                               // 16-row weight subtiles per wave
constexpr int kCUs = 256;

// The activations' LDS image of a batch: per step of 512 inputs and 16-row tile 16 KB, row m of 64
// 16-byte units (half, even / odd codes, word), unit v of a row stored at v ^ m in its low 4 bits so
// that the 16 rows read at one unit index start at 16 different slots of a 256-byte bank cycle.
// Per block: all 160 KB of a CU; 80 KB for two blocks; 32 KB (K <= 1024) for four of 4 waves.
template <int TM, int WV>
constexpr int lds_units() { return TM > 1 ? 10240 : WV == 8 ? 5120 : 2048; }
constexpr int kTileUnits = kMT * 64;

typedef uint32_t u32_a2 __attribute__((aligned(2)));     // two adjacent fp16 / bf16 values

// Cost of an item in the units of the shares: the weights' bytes and their dequantisation cost about
// what the multiplication of four tiles does.
constexpr uint32_t kItemCost = 4;

// PAIR: K is a multiple of 512 (no group past the end).  TM: M tiles per batch, at most.  WV: waves.
template <int MODE, int SBF, bool PAIR, int TM, int WV>
__global__ __launch_bounds__(64 * WV, TM == 1 ? 4 : 2) void k_q2g_mm(
    const __half* __restrict__ src, int n_src_rows, const int32_t* __restrict__ row_map,
    const int32_t* __restrict__ row_out, int n_out_rows,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot, int n_seg, int n_rows,
    Q2Experts E, int n_slots, int K, int N, int tiles, int mtmax, int span, int vec_out, __half* __restrict__ out) {
    constexpr int kCols = MODE == kGateUp ? 16 : 32;           // columns per wave
    const int batch_rows = kMT * mtmax;
    __shared__ uint4 a_lds[lds_units<TM, WV>()];
    unsigned long long* wsum = reinterpret_cast<unsigned long long*>(a_lds);        // the shares' scratch
    int(*bound)[6] = reinterpret_cast<int(*)[6]>(a_lds + 64);      // first / end item: segment, batch, tile; rows, slot

    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    auto seg_range = [&](int seg, int& r0, int& r1, int& slot) {
        r0 = seg_start[seg];
        r1 = seg_start[seg + 1];
        r0 = r0 < 0 ? 0 : (r0 > n_rows ? n_rows : r0);
        r1 = r1 < r0 ? r0 : (r1 > n_rows ? n_rows : r1);
        slot = seg_slot ? seg_slot[seg] : seg;
        if (slot < 0 || slot >= n_slots) r1 = r0;
    };

    int seg, batch, tile0, seg_e, batch_e, tile_e, r0, r1, slot;
    int first = 0;                                             // where the next batch's tiles begin
    if (TM == 1 && span) {
        // one block per segment and `span` column tiles, which takes the segment's batches in turn
        const int work = xcd_order(blockIdx.x, gridDim.x), per_seg = (tiles + span - 1) / span;
        seg = seg_e = work / per_seg;
        first = tile0 = work % per_seg * span;
        batch = 0;
        batch_e = 0x7FFFFFFF;
        tile_e = 0;
        seg_range(seg, r0, r1, slot);
    } else {
        // this block's share of the items, ordered by (segment, batch, column tile): those whose start
        // in the running cost lies in [total * b / nb, total * (b + 1) / nb)
        const int per = (n_seg + 64 * WV - 1) / (64 * WV), s0 = t * per;
        const int s1 = s0 + per < n_seg ? s0 + per : n_seg;
        auto cost = [&](int rows, uint32_t& full, uint32_t& rem) {
            full = (uint32_t)rows / batch_rows;
            rem = ((uint32_t)rows % batch_rows + kMT - 1) / kMT;
            return (unsigned long long)tiles * (full * (kItemCost + (uint32_t)mtmax) + (rem ? kItemCost + rem : 0u));
        };
        unsigned long long sum = 0;
        uint32_t full, rem;
        r0 = r1 = slot = 0;                                    // the thread's only segment, where it has one
        for (int s = s0; s < s1; ++s) {
            seg_range(s, r0, r1, slot);
            sum += cost(r1 - r0, full, rem);
        }
        unsigned long long inc = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned long long o = __shfl_up(inc, d, 64);
            if (lane >= d) inc += o;
        }
        if (lane == 63) wsum[wv] = inc;
        if (t < 2) {
            bound[t][0] = n_seg;
            bound[t][1] = bound[t][2] = bound[t][3] = bound[t][4] = bound[t][5] = 0;
        }
        __syncthreads();
        unsigned long long pre = inc - sum, total = 0;
#pragma unroll
        for (int w = 0; w < WV; ++w) {
            if (w < wv) pre += wsum[w];
            total += wsum[w];
        }
        // any function of b that does not fall, is 0 at 0 and total at nb gives every item one block
        const int me = xcd_order(blockIdx.x, gridDim.x);
        const double share = (double)total / (double)gridDim.x;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const unsigned long long at = me + e == (int)gridDim.x ? total : (unsigned long long)(share * (me + e));
            if (at < pre || at >= pre + sum) continue;
            unsigned long long p = pre;
            for (int s = s0; s < s1; ++s) {
                if (per > 1) seg_range(s, r0, r1, slot);
                const unsigned long long c = cost(r1 - r0, full, rem);
                if (at < p + c) {
                    uint32_t b = 0, tl = 0;
                    if (at > p) {
                        const uint32_t d = (uint32_t)(at - p), fb = (uint32_t)tiles * (kItemCost + (uint32_t)mtmax);
                        b = d / fb < full ? d / fb : full;
                        const uint32_t ic = kItemCost + (b < full ? (uint32_t)mtmax : rem);
                        tl = (d - b * fb + ic - 1) / ic;
                    }
                    bound[e][0] = s;
                    bound[e][1] = (int)b;
                    bound[e][2] = (int)tl;
                    bound[e][3] = r0;
                    bound[e][4] = r1;
                    bound[e][5] = slot;
                    break;
                }
                p += c;
            }
        }
        __syncthreads();
        seg = __builtin_amdgcn_readfirstlane(bound[0][0]);
        batch = __builtin_amdgcn_readfirstlane(bound[0][1]);
        tile0 = __builtin_amdgcn_readfirstlane(bound[0][2]);
        r0 = __builtin_amdgcn_readfirstlane(bound[0][3]);
        r1 = __builtin_amdgcn_readfirstlane(bound[0][4]);
        slot = __builtin_amdgcn_readfirstlane(bound[0][5]);
        seg_e = __builtin_amdgcn_readfirstlane(bound[1][0]);
        batch_e = __builtin_amdgcn_readfirstlane(bound[1][1]);
        tile_e = __builtin_amdgcn_readfirstlane(bound[1][2]);
    }

    const int kg = K / 64, nst = (kg + 7) / 8;                 // steps of 8 groups (K 512) per column tile
    // the last step of a K that is no multiple of 512: with at most 4 groups left it has one half
    const bool one_half = !PAIR && (kg & 7) >= 1 && (kg & 7) <= 4;
    const int n = lane & 15, kq = lane >> 4;
    const uint32_t code_row = (uint32_t)K / 4;
    // Weight row of lane n in subtile s: the wave's columns are dealt out so that a lane of the
    // product (4 rows of the subtile) holds adjacent columns over all its subtiles
    constexpr int kSubs = MODE == kGateUp ? 1 : 2;             // subtiles per projection
    const uint32_t lane_row = (uint32_t)(4 * kSubs * (n >> 2) + (n & 3));
    const uint32_t lane_code = lane_row * code_row, lane_sb = lane_row * (uint32_t)kg;
    constexpr uint32_t kStep = SBF == 0 ? 4 : 2;

    // Group of lane group q in half h of step p: the two adjacent groups 2q, 2q + 1 of the step's
    // eight, so a lane's codes are 32 contiguous bytes and its scales one word.  Groups past the
    // end read the last one; their activations are staged as zeros.
    auto group = [&](int p, int q, int h) {
        if constexpr (PAIR) return 8 * p + 2 * q + h;
        else return one_half && p == nst - 1 ? 8 * p + q : 8 * p + 2 * q + h;
    };
    auto clampg = [&](int g) { return PAIR ? g : (g < kg ? g : kg - 1); };
    const int sv = t & 15;                                     // staged word: lane group sv >> 2, word sv & 3
    constexpr int kPassRows = 4 * WV;                    // rows staged per pass of the block

    // Rows b0 .. of one batch (M tiles, rows up to r1) times the column tiles ta .. tb - 1.
    auto body = [&](auto mtc, int slot, int b0, int r1, int ta, int tb) {
        constexpr int M = decltype(mtc)::value;
        constexpr int U = (M * kMT + kPassRows - 1) / kPassRows;
        const int sm = t >> 4;
        const bool mine = M * kMT % kPassRows == 0 || (U - 1) * kPassRows + sm < M * kMT;   // last pass partial
        const __half* xp[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int r = b0 + u * kPassRows + sm;
            r = r < r1 ? r : r1 - 1;
            int v = row_map ? row_map[r] : r;
            v = v >= 0 && v < n_src_rows ? v : 0;
            xp[u] = src + (size_t)v * K + (sv & 3) * 16;
        }
        // the output row of this lane's row in each tile (-1: none), and for gate/up whether it names a
        // source row (one that names none gives zeros)
        int orow[M];
        bool live[M];
#pragma unroll
        for (int mt = 0; mt < M; ++mt) {
            const int r = b0 + mt * kMT + n, rc = r < r1 ? r : r1 - 1;
            int o = rc;
            live[mt] = true;
            if constexpr (MODE == kGateUp) {
                const int v = row_map ? row_map[rc] : rc;
                live[mt] = v >= 0 && v < n_src_rows;
            } else {
                if (row_out) o = row_out[rc];
                if (o >= n_out_rows) o = -1;
            }
            orow[mt] = r < r1 ? o : -1;
        }
        struct X {
            uint4 v[U][2][2];
        };
        auto load_x = [&](int p, X& xs) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int g = clampg(group(p, sv >> 2, h));
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint4* x = reinterpret_cast<const uint4*>(xp[u] + g * 64);
                    xs.v[u][h][0] = x[0];
                    xs.v[u][h][1] = x[1];
                }
            }
        };
        auto stage = [&](int p, const X& xs) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool uv = PAIR || group(p, sv >> 2, h) < kg;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    f16x8 ev, od;
                    split_even_odd(xs.v[u][h][0], xs.v[u][h][1], ev, od);
                    const int row = u * kPassRows + sm;
                    uint4* d = a_lds + p * (M * kTileUnits) + row * 64 + 32 * h + (sv ^ (row & 15));
                    if (u < U - 1 || mine) {
                        d[0] = uv ? __builtin_bit_cast(uint4, ev) : make_uint4(0, 0, 0, 0);
                        d[16] = uv ? __builtin_bit_cast(uint4, od) : make_uint4(0, 0, 0, 0);
                    }
                }
            }
        };

        // one step's weights: codes, and scale / bias words as loaded
        struct W {
            uint4 c[kMmSubs][2];
            uint32_t r0[kMmSubs], r1[kMmSubs];
        };
        uint32_t sb[kMmSubs][2];
        // Subtile s of column tile tl: 16 of the weight rows base .. of its projection.  N is a
        // multiple of 64, so a wave's columns are wholly in range or wholly out; a wave that is out
        // reads the last ones and does not write.
        auto base_of = [&](int tl) { return (tl * WV + wv) * kCols; };
        auto row_of = [&](int tl, int s) {
            int base = base_of(tl);
            base = base < N ? base : N - kCols;
            return base + 4 * (MODE == kGateUp ? s >> 1 : s);
        };
        auto load_w = [&](int tl, int p, W& w) {
            const uint32_t o0 = lane_code + (uint32_t)clampg(group(p, kq, 0)) * 16;
            const uint32_t o1 = PAIR ? o0 + 16 : lane_code + (uint32_t)clampg(group(p, kq, 1)) * 16;
#pragma unroll
            for (int s = 0; s < kMmSubs; ++s) {
                const Q2Proj& P = E.p[MODE == kGateUp ? (s & 1) : 2];
                const uint8_t* c = P.w + (size_t)slot * P.w_stride + (size_t)row_of(tl, s) * code_row;
                w.c[s][0] = *reinterpret_cast<const uint4*>(c + o0);
                w.c[s][1] = *reinterpret_cast<const uint4*>(c + o1);
            }
        };
        auto load_sb = [&](int tl, int p, W& w) {
            const int g0 = clampg(group(p, kq, 0)), g1 = PAIR ? g0 + 1 : clampg(group(p, kq, 1));
#pragma unroll
            for (int s = 0; s < kMmSubs; ++s) {
                const Q2Proj& P = E.p[MODE == kGateUp ? (s & 1) : 2];
                const size_t ro = (size_t)row_of(tl, s) * (kg * kStep);
                const uint8_t* sp = P.s + (size_t)slot * P.s_stride + ro;
                const uint8_t* bp = P.b + (size_t)slot * P.b_stride + ro;
                if constexpr (SBF == 0) {
                    w.r0[s] = *reinterpret_cast<const uint32_t*>(sp + (lane_sb + (uint32_t)g0) * kStep);
                    w.r1[s] = *reinterpret_cast<const uint32_t*>(sp + (lane_sb + (uint32_t)g1) * kStep);
                } else if (PAIR || kg > 1) {
                    // both groups with one load; from the last group of a row the one before it comes along
                    const int gp = PAIR || g0 < kg - 1 ? g0 : kg - 2;
                    const uint32_t o = (lane_sb + (uint32_t)gp) * kStep;
                    w.r0[s] = *reinterpret_cast<const u32_a2*>(sp + o);
                    w.r1[s] = *reinterpret_cast<const u32_a2*>(bp + o);
                } else {
                    w.r0[s] = *reinterpret_cast<const uint16_t*>(sp + lane_sb * kStep);
                    w.r1[s] = *reinterpret_cast<const uint16_t*>(bp + lane_sb * kStep);
                }
            }
        };
        // of the step p that w holds
        auto convert_sb = [&](int p, const W& w) {
            const int drop = SBF == 0 || PAIR || kg == 1 || clampg(group(p, kq, 0)) < kg - 1 ? 0 : 16;
#pragma unroll
            for (int s = 0; s < kMmSubs; ++s) {
                if constexpr (SBF == 0) {
                    sb[s][0] = w.r0[s];
                    sb[s][1] = w.r1[s];
                } else {
                    const uint32_t sc = PAIR ? w.r0[s] : w.r0[s] >> drop, bi = PAIR ? w.r1[s] : w.r1[s] >> drop;
                    sb[s][0] = sb_word<SBF>(sc & 0xFFFFu, bi & 0xFFFFu);
                    sb[s][1] = sb_word<SBF>(sc >> 16, bi >> 16);
                }
            }
        };

        f32x4 acc[M][kMmSubs];
        auto clear = [&]() {
#pragma unroll
            for (int mt = 0; mt < M; ++mt)
#pragma unroll
                for (int s = 0; s < kMmSubs; ++s) acc[mt][s] = (f32x4){0.f, 0.f, 0.f, 0.f};
        };
        // Eight phases per half (word q = ph / 2 of the lane's group, even or odd codes): a phase
        // multiplies its fragments while the next phase's are read from LDS and dequantised, the two
        // interleaved so that the matrix unit runs under the conversions.
        const uint4* aq[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) aq[q] = a_lds + n * 64 + ((4 * kq + q) ^ n);
        auto compute = [&](int p, const W& w, auto hc) {
            constexpr int h = decltype(hc)::value;
            const int po = p * (M * kTileUnits);
            auto frag_a = [&](int ph, f16x8 (&a)[M]) {
#pragma unroll
                for (int mt = 0; mt < M; ++mt)
                    a[mt] = __builtin_bit_cast(f16x8, aq[ph >> 1][po + mt * kTileUnits + 32 * h + 16 * (ph & 1)]);
            };
            auto frag_b = [&](int ph, f16x8 (&b)[kMmSubs]) {
#pragma unroll
                for (int s = 0; s < kMmSubs; ++s) {
                    const int q = ph >> 1;
                    const uint4 cv = w.c[s][h];
                    const uint32_t wq = q == 0 ? cv.x : q == 1 ? cv.y : q == 2 ? cv.z : cv.w;
                    b[s] = dequant8((wq >> (2 * (ph & 1))) & 0x33333333u, sb[s][h]);
                }
            };
            f16x8 fa[2][M], fb[2][kMmSubs];
            frag_a(0, fa[0]);
            frag_b(0, fb[0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ph = 0; ph < 8; ++ph) {
                if (ph < 7) {
                    frag_a(ph + 1, fa[(ph + 1) & 1]);
                    frag_b(ph + 1, fb[(ph + 1) & 1]);
                }
#pragma unroll
                for (int s = 0; s < kMmSubs; ++s)
#pragma unroll
                    for (int mt = 0; mt < M; ++mt)
                        acc[mt][s] =
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[ph & 1][s], fa[ph & 1][mt], acc[mt][s], 0, 0, 0);
                if (ph < 7) {
                    constexpr int kPer = (10 * kMmSubs + kMmSubs * M - 1) / (kMmSubs * M);
                    __builtin_amdgcn_sched_group_barrier(0x100, M, 0);
#pragma unroll
                    for (int i = 0; i < kMmSubs * M; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, kPer, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // lane: row n of each tile, 4 * kSubs adjacent columns
        auto write = [&](int tl) {
            if (base_of(tl) >= N) return;
#pragma unroll
            for (int mt = 0; mt < M; ++mt) {
                if (orow[mt] < 0) continue;
                __half* o = out + (size_t)orow[mt] * N + base_of(tl) + 4 * kSubs * kq;
                uint32_t hw[2 * kSubs];
#pragma unroll
                for (int i = 0; i < 2 * kSubs; ++i) {
                    uint32_t v[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int c = 2 * i + e, s = c >> 2;
                        if constexpr (MODE == kGateUp) {
                            const float g = acc[mt][2 * s][c & 3], u = acc[mt][2 * s + 1][c & 3];
                            v[e] = __half_as_ushort(__float2half_rn(live[mt] ? g / (1.0f + __expf(-g)) * u : 0.0f));
                        } else {
                            v[e] = __half_as_ushort(__float2half_rn(acc[mt][s][c & 3]));
                        }
                    }
                    hw[i] = v[0] | (v[1] << 16);
                }
                if (vec_out) {
                    if constexpr (kSubs == 1) {
                        *reinterpret_cast<uint2*>(o) = make_uint2(hw[0], hw[1]);
                    } else {
#pragma unroll
                        for (int i = 0; i < kSubs / 2; ++i)
                            reinterpret_cast<uint4*>(o)[i] =
                                make_uint4(hw[4 * i], hw[4 * i + 1], hw[4 * i + 2], hw[4 * i + 3]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4 * kSubs; ++i)
                        o[i] = __ushort_as_half((unsigned short)(hw[i >> 1] >> (16 * (i & 1))));
                }
            }
        };

        // The batch's activations are staged once for the whole K; after that the waves run without
        // barriers.  One step = 512 inputs of one column tile: its weights are loaded two steps ahead
        // (past the end the last step's are read again: no load is conditional).
        int tl = ta, p = 0, tl_w = ta, p_w = 0;
        // steps ahead; one at four waves per SIMD, whose 128 registers do not hold a third step (spills:
        // 2560 x 640, 37 tokens 134 us against 121)
        constexpr int kAhead = TM == 1 ? 1 : 2;
        W w0, w1, w2;
        auto fetch = [&](W& w) {
            load_w(tl_w, p_w, w);
            load_sb(tl_w, p_w, w);
            if (p_w + 1 < nst) {
                ++p_w;
            } else if (tl_w + 1 < tb) {
                ++tl_w;
                p_w = 0;
            }
        };
        {
            X xa, xb;
            load_x(0, xa);
            load_x(nst > 1 ? 1 : 0, xb);
            fetch(w0);
            if constexpr (kAhead == 2) fetch(w1);
            lds_barrier();                                     // every wave is done with the LDS
            stage(0, xa);
            if (nst > 1) stage(1, xb);
            for (int q = 2; q < nst; q += 2) {
                load_x(q, xa);
                load_x(q + 1 < nst ? q + 1 : q, xb);
                stage(q, xa);
                if (q + 1 < nst) stage(q + 1, xb);
            }
            lds_barrier();
        }
        clear();
        auto step = [&](const W& cur, W& nxt) {
            fetch(nxt);
            __builtin_amdgcn_sched_barrier(0);
            convert_sb(p, cur);
            compute(p, cur, std::integral_constant<int, 0>());
            if (PAIR || !(one_half && p == nst - 1)) compute(p, cur, std::integral_constant<int, 1>());
            if (++p < nst) return true;
            write(tl);
            clear();
            p = 0;
            return ++tl < tb;
        };
        for (;;) {
            if constexpr (kAhead == 2) {
                if (!step(w0, w2)) break;
                if (!step(w1, w0)) break;
                if (!step(w2, w1)) break;
            } else {
                if (!step(w0, w1)) break;
                if (!step(w1, w0)) break;
            }
        }
    };

    while (seg < n_seg && (seg < seg_e || (seg == seg_e && batch <= batch_e))) {
        const int b0 = r0 + batch * batch_rows;
        if (b0 >= r1) {
            batch = tile0 = 0;
            if (++seg < n_seg && seg <= seg_e) seg_range(seg, r0, r1, slot);
            continue;
        }
        const bool at_end = seg == seg_e && batch == batch_e;
        const int tb = TM == 1 && span ? (first + span < tiles ? first + span : tiles) : at_end ? tile_e : tiles;
        if (tile0 < tb) {
            const int mts = (r1 - b0 + kMT - 1) / kMT;
            if (TM == 1 || mtmax == 1 || mts == 1) body(std::integral_constant<int, 1>(), slot, b0, r1, tile0, tb);
            else if (mtmax == 2 || mts == 2) body(std::integral_constant<int, TM == 1 ? 1 : 2>(), slot, b0, r1, tile0, tb);
            else if (mtmax == 3 || mts == 3) body(std::integral_constant<int, TM == 1 ? 1 : 3>(), slot, b0, r1, tile0, tb);
            else body(std::integral_constant<int, TM>(), slot, b0, r1, tile0, tb);
        }
        if (at_end) break;
        ++batch;
        tile0 = first;
    }
}

// Short K in the whole-K form (K = 512, GPL 2; any K up to 256, GPL 1): a block takes one segment and 256
// output rows (128 of each projection for gate/up), each wave 4 subtiles of 16 rows whose whole K it
// requests at once and keeps in registers while the segment's rows pass through LDS (staged for the
// whole K, split into the MFMA's even / odd fragments; one barrier per pass).  row_idx names each row's
// source row (gate/up) or output row (down); without it they are the same.  Lane group kq takes groups
// GPL*kq .. GPL*kq + GPL - 1: at K = 512 and up to 256 these are k_q2g_mm's positions, and the sums have
// its bits.  Groups past a K below 256 read the last one; their activations are staged as zeros.
//
// What bounds it: one chain of dependent round trips per block (segment, rows, activations beside the
// weights) and the dequantisation.  Up to K 256 k_q2g_mm leaves half of every 512-input step empty, and
// its waves hold half as many weights; two M tiles per pass share the dequantisation.  Down in us, the
// chunked kernel of old / k_q2g_mm / this: 137 tokens x top-10 of 280, 1728 x 256: 17.2 / 26 / 16.7; 79 x
// top-5 of 66, 2304 x 256: 8.0 / 13.3 / 8.1; 222 x top-7 of 202, 512 x 256: 9.4 / 13.6 / 9.0; gate/up of
// 924 x top-4 of 338, 256 x 576: 19.5 / 23.5 / 19.0.  One tile per pass: 1-3 us slower where segments
// exceed 16 rows; 5 or 6 blocks per CU instead of 4: spills.
template <int GPL, int MODE>
constexpr bool two_pass() { return GPL == 2 || MODE == kGateUp; }

template <int GPL, int MODE, int SBF>
__global__ __launch_bounds__(256, 2) void k_q2g_wk(
    const __half* __restrict__ src, int n_src_rows, const int32_t* __restrict__ row_idx, int n_out_rows,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot, int n_seg, int n_rows,
    Q2Experts E, int n_slots, int N, int tiles_per_seg, __half* __restrict__ out, int k_len) {
    const int K = GPL == 1 ? k_len : 256 * GPL, kg = K / 64;
    constexpr int UPR = 32 * GPL;                     // 16-byte units per activation row in LDS
    constexpr int kPairsPerThread = UPR / 32;         // unit pairs a thread stages per tile
    constexpr int NT = GPL == 1 ? 2 : 1;              // M tiles per pass
    // segments of several passes first, in a grid of twice the items; a short K's down is as fast without
    constexpr bool kTwoPass = two_pass<GPL, MODE>();
    __shared__ uint4 a_lds[NT * 16 * UPR];
    const int items = n_seg * tiles_per_seg;
    const int pass = (int)blockIdx.x >= items ? 1 : 0;
    const int work = xcd_order((int)blockIdx.x - pass * items, items);
    const int seg = work / tiles_per_seg, tile = work % tiles_per_seg;
    if (seg >= n_seg) return;
    int r0 = seg_start[seg], r1 = seg_start[seg + 1];
    r0 = r0 < 0 ? 0 : (r0 > n_rows ? n_rows : r0);
    r1 = r1 < r0 ? r0 : (r1 > n_rows ? n_rows : r1);
    const int slot = seg_slot ? seg_slot[seg] : seg;
    if (r1 == r0 || slot < 0 || slot >= n_slots) return;
    if (kTwoPass && (pass == 0) != (r1 - r0 > NT * kMT)) return;

    const int t0 = threadIdx.x, lane0 = t0 & 63, wv = __builtin_amdgcn_readfirstlane(t0 >> 6);
    const int n0 = lane0 & 15, kq0 = lane0 >> 4;
    const int g0 = GPL > 1 || kq0 < kg ? GPL * kq0 : kg - 1;
    const size_t code_row = (size_t)K / 4;
    // the wave's 4 subtiles: rows base .. base + 15 of their projection (N is a multiple of 64)
    uint4 cw[4][GPL];
    uint32_t sw[4][GPL];
    bool rv[4];
    int col[4];
#pragma unroll
    for (int sIdx = 0; sIdx < 4; ++sIdx) {
        int base = MODE == kGateUp ? tile * 128 + wv * 32 + (sIdx >> 1) * 16 : tile * 256 + wv * 64 + sIdx * 16;
        const Q2Proj& P = E.p[MODE == kGateUp ? (sIdx & 1) : 2];
        rv[sIdx] = base < N;
        col[sIdx] = base + n0;
        if (base >= N) base = N - 16;
        const uint8_t* cr = P.w + (size_t)slot * P.w_stride + (size_t)(base + n0) * code_row + (size_t)g0 * 16;
#pragma unroll
        for (int i = 0; i < GPL; ++i) cw[sIdx][i] = *reinterpret_cast<const uint4*>(cr + (size_t)i * 16);
        const size_t o = (size_t)(base + n0) * kg + g0;
        if constexpr (SBF == 0) {
            const uint32_t* sr = reinterpret_cast<const uint32_t*>(P.s + (size_t)slot * P.s_stride) + o;
#pragma unroll
            for (int i = 0; i < GPL; ++i) sw[sIdx][i] = sr[i];
        } else {
            const uint16_t* scr = reinterpret_cast<const uint16_t*>(P.s + (size_t)slot * P.s_stride) + o;
            const uint16_t* bir = reinterpret_cast<const uint16_t*>(P.b + (size_t)slot * P.b_stride) + o;
#pragma unroll
            for (int i = 0; i < GPL; ++i) sw[sIdx][i] = sb_word<SBF>(scr[i], bir[i]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    const int sm = t0 >> 4, sv0 = t0 & 15;
#pragma unroll 1
    for (int m0 = r0; m0 < r1; m0 += NT * kMT) {     // block-uniform
        const int rows_t = (r1 - m0) < NT * kMT ? (r1 - m0) : NT * kMT;
        const bool two = NT > 1 && rows_t > kMT;
        int srow[NT];
        uint4 xv[NT][2 * kPairsPerThread];
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            if (u && !two) break;
            srow[u] = -1;
            if (u * kMT + sm < rows_t) {
                srow[u] = m0 + u * kMT + sm;
                if (MODE == kGateUp && row_idx) srow[u] = row_idx[srow[u]];
                if ((unsigned)srow[u] >= (unsigned)n_src_rows) srow[u] = -1;
            }
            const uint4* xr = reinterpret_cast<const uint4*>(src + (size_t)(srow[u] < 0 ? 0 : srow[u]) * K);
#pragma unroll
            for (int c = 0; c < kPairsPerThread; ++c) {
                const int pv = GPL == 1 && sv0 * 16 >= K ? 0 : sv0 + 16 * c;
                xv[u][2 * c] = xr[2 * pv];
                xv[u][2 * c + 1] = xr[2 * pv + 1];
            }
        }
        if (m0 > r0) lds_barrier();                   // every wave is done with the last pass
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            if (u && !two) break;
            const bool live = srow[u] >= 0 && (GPL > 1 || sv0 * 16 < K);
            uint4* d = a_lds + (u * kMT + sm) * UPR;
#pragma unroll
            for (int c = 0; c < kPairsPerThread; ++c) {
                const int v = 2 * (sv0 + 16 * c);
                f16x8 ev, od;
                split_even_odd(xv[u][2 * c], xv[u][2 * c + 1], ev, od);
                const uint4 e4 = __builtin_bit_cast(uint4, ev), o4 = __builtin_bit_cast(uint4, od);
                d[v ^ sm] = live ? e4 : make_uint4(0, 0, 0, 0);
                d[(v + 1) ^ sm] = live ? o4 : make_uint4(0, 0, 0, 0);
            }
        }
        lds_barrier();
        // opaque per pass: the converted weights and the fragment addresses are not kept across
        // passes
        uint32_t z;
        asm volatile("v_mov_b32 %0, 0" : "=v"(z));
        int tq = (int)threadIdx.x;
        asm volatile("" : "+v"(tq));
        const int n = tq & 15, kq = (tq & 63) >> 4;
        f32x4 acc[NT][4];
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int sIdx = 0; sIdx < 4; ++sIdx) acc[u][sIdx] = (f32x4){0.f, 0.f, 0.f, 0.f};
        const uint4* arow = a_lds + n * UPR;
#pragma unroll
        for (int i = 0; i < GPL; ++i) {
            uint32_t sb[4];
#pragma unroll
            for (int sIdx = 0; sIdx < 4; ++sIdx) sb[sIdx] = sw[sIdx][i] ^ z;
            const int u0 = 8 * (GPL * kq + i);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int v = u0 + 2 * q;
                f16x8 a_ev[NT], a_od[NT];
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    if (u && !two) break;
                    a_ev[u] = __builtin_bit_cast(f16x8, arow[u * kMT * UPR + (v ^ n)]);
                    a_od[u] = __builtin_bit_cast(f16x8, arow[u * kMT * UPR + ((v + 1) ^ n)]);
                }
#pragma unroll
                for (int sIdx = 0; sIdx < 4; ++sIdx) {
                    const uint4 cv = cw[sIdx][i];
                    const uint32_t wq = (q == 0 ? cv.x : q == 1 ? cv.y : q == 2 ? cv.z : cv.w) ^ z;
                    const f16x8 b_ev = dequant8(wq & 0x33333333u, sb[sIdx]);
                    const f16x8 b_od = dequant8((wq >> 2) & 0x33333333u, sb[sIdx]);
#pragma unroll
                    for (int u = 0; u < NT; ++u) {
                        if (u && !two) break;
                        acc[u][sIdx] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_ev[u], b_ev, acc[u][sIdx], 0, 0, 0);
                        acc[u][sIdx] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_od[u], b_od, acc[u][sIdx], 0, 0, 0);
                    }
                }
            }
        }
        // lane holds rows 4 kq + i of column n of each subtile
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            if (u && !two) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = u * kMT + 4 * kq + i;
                if (m >= rows_t) continue;
                const int r = m0 + m;
                if constexpr (MODE == kGateUp) {
#pragma unroll
                    for (int sIdx = 0; sIdx < 4; sIdx += 2) {
                        const float g = acc[u][sIdx][i], up = acc[u][sIdx + 1][i];
                        if (rv[sIdx]) out[(size_t)r * N + col[sIdx]] = __float2half_rn(g / (1.0f + __expf(-g)) * up);
                    }
                } else {
                    const int orow = row_idx ? row_idx[r] : r;
                    if (orow < 0 || orow >= n_out_rows) continue;
#pragma unroll
                    for (int sIdx = 0; sIdx < 4; ++sIdx)
                        if (rv[sIdx]) out[(size_t)orow * N + col[sIdx]] = __float2half_rn(acc[u][sIdx][i]);
                }
            }
        }
    }
}

template <int MODE, int SBF, int TM, int WV>
int launch_mm(int K, int span, const __half* src, int n_src_rows, const int32_t* row_map, const int32_t* row_out,
              int n_out_rows, const int32_t* seg_start, const int32_t* seg_slot, int n_seg, int n_rows,
              const Q2Experts& E, int n_slots, int N, __half* out, hipStream_t s) {
    constexpr int cols = WV * (MODE == kGateUp ? 16 : 32), cus = TM == 1 ? 2 * kCUs : kCUs;
    const int tiles = (N + cols - 1) / cols, nst = (K + 511) / 512;
    const int fit = lds_units<TM, WV>() / (nst * kTileUnits), mtmax = fit < TM ? fit : TM;
    const long long items = (long long)tiles * (n_seg + (long long)n_rows / (kMT * mtmax));   // at most
    const long long nbl = span ? (long long)n_seg * ((tiles + span - 1) / span) : items < cus ? items : cus;
    if (nbl > 0x7FFFFFFFLL) { moe_set_error("grouped q2: grid too large"); return -1; }
    const unsigned nb = (unsigned)nbl;
    const int vec_out = (uintptr_t)out % 16 == 0;              // rows are whole 128-byte lines; the base may not be
    if (K % 512 == 0)
        MOE_LAUNCH(MODE == kGateUp ? TK_PF_GATE_UP : TK_PF_DOWN, (k_q2g_mm<MODE, SBF, true, TM, WV>), dim3(nb),
                   dim3(64 * WV), 0, s, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                   n_rows, E, n_slots, K, N, tiles, mtmax, span, vec_out, out);
    else
        MOE_LAUNCH(MODE == kGateUp ? TK_PF_GATE_UP : TK_PF_DOWN, (k_q2g_mm<MODE, SBF, false, TM, WV>), dim3(nb),
                   dim3(64 * WV), 0, s, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                   n_rows, E, n_slots, K, N, tiles, mtmax, span, vec_out, out);
    HIP_TRY(hipGetLastError());
    return 0;
}

template <int SBF>
int launch_gu_wk(const __half* src, int n_src_rows, const int32_t* row_map, const int32_t* seg_start,
                 const int32_t* seg_slot, int n_seg, int n_rows, const Q2Experts& E, int n_slots, int inter,
                 __half* out, hipStream_t s) {
    const int tiles = (inter + 127) / 128;
    const long long nb = 2LL * n_seg * tiles;                  // two passes
    if (nb > 0x7FFFFFFFLL) { moe_set_error("grouped q2: grid too large"); return -1; }
    MOE_LAUNCH(TK_PF_GATE_UP, (k_q2g_gu_wk<8, SBF>), dim3((unsigned)nb), dim3(256), 0, s, src, n_src_rows, row_map,
               seg_start, seg_slot, n_seg, n_rows, E, n_slots, inter, tiles, out);
    HIP_TRY(hipGetLastError());
    return 0;
}

template <int GPL, int MODE, int SBF>
int launch_wk(int K, const __half* src, int n_src_rows, const int32_t* row_map, const int32_t* row_out, int n_out_rows,
              const int32_t* seg_start, const int32_t* seg_slot, int n_seg, int n_rows, const Q2Experts& E, int n_slots,
              int N, __half* out, hipStream_t s) {
    const int tiles = MODE == kGateUp ? (N + 127) / 128 : (N + 255) / 256;
    const long long nb = (two_pass<GPL, MODE>() ? 2LL : 1LL) * n_seg * tiles;
    if (nb > 0x7FFFFFFFLL) { moe_set_error("grouped q2: grid too large"); return -1; }
    MOE_LAUNCH(MODE == kGateUp ? TK_PF_GATE_UP : TK_PF_DOWN, (k_q2g_wk<GPL, MODE, SBF>), dim3((unsigned)nb), dim3(256), 0,
               s, src, n_src_rows, MODE == kGateUp ? row_map : row_out, n_out_rows, seg_start, seg_slot, n_seg, n_rows, E,
               n_slots, N, tiles, out, K);
    HIP_TRY(hipGetLastError());
    return 0;
}

template <int MODE, int SBF>
int dispatch_proj_f(int K, const __half* src, int n_src_rows, const int32_t* row_map, const int32_t* row_out,
                    int n_out_rows, const int32_t* seg_start, const int32_t* seg_slot, int n_seg, int n_rows,
                    const Q2Experts& E, int n_slots, int hidden, int inter, __half* out, hipStream_t s) {
    // column tiles of 4 and of 8 waves; the whole-K grids (at most twice n_seg * t4 blocks) fit in 31 bits
    const int N = MODE == kGateUp ? inter : hidden;
    const long long t4 = (N + (MODE == kGateUp ? 63 : 127)) / (MODE == kGateUp ? 64 : 128), t8 = (t4 + 1) / 2;
    const bool wk_fits = n_seg * t4 <= 0x3FFFFFFF;
    // Short segments at the two shapes the whole-K kernels are built for: those, whose short blocks
    // (512 or more, 2-4 per CU) hide each other's latencies; from about one full M tile per segment on,
    // k_q2g_mm's one pass over the weights per 64 rows wins (gate/up + down + combine in us, whole-K
    // against k_q2g_mm, top-4 of 512 experts of 2048 x 512: 128 tokens 78 and 97, 512 tokens 125 and 144,
    // 1024 tokens 157 and 159, 1536 tokens 190 and 170, 3584 tokens 426 and 240; one segment of 16 rows 20.8
    // and 23.5, of 40 rows 51 and 28; 250 segments of 28 rows 262 and 137).  The line is drawn on the
    // segments and not on the pool's slots: rows on a few experts of a large pool are long segments too,
    // and a plan cut into one-tile segments keeps the kernel that is made for it (2048 tokens, gate/up
    // over one-tile segments: 233 us whole-K, 266 in k_q2g_mm, which reads the weights once per segment).
    // Both kernels give the same bits.
    if (wk_fits && n_rows <= 16LL * n_seg) {
        if constexpr (MODE == kGateUp) {
            if (K == 2048)
                return launch_gu_wk<SBF>(src, n_src_rows, row_map, seg_start, seg_slot, n_seg, n_rows, E, n_slots, inter,
                                         out, s);
        } else if (K == 512) {
            return launch_wk<2, MODE, SBF>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                           n_rows, E, n_slots, hidden, out, s);
        }
    }
    // K up to 256: the whole-K form while the segments are short; the longest one sets its time, so the
    // line lies lower with few column tiles, whose other work is soon done.  Whole-K against k_q2g_mm in
    // us: 300 segments of 14 rows, down to 2304 x 256: 26 and 35, of 30 rows 42 and 41; 100 of 14 rows to
    // 1024 x 128: 10.4 and 12.1, of 30 rows 17.0 and 13.9; 133 of 17 rows to 512 x 192: 16.0 and 9.8; gate/up
    // of 300 segments of 20 rows, 256 x 512: 20.4 and 25; 8 segments of 20 rows, 128 x 256: 5.7 and 7.5.
    // The smallest down products stay with k_q2g_mm's one-segment blocks, which start sooner (4.6-4.7 us
    // against 5.0).
    if (K <= 256 && wk_fits) {
        const int most_rows = K > 128 ? K / 8 : 16, by_tiles = MODE == kGateUp ? N / 16 : N / 64;
        long long line = by_tiles < most_rows ? by_tiles : most_rows;
        const int least = MODE == kDown && K <= 192 ? 8 : 12;
        if (line < least) line = least;
        if (n_seg <= 16 && n_rows <= 256) line = 32;
        const long long tiny = n_seg <= 16 ? 16 : n_seg <= 32 ? 8 : 4;
        const bool smallest = MODE == kDown && n_seg * t4 <= kCUs && n_rows <= tiny * n_seg;
        if (n_rows <= line * n_seg && !smallest)
            return launch_wk<1, MODE, SBF>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                           n_rows, E, n_slots, N, out, s);
    }
    // Gate/up at K 512 likewise, while its blocks hide each other's latencies: the more there are, the longer
    // the segments may be.  Whole-K against k_q2g_mm in us: 255 segments of 4.3 rows, 512 x 512: 20.3 and
    // 23.4; 278 of 5 rows to 768: 23.3 and 28.9; 277 of 13 rows to 320: 25.0 and 26.3; 107 of 12 rows to 384: 18.1
    // and 14.1; 75 of 5 rows to 128: 7.1 and 6.2; 278 of 3.4 rows to 64: 11.2 and 7.3.
    if (MODE == kGateUp && K == 512 && N >= 128 && n_seg * t4 > kCUs && wk_fits) {
        const long long line = n_seg * t4 / 64 < 16 ? n_seg * t4 / 64 : 16;
        if (n_rows <= line * n_seg)
            return launch_wk<2, MODE, SBF>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                           n_rows, E, n_slots, N, out, s);
    }
    auto go = [&](auto tm, auto wv, int span) {
        return launch_mm<MODE, SBF, decltype(tm)::value, decltype(wv)::value>(
            K, span, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg, n_rows, E, n_slots,
            N, out, s);
    };
    using One = std::integral_constant<int, 1>;
    using Four = std::integral_constant<int, 4>;
    using Eight = std::integral_constant<int, 8>;
    // Short calls: blocks of one segment and a few column tiles instead of shares, so that no block starts
    // with the sum over the segments (2-3 us), while the blocks are few and the segments short; K up
    // to 1024 in blocks of 4 waves, four per CU.  Gate/up + down + combine in us (chunked kernel
    // before; shares; these): 12 tokens x top-7 of 28 experts, 512 x 256: 13.8, 19.2, 11.7; 251 x
    // top-4 of 381, 576 x 512: 45.5, 44.9, 40.4; 5 x top-7, 2176 x 576: 36.8, 33.7, 29.5.  The lines
    // lie where the shares win again.  Gate/up, these and shares: 427 segments of 8.4 rows, 1024 x 320, 51
    // and 41; 308 of 7.4 rows, 832 x 704, 51 and 46; 253 of 5.7 rows, 640 x 192, 15.4 and 20.9; 174 of 9.8
    // rows, 704 x 320, 20.7 and 22.0; 8 of 20 rows, 1024 x 128, 10.3 and 10.8 (64-row batches 13.7).
    // A block takes as many column tiles as keep the grid at 2,048 blocks, 1,024 with the shortest
    // segments (55 x top-3 of 401, 2240 x 256: 36.6 against 34.0; 415 x top-6 of 289: 65.7 against 75.3).
    const long long most = n_rows <= 4LL * n_seg ? 1024 : 2048;
    const long long short_rows = n_rows <= 256 ? 32 : n_rows <= 1024 ? 16 : n_seg * t4 > 2048 ? 7 : 10;
    if (K <= 1024 && n_rows <= short_rows * n_seg && n_seg * t4 <= 6144)
        return go(One(), Four(), (int)((n_seg * t4 + most - 1) / most));
    // Above K 1024, blocks of 8 waves.  54 x top-8 of 95, 1216 x 448 (4.5 rows): shares 34.0 against 39.3; 64 x
    // top-10 of 512, 2560 x 640 (367 segments, 1,835 blocks) 152 against 175.  Grids that leave CUs idle
    // wait for their longest segment, unless all are short (gate/up, these and shares: 208 blocks for 762
    // rows, 1856 x 128, 26.2 and 18.4; 200 for 320, 1280 x 192, 14.8 and 13.4; 108 for 280, 1600 x 64, 12.2 and
    // 14.1).
    if (K > 1024 && n_rows <= 4LL * n_seg && n_seg * t8 <= 1024 && (n_rows <= 300 || n_seg * t8 >= kCUs))
        return go(One(), Eight(), 1);
    // One-tile batches, two blocks per CU, for few rows per segment (256 tokens at 2560 x 640, 5 per
    // expert: 242 / 230 us against 246 / 232 with 64-row batches; 512 tokens, 10 per expert: 297 /
    // 286 against 296 / 275; up to K 1024 gate/up of 439 segments of 8.5 rows, 896 x 768, 64.5 against 70.6)
    // and for small work (1,660 x top-2 of 28, 256 x 512: 27.0 against 35.1; but down of 1,020 rows over 22
    // experts to 2304 x 256: 17.1 against 12.0).
    const bool small_work = K <= 512 && n_rows <= 4096 && (MODE == kGateUp || (long long)n_rows * N <= 2000000);
    if (n_rows <= (K <= 1024 ? 10LL : 8LL) * n_seg || small_work) return go(One(), Eight(), 0);
    return go(std::integral_constant<int, kMaxTiles>(), Eight(), 0);
}

template <int MODE>
int dispatch_proj(int K, const __half* src, int n_src_rows, const int32_t* row_map, const int32_t* row_out,
                  int n_out_rows, const int32_t* seg_start, const int32_t* seg_slot, int n_seg, int n_rows,
                  const Q2Experts& E, int n_slots, int hidden, int inter, __half* out, hipStream_t s) {
    if (E.p[0].sb_step == 4)
        return dispatch_proj_f<MODE, 0>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                        n_rows, E, n_slots, hidden, inter, out, s);
    if (E.bf16)
        return dispatch_proj_f<MODE, 2>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                        n_rows, E, n_slots, hidden, inter, out, s);
    return dispatch_proj_f<MODE, 1>(K, src, n_src_rows, row_map, row_out, n_out_rows, seg_start, seg_slot, n_seg,
                                    n_rows, E, n_slots, hidden, inter, out, s);
}

bool check_grouped(const char* who, int hidden, int inter, int group, int n_seg, int n_rows, const void* pool,
                   size_t stride, int n_slots, const void* a, const void* b, const void* c) {
    if (group != 64) { moe_set_error("%s: group=%d unsupported (kernels take group 64)", who, group); return false; }
    if (hidden <= 0 || inter <= 0 || hidden % 64 || inter % 64 || hidden > kMaxChunks * 256 || inter > kMaxChunks * 256) {
        moe_set_error("%s: hidden=%d inter=%d must be multiples of 64 in 64..%d", who, hidden, inter, kMaxChunks * 256);
        return false;
    }
    if (n_seg < 0 || n_rows < 0) { moe_set_error("%s: negative segment or row count", who); return false; }
    if (n_seg > 0 && (!pool || n_slots <= 0 || !a || !b || !c)) {
        moe_set_error("%s: empty pool or null pointer", who);
        return false;
    }
    BlobLayout L = blob_layout(hidden, inter, group);
    if (n_seg > 0 && stride < L.bytes) {
        moe_set_error("%s: expert stride %zu < blob bytes %zu", who, stride, L.bytes);
        return false;
    }
    return true;
}

__global__ __launch_bounds__(256) void k_pair_combine(const __half* __restrict__ y, const __half* __restrict__ scores,
                                                      const __half* __restrict__ residual, int k, int hidden,
                                                      float* __restrict__ out) {
    const int t = blockIdx.y;
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 2;
    if (c >= hidden) return;
    float a0 = 0.f, a1 = 0.f;
    for (int j = 0; j < k; ++j) {
        const float sj = __half2float(scores[(size_t)t * k + j]);
        const __half* row = y + ((size_t)t * k + j) * hidden;
        a0 += sj * __half2float(row[c]);
        if (c + 1 < hidden) a1 += sj * __half2float(row[c + 1]);
    }
    if (residual) {
        a0 += __half2float(residual[(size_t)t * hidden + c]);
        if (c + 1 < hidden) a1 += __half2float(residual[(size_t)t * hidden + c + 1]);
    }
    out[(size_t)t * hidden + c] = a0;
    if (c + 1 < hidden) out[(size_t)t * hidden + c + 1] = a1;
}

// The same sum for hidden a multiple of 8: each thread 8 consecutive columns, 16-byte loads of
// the fp16 rows and two 16-byte stores (the same operations per element in the same order, so
// bit-identical to k_pair_combine).
__global__ __launch_bounds__(256) void k_pair_combine8(const __half* __restrict__ y, const __half* __restrict__ scores,
                                                       const __half* __restrict__ residual, int k, int hidden,
                                                       float* __restrict__ out) {
    const int t = blockIdx.y;
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 8;
    if (c >= hidden) return;
    // every row's load first (k <= MOE_MAX_K), then the sums in row order
    uint4 rv[MOE_MAX_K];
#pragma unroll
    for (int j = 0; j < MOE_MAX_K; ++j)
        if (j < k) rv[j] = *reinterpret_cast<const uint4*>(y + ((size_t)t * k + j) * hidden + c);
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < MOE_MAX_K; ++j) {
        if (j < k) {
            const float sj = __half2float(scores[(size_t)t * k + j]);
            const uint4 v = rv[j];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[2 * i] += sj * __half2float(__ushort_as_half((unsigned short)(w[i] & 0xFFFFu)));
                a[2 * i + 1] += sj * __half2float(__ushort_as_half((unsigned short)(w[i] >> 16)));
            }
        }
    }
    if (residual) {
        const uint4 v = *reinterpret_cast<const uint4*>(residual + (size_t)t * hidden + c);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[2 * i] += __half2float(__ushort_as_half((unsigned short)(w[i] & 0xFFFFu)));
            a[2 * i + 1] += __half2float(__ushort_as_half((unsigned short)(w[i] >> 16)));
        }
    }
    float4* o = reinterpret_cast<float4*>(out + (size_t)t * hidden + c);
    o[0] = make_float4(a[0], a[1], a[2], a[3]);
    o[1] = make_float4(a[4], a[5], a[6], a[7]);
}

}  // namespace

int launch_q2_grouped_gate_up(const __half* x, int n_tokens, const int32_t* row_token, int n_rows,
                              const int32_t* seg_start, const int32_t* seg_slot, int n_seg, const uint8_t* pool,
                              size_t stride, int n_slots, int hidden, int inter, int group, __half* h_out,
                              hipStream_t s) {
    if (!check_grouped("q2_grouped_gate_up", hidden, inter, group, n_seg, n_rows, pool, stride, n_slots, x, seg_start,
                       h_out))
        return -1;
    if (n_seg == 0 || n_rows == 0) return 0;
    if (n_tokens <= 0) {                      // the kernel reads source row 0 unconditionally
        moe_set_error("q2_grouped_gate_up: %d rows but no tokens", n_rows);
        return -1;
    }
    const Q2Experts E = q2_experts_from_blob(pool, stride, blob_layout(hidden, inter, group));
    return dispatch_proj<kGateUp>(hidden, x, n_tokens, row_token, nullptr, 0, seg_start, seg_slot, n_seg, n_rows, E,
                                  n_slots, hidden, inter, h_out, s);
}

int launch_q2_grouped_down(const __half* h, int n_rows, const int32_t* row_out, int n_out_rows,
                           const int32_t* seg_start, const int32_t* seg_slot, int n_seg, const uint8_t* pool,
                           size_t stride, int n_slots, int hidden, int inter, int group, __half* y_out, hipStream_t s) {
    if (!check_grouped("q2_grouped_down", hidden, inter, group, n_seg, n_rows, pool, stride, n_slots, h, seg_start,
                       y_out))
        return -1;
    if (n_seg == 0 || n_rows == 0) return 0;
    const Q2Experts E = q2_experts_from_blob(pool, stride, blob_layout(hidden, inter, group));
    return dispatch_proj<kDown>(inter, h, n_rows, nullptr, row_out, row_out ? n_out_rows : n_rows, seg_start, seg_slot,
                                n_seg, n_rows, E, n_slots, hidden, inter, y_out, s);
}

// The same over the reference's 9 tensors (E from their pools; see q2t_shape_ok for the shapes the
// decode kernels take -- the grouped kernels take any multiple of 64 up to 2560).
int launch_q2t_grouped_gate_up(const __half* x, int n_tokens, const int32_t* row_token, int n_rows,
                               const int32_t* seg_start, const int32_t* seg_slot, int n_seg, const Q2Experts& E,
                               int n_slots, int hidden, int inter, int group, __half* h_out, hipStream_t s) {
    if (!check_grouped("q2t_grouped_gate_up", hidden, inter, group, n_seg, n_rows, E.p[0].w, ~size_t(0), n_slots, x,
                       seg_start, h_out))
        return -1;
    if (n_seg == 0 || n_rows == 0) return 0;
    if (n_tokens <= 0) {
        moe_set_error("q2t_grouped_gate_up: %d rows but no tokens", n_rows);
        return -1;
    }
    return dispatch_proj<kGateUp>(hidden, x, n_tokens, row_token, nullptr, 0, seg_start, seg_slot, n_seg, n_rows, E,
                                  n_slots, hidden, inter, h_out, s);
}

int launch_q2t_grouped_down(const __half* h, int n_rows, const int32_t* row_out, int n_out_rows,
                            const int32_t* seg_start, const int32_t* seg_slot, int n_seg, const Q2Experts& E,
                            int n_slots, int hidden, int inter, int group, __half* y_out, hipStream_t s) {
    if (!check_grouped("q2t_grouped_down", hidden, inter, group, n_seg, n_rows, E.p[2].w, ~size_t(0), n_slots, h,
                       seg_start, y_out))
        return -1;
    if (n_seg == 0 || n_rows == 0) return 0;
    return dispatch_proj<kDown>(inter, h, n_rows, nullptr, row_out, row_out ? n_out_rows : n_rows, seg_start, seg_slot,
                                n_seg, n_rows, E, n_slots, hidden, inter, y_out, s);
}

int launch_pair_combine(const __half* y, const __half* scores, const __half* residual, int n_tokens, int k,
                        int hidden, float* out, hipStream_t s) {
    if (n_tokens < 0 || k <= 0 || hidden <= 0 || n_tokens > 65535) {
        moe_set_error("pair_combine: n_tokens=%d (<= 65535) k=%d hidden=%d", n_tokens, k, hidden);
        return -1;
    }
    if (n_tokens == 0) return 0;
    if (!y || !scores || !out) { moe_set_error("pair_combine: null pointer"); return -1; }
    const bool aligned = ((uintptr_t)y | (uintptr_t)out | (uintptr_t)residual) % 16 == 0;
    if (hidden % 8 == 0 && aligned && k <= MOE_MAX_K) {
        dim3 grid((hidden / 8 + 255) / 256, n_tokens);
        MOE_LAUNCH(TK_COMBINE, k_pair_combine8, grid, dim3(256), 0, s, y, scores, residual, k, hidden, out);
    } else {
        dim3 grid(((hidden + 1) / 2 + 255) / 256, n_tokens);
        MOE_LAUNCH(TK_COMBINE, k_pair_combine, grid, dim3(256), 0, s, y, scores, residual, k, hidden, out);
    }
    HIP_TRY(hipGetLastError());
    return 0;
}
