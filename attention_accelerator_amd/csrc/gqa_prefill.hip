// gqa_prefill.hip -- chunked prefill (multi-query GQA) on MFMA for gfx950, and the KV
// append with RoPE on insert.
//
// The reference core computes one query token per start (gqa_controller.v:140-277;
// golden pyfiles/gen_gqa_wrapper_vectors.py:121-139).  A prefill chunk is that step for
// T consecutive tokens of a sequence: token t sits at position start+t and attends to
// keys p <= start+t (the causal half of gqa_attention_wrapper.v:279), where keys
// p < start are cache rows as stored (post-RoPE) and keys start..start+T-1 are the
// chunk's own K/V rows, rotated at their positions in double and not re-rounded, as
// the golden rotates K (gen_gqa_wrapper_vectors.py:124-126).
//
// Four launches, or five where few query blocks have their keys cut into runs, then the fp64
// rescore of flagged rows (gqa_decode.hip):
//
// kv_append_kernel writes the chunk's K rows (rotated, rounded double -> f32 -> BF16,
// pyfiles/gqa_reference.py:15-19) and V rows into the cache, and the rotated K rows in fp32
// (24 bits, not rounded to BF16) into the workspace.
//
// prefill_stage_kernel copies the K/V rows the attention reads -- cache rows before the
// chunk, the chunk's rows -- into fp16 planes in the workspace, one power-of-two scale per
// (sequence, KV head, block of 64 positions) putting the block's largest magnitude in
// [2^14, 2^15).  A BF16 value has an 8-bit significand, so it converts exactly unless it
// lies more than ~2^31 below that largest magnitude; a chunk key's fp32 value becomes two
// fp16 parts (leading + trailing, ~22 bits).  A block holding a non-finite value, a scale
// outside the fp32 range the attention kernel uses, or a row more than 2^12 below the
// block's largest magnitude is marked, and the attention kernel hands all rows that read
// it to the fp64 rescore.  It also leaves each block's K pair-group norm and |V| maxima.
//
// prefill_stat_reduce_kernel folds those block maxima into the maxima over the keys each
// chunk block's rows see (the rescore flag's statistics).
//
// prefill_attn_kernel: one workgroup of 8 waves per (sequence, KV head, 32 query
// positions); wave w computes Q head 4*kv_head + (w & 3) for 16 positions.  The staged
// rows of each 64-key block are copied once per workgroup into LDS and used by all 4
// heads of the group and all 32 positions (gqa_kv_broadcast.v:38-59 at block scale).
// K runs one block ahead of V, so that each wave forms block j's probabilities while its
// MFMAs form block j+1's scores, then accumulates block j's V^T P^T.
//
//  * Scores S^T = K Q^T with v_mfma_f32_16x16x32_f16: A = 16 keys x 32 dims of K from
//    LDS (row = key), B = Q^T (column = query) held in registers.  Q is rotated and
//    scaled by scale*log2(e) in double, scaled by a power of two per query row, and split
//    into two fp16 parts (11-bit significands: ~22 bits of Q); the products are exact in
//    fp32.  Blocks with chunk keys add the trailing part of K against Q's leading part.
//    Lane (g, n) ends with the scores of keys 4g+i (i = 0..3) of each 16-key tile for
//    query n, times 2^(q scale + block K scale), which one multiply removes.
//  * Online softmax per query with an integer-valued running max (every rescale is an
//    exact power of two), p = exp2(s - m) in fp32, masked keys p = 0 exactly.
//  * O^T += V^T P^T with the same MFMA: A = 16 dims x 32 keys of V^T from LDS, B = P^T.
//    The lane already holds P for keys {4g+i} of tiles 2w and 2w+1, which is its B
//    operand for the 32-key window w if V^T stores each window's keys in that order
//    (slot 8g+4h+i <-> key 16h+4g+i).  P, scaled by 2^12, is split into two fp16 parts
//    (rounded to nearest: ~22 bits).  The fp32 products of a group of up to four cached
//    blocks, or of one block holding chunk keys, are scaled by the group's V scale into an
//    fp64 accumulator, so that accumulation over thousands of keys adds no fp32 rounding.
//  * O / l, rounded double -> f32 -> BF16, written in Q-head order; the row's rescore flag
//    decided from those BF16 values (pf_flag_row).
//
// prefill_merge_kernel: where a query block's keys were cut into runs, a workgroup each, sums
// the runs' fp64 partials and ends the rows in the attention kernel's stead.
//
// Chunks of at most 16 new tokens take the multi-token decode path instead
// (gqa_multitoken.hip), which shares this file's LDS row layout (gqa_prefill_common.h).
#include <type_traits>

#include "gqa_device.h"
#include "gqa_internal.h"
#include "gqa_prefill_common.h"

namespace gqa {

namespace {

constexpr int kPfPos = 32;                 // query positions per workgroup
constexpr int kPfWaves = 8;                // 4 Q heads x 2 tiles of 16 positions
constexpr int kPfThreads = kPfWaves * kWave;
constexpr int kPfBlk = 64;                 // keys per K/V block
constexpr int kStgThreads = 256;           // staging workgroup: 4 threads per row of a block
constexpr int kStgMaxWgs = 8192;
constexpr int kPScaleExp = 12;             // P is formed as 2^12 * 2^(s - m) <= 4096

// Key splits of the attention kernel.  One workgroup per (sequence, KV head, 32 positions)
// leaves most of the chip idle for a short chunk of one or a few sequences (200 tokens of one
// sequence: 56 workgroups on 256 CUs), however long the context is.  When the CUs hold the
// query blocks at least twice over (a workgroup's LDS and registers fill a CU), each query
// block's keys are cut into up to n_split runs of whole blocks, one workgroup each, whose fp64
// partials prefill_merge_kernel combines: as many as fit in one round of the CUs, so that a
// split never adds a round.  Every run but the last has at least kPfMinRun blocks (a workgroup
// costs about 15 us, its launch included, besides its blocks of 1.6 us each, measured with 8
// to 128 blocks; and a partial is 136 KB to write and read).
constexpr int kPfMaxSplit = 32;
constexpr int kPfMinRun = 4;

size_t al256(size_t x) { return (x + 255) / 256 * 256; }

// A split workgroup's partial: per wave and lane 32 doubles of O, and (l, m, u).
constexpr size_t kSplitOB = size_t{kPfWaves} * kWave * 32 * sizeof(double);
struct SplitMl {
    double l;
    float m;
    float u;
};
constexpr size_t kSplitMlB = size_t{kPfWaves} * kWave * sizeof(SplitMl);

// Workgroups of the attention kernel without a split.
int64_t query_blocks(int32_t batch, int32_t n_new) {
    return static_cast<int64_t>(batch) * kHkv * ((n_new + kPfPos - 1) / kPfPos);
}

// Runs that the keys of `capacity` positions can be cut into: kPfMinRun blocks each, at most
// kPfMaxSplit.
int32_t most_runs(int32_t capacity) {
    const int32_t n = (capacity + kPfBlk - 1) / kPfBlk / kPfMinRun;
    return n < 2 ? 1 : n > kPfMaxSplit ? kPfMaxSplit : n;
}

// Partials a workspace has room for: at least those of this call's split, and of every smaller
// call's (fewer sequences or tokens may be cut into more runs), so that a workspace made for a
// program's largest chunk holds its shorter ones too.
size_t split_slots(int32_t batch, int32_t n_new, int32_t capacity, int32_t cus) {
    if (cus < 2 * kHkv || most_runs(capacity) == 1) return 0;      // (the smallest call has kHkv query blocks)
    const int64_t most = query_blocks(batch, n_new) * most_runs(capacity);
    return static_cast<size_t>(most < cus ? most : cus);
}

// The runs of a query block of n_blk key blocks: `per` blocks each, n of them (1: no partial).
__device__ __forceinline__ int pf_runs(int n_blk, int n_split, int& per) {
    const int want = max(1, min(n_split, n_blk / kPfMinRun));
    per = (n_blk + want - 1) / want;
    return (n_blk + per - 1) / per;
}

}  // namespace

// (The lengths are on the device: the capacity bounds what they can ask for.  A prompt of 200
// tokens in a cache of 256 has one run per query block: no idle workgroups, no merge launch.)
int32_t prefill_splits(int32_t batch, int32_t n_new, int32_t capacity, int32_t cus) {
    const int64_t n = cus / query_blocks(batch, n_new);
    const int64_t most = most_runs(capacity);
    return n < 2 ? 1 : static_cast<int32_t>(n < most ? n : most);
}

// ---------------------------------------------------------------------------------
// Workspace of the prefill attention path: the rotated new K rows in fp32, the fp16 K and
// V planes, the trailing-part planes of the chunk blocks and the block scale words.
size_t prefill_stage_bytes(int32_t batch, int32_t n_new, int32_t capacity, int32_t cus) {
    const size_t rows = static_cast<size_t>(batch) * n_new * kHkv;
    const size_t pos = (static_cast<size_t>(capacity) + kPfBlk - 1) / kPfBlk * kPfBlk;
    const size_t cb = static_cast<size_t>(prefill_chunk_blocks(n_new));
    const size_t bh = static_cast<size_t>(batch) * kHkv;
    return al256(rows * kD * sizeof(float)) + 2 * al256(bh * pos * kD * sizeof(uint16_t)) +
           al256(bh * cb * kPfBlk * kD * sizeof(uint16_t)) + al256(bh * (pos / kPfBlk) * sizeof(uint32_t)) +
           split_slots(batch, n_new, capacity, cus) * (kSplitOB + kSplitMlB);
}

void prefill_stage_layout(PrefillArgs& a, void* base) {
    const size_t rows = static_cast<size_t>(a.batch) * a.n_new * kHkv;
    a.stg_pos = (a.capacity + kPfBlk - 1) / kPfBlk * kPfBlk;
    a.stg_cb = prefill_chunk_blocks(a.n_new);
    const size_t bh = static_cast<size_t>(a.batch) * kHkv;
    char* p = static_cast<char*>(base);
    a.kx32 = reinterpret_cast<float*>(p);
    p += al256(rows * kD * sizeof(float));
    a.stg_k = reinterpret_cast<uint16_t*>(p);
    p += al256(bh * a.stg_pos * kD * sizeof(uint16_t));
    a.stg_v = reinterpret_cast<uint16_t*>(p);
    p += al256(bh * a.stg_pos * kD * sizeof(uint16_t));
    a.stg_klo = reinterpret_cast<uint16_t*>(p);
    p += al256(bh * a.stg_cb * kPfBlk * kD * sizeof(uint16_t));
    a.stg_scale = reinterpret_cast<uint32_t*>(p);
    p += al256(bh * (a.stg_pos / kPfBlk) * sizeof(uint32_t));
    a.sp_o = reinterpret_cast<double2*>(p);
    a.sp_ml = p + static_cast<size_t>(query_blocks(a.batch, a.n_new)) * a.n_split * kSplitOB;
}

// ---------------------------------------------------------------------------------
// KV append: one 4-wave workgroup per new (sequence, token), two KV heads per wave; lane i
// computes the angle of frequency i at position start+t (pyfiles/gen_gqa_wrapper_vectors.py:
// 30-31) and rotates the pair (i, i+64) of its heads' rows in double (:25-35).  The new rows do
// not depend on the start position or the block id, so they are requested together with
// them: a wave waits for memory once, or twice for a paged cache.  (All 8 heads per wave, the
// rows after the start: one token of 24 sequences, paged, 6.7 us, now 4.3 us.)
__global__ __launch_bounds__(256) void kv_append_kernel(PrefillArgs a) {
    constexpr int kHeads = 2;
    const int64_t bt = blockIdx.x;                  // b * T + t
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & (kWave - 1);
    if (bt == 0) rs_clear(a, threadIdx.x);
    const int t = static_cast<int>(bt % a.n_new);
    const int b = static_cast<int>(bt / a.n_new);
    const int st = a.start[b];
    const int h0 = kHeads * wave;
    uint16_t kx[kHeads], ky[kHeads], vx[kHeads], vy[kHeads];
#pragma unroll
    for (int h = 0; h < kHeads; ++h) {
        const int64_t row = (bt * kHkv + h0 + h) * kD + lane;
        kx[h] = a.k_new[row];
        ky[h] = a.k_new[row + kPairs];
        vx[h] = a.v_new[row];
        vy[h] = a.v_new[row + kPairs];
    }
    // The rescore's counters start at zero (also for a sequence whose start is out of range:
    // the tile counters are indexed by tile, not by row).
    if (a.rs_hdr) {
        if (threadIdx.x < kHq) a.rs_done[bt * kHq + threadIdx.x] = 0u;
        if (t == 0 && threadIdx.x < kHkv) a.rs_gcnt[b * kHkv + threadIdx.x] = 0u;
    }
    if (!prefill_start_ok(a, st)) return;
    const int64_t pos = static_cast<int64_t>(st) + t;
    const int64_t ce0 = cache_elem(a, b, h0, pos);
    const bool rope = (a.flags & 2u) != 0;
    double sn = 0.0, cs = 1.0;
    const bool any_rope = (a.flags & 3u) != 0;        // the rescore rotates Q with these too
    if (any_rope) rope_sincos(pos, a.rope.inv_freq[lane], sn, cs);
    if (a.rs_hdr && any_rope && wave == 0) a.rs_cs[bt * kPairs + lane] = make_double2(cs, sn);
#pragma unroll
    for (int h = 0; h < kHeads; ++h) {
        const double x = bf16_to_f32(kx[h]);
        const double y = bf16_to_f32(ky[h]);
        double xr = x, yr = y;
        if (rope) {
            xr = x * cs - y * sn;
            yr = x * sn + y * cs;
        }
        if (ce0 >= 0) {
            uint16_t* kdst = a.k + ce0 + h * a.kv_head_stride;
            uint16_t* vdst = a.v + ce0 + h * a.kv_head_stride;
            kdst[lane] = bf16_of(xr);
            kdst[lane + kPairs] = bf16_of(yr);
            vdst[lane] = vx[h];
            vdst[lane + kPairs] = vy[h];
        }
        if (a.kx32) {
            float* kr = a.kx32 + (bt * kHkv + h0 + h) * kD;
            kr[lane] = static_cast<float>(xr);
            kr[lane + kPairs] = static_cast<float>(yr);
        }
    }
}

hipError_t launch_kv_append(const PrefillArgs& a, hipStream_t stream) {
    const int64_t n_tok = static_cast<int64_t>(a.batch) * a.n_new;
    if (n_tok == 0) return hipSuccess;
    hipLaunchKernelGGL(kv_append_kernel, dim3(static_cast<unsigned>(n_tok)), dim3(256), 0, stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Staging.

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// Two floats -> two fp16 codes in one dword, each rounded to nearest (v_cvt_pk_f16_f32).
__device__ __forceinline__ uint32_t pk_f16(float lo, float hi) {
    f16x2_t h;
    h[0] = static_cast<_Float16>(lo);
    h[1] = static_cast<_Float16>(hi);
    return __builtin_bit_cast(uint32_t, h);
}

// A double rounded to fp32, opaque to the compiler: it merges the conversion with a following
// one to fp16 into a double -> fp16 conversion, which gfx950 does not have and which it
// expands to about 40 instructions (one v_cvt_f32_f64 and half a v_cvt_pk_f16_f32 here).
__device__ __forceinline__ float f32_of(double x) {
    float f = static_cast<float>(x);
    asm("" : "+v"(f));
    return f;
}

__device__ __forceinline__ float f16_lo(uint32_t w) { return static_cast<float>(__builtin_bit_cast(f16x2_t, w)[0]); }
__device__ __forceinline__ float f16_hi(uint32_t w) { return static_cast<float>(__builtin_bit_cast(f16x2_t, w)[1]); }

// x - (fp16 half of h), exact, in one instruction: v_fma_mix_f32 reads the half as fp16
// (op_sel_hi) and computes -h * 1 + x with one rounding, and x - h is representable.
__device__ __forceinline__ float sub_f16_lo(float x, uint32_t h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
__device__ __forceinline__ float sub_f16_hi(float x, uint32_t h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}

// Scale exponent putting magnitude bits `mb` (fp32, sign cleared) in [2^14, 2^15): 14 - floor(log2).
// 0 for zero.  Exponents outside [-100, 100] mark the block (the attention kernel keeps the
// factor 2^-scale in the fp32 normal range) and are clamped.
__device__ __forceinline__ int stg_scale_exp(uint32_t mb, bool& bad) {
    if (mb == 0u) return 0;
    const int e = static_cast<int>(mb >> 23) - 127;
    if (e < -100 || e > 100) bad = true;
    return 14 - (e < -100 ? -100 : e > 100 ? 100 : e);
}

__device__ __forceinline__ float pow2f(int e) { return __uint_as_float(static_cast<uint32_t>(127 + e) << 23); }

// Statistics of one staged block for the rescore flag: thread (r, qq) holds pair groups 2qq
// and 2qq+1 of row r whole (dims 16qq .. 16qq+15 and 64+16qq ..), so its two squared group
// norms need no other thread, and the |V| codes of its 32 dims.  stg_stats_put writes the
// block's rows to LDS ([64 rows][64 dwords] of |V| codes, dword c = dims 2c and 2c+1; [64
// rows][8] norms) before the kernel's own barrier; after it, stg_stats_take reduces
// columns, one wave per 16 dword columns and 2 norm groups: a block of cached rows stores
// its maxima (rs_kblk / rs_dblk, folded over the cache by prefill_stat_reduce_kernel), a
// block holding chunk keys the maxima over its rows up to each row (rs_kpre / rs_dpre).
struct StgStatLds {
    uint32_t v[kPfBlk][kD / 2];
    uint32_t k[kPfBlk][8];
};

// n0, n1: the squared norms of pair groups 2qq and 2qq + 1 of the row's K; vw: its V as
// BF16 codes (dims 16qq .. +7, 16qq + 8 .., 64 + 16qq .., 64 + 16qq + 8 ..).
__device__ __forceinline__ void stg_stats_put(int r, int qq, float n0, float n1, const uint4 (&vw)[4],
                                              StgStatLds& sl) {
    uint4* vrow = reinterpret_cast<uint4*>(&sl.v[r][0]);
    const uint32_t m = 0x7fff7fffu;
    vrow[2 * qq] = make_uint4(vw[0].x & m, vw[0].y & m, vw[0].z & m, vw[0].w & m);
    vrow[2 * qq + 1] = make_uint4(vw[1].x & m, vw[1].y & m, vw[1].z & m, vw[1].w & m);
    vrow[8 + 2 * qq] = make_uint4(vw[2].x & m, vw[2].y & m, vw[2].z & m, vw[2].w & m);
    vrow[8 + 2 * qq + 1] = make_uint4(vw[3].x & m, vw[3].y & m, vw[3].z & m, vw[3].w & m);
    sl.k[r][2 * qq] = __float_as_uint(n0);
    sl.k[r][2 * qq + 1] = __float_as_uint(n1);
}

// Largest |x| over 8 BF16 codes, as fp32 bits (NaN and infinity above every finite value).
__device__ __forceinline__ uint32_t stg_absmax8(const uint4& w) {
    const uint32_t m = pk_max_u16(pk_max_u16(w.x & 0x7fff7fffu, w.y & 0x7fff7fffu),
                                  pk_max_u16(w.z & 0x7fff7fffu, w.w & 0x7fff7fffu));
    return max(m << 16, m & 0x7fff0000u);
}

// Two BF16 codes (one dword) times f, as two fp16 codes.
__device__ __forceinline__ uint32_t stg_f16x2(uint32_t w, float f) {
    return pk_f16(__uint_as_float(w << 16) * f, __uint_as_float(w & 0xffff0000u) * f);
}

__device__ __forceinline__ void stg_stats_take(const PrefillArgs& a, int bh, int blk, int st, int wave, int lane,
                                               const StgStatLds& sl) {
    // Wave w: |V| dword columns 16w .. 16w+15 (lane: column 16w + (lane & 15), rows
    // 16 (lane >> 4) .. +15) and norm groups 2w, 2w+1 (lane: group 2w + (lane & 1), rows
    // 2 (lane >> 1) and +1).
    const int col = 16 * wave + (lane & 15);
    const int rg = lane >> 4;
    const int kg = 2 * wave + (lane & 1);
    const int kr = 2 * (lane >> 1);
    if (blk * kPfBlk + kPfBlk - 1 < st) {
        uint32_t x = 0u;
#pragma unroll
        for (int i = 0; i < 16; ++i) x = pk_max_u16(x, sl.v[16 * rg + i][col]);
        x = pk_max_u16(x, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), 16)));
        x = pk_max_u16(x, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), 32)));
        const int64_t e = static_cast<int64_t>(bh) * a.rs_nblk + blk;
        if (rg == 0) a.rs_dblk[e * (kD / 2) + col] = x;
        uint32_t y = max(sl.k[kr][kg], sl.k[kr + 1][kg]);
#pragma unroll
        for (int sh = 2; sh < kWave; sh <<= 1) y = max(y, static_cast<uint32_t>(__shfl_xor(static_cast<int>(y), sh)));
        if (lane < 2) a.rs_kblk[e * 8 + kg] = y;
        return;
    }
    // Running maxima down the rows: within each lane's 16 (or 2) rows, then the earlier
    // lanes' totals (row groups 16 and 32 lanes apart; norm rows 2, 4, .. lanes apart).
    const int cb = blk - st / kPfBlk;
    const int64_t e0 = (static_cast<int64_t>(bh) * a.rs_ncb + cb) * a.rs_nr;
    uint32_t run[16];
    uint32_t x = 0u;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        x = pk_max_u16(x, sl.v[16 * rg + i][col]);
        run[i] = x;
    }
    uint32_t carry = 0u;
    {
        const uint32_t t16 = static_cast<uint32_t>(__shfl_up(static_cast<int>(x), 16));
        const uint32_t t32 = static_cast<uint32_t>(__shfl_up(static_cast<int>(x), 32));
        const uint32_t t48 = static_cast<uint32_t>(__shfl_up(static_cast<int>(x), 48));
        if (rg >= 1) carry = pk_max_u16(carry, t16);
        if (rg >= 2) carry = pk_max_u16(carry, t32);
        if (rg >= 3) carry = pk_max_u16(carry, t48);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
        *reinterpret_cast<uint32_t*>(a.rs_dpre + (e0 + 16 * rg + i) * kD + 2 * col) = pk_max_u16(run[i], carry);
    const uint32_t y0 = sl.k[kr][kg];
    const uint32_t y1 = max(y0, sl.k[kr + 1][kg]);
    uint32_t yc = 0u;
#pragma unroll
    for (int sh = 2; sh < kWave; sh <<= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(max(y1, yc)), sh));
        if (lane >= sh) yc = max(yc, o);
    }
    a.rs_kpre[(e0 + kr) * 8 + kg] = max(y0, yc);
    a.rs_kpre[(e0 + kr + 1) * 8 + kg] = max(y1, yc);
}

// One workgroup per (sequence, KV head, 64-position block) of the positions the attention
// reads, [0, start + T); thread (r, qq) holds dims 16qq .. 16qq+15 and 64+16qq .. of row r.
// Rows past start + T in the last block are written as zeros (the attention kernel copies
// whole blocks and masks them).
__global__ __launch_bounds__(kStgThreads) void prefill_stage_kernel(PrefillArgs a) {
    __shared__ uint32_t red[2][kStgThreads / kWave];
    __shared__ StgStatLds stat_s;
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & (kWave - 1);
    const int r = tid >> 2;
    const int qq = tid & 3;
    const int nblk = a.stg_pos / kPfBlk;
    const int64_t n_items = static_cast<int64_t>(a.batch) * kHkv * nblk;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const int blk = static_cast<int>(item % nblk);
        const int bh = static_cast<int>(item / nblk);
        const int b = bh / kHkv;
        const int h = bh % kHkv;
        const int st = a.start[b];
        if (!prefill_start_ok(a, st)) continue;
        const int n_keys = st + a.n_new;
        if (blk * kPfBlk >= n_keys) continue;
        const int p = blk * kPfBlk + r;
        // This thread's 32 dims of the row (16-byte pieces c: dims 16qq + 8c for c < 2, 64 +
        // 16qq + 8(c - 2) after): V and cached K kept as BF16 codes; a chunk row's K (fp32,
        // from the append) is read here for its maxima and norms and again for conversion.
        uint4 vw[4], kw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) vw[c] = kw[c] = make_uint4(0u, 0u, 0u, 0u);
        bool bad = false;
        const bool chunk_row = p >= st && p < n_keys;
        const float* kx = a.kx32 + ((static_cast<int64_t>(b) * a.n_new + (p - st)) * kHkv + h) * kD;
        uint32_t rk = 0u, rv = 0u;
        float n0 = 0.f, n1 = 0.f;
        if (p < n_keys) {
            const int64_t ce = cache_elem(a, b, h, p);
            if (ce < 0) {
                bad = true;
            } else {
                const char* vr = reinterpret_cast<const char*>(a.v + ce);
#pragma unroll
                for (int c = 0; c < 4; ++c) vw[c] = load_stream16(vr + 128 * (c >> 1) + 32 * qq + 16 * (c & 1));
                if (!chunk_row) {
                    const char* kr = reinterpret_cast<const char*>(a.k + ce);
#pragma unroll
                    for (int c = 0; c < 4; ++c) kw[c] = load_stream16(kr + 128 * (c >> 1) + 32 * qq + 16 * (c & 1));
                    rk = max(max(stg_absmax8(kw[0]), stg_absmax8(kw[1])), max(stg_absmax8(kw[2]), stg_absmax8(kw[3])));
                    const uint32_t g0[8] = {kw[0].x, kw[0].y, kw[0].z, kw[0].w, kw[2].x, kw[2].y, kw[2].z, kw[2].w};
                    const uint32_t g1[8] = {kw[1].x, kw[1].y, kw[1].z, kw[1].w, kw[3].x, kw[3].y, kw[3].z, kw[3].w};
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        n0 = bf16x2_sq_acc(g0[i], n0);
                        n1 = bf16x2_sq_acc(g1[i], n1);
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        // dims 16qq + 4c (c < 4), 64 + 16qq + 4(c - 4): groups 2qq + ((c >> 1) & 1)
                        const float4 f = *reinterpret_cast<const float4*>(kx + 64 * (c >> 2) + 16 * qq + 4 * (c & 3));
                        rk = max(rk, max(max(__float_as_uint(f.x) & 0x7fffffffu, __float_as_uint(f.y) & 0x7fffffffu),
                                         max(__float_as_uint(f.z) & 0x7fffffffu, __float_as_uint(f.w) & 0x7fffffffu)));
                        const float sq = fmaf(f.x, f.x, fmaf(f.y, f.y, fmaf(f.z, f.z, f.w * f.w)));
                        if ((c >> 1) & 1) n1 += sq;
                        else n0 += sq;
                    }
                }
                rv = max(max(stg_absmax8(vw[0]), stg_absmax8(vw[1])), max(stg_absmax8(vw[2]), stg_absmax8(vw[3])));
            }
        }
        // Largest magnitudes as fp32 bit patterns: per row over its four threads, then over
        // the block.
        rk = max(rk, static_cast<uint32_t>(__shfl_xor(static_cast<int>(rk), 1)));
        rk = max(rk, static_cast<uint32_t>(__shfl_xor(static_cast<int>(rk), 2)));
        rv = max(rv, static_cast<uint32_t>(__shfl_xor(static_cast<int>(rv), 1)));
        rv = max(rv, static_cast<uint32_t>(__shfl_xor(static_cast<int>(rv), 2)));
        uint32_t wk = rk, wv = rv;
#pragma unroll
        for (int sh = 4; sh < kWave; sh <<= 1) {
            wk = max(wk, static_cast<uint32_t>(__shfl_xor(static_cast<int>(wk), sh)));
            wv = max(wv, static_cast<uint32_t>(__shfl_xor(static_cast<int>(wv), sh)));
        }
        __syncthreads();                      // red and stat_s are rewritten for every item
        if (lane == 0) {
            red[0][wave] = wk;
            red[1][wave] = wv;
        }
        if (a.rs_hdr) stg_stats_put(r, qq, n0, n1, vw, stat_s);
        __syncthreads();
        uint32_t bk = 0u, bv = 0u;
#pragma unroll
        for (int w = 0; w < kStgThreads / kWave; ++w) {
            bk = max(bk, red[0][w]);
            bv = max(bv, red[1][w]);
        }
        if (bk >= 0x7f800000u || bv >= 0x7f800000u) bad = true;
        const int sk = stg_scale_exp(bk, bad);
        const int sv = stg_scale_exp(bv, bad);
        // A row far below the block's largest magnitude would keep fewer bits of its small
        // elements than the attention's error bound allows.
        if (bk >= (13u << 23) && rk != 0u && rk < bk - (12u << 23)) bad = true;
        if (bv >= (13u << 23) && rv != 0u && rv < bv - (12u << 23)) bad = true;
        const bool any_bad = __syncthreads_or(bad);
        const float fk = pow2f(sk), fv = pow2f(sv);
        const int64_t row = static_cast<int64_t>(bh) * a.stg_pos + p;
        char* ko = reinterpret_cast<char*>(a.stg_k + row * kD);
        char* vo = reinterpret_cast<char*>(a.stg_v + row * kD);
        const bool chunk_blk = blk * kPfBlk + kPfBlk - 1 >= st;
        char* lo = reinterpret_cast<char*>(
            a.stg_klo + ((static_cast<int64_t>(bh) * a.stg_cb + (blk - st / kPfBlk)) * kPfBlk + r) * kD);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int off = 128 * (c >> 1) + 32 * qq + 16 * (c & 1);
            *reinterpret_cast<uint4*>(vo + off) = make_uint4(stg_f16x2(vw[c].x, fv), stg_f16x2(vw[c].y, fv),
                                                             stg_f16x2(vw[c].z, fv), stg_f16x2(vw[c].w, fv));
            uint4 kh, kl = make_uint4(0u, 0u, 0u, 0u);
            if (!chunk_row) {
                kh = make_uint4(stg_f16x2(kw[c].x, fk), stg_f16x2(kw[c].y, fk), stg_f16x2(kw[c].z, fk),
                                stg_f16x2(kw[c].w, fk));
            } else {
                // the fp32 row as two fp16 parts (leading, trailing)
                const float* src = kx + 64 * (c >> 1) + 16 * qq + 8 * (c & 1);
                const float4 f0 = *reinterpret_cast<const float4*>(src);
                const float4 f1 = *reinterpret_cast<const float4*>(src + 4);
                const float x[8] = {f0.x * fk, f0.y * fk, f0.z * fk, f0.w * fk, f1.x * fk, f1.y * fk, f1.z * fk, f1.w * fk};
                uint32_t hh[4], ll[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    hh[j] = pk_f16(x[2 * j], x[2 * j + 1]);
                    ll[j] = pk_f16(x[2 * j] - f16_lo(hh[j]), x[2 * j + 1] - f16_hi(hh[j]));
                }
                kh = make_uint4(hh[0], hh[1], hh[2], hh[3]);
                kl = make_uint4(ll[0], ll[1], ll[2], ll[3]);
            }
            *reinterpret_cast<uint4*>(ko + off) = kh;
            if (chunk_blk) *reinterpret_cast<uint4*>(lo + off) = kl;
        }
        if (tid == 0)
            a.stg_scale[static_cast<int64_t>(bh) * nblk + blk] =
                (static_cast<uint32_t>(sk) & 0xffu) | ((static_cast<uint32_t>(sv) & 0xffu) << 8) |
                (any_bad ? 0x80000000u : 0u);
        if (a.rs_hdr) stg_stats_take(a, bh, blk, st, wave, lane, stat_s);
    }
}

// The maxima over the keys before each chunk block of a (sequence, KV head): the blocks of
// cached rows only (the block maxima the staging kernel wrote) folded by 16 partial sweeps
// (thread t: dword column t % 64 of every 16th block; norm group t % 8 of every 64th),
// meeting in LDS; then, chunk block by chunk block, the previous chunk blocks' maxima (row
// 63 of their running maxima).
// Bound by its round trips: a chunk block's row read only after the one before was stored was 17
// of them for 1000 tokens; eight at a time, two prompts of 1000 tokens step 120.1 -> 117.2 us.
__global__ __launch_bounds__(1024) void prefill_stat_reduce_kernel(PrefillArgs a) {
    __shared__ uint32_t vpart[16][kD / 2];
    __shared__ uint32_t kpart[64][8];
    constexpr int kAhead = 8;             // chunk blocks whose last rows are requested together
    const int bh = blockIdx.x;
    const int tid = threadIdx.x;
    const int st = a.start[bh / kHkv];
    const int n_cached = prefill_start_ok(a, st) ? st / kPfBlk : 0;
    {
        const int col = tid & 63, sub = tid >> 6;
        const uint32_t* vb = a.rs_dblk + static_cast<int64_t>(bh) * a.rs_nblk * (kD / 2) + col;
        uint32_t x = 0u;
        for (int i0 = sub; i0 < n_cached; i0 += 16 * 8) {
            uint32_t w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                w[j] = i0 + 16 * j < n_cached ? vb[static_cast<int64_t>(i0 + 16 * j) * (kD / 2)] : 0u;
#pragma unroll
            for (int j = 0; j < 8; ++j) x = pk_max_u16(x, w[j]);
        }
        vpart[sub][col] = x;
    }
    if (tid < 512) {
        const int g = tid & 7, ks = tid >> 3;
        const uint32_t* kb = a.rs_kblk + static_cast<int64_t>(bh) * a.rs_nblk * 8 + g;
        uint32_t y = 0u;
        for (int i0 = ks; i0 < n_cached; i0 += 64 * 4) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = i0 + 64 * j < n_cached ? kb[static_cast<int64_t>(i0 + 64 * j) * 8] : 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) y = max(y, w[j]);
        }
        kpart[ks][g] = y;
    }
    __syncthreads();
    if (tid < kD / 2) {
        uint32_t v = 0u;
#pragma unroll
        for (int i = 0; i < 16; ++i) v = pk_max_u16(v, vpart[i][tid]);
        // Chunk block cb: the cached maxima and chunk blocks 0 .. cb-1 (their last row).
        const int64_t pre0 = static_cast<int64_t>(bh) * a.rs_ncb * a.rs_nr;
        for (int cb = 0; cb < a.rs_ncb; cb += kAhead) {
            uint32_t w[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                w[j] = *reinterpret_cast<const uint32_t*>(
                    a.rs_dpre + (pre0 + static_cast<int64_t>(min(cb + j, a.rs_ncb - 1)) * a.rs_nr + a.rs_nr - 1) * kD + 2 * tid);
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                if (cb + j < a.rs_ncb)
                    *reinterpret_cast<uint2*>(a.rs_dc + (static_cast<int64_t>(bh) * a.rs_ncb + cb + j) * kD + 2 * tid) =
                        make_uint2(v & 0xffffu, v >> 16);
                v = pk_max_u16(v, w[j]);
            }
        }
    } else if (tid < kD / 2 + 8) {
        const int g = tid - kD / 2;
        uint32_t y = 0u;
#pragma unroll 8
        for (int i = 0; i < 64; ++i) y = max(y, kpart[i][g]);
        const int64_t pre0 = static_cast<int64_t>(bh) * a.rs_ncb * a.rs_nr;
        for (int cb = 0; cb < a.rs_ncb; cb += kAhead) {
            uint32_t w[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                w[j] = a.rs_kpre[(pre0 + static_cast<int64_t>(min(cb + j, a.rs_ncb - 1)) * a.rs_nr + a.rs_nr - 1) * 8 + g];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                if (cb + j < a.rs_ncb) a.rs_kc[(static_cast<int64_t>(bh) * a.rs_ncb + cb + j) * 8 + g] = y;
                y = max(y, w[j]);
            }
        }
    }
}

hipError_t launch_prefill_stat_reduce(const PrefillArgs& a, hipStream_t stream) {
    if (!a.rs_hdr) return hipSuccess;
    hipLaunchKernelGGL(prefill_stat_reduce_kernel, dim3(static_cast<unsigned>(a.batch * kHkv)), dim3(1024), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_prefill_stage(const PrefillArgs& a, hipStream_t stream) {
    const int64_t n_items = static_cast<int64_t>(a.batch) * kHkv * (a.stg_pos / kPfBlk);
    if (n_items == 0) return hipSuccess;
    const int64_t grid = n_items < kStgMaxWgs ? n_items : kStgMaxWgs;
    hipLaunchKernelGGL(prefill_stage_kernel, dim3(static_cast<unsigned>(grid)), dim3(kStgThreads), 0, stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Attention.

// LDS: six 16 KB planes of 64 rows x 256 B -- K of buffers 0 and 1, V of buffers 0 and 1,
// the trailing parts of chunk keys for buffers 0 and 1 (96 KB in all).  K runs one block
// ahead of V: while block j's probabilities are formed and its V^T P^T accumulated, block
// j+1's scores are formed from the other K buffer.  Rows are copied from the staging planes
// straight into LDS (global_load_lds_dwordx4: lane l of an instruction writes bytes
// [16l, 16l + 16) of a 1 KB stretch = 4 rows), so a row's 16 16-byte chunks are placed by
// choosing which chunk each lane fetches: chunk c of row r sits at position c ^ pf_swz(r & 15).
// With that swizzle the K operand and V^T transpose reads hit no bank twice, and because it
// depends on r & 15 only, the rows 16 apart that one lane reads differ by a constant offset.
constexpr int kPlaneB = kPfBlk * kRowB;     // 16 KB per plane
constexpr int kOffK = 0;                    // + buffer * kPlaneB
constexpr int kOffV = 2 * kPlaneB;
constexpr int kOffKlo = 4 * kPlaneB;
// Then a ring of block scale words: words for blocks [0, 512) are copied at the start and
// words for blocks [256k + 256, 256k + 512) at step 256k + 128, into the half whose blocks are
// done, so that a word is in LDS 126 steps before it is read.  Copied like the rows (straight into
// LDS, completed by the step's vmcnt(0) wait), it costs no wait of its own: a plain load's
// wait would also wait for the K/V copies in flight.
constexpr int kOffSw = 6 * kPlaneB;
constexpr int kSwRing = 512;
constexpr int kLdsB = 6 * kPlaneB + kSwRing * 4;

// Wave w of the workgroup copies rows 8w .. 8w+7 of a plane (two 4-row instructions).
__device__ __forceinline__ int pf_copy_row(int wave, int ii, int lane) { return 4 * (2 * wave + ii) + (lane >> 4); }

// The lane's byte offset within a staged 64-row block for its two copy instructions.
__device__ __forceinline__ void pf_copy_offsets(int wave, int lane, uint32_t (&loff)[2]) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
        const int r = pf_copy_row(wave, ii, lane);
        loff[ii] = static_cast<uint32_t>(r * kRowB + 16 * ((lane & 15) ^ pf_swz(r)));
    }
}

// Request one staged 64-row block (16 KB at `src`, uniform) into the LDS plane at `dst`.  The
// block's address stays a scalar pair and the lane's offset a 32-bit register (the empty asm
// keeps the compiler from carrying a 64-bit address per lane and plane through the loop).
__device__ __forceinline__ void pf_issue(const char* src, const uint32_t (&loff)[2], uint8_t* dst, int wave) {
    asm("" : "+s"(src));
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
        __builtin_amdgcn_global_load_lds(src + loff[ii], (lds_void_t*)(dst + (2 * wave + ii) * 1024), 16, 0, 0);
}

__device__ __forceinline__ f16x8_t as_f16x8(const uint4& w) { return __builtin_bit_cast(f16x8_t, w); }

// Lane (g, n)'s byte offset in a K plane of its operand for 16-key tile 0, dims 8g .. 8g+7
// (slice 0); slice q is that offset ^ 64 q (the chunk index is swizzled by exclusive or),
// tile kt 4096 kt further.
__device__ __forceinline__ uint32_t pf_k_offset(int n, int g) { return n * kRowB + 16 * (g ^ pf_swz(n)); }

// K operands of half a 32-dim slice: dims 32 (i / 2) .., 16-key tiles 2 (i % 2) and the next.
__device__ __forceinline__ void pf_k_pair(const uint8_t* kplane, int i, uint32_t koff, f16x8_t (&ak)[2]) {
    const uint8_t* p = kplane + (koff ^ (64u * (i >> 1))) + 32 * (i & 1) * kRowB;
    ak[0] = *reinterpret_cast<const f16x8_t*>(p);
    ak[1] = *reinterpret_cast<const f16x8_t*>(p + 16 * kRowB);
}

// The scores S^T[key][query] those operands add to: the 2 fp16 parts of Q against the K
// plane, and for chunk keys the trailing part of K against Q's leading part.
template <bool kNew>
__device__ __forceinline__ void pf_qk_pair(const uint8_t* kplane, const f16x8_t (&ak)[2], const f16x8_t (&qop)[2][4],
                                           int i, uint32_t koff, f32x4_t (&sacc)[4]) {
    const int q = i >> 1, kt = 2 * (i & 1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < 2; ++e)
            sacc[kt + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ak[e], qop[s][q], sacc[kt + e], 0, 0, 0);
    if (kNew) {
        f16x8_t al[2];
        pf_k_pair(kplane + (kOffKlo - kOffK), i, koff, al);
#pragma unroll
        for (int e = 0; e < 2; ++e)
            sacc[kt + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[e], qop[0][q], sacc[kt + e], 0, 0, 0);
    }
}

// Per-tile softmax state: the running max (integer-valued, log2 units), sum and O (fp64,
// lane (g, n): O^T[16dt + 4g + i][query n]), both in units of 2^12 p, and the fp32 sum of
// V^T P^T over the current group of up to kPfGroup blocks (moved into the fp64 O when the
// group closes: fp32 sums over 256 keys add no error measurable against per-block sums).
constexpr int kPfGroup = 4;
struct PfTile {
    double o64[8][4];
    f32x4_t acc[8];
    double l64;
    float m_run;
    float u;           // bound on what fp16's subnormal quantum adds to O (O's units, this lane's keys)
};

// Closes a group: O += acc * cv (cv = 2^-(V scale of the group's blocks), exact).
__device__ __forceinline__ void pf_flush(PfTile& t, double cv) {
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) t.o64[dt][i] = fma(static_cast<double>(t.acc[dt][i]), cv, t.o64[dt][i]);
        t.acc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
}

// Masks a diagonal block's keys past the query at pos_n.
__device__ __forceinline__ void pf_mask(f32x4_t (&sacc)[4], int key0, int g, int pos_n) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (key0 + 16 * kt + 4 * g + i > pos_n) sacc[kt][i] = -INFINITY;
}

// Running max after a block, in two steps: the lane's largest raw score, then ceil(block max)
// where that exceeds the running max m (integer-valued, so every rescale is an exact power of
// two), else m.  `mult` turns the block's raw scores into log2 units.  The two cross-row steps
// are gfx950 lane swaps (rows 16 and 32 lanes apart), not LDS permutes.
__device__ __forceinline__ float pf_lane_max(const f32x4_t (&sacc)[4]) {
    float bmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) bmax = fmaxf(bmax, sacc[kt][i]);
    return bmax;
}

__device__ __forceinline__ float pf_next_max(float bmax, float m, float mult) {
    bmax = swap32_max(swap16_max(bmax)) * mult;
    return bmax > m ? ceilf(bmax) : m;
}

// Moves O, the open group's sum and l to the running max m_new (exact power-of-two scaling;
// an fp32 group term pushed below 2^-149 is below 2^-149 of the new maximum's weight).
__device__ __forceinline__ void pf_rescale(PfTile& t, float m_new) {
    if (__ballot(m_new != t.m_run)) {
        const int shift = (t.m_run == -INFINITY) ? 0 : max_shift(t.m_run, m_new);
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                t.o64[dt][i] = ldexp(t.o64[dt][i], shift);
                t.acc[dt][i] = ldexpf(t.acc[dt][i], shift);
            }
        t.l64 = ldexp(t.l64, shift);
        t.u = ldexpf(t.u, shift);
        t.m_run = m_new;
    }
}

// p = 2^12 * 2^(s - m) of half j of key tile kt (keys 4g + 2j, + 1; 0 for masked keys; s = raw
// score * mult), summed into lsum and split into two fp16 parts rounded to nearest (p = p1 + p2 to 2^-22 relative),
// packed as the P^T B operand: ph[part][window][dword].
__device__ __forceinline__ void pf_probs_half16(const f32x4_t& s, float mult, float off, float& lsum,
                                                uint32_t (&ph)[2][2][4], int kt, int j) {
    float p[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // v_exp_f32: 2^x, 0 for -inf (masked keys); results below 2^-126 flush to 0.
        p[i] = __builtin_amdgcn_exp2f(fmaf(s[2 * j + i], mult, off));
        lsum += p[i];
    }
    const int w = kt >> 1, d0 = (kt & 1) * 2;
    const uint32_t h1 = pk_f16(p[0], p[1]);
    ph[0][w][d0 + j] = h1;
    ph[1][w][d0 + j] = pk_f16(sub_f16_lo(p[0], h1), sub_f16_hi(p[1], h1));
}

// V^T operands of one 16-dim tile dt for both 32-key windows: lane (g, m) gets keys
// 32w + 4g + i (slots 0..3) and 32w + 16 + 4g + i (slots 4..7) of dim 16dt + m, through
// transpose reads (ds_read_b64_tr_b16: lane i of a 16-lane group receives element i%4 of the
// 8 bytes addressed by lane 4j + i/4, j = 0..3).  Supplying lane a addresses row
// 32w + 4g + a/4 (+16), dims 16dt + 4(a%4) .. +3; `addr` is that address for w = 0 without
// the +16, and the other three rows are 16, 32 and 48 rows further.
//
// The reads are issued from inline assembly and waited for by pf_vt_wait: the compiler
// treats every transpose read as possibly reading LDS that an outstanding copy writes and
// would wait for all of them (the next block's copies included) before the first one.  The
// copies that fill the buffer read here completed before the barrier that opened this block.
struct VtPair {
    short4_t r[2][2];   // [window][half]
};

__device__ __forceinline__ VtPair pf_vt_issue(uint32_t addr) {
    VtPair v;
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v.r[0][0]) : "v"(addr));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:4096" : "=v"(v.r[0][1]) : "v"(addr));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:8192" : "=v"(v.r[1][0]) : "v"(addr));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:12288" : "=v"(v.r[1][1]) : "v"(addr));
    return v;
}

// Waits for every outstanding LDS read (lgkmcnt(0)); tied to the operands so that their uses
// stay behind it.
__device__ __forceinline__ void pf_vt_wait(VtPair& v0, VtPair& v1) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(v0.r[0][0]), "+v"(v0.r[0][1]), "+v"(v0.r[1][0]), "+v"(v0.r[1][1]), "+v"(v1.r[0][0]),
                   "+v"(v1.r[0][1]), "+v"(v1.r[1][0]), "+v"(v1.r[1][1]));
}

__device__ __forceinline__ f16x8_t pf_vt_operand(const VtPair& v, int w) {
    union {
        short4_t h[2];
        f16x8_t v;
    } u;
    u.h[0] = v.r[w][0];
    u.h[1] = v.r[w][1];
    return u.v;
}

// A step's instructions are laid out in chunks that the scheduler keeps in this order (it may
// only move instructions inside a chunk): left to itself it hoists the probabilities' VALU
// work out of the MFMAs it should run beside, and sinks LDS reads to just before their use.
__device__ __forceinline__ void pf_chunk_end() { __builtin_amdgcn_sched_barrier(0); }

// The scores of the next block from K buffer `kplane` (kNext: there is one; kNew: it holds chunk
// keys), beside the second half of the current block's probabilities (key tiles 2 and 3: raw
// scores `scur`; the first half was formed beside the previous block's V^T P^T).  Four
// chunks, each two K operand pairs (8 MFMAs), the reads of the pairs two on, and half a key
// tile of probabilities; with kVt the last one also requests the first V^T operands (cur):
// only where no branch lies between the request and its wait.
template <bool kNext, bool kNew, bool kVt>
__device__ __forceinline__ void pf_scores_beside(const f32x4_t (&scur)[4], float mult, float off, float& lsum,
                                                 const uint8_t* kplane, const f16x8_t (&qop)[2][4], uint32_t koff,
                                                 uint32_t vaddr, uint32_t (&ph)[2][2][4], f32x4_t (&snext)[4],
                                                 VtPair (&cur)[2]) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)       // (no next block: as if every key were masked)
        snext[kt] = kNext ? f32x4_t{0.f, 0.f, 0.f, 0.f} : f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    f16x8_t ak[3][2];
    if (kNext) {
        pf_k_pair(kplane, 0, koff, ak[0]);
        pf_k_pair(kplane, 1, koff, ak[1]);
        pf_chunk_end();
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (kNext && i < 6) pf_k_pair(kplane, i + 2, koff, ak[(i + 2) % 3]);
        if (kVt && i == 7) {
            // (after the last K operands have arrived: LDS reads complete in order)
            asm volatile("" : "+v"(ak[1][0]), "+v"(ak[1][1]));
            cur[0] = pf_vt_issue(vaddr);
            cur[1] = pf_vt_issue(vaddr ^ 32u);
        }
        if (kNext) pf_qk_pair<kNew>(kplane, ak[i % 3], qop, i, koff, snext);
        if (!(i & 1)) pf_probs_half16(scur[2 + (i >> 2)], mult, off, lsum, ph, 2 + (i >> 2), (i >> 1) & 1);
        if (kNext && (i & 1)) pf_chunk_end();
    }
}

// The group's fp32 sum += the block's V^T P^T: per 16-dim tile, V^T (transpose reads) against
// the two P parts of both 32-key windows; two tiles at a time, the next two tiles' operands
// requested before the current two's products (cur: tiles 0 and 1, requested already).
// vaddr: the lane's transpose-read address of dim tile 0; tile dt is vaddr ^ 32 dt (its chunk
// index 2 dt is swizzled by exclusive or, and the planes are aligned).  beside(i), i < 4:
// work to place among the products of tiles 2i and 2i + 1.
template <class F>
__device__ __forceinline__ void pf_pv(uint32_t vaddr, const uint32_t (&ph)[2][2][4], VtPair (&cur)[2], PfTile& t,
                                      F&& beside) {
    f16x8_t pb[2][2];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int s = 0; s < 2; ++s) pb[w][s] = as_f16x8(make_uint4(ph[s][w][0], ph[s][w][1], ph[s][w][2], ph[s][w][3]));
#pragma unroll
    for (int d0 = 0; d0 < 8; d0 += 2) {
        pf_vt_wait(cur[0], cur[1]);
        VtPair nxt[2];
        if (d0 + 2 < 8) {
            nxt[0] = pf_vt_issue(vaddr ^ (32u * (d0 + 2)));
            nxt[1] = pf_vt_issue(vaddr ^ (32u * (d0 + 3)));
        }
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    t.acc[d0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pf_vt_operand(cur[e], w), pb[w][s],
                                                                           t.acc[d0 + e], 0, 0, 0);
        beside(d0 >> 1);
        pf_chunk_end();
        if (d0 + 2 < 8) {
            cur[0] = nxt[0];
            cur[1] = nxt[1];
        }
    }
}

// The rescore flag of one output row, in the attention kernel's layout: lane (g, n) holds
// dims 16 dt + 4 g + i of query n's row (BF16 codes, pk[dt]).  The same decision as the
// multi-token merge's (rs_flag_decide over the row's elements in units of each dim's largest |V|
// and the scores' bound E = scale log2(e) sum_G |q_G| max|k_G|), over the keys the row at
// position pos sees: the keys before its chunk block (rs_kc, rs_dc at that block, reduced
// before this kernel runs) and the block's rows up to its own (rs_kpre, rs_dpre).  Q's
// pair-group norms come from the row as given (rotation leaves them unchanged): this lane
// reads dims 8g .. 8g+7 and 32 + 8g .. (and their pairs 64 on), pair groups g and 4 + g.
// The decision is formed in fp32 first, and where that cannot tell with y and its square in
// double, as in the multi-token merge (in fp32 y^2 underflows in every dim of a row whose
// elements lie ~2^63 below their dims' largest |V|).  ul bounds the error fp16's subnormal
// quantum added to every element (the attention loop's u over l; infinite for rows that are
// always rescored): a row with an element below 8 ul, where that error could reach 64 ULP with
// a margin of 2, is rescored as well.  Returns the decision for the row in every lane of its
// column.
__device__ __forceinline__ bool pf_flag_row(const PrefillArgs& a, int b, int kvh, int st, int pos, int64_t row,
                                            float m, double ul, const uint2 (&pk)[8], int lane) {
    const int g = lane >> 4;
    const int cb = pos / kPfBlk - st / kPfBlk;
    const int r = pos % kPfBlk;
    const int64_t ec = (static_cast<int64_t>(b) * kHkv + kvh) * a.rs_ncb + cb;
    const int64_t er = ec * a.rs_nr + r;
    const uint16_t* qrow = a.q + row * kD;
    const uint4 q0 = *reinterpret_cast<const uint4*>(qrow + 8 * g);
    const uint4 q1 = *reinterpret_cast<const uint4*>(qrow + 32 + 8 * g);
    const uint4 q2 = *reinterpret_cast<const uint4*>(qrow + kPairs + 8 * g);
    const uint4 q3 = *reinterpret_cast<const uint4*>(qrow + kPairs + 32 + 8 * g);
    const uint32_t k0 = max(a.rs_kc[ec * 8 + g], a.rs_kpre[er * 8 + g]);
    const uint32_t k1 = max(a.rs_kc[ec * 8 + 4 + g], a.rs_kpre[er * 8 + 4 + g]);
    float qq0 = 0.f, qq1 = 0.f;
    {
        const uint32_t w0[8] = {q0.x, q0.y, q0.z, q0.w, q2.x, q2.y, q2.z, q2.w};
        const uint32_t w1[8] = {q1.x, q1.y, q1.z, q1.w, q3.x, q3.y, q3.z, q3.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            qq0 = bf16x2_sq_acc(w0[i], qq0);
            qq1 = bf16x2_sq_acc(w1[i], qq1);
        }
    }
    float e = sqrtf(qq0) * sqrtf(__uint_as_float(k0)) + sqrtf(qq1) * sqrtf(__uint_as_float(k1));
    // Element magnitudes as packed codes: the largest (infinity and NaN above every finite
    // one) and the smallest; and the D_j, the largest of them likewise.
    uint32_t d[8][4], d_max = 0u, x_max = 0u, x_min = 0x7fff7fffu;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
        const uint4 dc = *reinterpret_cast<const uint4*>(a.rs_dc + ec * kD + 16 * dt + 4 * g);
        const uint2 dp = *reinterpret_cast<const uint2*>(a.rs_dpre + er * kD + 16 * dt + 4 * g);
        d[dt][0] = max(dc.x, dp.x & 0xffffu);
        d[dt][1] = max(dc.y, dp.x >> 16);
        d[dt][2] = max(dc.z, dp.y & 0xffffu);
        d[dt][3] = max(dc.w, dp.y >> 16);
        d_max = max(d_max, max(max(d[dt][0], d[dt][1]), max(d[dt][2], d[dt][3])));
        const uint32_t m0 = pk[dt].x & 0x7fff7fffu, m1 = pk[dt].y & 0x7fff7fffu;
        x_max = pk_max_u16(x_max, pk_max_u16(m0, m1));
        x_min = pk_min_u16(x_min, pk_min_u16(m0, m1));
    }
    auto elem = [&](int dt, int i) {
        const uint32_t w = i < 2 ? pk[dt].x : pk[dt].y;
        return __uint_as_float((i & 1) ? w & 0xffff0000u : w << 16);
    };
    // A first decision in fp32.  Where it can tell -- every square at or above kMinY2, so that
    // none has lost bits to fp32's subnormals (an element 2^59 below its D_j and further), and
    // no infinite or NaN sum (a zero or subnormal D_j has no reciprocal) -- its relative error
    // is far below the 1 % margin, so a row it clears is clear.  About 1 % of the N(0,1) waves
    // hold a row that it does not clear and form the decision in double below.  (The double
    // version for every wave cost about 2 us at the end of each workgroup.)
    constexpr float kMinY2 = 3.0092655e-36f;             // 2^-118
    float ss32 = 0.f, mn32 = INFINITY;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float y = elem(dt, i) * __builtin_amdgcn_rcpf(__uint_as_float(d[dt][i] << 16));
            ss32 = fmaf(y, y, ss32);
            mn32 = fminf(mn32, y * y);
        }
    // the row's four lanes: n, n + 16, n + 32, n + 48
    e += __shfl_xor(e, 16);
    e += __shfl_xor(e, 32);
    ss32 += __shfl_xor(ss32, 16);
    ss32 += __shfl_xor(ss32, 32);
    mn32 = swap32_max(swap16_max(-mn32));
    x_max = pk_max_u16(x_max, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x_max), 16)));
    x_max = pk_max_u16(x_max, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x_max), 32)));
    x_min = pk_min_u16(x_min, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x_min), 16)));
    x_min = pk_min_u16(x_min, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x_min), 32)));
    d_max = max(d_max, static_cast<uint32_t>(__shfl_xor(static_cast<int>(d_max), 16)));
    d_max = max(d_max, static_cast<uint32_t>(__shfl_xor(static_cast<int>(d_max), 32)));
    const float mnx = __uint_as_float(min(x_min & 0xffffu, x_min >> 16) << 16);
    const bool bad = max(x_max & 0xffffu, x_max >> 16) >= 0x7f80u || !(static_cast<double>(mnx) >= 8.0 * ul);
    // an infinite or NaN V among the row's keys (its y is 0: the row is flagged)
    if (d_max >= 0x7f80u && (lane >> 4) == 0) atomicOr(a.rs_hdr + 2, 1u);
    const double ed = static_cast<double>(e) * fabs(a.qk_scale_log2);
    const double md = static_cast<double>(m);
    bool flagged = bad || !(-mn32 >= kMinY2) ||
                   rs_flag_decide(-static_cast<double>(mn32), 1.01 * static_cast<double>(ss32), md, ed);
    if (__ballot(flagged && !bad)) {
        double ss = 0.0, mn2 = INFINITY;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dv = __uint_as_float(d[dt][i] << 16);
                const double y =
                    dv > 0.f ? static_cast<double>(elem(dt, i)) * __builtin_amdgcn_rcp(static_cast<double>(dv)) : 0.0;
                ss = fma(y, y, ss);
                if (dv > 0.f) mn2 = fmin(mn2, y * y);
            }
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        mn2 = fmin(mn2, __shfl_xor(mn2, 16));
        mn2 = fmin(mn2, __shfl_xor(mn2, 32));
        flagged = bad || rs_flag_decide(mn2, ss, md, ed);
    }
    return flagged;
}

// Ends the rows of one wave's 16 queries (lane (g, n): dims 16dt + 4g + i of query n at
// position st + t; O, this lane's share of l, the running max and this lane's share of the
// bound u, infinite for rows that always go to the rescore): normalises, rounds double -> f32 ->
// BF16, decides the rescore flag from the rounded row and writes it.  q_ok: the lane's query
// exists (waves past the last query decide and write nothing).
__device__ __forceinline__ void pf_finish(const PrefillArgs& a, int b, int kvh, int st, int t, bool q_ok, int hq,
                                          const double (&o64)[8][4], double l64, float m, float u, int lane) {
    const int g = lane >> 4;
    double l = l64 + __shfl_xor(l64, 16);
    l += __shfl_xor(l, 32);
    u += __shfl_xor(u, 16);
    u += __shfl_xor(u, 32);
    const double ul = static_cast<double>(u) / l;     // bound on that error in the row's elements
    const double inv_l = 1.0 / l;
    const int64_t row = (static_cast<int64_t>(b) * a.n_new + t) * kHq + hq;
    uint2 pk[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = static_cast<float>(quotient(o64[dt][i], l, inv_l));
        pk[dt].x = f32x2_to_bf16_out(x[0], x[1]);
        pk[dt].y = f32x2_to_bf16_out(x[2], x[3]);
    }
    if (a.rs_hdr && __ballot(q_ok)) {
        if (pf_flag_row(a, b, kvh, st, st + t, row, m, ul, pk, lane) && q_ok && g == 0)
            rs_append(a, static_cast<uint32_t>(row));
    }
    if (!q_ok) return;
    uint16_t* orow = a.out + row * kD;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * g) = pk[dt];
}

__global__ __launch_bounds__(kPfThreads) void prefill_attn_kernel(PrefillArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsB];

    // Workgroup -> (sequence, KV head, query block).  Workgroups are dealt to the 8 XCDs
    // round-robin; all query blocks of a pair (8 per sequence) go to one XCD so that its K/V
    // blocks are shared in that XCD's L2.  A pair's query blocks are dealt last first: the
    // last ones see the most keys, and the short ones then fill the CUs that finish early.
    // Then the runs of a query block (n_split > 1), neighbours on the same XCD.
    const int unit = (blockIdx.x >> 3) / a.n_split;
    const int run = (blockIdx.x >> 3) % a.n_split;
    const int qb = a.n_qblk - 1 - unit % a.n_qblk;
    const int pair = (unit / a.n_qblk) * 8 + (blockIdx.x & 7);
    const int b = pair / kHkv;
    const int kvh = pair % kHkv;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & (kWave - 1);
    const int n = lane & 15;
    const int g = lane >> 4;
    const int hq = kvh * kGroup + (wave & 3);
    const int pt = wave >> 2;
    const int T = a.n_new;
    const int t_wave0 = qb * kPfPos + pt * 16;
    const int tq = t_wave0 + n;
    const bool q_ok = tq < T;
    const int st = a.start[b];

    if (!prefill_start_ok(a, st)) {
        if (q_ok && g == 0 && run == 0) {
            uint4* o = reinterpret_cast<uint4*>(a.out + ((static_cast<int64_t>(b) * T + tq) * kHq + hq) * kD);
            for (int i = 0; i < kD / 8; ++i) o[i] = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
        }
        return;
    }

    // Every wave runs every block of the workgroup; a block past the keys of this wave's
    // queries is masked for all of them (without a split block 0 always holds a valid key, so
    // the running max is finite from the first block on; in a later run it may stay -inf, and
    // p is formed against 0 then).  Waves past the last query compute the last query and write
    // nothing.
    const int tq_c = min(tq, T - 1);
    const int pos_n = st + tq_c;            // this lane's query position
    const int n_keys = st + min(T, qb * kPfPos + kPfPos);
    const int all_blk = (n_keys + kPfBlk - 1) / kPfBlk;
    int per_run;
    const int n_run = pf_runs(all_blk, a.n_split, per_run);
    if (run >= n_run) return;
    const int blk0 = run * per_run;
    const int n_blk = min(all_blk, blk0 + per_run);        // this run: blocks blk0 .. n_blk - 1
    const int nblk_stg = a.stg_pos / kPfBlk;
    const char* kseg = reinterpret_cast<const char*>(a.stg_k + static_cast<int64_t>(pair) * a.stg_pos * kD);
    const char* vseg = reinterpret_cast<const char*>(a.stg_v + static_cast<int64_t>(pair) * a.stg_pos * kD);
    const char* kloseg = reinterpret_cast<const char*>(a.stg_klo + static_cast<int64_t>(pair) * a.stg_cb * kPfBlk * kD);
    const uint32_t* sw = a.stg_scale + static_cast<int64_t>(pair) * nblk_stg;
    const int cb0 = st / kPfBlk;            // first block holding chunk keys
    auto blk_new = [&](int blk) { return blk >= cb0; };
    auto blk_diag = [&](int blk) { return blk * kPfBlk + kPfBlk - 1 > st + t_wave0; };
    auto issue_k = [&](int blk, int buf, const uint32_t (&loff)[2]) {
        pf_issue(kseg + static_cast<int64_t>(blk) * kPlaneB, loff, lds + kOffK + buf * kPlaneB, wave);
        if (blk_new(blk))
            pf_issue(kloseg + static_cast<int64_t>(blk - cb0) * kPlaneB, loff, lds + kOffKlo + buf * kPlaneB, wave);
    };
    auto issue_v = [&](int blk, int buf, const uint32_t (&loff)[2]) {
        pf_issue(vseg + static_cast<int64_t>(blk) * kPlaneB, loff, lds + kOffV + buf * kPlaneB, wave);
    };

    // K of the first two blocks and V of the first are requested before the Q operands are
    // formed.
    uint32_t loff[2];
    pf_copy_offsets(wave, lane, loff);
    issue_k(blk0, blk0 & 1, loff);
    issue_v(blk0, blk0 & 1, loff);
    if (blk0 + 1 < n_blk) issue_k(blk0 + 1, (blk0 + 1) & 1, loff);
    // Scale words of 64 blocks per wave, from the ring half that holds the first block (entries
    // past the last block repeat it).
    auto issue_sw = [&](int first) {
        __builtin_amdgcn_global_load_lds(sw + min(first + lane, nblk_stg - 1),
                                         (lds_void_t*)(lds + kOffSw + 4 * (first & (kSwRing - 1))), 4, 0, 0);
    };
    issue_sw((blk0 & ~255) + 64 * wave);
    // The first scale words again, for their maximum below (requested with the rest).
    constexpr int kSwAhead = 3;
    uint32_t sw_ahead[kSwAhead];
#pragma unroll
    for (int i = 0; i < kSwAhead; ++i) sw_ahead[i] = sw[min(i * kWave + lane, nblk_stg - 1)];
    auto sw_lds = [&](int blk) {
        return *reinterpret_cast<const uint32_t*>(lds + kOffSw + 4 * (blk & (kSwRing - 1)));
    };

    // Q operands: query n = this lane's column, dims 32kb + 8g + j, two fp16 parts of Q
    // scaled by 2^sq, sq putting the row's largest magnitude in [2^14, 2^15).
    f16x8_t qop[2][4];
    float cq;                               // 2^-sq
    bool q_bad = false;
    {
        const int64_t tok = static_cast<int64_t>(b) * T + tq_c;
        const char* qrow = reinterpret_cast<const char*>(a.q + (tok * kHq + hq) * kD) + 16 * g;
        // The token's (cos, sin) row, from the append kernel: rotating here (16 double sincos
        // per lane) took about 20 us at the start of every workgroup.
        const double2* csr = a.rs_cs + tok * kPairs + 8 * g;
        uint4 qw[4];
        double2 cs[2][8];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) qw[kb] = *reinterpret_cast<const uint4*>(qrow + 64 * kb);
        if (a.flags & 1u) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int j = 0; j < 8; ++j) cs[kb][j] = csr[32 * kb + j];
        }
        float qf[4][8];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) unpack8(qw[kb], qf[kb]);
        double qv[4][8];
        double mx = 0.0;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const double x = qf[kb][j];
                const double y = qf[kb + 2][j];
                double xr = x, yr = y;
                if (a.flags & 1u) {
                    xr = x * cs[kb][j].x - y * cs[kb][j].y;
                    yr = x * cs[kb][j].y + y * cs[kb][j].x;
                }
                qv[kb][j] = xr * a.qk_scale_log2;
                qv[kb + 2][j] = yr * a.qk_scale_log2;
                mx = fmax(mx, fmax(fabs(qv[kb][j]), fabs(qv[kb + 2][j])));
            }
        }
        // Out of range: an element that is not finite as given, or a rotated and scaled one
        // past 1e300 (finite elements rotate and scale without a NaN).
        uint32_t qm = 0u;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
            qm = pk_max_u16(qm, pk_max_u16(pk_max_u16(qw[kb].x & 0x7fff7fffu, qw[kb].y & 0x7fff7fffu),
                                           pk_max_u16(qw[kb].z & 0x7fff7fffu, qw[kb].w & 0x7fff7fffu)));
        if (max(qm & 0xffffu, qm >> 16) >= 0x7f80u || !(mx <= 1e300)) q_bad = true;
        mx = fmax(mx, __shfl_xor(mx, 16));
        mx = fmax(mx, __shfl_xor(mx, 32));
        int e = 0;
        if (mx > 0.0) {
            e = ilogb(mx);
            if (e < -100 || e > 100) q_bad = true;
            e = e < -100 ? -100 : e > 100 ? 100 : e;
        }
        const int sq = mx > 0.0 ? 14 - e : 0;
        cq = pow2f(-sq);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            uint32_t w0[4], w1[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double x0 = ldexp(qv[kb][2 * j], sq), x1 = ldexp(qv[kb][2 * j + 1], sq);
                w0[j] = pk_f16(f32_of(x0), f32_of(x1));
                w1[j] = pk_f16(f32_of(x0 - static_cast<double>(f16_lo(w0[j]))),
                               f32_of(x1 - static_cast<double>(f16_hi(w0[j]))));
            }
            // Pin the operands: without this the compiler re-derives them from the double
            // rows inside the block loop to save registers.
            asm volatile("" : "+v"(w0[0]), "+v"(w0[1]), "+v"(w0[2]), "+v"(w0[3]));
            asm volatile("" : "+v"(w1[0]), "+v"(w1[1]), "+v"(w1[2]), "+v"(w1[3]));
            qop[0][kb] = as_f16x8(make_uint4(w0[0], w0[1], w0[2], w0[3]));
            qop[1][kb] = as_f16x8(make_uint4(w1[0], w1[1], w1[2], w1[3]));
        }
    }

    const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_t*)(lds)));
    const uint32_t vaddr = lds_base + kOffV + vt_tr_offset(0, lane);
    const uint32_t koff = pf_k_offset(n, g);

    PfTile tl;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) tl.o64[dt][i] = 0.0;
        tl.acc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    tl.l64 = 0.0;
    tl.m_run = -INFINITY;
    tl.u = 0.f;
    // The open group: blocks summed into tl.acc so far and their V scale exponent.  A block
    // whose V scale differs from the group's by more than 3 (its P would leave fp16's range
    // or its precision) closes the group first.  A block holding chunk keys is summed alone.
    // Its scales may depend on rows that later tokens see and this token does not, and within a
    // group a different scale would change how the other blocks' terms round, so this token's
    // output would depend on keys its mask hides; alone, its sum only scales by a power of two.
    // And a prompt's blocks, all of them chunk blocks, meet in fp64: joined in fp32 (those that
    // every query of the wave sees) two prompts of 1000 tokens took 116.6 us, so 119.1.
    int grp_n = 0, grp_sv = 0;
    int shut_sv = 0;                        // a group to close before the next products, its exponent
    bool shut = false;

    // Raw scores carry 2^(sq + sk): mult = 2^-sq * 2^-sk(block) turns them into log2 units.
    // (Kept at least 2^-126: a smaller factor means scores below ~2^-90, all p = 1 either way,
    // and 0 would turn masked keys' -inf into NaN.)
    auto blk_mult = [&](uint32_t w) {
        return fmaxf(cq * pow2f(-static_cast<int>(static_cast<int8_t>(w & 0xffu))), 1.17549435e-38f);
    };
    auto blk_sv = [&](uint32_t w) { return static_cast<int>(static_cast<int8_t>((w >> 8) & 0xffu)); };
    // The largest V scale exponent among the query block's blocks (the smallest-V block's).
    int sv_hi = -128;
#pragma unroll
    for (int i = 0; i < kSwAhead; ++i)
        if (i * kWave + lane < all_blk) sv_hi = max(sv_hi, blk_sv(sw_ahead[i]));
    for (int j = kSwAhead * kWave + lane; j < all_blk; j += kWave) sv_hi = max(sv_hi, blk_sv(sw[j]));
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) sv_hi = max(sv_hi, __shfl_xor(sv_hi, sh));
    sv_hi = __builtin_amdgcn_readfirstlane(sv_hi);

    // The first block's scores.  The barrier after them frees its K buffer.
    __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0)
    __syncthreads();
    f32x4_t scur[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) scur[kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint8_t* kfirst = lds + kOffK + (blk0 & 1) * kPlaneB;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        f16x8_t ak[2];
        pf_k_pair(kfirst, i, koff, ak);
        if (blk_new(blk0))
            pf_qk_pair<true>(kfirst, ak, qop, i, koff, scur);
        else
            pf_qk_pair<false>(kfirst, ak, qop, i, koff, scur);
    }
    uint32_t w_cur = __builtin_amdgcn_readfirstlane(sw_lds(blk0));
    uint32_t w_ahead = sw_lds(blk0 + 1);          // block blk+1's word, read a step ahead
    uint32_t unsafe = w_cur;                // bit 31 of any block read marks all rows
    float mult_cur = blk_mult(w_cur);
    if (blk_diag(blk0)) pf_mask(scur, blk0 * kPfBlk, g, pos_n);
    pf_rescale(tl, pf_next_max(pf_lane_max(scur), tl.m_run, mult_cur));
    // The group of the next block to be summed (its scale word w; solo: alone) and the factor
    // 2^vshift its P carries, the group's V scale over the block's (|vshift| <= 3).
    auto open_group = [&](uint32_t w, bool solo) {
        const int sv = blk_sv(w);
        const int far = static_cast<int>(solo) | static_cast<int>(abs(grp_sv - sv) > 3);
        const int sh = static_cast<int>(grp_n == kPfGroup) | (static_cast<int>(grp_n > 0) & far);
        shut = sh != 0;
        shut_sv = grp_sv;
        const int start = sh | static_cast<int>(grp_n == 0);
        grp_sv = start ? sv : grp_sv;
        grp_n = solo ? kPfGroup : (start ? 1 : grp_n + 1);
        return grp_sv - sv;
    };
    // The first half of the first block's probabilities.  lsum: the block's sum of p (with
    // 2^vshift).  p = 2^(s + off); a running max still at -inf (every key so far masked) counts
    // as 0, so that p = 0.
    auto p_off = [&](int shift, float m) {
        return static_cast<float>(kPScaleExp + shift) - (m == -INFINITY ? 0.f : m);
    };
    int vshift = open_group(w_cur, blk_new(blk0));
    float off = p_off(vshift, tl.m_run);
    float lsum = 0.f;
    uint32_t ph[2][2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pf_probs_half16(scur[i >> 1], mult_cur, off, lsum, ph, i >> 1, i & 1);
    __syncthreads();

    // One step of the block loop.  Resident: K of block blk+1 (K buffer (blk+1)&1) and V of
    // block blk (V buffer blk&1).  Free: K buffer blk&1 (block blk, scored in the previous step)
    // and V buffer (blk+1)&1 (block blk-1).  Half of a block's probabilities are formed beside
    // the next block's scores and half (of the block after) beside V^T P^T, so that both runs of
    // 32 MFMAs have about as much VALU work beside them as fits: a SIMD's two waves issue
    // 2 x 32 MFMAs in 1024 cycles, and with all 80 VALU instructions of the probabilities beside
    // the scores that run took 1700-2400.  kPlain: blocks blk and blk+1 hold cached keys only (no
    // masks, no trailing K parts), so that the step is one straight run.  With the branches of
    // the general step in the loop, the compiler formed most probabilities before the scores'
    // MFMAs: 4 x 512 tokens over 8192 566 us, now 540 us (MFMAs alone 254 us; timing builds:
    // without the probabilities 64 us less, the copies 38, the LDS reads 30, the rescale of O and
    // the fp64 sums 17 each).
    auto step = [&](auto plain, int blk) {
        constexpr bool kPlain = decltype(plain)::value;
        const bool next = kPlain || blk + 1 < n_blk;
        if (blk + 2 < n_blk) issue_k(blk + 2, blk & 1, loff);
        if (next) issue_v(blk + 1, (blk + 1) & 1, loff);
        if ((blk & 255) == 128 && wave < 4 && blk + 128 < n_blk) issue_sw(blk + 128 + 64 * wave);
        const uint32_t w_next = next ? __builtin_amdgcn_readfirstlane(w_ahead) : w_cur;
        unsafe |= w_next;
        if (shut) pf_flush(tl, static_cast<double>(pow2f(-shut_sv)));
        const int sv_blk = grp_sv;               // this block's group
        const int l_shift = -vshift;
        if (next) vshift = open_group(w_next, !kPlain && blk_new(blk + 1));

        f32x4_t snext[4];
        VtPair vt[2];
        const uint32_t va = vaddr + (blk & 1) * kPlaneB;
        const uint8_t* knext = lds + kOffK + ((blk + 1) & 1) * kPlaneB;
        // The two waves of a SIMD run the same steps; the one in this MFMA + VALU mix gets
        // issue priority over the other's V^T P^T.
        __builtin_amdgcn_s_setprio(1);
        if (kPlain)
            pf_scores_beside<true, false, true>(scur, mult_cur, off, lsum, knext, qop, koff, va, ph, snext, vt);
        else if (!next)
            pf_scores_beside<false, false, false>(scur, mult_cur, off, lsum, knext, qop, koff, va, ph, snext, vt);
        else if (blk_new(blk + 1))
            pf_scores_beside<true, true, false>(scur, mult_cur, off, lsum, knext, qop, koff, va, ph, snext, vt);
        else
            pf_scores_beside<true, false, false>(scur, mult_cur, off, lsum, knext, qop, koff, va, ph, snext, vt);
        __builtin_amdgcn_s_setprio(0);

        // The next block's running max is found beside this block's V^T P^T (which still
        // accumulates at the current max); O and l move to it afterwards.
        const float l_blk = lsum;
        const float mult_next = blk_mult(w_next);
        float m_next = tl.m_run;
        uint32_t pn[2][2][4];
        if (!kPlain && next && blk_diag(blk + 1)) pf_mask(snext, (blk + 1) * kPfBlk, g, pos_n);
        lsum = 0.f;
        if (!kPlain) {
            vt[0] = pf_vt_issue(va);
            vt[1] = pf_vt_issue(va ^ 32u);
        }
        pf_pv(va, ph, vt, tl, [&](int i) {
            // (no branches here: V^T operands are in flight)
            if (i == 0) {
                w_ahead = sw_lds(blk + 2);
                m_next = pf_next_max(pf_lane_max(snext), tl.m_run, mult_next);
                off = kPlain ? static_cast<float>(kPScaleExp + vshift) - m_next : p_off(vshift, m_next);
                tl.l64 += ldexp(static_cast<double>(l_blk), l_shift);
            }
            if (i == 1) pf_probs_half16(snext[0], mult_next, off, lsum, pn, 0, 0);
            if (i == 2) {
                pf_probs_half16(snext[0], mult_next, off, lsum, pn, 0, 1);
                pf_probs_half16(snext[1], mult_next, off, lsum, pn, 1, 0);
            }
            if (i == 3) pf_probs_half16(snext[1], mult_next, off, lsum, pn, 1, 1);
        });

        // fp16's subnormal quantum: a p below 2^-2 (in the units the MFMAs see) has a second part
        // below 2^-14, and the split carries it to within 2^-25 absolutely, not 2^-22 of itself
        // (a p below 2^-25 is dropped).  Harmless while those keys' V is about as large as the
        // rest's (what is lost is then below the calibrated rounding), not when keys of tiny
        // weight carry V far larger than the output.  So on blocks whose V is 2^6 times the
        // smallest-V block's or more (a uniform test), a lane with a p below 2^-2 among its 16
        // keys (the fp16 codes of the first parts, below 0x3400; masked keys count,
        // conservatively) adds their bound 16 * 2^-25 * 2^15 (staged |V| < 2^15) = 2^-6, times
        // 2^-sv_blk, to u, which the epilogue compares with the row's elements.
        if (sv_blk < sv_hi - 6) {
            uint32_t m16 = ph[0][0][0];
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
                for (int d = 0; d < 4; ++d) m16 = pk_min_u16(m16, ph[0][w][d]);
            if (min(m16 & 0xffffu, m16 >> 16) < 0x3400u) tl.u += pow2f(-6 - sv_blk);
        }
        pf_rescale(tl, m_next);
#pragma unroll
        for (int kt = 2; kt < 4; ++kt) scur[kt] = snext[kt];
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
            for (int d = 0; d < 4; ++d) ph[part][0][d] = pn[part][0][d];
        w_cur = w_next;
        mult_cur = mult_next;
        // This wave's copies into LDS are complete; after the barrier every wave's are, and
        // every wave is done with the buffers the next step's copies go to.
        __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0)
        __syncthreads();
    };
    int blk = blk0;
    for (; blk + 1 < min(cb0, n_blk); ++blk) step(std::true_type{}, blk);
    for (; blk < n_blk; ++blk) step(std::false_type{}, blk);
    pf_flush(tl, static_cast<double>(pow2f(-grp_sv)));

    // Rows that read a marked block or whose Q row is out of range always go to the rescore:
    // their error bound is infinite.
    if ((unsafe >> 31) != 0u || q_bad) tl.u = INFINITY;
    if (n_run > 1) {
        const int64_t slot = (static_cast<int64_t>(pair) * a.n_qblk + qb) * a.n_split + run;
        double2* po = a.sp_o + (slot * kPfWaves + wave) * 16 * kWave + lane;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                po[(2 * dt + j) * kWave] = make_double2(tl.o64[dt][2 * j], tl.o64[dt][2 * j + 1]);
        static_cast<SplitMl*>(a.sp_ml)[(slot * kPfWaves + wave) * kWave + lane] = SplitMl{tl.l64, tl.m_run, tl.u};
        return;
    }
    pf_finish(a, b, kvh, st, tq_c, q_ok, hq, tl.o64, tl.l64, tl.m_run, tl.u, lane);
}

// Combines the runs of one wave's 16 queries (grid: 8 waves per query block and pair): wave v
// of the workgroup sums dim tile v over the runs in order, each scaled by the exact power of two
// between its running max and the largest so far, and the sums meet in LDS for the first
// wave, which ends the rows as the attention kernel does.
__global__ __launch_bounds__(kPfThreads) void prefill_merge_kernel(PrefillArgs a) {
    __shared__ double2 o_s[kPfWaves][2][kWave];
    const int unit = blockIdx.x / kPfWaves;
    const int wt = blockIdx.x % kPfWaves;
    const int pair = unit / a.n_qblk;
    const int qb = unit % a.n_qblk;
    const int b = pair / kHkv;
    const int kvh = pair % kHkv;
    const int v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    const int T = a.n_new;
    const int st = a.start[b];
    if (!prefill_start_ok(a, st)) return;
    int per;
    const int n_run = pf_runs((st + min(T, qb * kPfPos + kPfPos) + kPfBlk - 1) / kPfBlk, a.n_split, per);
    if (n_run == 1) return;
    const int t_wave0 = qb * kPfPos + (wt >> 2) * 16;
    if (t_wave0 >= T) return;
    const int tq = t_wave0 + (lane & 15);
    const int64_t slot0 = (static_cast<int64_t>(pair) * a.n_qblk + qb) * a.n_split;
    const double2* po = a.sp_o + ((slot0 * kPfWaves + wt) * 16 + 2 * v) * kWave + lane;
    const SplitMl* pml = static_cast<const SplitMl*>(a.sp_ml) + (slot0 * kPfWaves + wt) * kWave + lane;
    double o[4] = {0.0, 0.0, 0.0, 0.0};
    double l = 0.0;
    float m = -INFINITY, u = 0.f;
    constexpr int kAhead = 8;
    for (int r0 = 0; r0 < n_run; r0 += kAhead) {
        double2 x[kAhead][2];
        SplitMl ml[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int64_t r = min(r0 + i, n_run - 1);
            ml[i] = pml[r * kPfWaves * kWave];
            x[i][0] = po[r * kPfWaves * 16 * kWave];
            x[i][1] = po[r * kPfWaves * 16 * kWave + kWave];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (r0 + i >= n_run) break;                       // (uniform)
            const float m_new = fmaxf(m, ml[i].m);
            const int sa = m == m_new ? 0 : max_shift(m, m_new);
            const int sx = ml[i].m == m_new ? 0 : max_shift(ml[i].m, m_new);
            o[0] = ldexp(o[0], sa) + ldexp(x[i][0].x, sx);
            o[1] = ldexp(o[1], sa) + ldexp(x[i][0].y, sx);
            o[2] = ldexp(o[2], sa) + ldexp(x[i][1].x, sx);
            o[3] = ldexp(o[3], sa) + ldexp(x[i][1].y, sx);
            l = ldexp(l, sa) + ldexp(ml[i].l, sx);
            u = ldexpf(u, sa) + ldexpf(ml[i].u, sx);
            m = m_new;
        }
    }
    o_s[v][0][lane] = make_double2(o[0], o[1]);
    o_s[v][1][lane] = make_double2(o[2], o[3]);
    __syncthreads();
    if (v > 0) return;
    double o64[8][4];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            o64[dt][2 * j] = o_s[dt][j][lane].x;
            o64[dt][2 * j + 1] = o_s[dt][j][lane].y;
        }
    pf_finish(a, b, kvh, st, min(tq, T - 1), tq < T, kvh * kGroup + (wt & 3), o64, l, m, u, lane);
}

hipError_t launch_prefill_attention(const PrefillArgs& a, hipStream_t stream) {
    const int64_t n_unit = static_cast<int64_t>(a.batch) * kHkv * a.n_qblk;
    if (n_unit == 0) return hipSuccess;
    hipLaunchKernelGGL(prefill_attn_kernel, dim3(static_cast<unsigned>(n_unit * a.n_split)), dim3(kPfThreads), 0,
                       stream, a);
    if (a.n_split > 1)
        hipLaunchKernelGGL(prefill_merge_kernel, dim3(static_cast<unsigned>(n_unit * kPfWaves)), dim3(kPfThreads), 0,
                           stream, a);
    return hipGetLastError();
}

}  // namespace gqa
