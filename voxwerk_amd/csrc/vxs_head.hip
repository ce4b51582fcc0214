// vxs_head.hip — the logit heads on the GPU, the step before the sampler.
//
// CodecHead and CodePredictorHead (src/Voxwerk/Talker/TalkerModel.cs:133-137) multiply fp32 hidden
// rows by a bf16 weight (the checkpoint's [out, in] layout, WeightPrecision.BFloat16,
// DecoderStack.cs:7-15): out[r][n] = sum_k x[r][k] * W[n][k]; the logits stay in HBM for the sampler.
// One to three rows are a GEMV on the VALU; from there the matrix cores take it (x split exactly into
// three bf16 parts): a split-K form while the call has few tiles, a tiled form for large batches
// (launch_head has the rule and what it was measured on).
//
// VALU layout: a wave owns two consecutive outputs; lane l holds W[n][k] for k = 512 j + 8 l + 0..7
// (one 16-byte load per output and j, 1 KiB contiguous per wave instruction), all of its rows in
// registers for the whole call. Per hidden row the lane loads its x slice (the next row's loads
// issued before the current row's products), forms its partial dots and reduces them across the wave by
// a halving exchange (xor 32: each lane keeps one of the two outputs and adds its partner's copy of it)
// and then plain butterflies (xor 16 .. 1). The fp32 sum order is each kernel's own; it differs from the
// reference's AVX-512 order by rounding only (bounded by K 2^-24 sum |x w|).
//
// The int8 form (WeightPrecision.Int8, DecoderStack.cs:7-16) keeps W as q[n][k] in [-127, 127] and
// one fp32 scale per output (PackedMatrix.FromBf16LinearInt8, PackedMatrix.cs:124-154):
// out[r][n] = scale[n] * sum_k x[r][k] * q[n][k], the scale applied to the fp32 dot as the decode
// path does (Gemm.cs:650-680, PanelPairDotInt8 / PanelDotInt8). Same layouts and reductions, half the
// weight bytes. The packing itself runs on the GPU too (head_pack_i8_kernel): per output the largest
// |w|, scale = amax / 127 (1 for an all-zero row), q = clamp(round-half-even(w * (1 / scale)), -127,
// 127), all in correctly rounded fp32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "vxs_internal.h"

namespace vxs {
namespace {

constexpr int kHT = 256;  // threads per workgroup

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float lo16(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi16(unsigned w) { return __uint_as_float(w & 0xFFFF0000u); }

// 8 bf16 (packed in u4) times 8 fp32, added to acc in k order.
__device__ __forceinline__ float dot8(u4 w, f4 xa, f4 xb, float acc) {
    acc = __builtin_fmaf(lo16(w.x), xa.x, acc);
    acc = __builtin_fmaf(hi16(w.x), xa.y, acc);
    acc = __builtin_fmaf(lo16(w.y), xa.z, acc);
    acc = __builtin_fmaf(hi16(w.y), xa.w, acc);
    acc = __builtin_fmaf(lo16(w.z), xb.x, acc);
    acc = __builtin_fmaf(hi16(w.z), xb.y, acc);
    acc = __builtin_fmaf(lo16(w.w), xb.z, acc);
    acc = __builtin_fmaf(hi16(w.w), xb.w, acc);
    return acc;
}

// One lane's slice of hidden row m: x[m][512 j + 8 lane + 0..7] for each j. FULL: k = 512 KJ, every
// slice inside the row; otherwise slices past k read the row's start and are zeroed (a select that
// waits for the load, so only the partial shapes pay it).
template <int KJ>
struct XSlice {
    f4 a[KJ], b[KJ];
};

template <int KJ, bool FULL>
__device__ __forceinline__ XSlice<KJ> load_x(const HeadArgs& h, int m, int lane) {
    XSlice<KJ> r;
#pragma unroll
    for (int j = 0; j < KJ; j++) {
        const int k = 512 * j + 8 * lane;
        const bool in = FULL || k < h.k;
        const float* p = h.x + (int64_t)m * h.ldx + (in ? k : 0);
        const f4 a = *reinterpret_cast<const f4*>(p);
        const f4 b = *reinterpret_cast<const f4*>(p + 4);
        r.a[j] = FULL || in ? a : f4{0.f, 0.f, 0.f, 0.f};
        r.b[j] = FULL || in ? b : f4{0.f, 0.f, 0.f, 0.f};
    }
    return r;
}

// The wave's two partial dots of one row, reduced: lanes 0..31 end with the first, 32..63 the second.
__device__ __forceinline__ float reduce_outputs(const float (&v)[2], int lane) {
    const bool hi = lane >= 32;
    float sum = (hi ? v[1] : v[0]) + __shfl_xor(hi ? v[0] : v[1], 32);
#pragma unroll
    for (int mask = 16; mask >= 1; mask /= 2) sum += __shfl_xor(sum, mask);
    return sum;
}

constexpr int R = 2;  // outputs per wave

// KJ slices of 8 per lane (k <= 512 KJ).
template <int KJ, bool FULL>
__global__ __launch_bounds__(kHT) void head_kernel(HeadArgs a) {
    const int lane = threadIdx.x & 63;
    const int n0 = (blockIdx.x * (kHT / 64) + (threadIdx.x >> 6)) * R;
    if (n0 >= a.n) return;  // whole wave past the last output (wave-uniform)

    // this lane's weights, kept as bf16 pairs
    u4 w[R][KJ];
#pragma unroll
    for (int o = 0; o < R; o++)
#pragma unroll
        for (int j = 0; j < KJ; j++) {
            const int k = 512 * j + 8 * lane;
            const bool in = n0 + o < a.n && (FULL || k < a.k);
            // every lane loads from inside W (a clamped address) and zeroes what lies outside
            const uint16_t* p = a.w + (int64_t)min(n0 + o, a.n - 1) * a.ldw + (FULL || k < a.k ? k : 0);
            const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
            w[o][j] = in ? v : u4{0u, 0u, 0u, 0u};
        }

    const int o_mine = lane >> 5;  // the output this lane holds after the reduction
    // rows two at a time with two slice buffers, each reloaded in place while the other is used,
    // so a row's loads are in flight during the previous row's products and exchanges
    auto row = [&](int m, const XSlice<KJ>& x) {
        float v[R];
#pragma unroll
        for (int o = 0; o < R; o++) {
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < KJ; j++) acc = dot8(w[o][j], x.a[j], x.b[j], acc);
            v[o] = acc;
        }
        const float sum = reduce_outputs(v, lane);
        if ((lane & 31) == 0 && n0 + o_mine < a.n) a.out[(int64_t)m * a.ldo + n0 + o_mine] = sum;
    };
    // this workgroup's rows: group blockIdx.y of a.row_group rows
    const int first = blockIdx.y * a.row_group;
    const int last = min(a.rows, first + a.row_group) - 1;
    XSlice<KJ> x0 = load_x<KJ, FULL>(a, first, lane);
    for (int m = first; m <= last; m += 2) {
        XSlice<KJ> x1 = load_x<KJ, FULL>(a, min(m + 1, last), lane);
        row(m, x0);
        if (m + 1 > last) break;
        x0 = load_x<KJ, FULL>(a, min(m + 2, last), lane);
        row(m + 1, x1);
    }
}

typedef unsigned int u2 __attribute__((ext_vector_type(2)));

// int8 weights, widened once: KJ slices of 8 per lane (k <= 512 KJ).
template <int KJ, bool FULL>
__global__ __launch_bounds__(kHT) void head_i8_kernel(HeadArgs a) {
    const int lane = threadIdx.x & 63;
    const int n0 = (blockIdx.x * (kHT / 64) + (threadIdx.x >> 6)) * R;
    if (n0 >= a.n) return;  // whole wave past the last output (wave-uniform)

    // every lane loads from inside q (a clamped address) and zeroes what lies outside; all loads
    // are issued before the first conversion
    u2 raw[R][KJ];
#pragma unroll
    for (int o = 0; o < R; o++)
#pragma unroll
        for (int j = 0; j < KJ; j++) {
            const int k = 512 * j + 8 * lane;
            const int8_t* p = a.q + (int64_t)min(n0 + o, a.n - 1) * a.ldw + (FULL || k < a.k ? k : 0);
            raw[o][j] = __builtin_nontemporal_load(reinterpret_cast<const u2*>(p));
        }
    // q = (q + 128) - 128: the biased byte (sign bit flipped) converted as unsigned, then an exact
    // fp32 subtraction. (A sign-extended byte fed straight to the conversion was compiled here into
    // an unsigned conversion of the extended value.)
    float w[R][KJ][8];
#pragma unroll
    for (int o = 0; o < R; o++)
#pragma unroll
        for (int j = 0; j < KJ; j++) {
            const int k = 512 * j + 8 * lane;
            const bool in = n0 + o < a.n && (FULL || k < a.k);
            const uint32_t lo = raw[o][j].x ^ 0x80808080u, hi = raw[o][j].y ^ 0x80808080u;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float f = (float)(((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xffu) - 128.0f;
                w[o][j][i] = in ? f : 0.0f;
            }
        }
    const int o_mine = lane >> 5;
    const float sc = a.scale[min(n0 + o_mine, a.n - 1)];
    auto row = [&](int m, const XSlice<KJ>& x) {
        float v[R];
#pragma unroll
        for (int o = 0; o < R; o++) {
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < KJ; j++) {
                const float xs[8] = {x.a[j].x, x.a[j].y, x.a[j].z, x.a[j].w, x.b[j].x, x.b[j].y, x.b[j].z, x.b[j].w};
#pragma unroll
                for (int i = 0; i < 8; i++) acc = __builtin_fmaf(w[o][j][i], xs[i], acc);
            }
            v[o] = acc;
        }
        const float sum = reduce_outputs(v, lane) * sc;
        if ((lane & 31) == 0 && n0 + o_mine < a.n) a.out[(int64_t)m * a.ldo + n0 + o_mine] = sum;
    };
    const int first = blockIdx.y * a.row_group;
    const int last = min(a.rows, first + a.row_group) - 1;
    XSlice<KJ> x0 = load_x<KJ, FULL>(a, first, lane);
    for (int m = first; m <= last; m += 2) {
        XSlice<KJ> x1 = load_x<KJ, FULL>(a, min(m + 1, last), lane);
        row(m, x0);
        if (m + 1 > last) break;
        x0 = load_x<KJ, FULL>(a, min(m + 2, last), lane);
        row(m + 1, x1);
    }
}

// ---- matrix-core forms, from 3 or 4 rows up -----------------------------------------------------
// The hidden rows are fp32 and v_mfma_f32_16x16x32_bf16 multiplies bf16, so each x is scaled by 2^32
// and split exactly into three bf16 parts, 2^32 x = h + m + l: h keeps the top 8 significand bits
// (truncation), m the next 8 of the remainder (exact in fp32), l what is left (at most 8 bits: exact in
// bf16). The scale keeps every bit of the smallest x: unscaled, a part below bf16's last place of 2^-133
// is cut short (x near 2^-120 then had 13 bits of 24); it costs one multiplication per x (256 x 1024 ->
// 3072 10.35 -> 10.48 us, 4096 rows 89.9 -> 90.7). A bf16 weight times a part is exact in fp32, so
// the matrix cores sum exact products: out = 2^-32 (W h + W m + W l), with fp32 roundings only in the
// accumulation (each kernel says how its sums are kept short; the test bound is that of K sequential
// fp32 additions). An int8 weight widens to bf16 exactly (|q| <= 127).
//
// +-inf and NaN need no care in the split: such an x (its remainders are NaN) or weight (inf times a
// zero part is NaN) leaves NaN in its outputs, and so do an |x| or a sum of 2^96 and more, which the
// scale takes out of range. An output that is not finite is formed again on the VALU (redo_rows), whose
// products and sums follow IEEE. Finite outputs had finite operands.
//
// MFMA operand layout (16x16x32): lane l supplies A[l % 16][8 (l / 16) + 0..7] and
// B[8 (l / 16) + 0..7][l % 16], and holds C[4 (l / 16) + i][l % 16], i = 0..3. Here A = W (outputs by
// k), B = x^T (k by rows), so lane l reads 8 consecutive k of one weight row and of one hidden row and
// ends with four consecutive outputs of one hidden row. Tile rows past the last hidden row or output,
// and entries past the end of k, read as zero (each result depends on its own row of A and column of B
// alone; what they compute is not stored).
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
constexpr float kUp = 0x1p32f, kDown = 0x1p-32f;

// three exact bf16 parts of 8 fp32 values below 2^96, times kUp
struct Parts {
    u4 h, m, l;
};
__device__ __forceinline__ Parts split3(const f4& a, const f4& b) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t th[8], tm[8], tl[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float x = v[i] * kUp;
        th[i] = __float_as_uint(x);
        const float r1 = x - __uint_as_float(th[i] & 0xFFFF0000u);
        tm[i] = __float_as_uint(r1);
        tl[i] = __float_as_uint(r1 - __uint_as_float(tm[i] & 0xFFFF0000u));
    }
    Parts p;
#pragma unroll
    for (int i = 0; i < 4; i++) {  // high halves of elements 2i (low) and 2i + 1 (high)
        p.h[i] = __builtin_amdgcn_perm(th[2 * i + 1], th[2 * i], 0x07060302u);
        p.m[i] = __builtin_amdgcn_perm(tm[2 * i + 1], tm[2 * i], 0x07060302u);
        p.l[i] = __builtin_amdgcn_perm(tl[2 * i + 1], tl[2 * i], 0x07060302u);
    }
    return p;
}

// 8 int8 weights (two dwords) as 8 bf16: the biased byte converted, 128 subtracted (exact), the
// high halves packed
__device__ __forceinline__ bf8 i8_to_bf16(uint32_t lo, uint32_t hi) {
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    uint32_t f[8];
#pragma unroll
    for (int i = 0; i < 8; i++)
        f[i] = __float_as_uint((float)(((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xffu) - 128.0f);
    u4 p;
#pragma unroll
    for (int i = 0; i < 4; i++) p[i] = __builtin_amdgcn_perm(f[2 * i + 1], f[2 * i], 0x07060302u);
    return __builtin_bit_cast(bf8, p);
}

// Operands reach the matrix cores through LDS. A wave's 16 consecutive lanes want 16 different rows,
// and loads in that order cost a cache line per lane (measured per compute unit, rows of 2 KiB that
// hit the L2: 16 rows x 64 bytes per wave load 27 bytes per ns, 8 rows x 128 bytes 78). So a tile of 16
// rows x 64 k is loaded with consecutive lanes along k (whole lines), written to LDS and read back one
// fragment per lane; the 16-byte units of a row are placed at their index xor the row, so eight
// consecutive lanes touch all 32 banks once in either order.
//
// Loads are raw buffer loads from the first row of the workgroup's tile: entries past the last row, or
// past k (an offset out of range), read as zero without touching memory. Offsets are 32-bit, which
// mfma_fits checks.
template <bool I8>
using WRaw = typename std::conditional<I8, u2, u4>::type;  // 8 weights as loaded
constexpr uint32_t kOut = 0x80000000u;                       // an offset past every tile

struct Tile {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t ld;  // row length in bytes
};
__device__ __forceinline__ Tile tile_of(const void* base, int64_t ld_bytes, int row0, int rows, int row_bytes) {
    const uint32_t ld = (uint32_t)ld_bytes;
    const char* p = static_cast<const char*>(base) + (int64_t)row0 * ld_bytes;
    return {__builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)((uint32_t)(rows - 1) * ld + (uint32_t)row_bytes), 0x00020000),
            ld};
}
// the 8 weights of tile row `row` from k on (k >= K: zeros)
template <bool I8>
__device__ __forceinline__ WRaw<I8> load_w8(const Tile& t, uint32_t row_off, int k, int K) {
    const uint32_t off = k < K ? row_off + (uint32_t)k * (I8 ? 1u : 2u) : kOut;
    if constexpr (I8)
        return __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(t.rsrc, off, 0, 0));
    else
        return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(t.rsrc, off, 0, 0));
}
__device__ __forceinline__ f4 load_x4(const Tile& t, uint32_t row_off, int k, int K) {
    const uint32_t off = k < K ? row_off + 4u * (uint32_t)k : kOut;
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(t.rsrc, off, 0, 0));
}
// Keeps the compiler from reordering a wave's LDS accesses. The hardware executes them in order, so a
// buffer of the wave's own is written again as soon as its reads are issued, with no wait.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The workgroup meets and sees each other's LDS writes; global stores are not waited for.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool I8>
__device__ __forceinline__ bf8 w_operand(const WRaw<I8>& r) {
    if constexpr (I8)
        return i8_to_bf16(r.x, r.y);
    else
        return __builtin_bit_cast(bf8, r);
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < __builtin_huge_valf(); }

// The outputs that are not finite among the `cols` from n0 on of the tile rows `rows` (a bit each), formed
// again as the VALU form does, by a workgroup whose waves have stored theirs (`lds`: two words that are free
// once it has met). A row with a NaN is done, as its outputs are NaN: the waves look through a row each. Of
// the others' outputs the waves (a power of two) take four each, the lanes along k, so that their loads are in
// flight together. (us, finite / one row with a NaN / one with an infinity / a NaN in every row; before, each lane
// formed its own outputs in k order: 24 x 1024 -> 2048 4.4 / 5.7 / 7.9 / 8.3, before 4.4 / 74 / 74 / 121; 256 x
// 1024 -> 3072 11.4 / 13.8 / 18.9 / 26.6, before 11.4 / 95 / 95 / 1411; 4096 rows 96 / 97 / 110 / 145, before 97 /
// 1230 / 1230 / 22460.)
template <bool I8>
__device__ __forceinline__ void redo_rows(const HeadArgs& a, int r0, int n0, int cols, uint64_t rows, uint32_t* lds, int wv, int nwaves,
                                          int lane) {
    const int end = min(n0 + cols, a.n);
    __syncthreads();
    if (threadIdx.x < 2) lds[threadIdx.x] = (uint32_t)(rows >> (32 * threadIdx.x));
    __syncthreads();
#pragma unroll 1
    for (uint64_t left = rows; left; left &= left - 1) {
        const int row = (int)__builtin_ctzll(left);
        if ((row & (nwaves - 1)) != wv) continue;
        const float* x = a.x + (int64_t)(r0 + row) * a.ldx;
        bool nan = false;
#pragma unroll 1
        for (int k = 4 * lane; k < a.k; k += 256) {
            const f4 v = *reinterpret_cast<const f4*>(x + k);
            nan = nan || v.x != v.x || v.y != v.y || v.z != v.z || v.w != v.w;
        }
        if (__ballot(nan) && lane == 0) atomicAnd(&lds[row >> 5], ~(1u << (row & 31)));
    }
    __syncthreads();
#pragma unroll 1
    for (rows = lds[0] | (uint64_t)lds[1] << 32; rows; rows &= rows - 1) {
        const int row = (int)__builtin_ctzll(rows), r = r0 + row;
        const float* x = a.x + (int64_t)r * a.ldx;
        float* o = a.out + (int64_t)r * a.ldo;
        uint64_t bad[2];  // a bit per output (of which this wave's own are not changing)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int n = n0 + 64 * h + lane;
            bad[h] = __ballot(n < end && !finite(o[min(n, end - 1)]));
        }
#pragma unroll 1
        for (int g = 0; 4 * g < cols; g++) {
            const uint32_t four = (uint32_t)(bad[g >> 4] >> (4 * (g & 15))) & 15u;
            if (!four || ((g + row) & (nwaves - 1)) != wv) continue;
            const int n = n0 + 4 * g;
            float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int k = 8 * lane; k < a.k; k += 512) {
                const f4 xa = *reinterpret_cast<const f4*>(x + k), xb = *reinterpret_cast<const f4*>(x + k + 4);
                WRaw<I8> w[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int64_t at = (int64_t)min(n + j, end - 1) * a.ldw + k;
                    if constexpr (I8)
                        w[j] = *reinterpret_cast<const u2*>(a.q + at);
                    else
                        w[j] = *reinterpret_cast<const u4*>(a.w + at);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) acc[j] = dot8(__builtin_bit_cast(u4, w_operand<I8>(w[j])), xa, xb, acc[j]);
            }
#pragma unroll
            for (int mask = 32; mask >= 1; mask /= 2)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[j] += __shfl_xor(acc[j], mask);
            if (lane < 4 && (four >> lane & 1u)) {
                const float sum = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
                o[n + lane] = I8 ? sum * a.scale[n + lane] : sum;
            }
        }
    }
}

// XCD-aware tile order: workgroups go to the 8 XCDs in turn, each with an L2 of its own, so workgroup
// b takes tile (b % 8) * per + b / 8 of the column-major tile list (row tiles fastest): an XCD's
// workgroups then share a few column tiles of W, read from memory once per XCD. False past the end.
__device__ __forceinline__ bool xcd_tile(int row_tiles, int tiles, int& rt, int& ct) {
    const int per = (tiles + 7) / 8;
    const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return false;
    rt = t % row_tiles;
    ct = t / row_tiles;
    return true;
}
inline int xcd_grid(int tiles) { return (tiles + 7) / 8 * 8; }

// Split-K form, for calls with few tiles: a workgroup owns 16 CT outputs of 16 RT rows; its NW waves
// split K in chunks of 64 (two 32-deep steps), chunk c to wave c % NW, each through operand buffers of
// its own (no barrier before the end). A tile's registers take the next chunk's loads as soon as the
// tile is in LDS. The waves' partial sums are added in LDS in a fixed order (waves w and w + NW / 2
// first, then over w).
template <int RT, int CT, int NW, bool I8>
__global__ __launch_bounds__(64 * NW) void head_mfma_kernel(HeadArgs a, int row_tiles, int tiles) {
    constexpr int NH = NW / 2;
    struct Turn {
        f4 x[16][16];
        WRaw<I8> w[CT > 1 ? 2 : 1][16][8];
    };
    __shared__ union {
        Turn turn[NW];
        struct {
            f4 part[NH][RT * CT][64];
            uint32_t redo;  // tile rows with an output that is not finite
        };
    } sm;
    int rt, ct;
    if (!xcd_tile(row_tiles, tiles, rt, ct)) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c16 = lane & 15;
    const int n0 = ct * 16 * CT, r0 = rt * 16 * RT;
    const int K = a.k, nchunks = (K + 63) / 64;
    const Tile tw = I8 ? tile_of(a.q, a.ldw, n0, min(16 * CT, a.n - n0), K)
                       : tile_of(a.w, a.ldw * 2, n0, min(16 * CT, a.n - n0), 2 * K);
    const Tile tx = tile_of(a.x, a.ldx * 4, r0, min(16 * RT, a.rows - r0), 4 * K);
    // a wave load holds 8 weight rows x 8 k, or 4 hidden rows x 4 k, per lane
    const uint32_t wl = (uint32_t)(lane >> 3) * tw.ld, xl = (uint32_t)(lane >> 4) * tx.ld;
    const int kw = 8 * (lane & 7), kx = 4 * (lane & 15);
    f4 acc[CT][RT];
#pragma unroll
    for (int t = 0; t < CT; t++)
#pragma unroll
        for (int q = 0; q < RT; q++) acc[t][q] = f4{0.f, 0.f, 0.f, 0.f};
    WRaw<I8> wr[CT][2];
    f4 xr[RT][4];
    auto load_wt = [&](int c, int t) {
#pragma unroll
        for (int j = 0; j < 2; j++) wr[t][j] = load_w8<I8>(tw, wl + (uint32_t)(16 * t + 8 * j) * tw.ld, 64 * c + kw, K);
    };
    auto load_xt = [&](int c, int q) {
#pragma unroll
        for (int j = 0; j < 4; j++) xr[q][j] = load_x4(tx, xl + (uint32_t)(16 * q + 4 * j) * tx.ld, 64 * c + kx, K);
    };
    Turn& tb = sm.turn[wv];
    if (wv < nchunks) {
#pragma unroll
        for (int q = 0; q < RT; q++) load_xt(wv, q);
#pragma unroll
        for (int t = 0; t < CT; t++) load_wt(wv, t);
    }
#pragma unroll 1
    for (int c = wv; c < nchunks; c += NW) {
        const int nx = c + NW;  // past the last chunk its loads are out of range
        Parts p[RT][2];
#pragma unroll
        for (int q = 0; q < RT; q++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 4 * j + (lane >> 4);
                tb.x[row][(lane & 15) ^ (row & 7)] = xr[q][j];
            }
            wave_order();
            f4 f[2][2];
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int h = 0; h < 2; h++) f[st][h] = tb.x[c16][(8 * st + 2 * g + h) ^ (c16 & 7)];
            wave_order();
            load_xt(nx, q);
#pragma unroll
            for (int st = 0; st < 2; st++) p[q][st] = split3(f[st][0], f[st][1]);
        }
        WRaw<I8> f[2][2];
        auto turn_w = [&](int t) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int row = 8 * j + (lane >> 3);
                tb.w[t & 1][row][(lane & 7) ^ (row & 7)] = wr[t][j];
            }
            wave_order();
#pragma unroll
            for (int st = 0; st < 2; st++) f[t & 1][st] = tb.w[t & 1][c16][(4 * st + g) ^ (c16 & 7)];
            wave_order();
            load_wt(nx, t);
        };
        turn_w(0);
#pragma unroll
        for (int t = 0; t < CT; t++) {
            if (t + 1 < CT) turn_w(t + 1);
            bf8 wa[2];
#pragma unroll
            for (int st = 0; st < 2; st++) wa[st] = w_operand<I8>(f[t & 1][st]);
            // the chunk's sums from zero, smallest parts first, then added to the wave's: six roundings of
            // which three are of the size of the sum
            f4 s[RT];
#pragma unroll
            for (int q = 0; q < RT; q++) s[q] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int part = 0; part < 3; part++)
#pragma unroll
                for (int st = 0; st < 2; st++)
#pragma unroll
                    for (int q = 0; q < RT; q++)
                        s[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            wa[st], __builtin_bit_cast(bf8, part == 0 ? p[q][st].l : part == 1 ? p[q][st].m : p[q][st].h), s[q], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < RT; q++) acc[t][q] += s[q];
        }
    }
    __syncthreads();  // every wave is done with its operand buffers
    if (threadIdx.x == 0) sm.redo = 0;
    if (wv >= NH)
#pragma unroll
        for (int t = 0; t < CT; t++)
#pragma unroll
            for (int q = 0; q < RT; q++) sm.part[wv - NH][t * RT + q][lane] = acc[t][q];
    __syncthreads();
    if (wv < NH)
#pragma unroll
        for (int t = 0; t < CT; t++)
#pragma unroll
            for (int q = 0; q < RT; q++) sm.part[wv][t * RT + q][lane] = acc[t][q] + sm.part[wv][t * RT + q][lane];
    __syncthreads();
    // (output, row) pairs of the tile, consecutive threads on consecutive outputs
    for (int e = threadIdx.x; e < 16 * CT * 16 * RT; e += 64 * NW) {
        const int nl = e % (16 * CT), rl = e / (16 * CT);
        const int l = 16 * ((nl % 16) / 4) + rl % 16;
        double dsum = 0.0;
#pragma unroll
        for (int w = 0; w < NH; w++) dsum += (double)sm.part[w][(nl / 16) * RT + rl / 16][l][nl % 4];
        float sum = (float)(dsum * (double)kDown);
        const int n = n0 + nl, r = r0 + rl;
        if (n >= a.n || r >= a.rows) continue;
        if constexpr (I8) sum *= a.scale[n];
        if (!finite(sum)) atomicOr(&sm.redo, 1u << rl);
        a.out[(int64_t)r * a.ldo + n] = sum;
    }
    lds_barrier();
    const uint32_t rows = sm.redo;
    if (__builtin_expect(rows != 0, 0)) redo_rows<I8>(a, r0, n0, 16 * CT, rows, reinterpret_cast<uint32_t*>(&sm.part), wv, NW, lane);
}

template <int RT, int CT, int NW>
hipError_t launch_mfma(const HeadArgs& a, hipStream_t stream) {
    const int row_tiles = (a.rows + 16 * RT - 1) / (16 * RT);
    const int tiles = row_tiles * ((a.n + 16 * CT - 1) / (16 * CT));
    if (a.q)
        hipLaunchKernelGGL((head_mfma_kernel<RT, CT, NW, true>), dim3(xcd_grid(tiles)), dim3(64 * NW), 0, stream, a, row_tiles, tiles);
    else
        hipLaunchKernelGGL((head_mfma_kernel<RT, CT, NW, false>), dim3(xcd_grid(tiles)), dim3(64 * NW), 0, stream, a, row_tiles, tiles);
    return hipGetLastError();
}

// Tiled form, for calls with tiles enough to fill the chip: a workgroup of 2 x 2 waves owns 32 WR rows
// x 32 WC outputs, a wave 16 WR x 16 WC, over the whole of K in steps of 64. Both operands are staged
// in LDS once per workgroup, the hidden rows split there into their three parts (int8 weights widened);
// the next step's loads are in flight during a step's products, and other workgroups of the compute
// unit fill the rest.
template <int WR, int WC, bool I8>
__global__ __launch_bounds__(kHT) __attribute__((amdgpu_waves_per_eu(2))) void head_mfma_tiled_kernel(HeadArgs a, int row_tiles,
                                                                                                      int tiles) {
    constexpr int BM = 32 * WR, BN = 32 * WC;
    __shared__ u4 xs[3][BM][8], ws[BN][8];  // rows of 64 bf16, the 16-byte units of a row xor-ed with it
    int rt, ct;
    if (!xcd_tile(row_tiles, tiles, rt, ct)) return;
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int g = lane >> 4, c16 = lane & 15;
    const int r0 = rt * BM, n0 = ct * BN;
    const int rw = (wv & 1) * 16 * WR, nw = (wv >> 1) * 16 * WC;  // the wave's part of the tile
    const int K = a.k, nchunks = (K + 63) / 64;
    const Tile tw = I8 ? tile_of(a.q, a.ldw, n0, min(BN, a.n - n0), K) : tile_of(a.w, a.ldw * 2, n0, min(BN, a.n - n0), 2 * K);
    const Tile tx = tile_of(a.x, a.ldx * 4, r0, min(BM, a.rows - r0), 4 * K);
    // a load of the workgroup holds 32 weight rows x 8 k, or 16 hidden rows x 4 k, per thread
    const uint32_t wl = (uint32_t)(t >> 3) * tw.ld, xl = (uint32_t)(t >> 4) * tx.ld;
    const int kw = 8 * (t & 7), kx = 4 * (t & 15);
    // The sums of the high parts in acc, moved to tot every 128 k; those of the others, 2^-8 of their
    // size, in low, which also takes what the addition to tot rounds off (Fast2Sum): so the roundings
    // of the size of the sum are the four of each 128 k and the last. Relative 2-norm error against
    // 64 bits, normal data, k = 1024: 0.7e-7 (the VALU form: 1.0e-7; one chain over all of k: 3.4e-7).
    f4 acc[WC][WR], low[WC][WR], tot[WC][WR];
#pragma unroll
    for (int i = 0; i < WC; i++)
#pragma unroll
        for (int q = 0; q < WR; q++) acc[i][q] = low[i][q] = tot[i][q] = f4{0.f, 0.f, 0.f, 0.f};
    WRaw<I8> wr[WC];
    f4 xr[2 * WR];
    auto load = [&](int c) {  // past the last chunk: out of range
#pragma unroll
        for (int j = 0; j < 2 * WR; j++) xr[j] = load_x4(tx, xl + (uint32_t)(16 * j) * tx.ld, 64 * c + kx, K);
#pragma unroll
        for (int j = 0; j < WC; j++) wr[j] = load_w8<I8>(tw, wl + (uint32_t)(32 * j) * tw.ld, 64 * c + kw, K);
    };
    load(0);
#pragma unroll 1
    for (int c = 0; c < nchunks; c++) {
#pragma unroll
        for (int j = 0; j < 2 * WR; j++) {
            const int row = 16 * j + (t >> 4);
            uint32_t th[4], tm[4], tl[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float x = xr[j][i] * kUp;
                th[i] = __float_as_uint(x);
                const float r1 = x - __uint_as_float(th[i] & 0xFFFF0000u);
                tm[i] = __float_as_uint(r1);
                tl[i] = __float_as_uint(r1 - __uint_as_float(tm[i] & 0xFFFF0000u));
            }
            const int unit = ((t & 15) >> 1) ^ (row & 7), half = t & 1;
            auto put = [&](int part, const uint32_t (&v)[4]) {
                reinterpret_cast<u2*>(&xs[part][row][unit])[half] = u2{__builtin_amdgcn_perm(v[1], v[0], 0x07060302u),
                                                                       __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)};
            };
            put(0, th);
            put(1, tm);
            put(2, tl);
        }
#pragma unroll
        for (int j = 0; j < WC; j++) {
            const int row = 32 * j + (t >> 3);
            ws[row][(t & 7) ^ (row & 7)] = __builtin_bit_cast(u4, w_operand<I8>(wr[j]));
        }
        __syncthreads();
        load(c + 1);
#pragma unroll
        for (int st = 0; st < 2; st++) {
            const int unit = (4 * st + g) ^ (c16 & 7);
            bf8 wa[WC];
#pragma unroll
            for (int i = 0; i < WC; i++) wa[i] = __builtin_bit_cast(bf8, ws[nw + 16 * i + c16][unit]);
#pragma unroll
            for (int part = 0; part < 3; part++) {
                bf8 xb[WR];
#pragma unroll
                for (int q = 0; q < WR; q++) xb[q] = __builtin_bit_cast(bf8, xs[part][rw + 16 * q + c16][unit]);
#pragma unroll
                for (int q = 0; q < WR; q++)
#pragma unroll
                    for (int i = 0; i < WC; i++) {
                        f4& s = part == 0 ? acc[i][q] : low[i][q];
                        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[i], xb[q], s, 0, 0, 0);
                    }
            }
        }
        if ((c & 1) || c + 1 == nchunks) {
#pragma unroll
            for (int i = 0; i < WC; i++)
#pragma unroll
                for (int q = 0; q < WR; q++) {
                    const f4 t2 = tot[i][q] + acc[i][q];
                    low[i][q] += acc[i][q] - (t2 - tot[i][q]);
                    tot[i][q] = t2;
                    acc[i][q] = f4{0.f, 0.f, 0.f, 0.f};
                }
        }
        __syncthreads();
    }
    const bool vec = a.ldo % 4 == 0 && ((uintptr_t)a.out & 15u) == 0;
    bool bad[WR] = {};
#pragma unroll
    for (int i = 0; i < WC; i++) {
        const int n = n0 + nw + 16 * i + 4 * g;
        f4 sc = {1.f, 1.f, 1.f, 1.f};
        if constexpr (I8) {
#pragma unroll
            for (int e = 0; e < 4; e++) sc[e] = a.scale[min(n + e, a.n - 1)];
        }
#pragma unroll
        for (int q = 0; q < WR; q++) {
            const int r = r0 + rw + 16 * q + c16;
            float* o = a.out + (int64_t)r * a.ldo + n;
            f4 v = (tot[i][q] + low[i][q]) * kDown;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if constexpr (I8) v[e] *= sc[e];
                bad[q] = bad[q] || !finite(v[e]);
            }
            if (r >= a.rows) continue;
            if (vec && n + 3 < a.n) {
                *reinterpret_cast<f4*>(o) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < a.n) o[e] = v[e];
            }
        }
    }
    // each wave's rows with an output that is not finite, in LDS (the operands are done with)
    uint32_t mine = 0;
#pragma unroll
    for (int q = 0; q < WR; q++) {
        const uint64_t m = __ballot(bad[q] && r0 + rw + 16 * q + c16 < a.rows);
        mine |= (uint32_t)((m | m >> 16 | m >> 32 | m >> 48) & 0xffffu) << (16 * q);
    }
    uint32_t* redo = reinterpret_cast<uint32_t*>(&xs[0][0][0]);
    if (lane == 0) redo[wv] = mine;
    lds_barrier();
    const uint64_t rows = (uint64_t)(redo[0] | redo[2]) | (uint64_t)(redo[1] | redo[3]) << (16 * WR);
    if (__builtin_expect(rows != 0, 0)) redo_rows<I8>(a, r0, n0, BN, rows, redo, wv, 4, lane);
}

template <int WR, int WC>
hipError_t launch_tiled(const HeadArgs& a, hipStream_t stream) {
    const int row_tiles = (a.rows + 32 * WR - 1) / (32 * WR);
    const int tiles = row_tiles * ((a.n + 32 * WC - 1) / (32 * WC));
    if (a.q)
        hipLaunchKernelGGL((head_mfma_tiled_kernel<WR, WC, true>), dim3(xcd_grid(tiles)), dim3(kHT), 0, stream, a, row_tiles, tiles);
    else
        hipLaunchKernelGGL((head_mfma_tiled_kernel<WR, WC, false>), dim3(xcd_grid(tiles)), dim3(kHT), 0, stream, a, row_tiles, tiles);
    return hipGetLastError();
}

// FromBf16LinearInt8 for one output row per workgroup.
__global__ __launch_bounds__(kHT) void head_pack_i8_kernel(int k, const uint16_t* __restrict__ w, int64_t ldw,
                                                          int8_t* __restrict__ q, int64_t ldq, float* __restrict__ scale) {
    __shared__ float wmax[kHT / 64];
    const int n = blockIdx.x;
    const uint16_t* row = w + (int64_t)n * ldw;
    float amax = 0.0f;
    for (int i = threadIdx.x; i < k; i += kHT) amax = fmaxf(amax, fabsf(__uint_as_float((uint32_t)row[i] << 16)));
#pragma unroll
    for (int mask = 32; mask >= 1; mask /= 2) amax = fmaxf(amax, __shfl_xor(amax, mask));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const float scl = amax > 0.0f ? amax / 127.0f : 1.0f;  // correctly rounded fp32 divisions
    const float inv = 1.0f / scl;
    int8_t* qr = q + (int64_t)n * ldq;
    for (int i = threadIdx.x; i < k; i += kHT) {
        const float t = rintf(__uint_as_float((uint32_t)row[i] << 16) * inv);  // half to even, as MathF.Round
        // (int) then Math.Clamp, with .NET's saturating conversion: NaN (0 * inf, when 1 / scale
        // overflowed) gives 0, +-inf the clamp's ends; clamped in fp32 first, so the cast is exact
        qr[i] = (int8_t)(t != t ? 0 : (int)fminf(fmaxf(t, -127.0f), 127.0f));
    }
    if (threadIdx.x == 0) scale[n] = scl;
}

// Rows are split into groups of at least two, one grid row each, while the launch has fewer than 2048
// waves for the chip's 1024 SIMDs; every group reads the weight again.
template <int KJ>
hipError_t launch_k(HeadArgs a, hipStream_t stream) {
    const int tiles = (a.n + (kHT / 64) * R - 1) / ((kHT / 64) * R);
    const int waves = tiles * (kHT / 64);
    const int groups = std::max(1, std::min(2048 / waves, a.rows / 2));
    a.row_group = (a.rows + groups - 1) / groups;
    const dim3 grid(tiles, (a.rows + a.row_group - 1) / a.row_group);
    if (a.q) {
        if (a.k == 512 * KJ)
            hipLaunchKernelGGL((head_i8_kernel<KJ, true>), grid, dim3(kHT), 0, stream, a);
        else
            hipLaunchKernelGGL((head_i8_kernel<KJ, false>), grid, dim3(kHT), 0, stream, a);
    } else if (a.k == 512 * KJ) {
        hipLaunchKernelGGL((head_kernel<KJ, true>), grid, dim3(kHT), 0, stream, a);
    } else {
        hipLaunchKernelGGL((head_kernel<KJ, false>), grid, dim3(kHT), 0, stream, a);
    }
    return hipGetLastError();
}

// The matrix forms address a tile (at most 128 outputs, 64 rows) by 31-bit byte offsets.
bool mfma_fits(const HeadArgs& a) {
    constexpr int64_t kMax = int64_t(1) << 31;
    return a.ldw < kMax / (128 * (a.q ? 1 : 2)) && a.ldx < kMax / (64 * 4);
}

}  // namespace

hipError_t launch_head(const HeadArgs& a, hipStream_t stream) {
    if (a.rows <= 0 || a.n <= 0) return hipSuccess;
    if (a.k <= 0 || a.k > 2048) return hipErrorInvalidValue;
    // One to three rows (two above k = 1024) on the VALU: one pass over the weight with no operand to
    // turn, 1 x 1024 -> 2048 2.5 us (split-K form 3.9), 3 x 1024 -> 2048 3.6 (3.9), but 4 x 1024 -> 3072
    // 4.5 (4.1) and 3 x 2048 -> 3072 6.2 (5.0). (bf16, back to back, 6 weights in turn; int8 alike up to
    // k = 1024. Above, int8 calls of at most 8192 outputs are 0.1 to 0.9 us faster on the VALU (4 x 2048 -> 512 4.5,
    // here 5.2; 12 x 2048 -> 64 4.3, 5.1), but with a rounding error of 1.0e-7 where this form's is 0.7e-7.)
    const bool few = a.rows <= 2 || (a.rows == 3 && a.k <= 1024);
    if (!few && mfma_fits(a)) {
        // The split-K form with the smallest tile that leaves at most one workgroup per compute unit:
        // its time is that of loading a tile (us, one round, k = 1024: 16 x 16 4.1, 16 x 32 4.5, 16 x 48
        // 5.1, 32 x 48 7.5, 32 x 64 8.6, 32 x 96 10.3) and a second round adds the same again (32 x 48
        // at 2 rounds 13.3). The two largest need k >= 512, as their eight waves take 64 k each
        // (256 x 256 -> 3072: 32 x 96 6.7, tiled 5.3).
        auto tiles = [&](int rt, int ct) { return (int64_t)((a.rows + 16 * rt - 1) / (16 * rt)) * ((a.n + 16 * ct - 1) / (16 * ct)); };
        constexpr int kCUs = 256;
        if (tiles(1, 1) <= kCUs) return launch_mfma<1, 1, 16>(a, stream);
        if (tiles(1, 2) <= kCUs) return launch_mfma<1, 2, 8>(a, stream);
        if (tiles(1, 3) <= kCUs) return launch_mfma<1, 3, 8>(a, stream);
        if (tiles(2, 3) <= kCUs) return launch_mfma<2, 3, 8>(a, stream);
        if (a.k >= 512 && tiles(2, 4) <= kCUs) return launch_mfma<2, 4, 8>(a, stream);
        if (a.k >= 512 && tiles(2, 6) <= kCUs) return launch_mfma<2, 6, 8>(a, stream);
        // The tiled form beyond: 64 x 128 tiles from one and a half workgroups per compute unit, else
        // 32 x 64 (us, 32 x 64 / 64 x 128: 512 x 1024 -> 3072 18.6 / 23.9, 1024 x 1024 -> 3072 32.8 / 31.3,
        // 2048 x 2048 -> 2048 85 / 61, 4096 x 1024 -> 3072 122 / 91; split-K 32 x 96: 19.5, 42, 95, 167).
        if (2 * tiles(4, 8) >= 3 * kCUs) return launch_tiled<2, 4>(a, stream);
        return launch_tiled<1, 2>(a, stream);
    }
    switch ((a.k + 511) / 512) {
        case 1: return launch_k<1>(a, stream);
        case 2: return launch_k<2>(a, stream);
        case 3: return launch_k<3>(a, stream);
        default: return launch_k<4>(a, stream);
    }
}

hipError_t launch_head_pack_int8(int k, int n, const uint16_t* w, int64_t ldw, int8_t* q, int64_t ldq, float* scale,
                                 hipStream_t stream) {
    if (n <= 0 || k <= 0) return hipSuccess;
    hipLaunchKernelGGL(head_pack_i8_kernel, dim3(n), dim3(kHT), 0, stream, k, w, ldw, q, ldq, scale);
    return hipGetLastError();
}

}  // namespace vxs
