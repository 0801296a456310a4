// Batched projections of some dozens to some hundreds of rows: C = X . [W0 | W1 | ...]^T with the weights
// decoded in registers, between the matrix instructions.
//
// Takes the place of the reference's decode-then-multiply prefill GEMM (dequantize*ToFP16 and gemmMMA,
// J/backend/tornado/kernels/TransformerBatchPrefillKernels.java:917-1076,2325-2363) where a call has too
// few rows to pay for a decoded copy of its weights in memory (jl_gemm_dense.hip) and too many for one
// pass over the weights per 32 rows (jl_gemm_skinny_kernels.h).  The kernel that decoded in its loop
// before (jl_gemm.hip) passes every decoded weight through LDS, written by one wave and read by others, in
// steps of 64 columns with three kinds of waves behind one barrier; here a weight goes to the wave that
// multiplies it and nowhere else:
//
//   * a wave owns 32 weight rows (gate/up: 16 of each) and 16 MB activation rows; the WN waves of a
//     workgroup that share activations read them from one LDS ring, filled by LDS-DMA; KW sets of such
//     waves take every KW-th 256-column block and add their sums at the end, in a fixed order, inside the
//     workgroup: no partial sums in memory and no launch behind the call;
//   * a wave brings its rows' raw bytes in as 16-byte pieces (whole cache lines: asked for slice by slice
//     as the lanes want them, the lines of 16 rows came from L2 several times over), puts them into LDS
//     of its own and reads them back as what each lane decodes: 32 columns of one row;
//   * a step is 128 columns: four fragments per row group, each multiplied with MB row blocks.  While
//     the matrix instructions of a step run, the wave decodes the next step's fragments; the loads of the
//     block after next go out between them.
//
// What bounds it: at MB = 8 a step issues 64 matrix instructions, 1 024 cycles a wave, two waves to a SIMD; LDS
// (8 waves x 32 KB of activations), vector instructions and loads take about half of those cycles each,
// and the parts hide each other by half: 41 % of the matrix rate at the clock it runs at (rocprofv3:
// SQ_VALU_MFMA_BUSY_CYCLES against SQ_BUSY_CYCLES).  Without the raw bytes' way a launch is a sixth
// shorter, without the decode a tenth, without either and the stage loads a third.
// Measured (one box, weights from HBM, before -> now): Q4_K gate/up 2 x [11008 x 4096] at 201 rows 107 -> 55
// us, q | k | v 12288 x 4096 61 -> 37, Q4_0 gate/up 2 x [14592 x 4096] at 99 rows 53 -> 43, Q8_0 q | k | v
// 13824 x 4608 at 408 rows 123 -> 84, Q6_K gate/up 2 x [13824 x 5120] at 128 rows 179 -> 80.
// Tried and taken back: activation fragments two row blocks ahead (55.2 against 56.4 us, and it spills
// with Q8_0); three stages (no change); matrix instructions at raised priority (no change); 32-byte quant
// runs read from LDS unaligned instead of funnel-shifted (68 against 46 us).
#include "jl_device.h"
#include "jl_internal.h"
#include "jl_slice_decode.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef __attribute__((address_space(1))) const uint8_t gbyte;
typedef __attribute__((address_space(1))) const u32x4u gpiece;
typedef __attribute__((address_space(3))) void lvoid;

#define JL_WAIT_VM(N) \
    __builtin_amdgcn_s_waitcnt(((N)&0xF) | (((N) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

constexpr int kMaxSeg = 8;
constexpr int kGroup = 16;      // weight rows of a matrix instruction
constexpr int NR = 2;           // such groups per wave

struct RegParams {
    const uint8_t *w[kMaxSeg];
    int seg_rows[kMaxSeg];
    int seg_group_begin[kMaxSeg + 1];  // first row group of each weight; [nseg] = all groups
    int seg_col_begin[kMaxSeg];        // first output column of each weight
    int nseg;
    const uint8_t *w_up;       // JL_SWIGLU: the up weight
    const _Float16 *A;         // [rows x k]
    const float *row_scale;    // null: every scale is 1
    const float *X;            // set: rows whose scale is marked by a minus sign are multiplied from here
    float *C;
    int c_f16;                 // JL_SWIGLU: C holds binary16 values, ldo and col_offset count them
    int rows, k;
    int64_t ldo, col_offset;
    int epilogue;
    int row_bytes;
    int ntiles, mtiles;
};

// ---- weights --------------------------------------------------------------------------------------

// 16-byte pieces of a row's 256 columns (Q6_K: 210 bytes, the last piece overlaps the one before), and
// the 1 KB loads that bring in a group's
constexpr int pieces_of(int type) { return (quad_bytes(type) + 15) / 16; }
constexpr int raw_loads(int type) { return (16 * pieces_of(type) + 63) / 64; }
constexpr int raw_bytes(int type) { return 16 * pieces_of(type) * 16; }

// LDS by hand: the compiler would drain the LDS-DMA loads before any LDS access that it sees
template <int N>
__device__ __forceinline__ void lds_issue_b128(uint32_t addr, u32x4 (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v[i]) : "v"(addr), "n"(16 * i) : "memory");
}
template <int N>
__device__ __forceinline__ void lds_issue_2b32(uint32_t addr, u32x2 (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "=&v"(v[i]) : "v"(addr), "n"(2 * i), "n"(2 * i + 1) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_issue_b32(uint32_t addr, uint32_t &v) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_issue_u16(uint32_t addr, uint32_t &v) {
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
template <typename T, int N>
__device__ __forceinline__ void settled(T (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) {
        T t = v[i];
        asm volatile("" : "+v"(t));
        v[i] = t;
    }
}
__device__ __forceinline__ void settled(uint32_t &v) { asm volatile("" : "+v"(v)); }

// what a lane reads for half t of its row's block: 32 columns, 128 t + 32 g ..
template <int TYPE> struct HalfWords;
template <> struct HalfWords<JL_Q8_0> {
    u32x2 w[4];
    uint32_t last, d;
    __device__ __forceinline__ uint32_t word(int i) const { return i == 8 ? last : w[i >> 1][i & 1]; }
    __device__ __forceinline__ void issue(uint32_t row, int t, int g) {
        const uint32_t at = 34 * (4 * t + g);
        lds_issue_2b32(row + ((at + 2) & ~3u), w);
        lds_issue_b32<32>(row + ((at + 2) & ~3u), last);
        lds_issue_u16<0>(row + at, d);
    }
    __device__ __forceinline__ void settle() { settled(w); settled(last); settled(d); }
};
template <> struct HalfWords<JL_Q4_0> {
    u32x2 w[2];
    uint32_t last, d;
    __device__ __forceinline__ uint32_t word(int i) const { return i == 4 ? last : w[i >> 1][i & 1]; }
    __device__ __forceinline__ void issue(uint32_t row, int t, int g) {
        const uint32_t at = 18 * (4 * t + g);
        lds_issue_2b32(row + ((at + 2) & ~3u), w);
        lds_issue_b32<16>(row + ((at + 2) & ~3u), last);
        lds_issue_u16<0>(row + at, d);
    }
    __device__ __forceinline__ void settle() { settled(w); settled(last); settled(d); }
};
template <> struct HalfWords<JL_Q4_K> {
    u32x4 h[1], q[2];
    __device__ __forceinline__ void issue(uint32_t row, int t, int g) {
        lds_issue_b128(row, h);
        lds_issue_b128(row + 16 + 64 * t + 32 * (g >> 1), q);
    }
    __device__ __forceinline__ void settle() { settled(h); settled(q); }
};
template <> struct HalfWords<JL_Q6_K> {
    u32x4 ql[2], qh[2];
    uint32_t sc;
    __device__ __forceinline__ void issue(uint32_t row, int t, int g) {
        lds_issue_b128(row + 64 * t + 32 * (g & 1), ql);
        lds_issue_b128(row + 128 + 32 * t, qh);
        lds_issue_u16<0>(row + 192 + 8 * t + 2 * g, sc);
    }
    __device__ __forceinline__ void settle() { settled(ql); settled(qh); settled(sc); }
};

// Eight bytes 0..15 -> byte * ds - dm, one rounding each.  A byte q of 0..15 is the e4m3 number q 2^-9 (its
// subnormals and its first binade are one even grid), so the fp8 conversion with a scale of 2^9 is the
// number itself, one instruction for two where the exponent trick (bytes_to_h2) takes two.
__device__ __forceinline__ half8 frag_affine(uint32_t q0, uint32_t q1, h2 ds, h2 dm) {
    const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(q0, 512.f, false) * ds - dm;
    const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(q0, 512.f, true) * ds - dm;
    const h2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(q1, 512.f, false) * ds - dm;
    const h2 e = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(q1, 512.f, true) * ds - dm;
    return half8{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
}

// Fragment i: columns 8 i .. of the lane's 32, the weight rounded to fp16 as jl_decode_to_f16 leaves it
// (Q6_K: scale x quant, an integer of at most 4096 in magnitude; d multiplies the products).
template <int TYPE>
__device__ __forceinline__ half8 decode_frag(const HalfWords<TYPE> &s, int t, int g, int i) {
    if constexpr (TYPE == JL_Q8_0) {
        // (block 4 t + g starts two bytes off a dword when g is odd: its quants then lie on dwords)
        const uint32_t shift = g & 1 ? 0 : 16;
        const _Float16 d = __builtin_bit_cast(_Float16, (unsigned short)s.d);
        const h2 bias = {(_Float16)1152.f, (_Float16)1152.f}, d2 = {d, d};
        const uint32_t q0 = __builtin_amdgcn_alignbit(s.word(2 * i + 1), s.word(2 * i), shift) ^ 0x80808080u;
        const uint32_t q1 = __builtin_amdgcn_alignbit(s.word(2 * i + 2), s.word(2 * i + 1), shift) ^ 0x80808080u;
        return frag_scaled(q0, q1, bias, d2);
    } else if constexpr (TYPE == JL_Q4_0) {
        const uint32_t shift = g & 1 ? 0 : 16;
        const _Float16 d = __builtin_bit_cast(_Float16, (unsigned short)s.d);
        const h2 bias = {(_Float16)1032.f, (_Float16)1032.f}, d2 = {d, d};
        const int at = 2 * (i & 1), nib = 4 * (i >> 1);
        const uint32_t q0 = __builtin_amdgcn_alignbit(s.word(at + 1), s.word(at), shift);
        const uint32_t q1 = __builtin_amdgcn_alignbit(s.word(at + 2), s.word(at + 1), shift);
        return frag_scaled((q0 >> nib) & 0x0F0F0F0Fu, (q1 >> nib) & 0x0F0F0F0Fu, bias, d2);
    } else if constexpr (TYPE == JL_Q4_K) {
        // sub-block 4 t + g: scale and minimum from the header's twelve packed bytes
        const uint32_t hx = s.h[0].x, hy = s.h[0].y, hz = s.h[0].z, hw = s.h[0].w;
        const int sh = 8 * g, nib = 4 * (g & 1);
        const uint32_t sc = t == 0 ? (hy >> sh) & 63u : ((hw >> sh) & 0xFu) | (((hy >> sh) & 0xC0u) >> 2);
        const uint32_t mn = t == 0 ? (hz >> sh) & 63u : ((hw >> (sh + 4)) & 0xFu) | (((hz >> sh) & 0xC0u) >> 2);
        const _Float16 ds = (_Float16)(jl_half_bits_to_float(hx) * (float)sc);
        const _Float16 dm = (_Float16)(jl_half_bits_to_float(hx >> 16) * (float)mn);
        const uint32_t q0 = (s.q[i >> 1][2 * (i & 1)] >> nib) & 0x0F0F0F0Fu, q1 = (s.q[i >> 1][2 * (i & 1) + 1] >> nib) & 0x0F0F0F0Fu;
        return frag_affine(q0, q1, h2{ds, ds}, h2{dm, dm});
    } else {
        static_assert(TYPE == JL_Q6_K, "no decoder for this type");
        const h2 bias = {(_Float16)1056.f, (_Float16)1056.f};
        const int nib = 4 * (g >> 1), top = 2 * g;
        const uint32_t l0 = s.ql[i >> 1][2 * (i & 1)], l1 = s.ql[i >> 1][2 * (i & 1) + 1];
        const uint32_t h0 = s.qh[i >> 1][2 * (i & 1)], h1 = s.qh[i >> 1][2 * (i & 1) + 1];
        return frag_scaled(((l0 >> nib) & 0x0F0F0F0Fu) | (((h0 >> top) & 0x03030303u) << 4),
                           ((l1 >> nib) & 0x0F0F0F0Fu) | (((h1 >> top) & 0x03030303u) << 4), bias, sbyte_h2(s.sc, i >> 1));
    }
}

// One output of a row that no power of two brings into fp16's range block by block: fp32 products of the
// activations as they came, lanes across the columns.  The sum is in every lane.
template <int TYPE>
__device__ __forceinline__ float plain_dot(const uint8_t *w, const float *x, int k, int lane) {
    float sum = 0.f;
    for (int c = lane; c < k; c += 64) {
        const uint8_t *b = w + (c >> 5) * (quad_bytes(TYPE) / 8);
        const float d = jl_half_bits_to_float(*(const uint16_t *)b);
        const int q = TYPE == JL_Q8_0 ? (int)(int8_t)b[2 + (c & 31)] : ((b[2 + (c & 15)] >> ((c & 16) >> 2)) & 15) - 8;
        sum += d * (float)q * x[c];
    }
    return jl_group_sum<64>(sum);
}

// What the chunk position of an activation row is exclusive-ored with.  A 128-bit LDS read serves 16
// lanes a cycle, rows 0-3 and 12-15 of one slice with rows 4-11 of the next: with slices four chunks
// apart these keys give the sixteen different 16-byte places (with row / 2 as the key they met in pairs:
// 8 cycles a read instead of 4, by SQ_LDS_BANK_CONFLICT).
__device__ __forceinline__ int row_key(int row) {
    const int v = (row >> 1) & 7;
    return v ^ ((v & 4) >> 1);
}

// LDS: per set of waves two stages of activations (128 columns of 16 MB rows each), then every wave's raw
// bytes (the last word that a lane reads may lie past them)
constexpr int kStages = 2;
template <int TYPE, int MB, int WN, int KW> constexpr int lds_bytes() {
    constexpr int ring = KW * kStages * MB * 4096 + WN * KW * NR * raw_bytes(TYPE) + 16;
    constexpr int fold = KW > 1 ? KW * WN * MB * NR * 1024 : 0;
    return ring > fold ? ring : fold;
}

template <int TYPE, int MB, int WN, int KW>
__global__ void __launch_bounds__(64 * WN * KW) __attribute__((amdgpu_waves_per_eu(2, 2)))
jl_gemm_reg(RegParams p) {
    extern __shared__ __attribute__((aligned(128))) uint8_t lds[];
    constexpr int LA = (4 * MB + WN - 1) / WN;   // 1 KB loads of a stage per wave (past the last one: that one again)
    constexpr int STAGE = MB * 4096;
    constexpr int PL = raw_loads(TYPE), PIECES = pieces_of(TYPE), RAW = raw_bytes(TYPE), RAW_ROW = 16 * PIECES;
    constexpr int QUAD = quad_bytes(TYPE);
    constexpr int ROWS = 16 * MB;
    constexpr bool POST = TYPE == JL_Q6_K;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int wn = wave % WN, kw = wave / WN;
    const int r16 = lane & 15, g = lane >> 4;

    // XCD x (workgroups blockIdx % 8 == x) takes the x-th eighth of the tiles, the row tiles of one set of
    // weight rows next to each other: they find the raw bytes in its L2
    const int total_tiles = p.ntiles * p.mtiles;
    const int per_xcd = (total_tiles + 7) / 8;
    const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || logical >= total_tiles) return;
    const int nt = logical / p.mtiles, mt = logical - nt * p.mtiles;
    const int m0 = mt * ROWS;
    const bool swiglu = p.epilogue == JL_SWIGLU;
    const int nb = p.k / 256;
    const int iters = (nb + KW - 1) / KW;

    // the wave's two groups of 16 weight rows (the table is walked with constant indices: it stays in
    // scalar registers)
    const int total_groups = p.seg_group_begin[p.nseg];
    const uint8_t *group_ptr[NR];
    int out_col[NR], out_from[NR];     // output column of the group's first row; rows before out_from are not stored
#pragma unroll
    for (int j = 0; j < NR; j++) {
        int group = swiglu ? nt * WN + wn : (nt * WN + wn) * NR + j;
        const bool real = group < total_groups;
        group = real ? group : total_groups - 1;
        const uint8_t *w = p.w[0];
        int rows = p.seg_rows[0], begin = 0, col = 0;
#pragma unroll
        for (int i = 1; i < kMaxSeg; i++) {
            if (i < p.nseg && group >= p.seg_group_begin[i]) {
                w = p.w[i];
                rows = p.seg_rows[i];
                begin = p.seg_group_begin[i];
                col = p.seg_col_begin[i];
            }
        }
        if (swiglu && j == 1) w = p.w_up;
        const int local = (group - begin) * kGroup;
        // a weight's last group is its last 16 rows: those that the group before has are not stored again
        const int base = local + kGroup <= rows ? local : rows - kGroup;
        out_col[j] = col + base;
        out_from[j] = real ? local - base : kGroup;
        group_ptr[j] = w + (int64_t)base * p.row_bytes;
    }

    // A stage: [half of the 128 columns][row][eight 16-byte chunks, at chunk ^ row_key(row)].  This wave's
    // loads are every WN-th octet of rows (rows past the call's last one re-read that one; their results
    // are not stored).
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lvoid *)lds;
    uint8_t *ring = lds + kw * kStages * STAGE;
    uint32_t a_off[LA];
#pragma unroll
    for (int n = 0; n < LA; n++) {
        const int o = n * WN + wn < 4 * MB ? n * WN + wn : 4 * MB - 1;
        const int hi = o / (2 * MB), row = (o % (2 * MB)) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ row_key(row);
        const int m = m0 + row < p.rows ? m0 + row : p.rows - 1;
        a_off[n] = (uint32_t)m * (uint32_t)(p.k * 2) + hi * 128 + c * 16;
    }
    // step s = half s % 2 of block (s / 2) KW + kw; steps past the last one: that one again, so that the count
    // of loads does not change
    // (Buffer loads: 141 calls of 65 ... 511 rows, all four types, take 0.8 % less time with them than with global ones,
    // 0.2 % more in the worst of 28 pairs of type and tiling.  What they bring in lies in the caches, where how far apart rows
    // are does not matter to them; it does in jl_gemm_hh, which has global ones.)
    const int last_step = 2 * iters - 1;
    auto issue_stage = [&](int s, int slot) {
        s = s < last_step ? s : last_step;
        int b = (s >> 1) * KW + kw;
        b = b < nb ? b : nb - 1;
        uint8_t *dst = ring + slot * STAGE;
#pragma unroll
        for (int n = 0; n < LA; n++)
            jl_load_to_lds<16>(p.A, dst + (n * WN + wn < 4 * MB ? n * WN + wn : 4 * MB - 1) * 1024, a_off[n], b * 512 + (s & 1) * 256);
        asm volatile("" ::: "memory");
    };

    // The raw bytes of a block, piece i (of 16 bytes) of a group from row i / PIECES.  Loaded a block
    // ahead into registers, written to the wave's own LDS once the block before has been read from it.
    uint32_t p_off[PL];
#pragma unroll
    for (int n = 0; n < PL; n++) {
        int i = n * 64 + lane;
        i = i < 16 * PIECES ? i : 16 * PIECES - 1;
        const int row = i / PIECES, off = i - row * PIECES;
        p_off[n] = (uint32_t)row * (uint32_t)p.row_bytes + (16 * off + 16 <= QUAD ? 16 * off : QUAD - 16);
    }
    const uint32_t raw0 = lds0 + KW * kStages * STAGE + wave * (NR * RAW);
    const uint32_t raw_put = raw0 + lane * 16;
    const uint32_t raw_put_last = raw0 + ((PL - 1) * 64 + lane < 16 * PIECES ? (PL - 1) * 64 + lane : 16 * PIECES - 1) * 16;
    const uint32_t raw_row = raw0 + r16 * RAW_ROW;
    constexpr int RL = NR * PL;      // vector memory operations of a block's raw bytes, at the least
    u32x4 raw[NR][PL];
    auto load_raw = [&](int it, int from, int to) {
        int b = it * KW + kw;
        b = b < nb ? b : nb - 1;
#pragma unroll
        for (int j = 0; j < NR; j++) {
            gbyte *base = (gbyte *)group_ptr[j] + (int64_t)b * QUAD;
#pragma unroll
            for (int n = 0; n < PL; n++) {
                if (j * PL + n < from || j * PL + n >= to) continue;
                const u32x4u v = *(gpiece *)(base + p_off[n]);
                raw[j][n] = u32x4{v.x, v.y, v.z, v.w};
            }
        }
        asm volatile("" ::: "memory");
    };
    auto store_raw = [&]() {
#pragma unroll
        for (int j = 0; j < NR; j++) {
#pragma unroll
            for (int n = 0; n + 1 < PL; n++)
                asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(raw_put), "v"(raw[j][n]), "n"(j * RAW + n * 1024) : "memory");
            asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(raw_put_last), "v"(raw[j][PL - 1]), "n"(j * RAW) : "memory");
        }
        asm volatile("s_nop 1" ::: "memory");
    };

    floatx4 total[MB][NR];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int j = 0; j < NR; j++) total[m][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // slice g of the 128 columns is chunks 4 (g % 2) .. of half g / 2; fragment i of row block m lies at
    // (a_base ^ (i << 4)) + m * 2048
    const uint32_t a_base = lds0 + kw * kStages * STAGE + (g >> 1) * (ROWS * 128) + r16 * 128 + ((row_key(r16) ^ ((g & 1) * 4)) << 4);

    HalfWords<TYPE> hw[NR];              // raw words of the next step
    half8 wf[2][NR][4];                  // fragments of this step and of the next
    uint32_t dd[2][NR][POST ? 4 : 1];    // POST: scales of weight rows 4 g .., those of the lane's results
    auto read_half = [&](int t, int set) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            hw[j].issue(raw_row + j * RAW, t, g);
            if (POST && t == 0) {
                const uint32_t at = raw0 + j * RAW + 4 * g * RAW_ROW;
                lds_issue_u16<222>(at, dd[set][j][0]);
                lds_issue_u16<222 + RAW_ROW>(at, dd[set][j][POST ? 1 : 0]);
                lds_issue_u16<222 + 2 * RAW_ROW>(at, dd[set][j][POST ? 2 : 0]);
                lds_issue_u16<222 + 3 * RAW_ROW>(at, dd[set][j][POST ? 3 : 0]);
            }
        }
    };
    auto settle_half = [&](int t, int set) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < NR; j++) {
            hw[j].settle();
            if (POST && t == 0) settled(dd[set][j]);
        }
    };

    __builtin_amdgcn_sched_barrier(0);
    load_raw(0, 0, RL);
    issue_stage(0, 0);
    store_raw();
    load_raw(1, 0, RL);
    read_half(0, 0);
    settle_half(0, 0);
#pragma unroll
    for (int j = 0; j < NR; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) wf[0][j][i] = decode_frag<TYPE>(hw[j], 0, g, i);
    read_half(1, 0);
    settle_half(1, 0);
    JL_WAIT_VM(0);

    // One step: half t of block `it`, whose parity is `set`.
    auto step = [&](int it, int t, int set) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        // This wave's part of the step's stage has landed.  Asked for after it, and left in flight: the
        // raw bytes, which go out in the second half behind its stage loads.
        if (t == 0) JL_WAIT_VM(RL);
        else JL_WAIT_VM(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t at = a_base + t * STAGE;
        half8 fa[2][4];
        auto read = [&](int m) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(fa[m & 1][i]) : "v"(at ^ (i << 4)), "n"(m * 2048) : "memory");
        };
        read(0);
        // (the slot held the step before, which every wave has read)
        issue_stage(2 * it + t + 1, t ^ 1);
        floatx4 acc[2][NR], d4[NR];
        if constexpr (POST) {
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) d4[j][e] = jl_half_bits_to_float(dd[set][j][e]);
        }
        auto post = [&](int m) {
#pragma unroll
            for (int j = 0; j < NR; j++)
                if constexpr (POST) total[m][j] += acc[m & 1][j] * d4[j];
        };
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const int k = m & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (t == 1) load_raw(it + 2, m * RL / MB, (m + 1) * RL / MB);
            if (m + 1 < MB) {
                read(m + 1);
                asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
            asm volatile("" : "+v"(fa[k][0]), "+v"(fa[k][1]), "+v"(fa[k][2]), "+v"(fa[k][3]));
            __builtin_amdgcn_sched_barrier(0);
            if (m > 0) post(m - 1);
            if constexpr (POST) {
#pragma unroll
                for (int j = 0; j < NR; j++) acc[k][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
            // a share of the next step's fragments, between the matrix instructions -- in the last group
            // before them, and behind the fragments the words of the step after
            auto decode_share = [&]() {
#pragma unroll
                for (int f = m * 8 / MB; f < (m + 1) * 8 / MB; f++) wf[t ^ 1][f >> 2][f & 3] = decode_frag<TYPE>(hw[f >> 2], t ^ 1, g, f & 3);
            };
            if (m == MB - 1) {
                decode_share();
                __builtin_amdgcn_sched_barrier(0);
                if (t == 0) store_raw();           // block it + 1
                read_half(t, set ^ 1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < NR; j++) {
                    if constexpr (POST) acc[k][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[t][j][i], fa[k][i], acc[k][j], 0, 0, 0);
                    else total[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[t][j][i], fa[k][i], total[m][j], 0, 0, 0);
                }
            if (m < MB - 1) {
                decode_share();
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, MB >= 7 ? (POST ? 4 : 2) : MB >= 4 ? (POST ? 6 : 4) : 8, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        settle_half(t, set ^ 1);
        post(MB - 1);
    };
    // (a wave whose set has a block less than others takes part in the barriers)
    auto block = [&](int it, int set) __attribute__((always_inline)) {
        if (KW == 1 || it * KW + kw < nb) {
            step(it, 0, set);
            step(it, 1, set);
        } else {
            JL_WAIT_VM(0);
            asm volatile("s_barrier\n\ts_barrier" ::: "memory");
        }
    };
    for (int it = 0; it < iters; it += 2) {
        block(it, 0);
        if (it + 1 < iters) block(it + 1, 1);
    }
    // (the loads past the end are not to be dropped: the waits above count them)
#pragma unroll
    for (int j = 0; j < NR; j++)
#pragma unroll
        for (int n = 0; n < PL; n++) asm volatile("" : : "v"(raw[j][n]));
    JL_WAIT_VM(0);   // nothing may land in LDS that is no longer this workgroup's

    // The weight fragment is the matrix instruction's row operand: a lane has output columns 4 g .. of the
    // group for activation row 16 m + r16.
    // What it reads, the row scales and (where everything lies on 16-byte boundaries) the values it adds to, is asked
    // for in front of the first store: where they are used each would be a round trip to memory.
    const bool quads = (p.ldo & 3) == 0 && ((uintptr_t)(p.C + p.col_offset) & 15) == 0 && ((out_col[0] | out_col[NR - 1]) & 3) == 0;
    const bool adds = quads && p.epilogue == JL_RESIDUAL;
    constexpr int MINE = (MB + KW - 1) / KW;   // row blocks a set of waves ends
    float scales[MINE];
    floatx4 old[MINE][NR];
#pragma unroll
    for (int i = 0; i < MINE; i++) {
        const int at = m0 + 16 * (i * KW + kw) + r16, row = at < p.rows ? at : p.rows - 1;
        scales[i] = p.row_scale ? p.row_scale[row] : 1.f;
        if (!adds) continue;
#pragma unroll
        for (int j = 0; j < NR; j++) old[i][j] = *(const floatx4 *)(p.C + (int64_t)row * p.ldo + p.col_offset + 4 * g + out_col[j]);
    }
    auto finish = [&](int m, const floatx4 (&t)[NR]) {
        const int row = m0 + 16 * m + r16;
        if (row >= p.rows) return;
        const float rs = scales[m / KW];
        if (rs < 0.f) return;   // (done apart, below)
        const int64_t at = (int64_t)row * p.ldo + p.col_offset + 4 * g;
        if (swiglu) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = jl_swiglu_single(t[0][e] * rs, t[1][e] * rs);
            const int64_t to = at + out_col[0];
            if (p.c_f16 && out_from[0] == 0) {
                jl_store4_f16((_Float16 *)p.C + to, v, 4);
            } else if (!p.c_f16 && out_from[0] == 0 && (((uintptr_t)(p.C + to)) & 15) == 0) {
                *(floatx4 *)(p.C + to) = floatx4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (4 * g + e < out_from[0]) continue;
                    if (p.c_f16) ((_Float16 *)p.C)[to + e] = (_Float16)v[e];
                    else p.C[to + e] = v[e];
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < NR; j++) {
            float *dst = p.C + at + out_col[j];
            floatx4 v = t[j] * rs;
            if (out_from[j] == 0 && quads) {
                if (adds) v += old[m / KW][j];
                *(floatx4 *)dst = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (4 * g + e < out_from[j]) continue;
                    if (p.epilogue == JL_RESIDUAL) dst[e] += v[e];
                    else dst[e] = v[e];
                }
            }
        }
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int m = 0; m < MB; m++) finish(m, total[m]);
    } else {
        // the sets' sums, added in the order of the sets; row block m by set m % KW
        __syncthreads();
        floatx4 *fold = (floatx4 *)lds;   // [kw][wn][m][j][lane]
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int j = 0; j < NR; j++) fold[((((kw * WN + wn) * MB + m) * NR) + j) * 64 + lane] = total[m][j];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MB; m++) {
            if (m % KW != kw) continue;
            floatx4 t[NR];
#pragma unroll
            for (int j = 0; j < NR; j++) t[j] = fold[(((wn * MB + m) * NR) + j) * 64 + lane];
#pragma unroll
            for (int z = 1; z < KW; z++)
#pragma unroll
                for (int j = 0; j < NR; j++) t[j] += fold[((((z * WN + wn) * MB + m) * NR) + j) * 64 + lane];
            finish(m, t);
        }
    }
    // Rows with a marked scale, which hardly any call has (a wave looks through its tile's scales: 0.1 us)
    if constexpr (TYPE == JL_Q8_0 || TYPE == JL_Q4_0) {
        if (!p.X || kw != 0) return;
        for (int first = 0; first < ROWS; first += 64) {
            const int mine = first + lane;
            uint64_t marked = __ballot(mine < ROWS && m0 + mine < p.rows && p.row_scale[m0 + mine] < 0.f);
            for (; marked; marked &= marked - 1) {
                const int row = m0 + first + __builtin_ctzll(marked);
                const float *x = p.X + (int64_t)row * p.k;
                float *dst = p.C + (int64_t)row * p.ldo + p.col_offset;
                for (int e = 0; e < kGroup; e++) {
                    float v[NR];
#pragma unroll
                    for (int j = 0; j < NR; j++) v[j] = e < out_from[j] ? 0.f : plain_dot<TYPE>(group_ptr[j] + (int64_t)e * p.row_bytes, x, p.k, lane);
                    if (lane != 0) continue;
                    if (swiglu) {
                        if (e >= out_from[0]) dst[out_col[0] + e] = jl_swiglu_single(v[0], v[1]);
                        continue;
                    }
#pragma unroll
                    for (int j = 0; j < NR; j++) {
                        if (e < out_from[j]) continue;
                        if (p.epilogue == JL_RESIDUAL) dst[out_col[j] + e] += v[j];
                        else dst[out_col[j] + e] = v[j];
                    }
                }
            }
        }
    }
}

template <int TYPE, int MB, int WN, int KW>
int launch_reg(jl_context *ctx, const RegParams &p) {
    auto fn = jl_gemm_reg<TYPE, MB, WN, KW>;
    constexpr int lds = lds_bytes<TYPE, MB, WN, KW>();
    if constexpr (lds <= 160 * 1024) {
        static jl_lds_limit_flags configured;
        const int st = jl_raise_lds_limit(configured, ctx->device, (const void *)fn, lds);
        if (st != JL_OK) return st;
        hipLaunchKernelGGL(fn, dim3((p.ntiles * p.mtiles + 7) / 8 * 8), dim3(64 * WN * KW), lds, ctx->stream, p);
        JL_HIP(hipGetLastError());
        return JL_OK;
    } else {
        return jl_fail(JL_ERR_INVALID, "jl_gemm: a tiling without room in LDS");
    }
}

// The tilings and what they cost, in microseconds a step (measured with every compute unit at work, and
// with half of the places of the chip filled, at 2 048 and 8 192 columns, weights from HBM) and beside the
// steps (launch, first stage, last stores).  Tilings of four waves have two workgroups to a compute unit,
// so that half of the places is one workgroup on each.  Five and six row blocks are there for the row counts
// just past 64, 128 and 256, where eight or seven leave a third of their rows empty or the chip two thirds
// full (Q8_0 gate/up 2 x [13824 x 5120] at 65 rows 111 -> 53 us, Q4_0 q | k | v 7168 x 5120 at 270 rows 65 ->
// 38); four row blocks with eight waves a set and two with four were never the cheapest.
struct Tiling {
    int mb, wn, kw, places;          // places: workgroups a compute unit holds
    float base;
    float full[4], half[4];          // Q8_0, Q4_0, Q4_K, Q6_K; 0: no such instance
};
constexpr Tiling kTilings[] = {
    {8, 8, 1, 1, 11.f, {2.48f, 2.05f, 2.11f, 0.f}, {1.90f, 1.53f, 1.45f, 0.f}},
    {7, 8, 1, 1, 9.f, {2.29f, 1.96f, 1.92f, 0.f}, {1.80f, 1.49f, 1.39f, 0.f}},
    {6, 8, 1, 1, 8.5f, {2.15f, 1.87f, 1.71f, 0.f}, {1.68f, 1.42f, 1.23f, 0.f}},
    {5, 8, 1, 1, 8.5f, {2.03f, 1.67f, 1.60f, 0.f}, {1.58f, 1.27f, 1.16f, 0.f}},
    {7, 4, 2, 1, 8.f, {0.f, 2.08f, 2.00f, 0.f}, {0.f, 1.69f, 1.66f, 0.f}},
    {6, 4, 2, 1, 8.f, {0.f, 1.98f, 1.90f, 0.f}, {0.f, 1.65f, 1.55f, 0.f}},
    {5, 4, 2, 1, 8.f, {2.27f, 1.86f, 1.80f, 0.f}, {1.93f, 1.55f, 1.50f, 0.f}},
    {4, 4, 2, 1, 7.f, {2.09f, 1.54f, 1.55f, 2.17f}, {1.88f, 1.34f, 1.28f, 2.14f}},
    {4, 4, 1, 2, 7.f, {1.95f, 1.60f, 1.50f, 2.13f}, {0.99f, 0.83f, 0.82f, 1.12f}},
    {4, 2, 2, 2, 6.f, {2.26f, 1.90f, 1.83f, 2.35f}, {1.14f, 0.90f, 0.86f, 1.24f}},
    {2, 2, 2, 2, 5.f, {1.61f, 1.20f, 0.f, 1.75f}, {0.99f, 0.70f, 0.f, 1.15f}},
};
constexpr int kTilingCount = sizeof(kTilings) / sizeof(kTilings[0]);
int type_column(int type) { return type == JL_Q8_0 ? 0 : type == JL_Q4_0 ? 1 : type == JL_Q4_K ? 2 : type == JL_Q6_K ? 3 : -1; }

template <int TYPE, int I>
int launch_tiling(jl_context *ctx, const RegParams &p, int tiling) {
    if constexpr (I < kTilingCount) {
        constexpr Tiling t = kTilings[I];
        constexpr int column = TYPE == JL_Q8_0 ? 0 : TYPE == JL_Q4_0 ? 1 : TYPE == JL_Q4_K ? 2 : 3;
        if constexpr (t.full[column] > 0.f) {
            if (tiling == I) return launch_reg<TYPE, t.mb, t.wn, t.kw>(ctx, p);
        }
        return launch_tiling<TYPE, I + 1>(ctx, p, tiling);
    } else {
        return jl_fail(JL_ERR_INVALID, "jl_gemm: no such tiling");
    }
}

// workgroup tiles of a call: row tiles x sets of WN wave tiles (32 columns each, or 16 of gate and of up)
int tiles_of(const Tiling &t, int rows, int groups, bool dual, int *ntiles, int *mtiles) {
    const int pairs = dual ? groups : (groups + NR - 1) / NR;
    *ntiles = (pairs + t.wn - 1) / t.wn;
    *mtiles = (rows + 16 * t.mb - 1) / (16 * t.mb);
    return *ntiles * *mtiles;
}

int groups_of(const jl_weight *const *weights, int count) {
    int groups = 0;
    for (int i = 0; i < count; i++) groups += ((int)weights[i]->rows + kGroup - 1) / kGroup;
    return groups;
}

}  // namespace

double jl_gemm_reg_price(const jl_context *ctx, const jl_weight *const *weights, int count, int rows, int epilogue,
                         int *tiling) {
    *tiling = -1;
    const int type = weights[0]->type, k = (int)weights[0]->cols, column = type_column(type);
    const bool dual = epilogue == JL_SWIGLU;
    // (32-bit offsets into the activations; sums of a row are cut by KW, which depends on the row count, so
    // a context that wants one order of addition whatever the row count goes another way)
    if (column < 0 || k % 256 != 0 || count > kMaxSeg || !ctx->split_k || (int64_t)rows * k >= (int64_t)1 << 30) return 1e30;
    for (int i = 0; i < count; i++)
        if (weights[i]->type != type || weights[i]->rows < kGroup || ((uintptr_t)weights[i]->blocks & 15)) return 1e30;
    const int groups = groups_of(weights, dual ? 1 : count);
    double best = 1e30;
    for (int i = 0; i < kTilingCount; i++) {
        const Tiling &t = kTilings[i];
        if (t.full[column] == 0.f) continue;
        int ntiles, mtiles;
        const int tiles = tiles_of(t, rows, groups, dual, &ntiles, &mtiles);
        const int places = ctx->compute_units * t.places;
        const int rounds = tiles / places, rest = tiles - rounds * places;
        // (measured with two row tiles to a set of weight rows; with four or more of them the raw bytes come
        // from the L2 mostly: gate/up of 2 x 8192 at 512 rows 2.08 us a step of the 8 x 8 tiling, not 2.48)
        const double full = mtiles >= 4 && t.places == 1 ? t.half[column] + 0.35 * (t.full[column] - t.half[column]) : t.full[column];
        double passes = rounds * full;
        if (rest > 0) {
            const double share = (double)rest / places;
            // (two workgroups of which only some share a compute unit take as long as if all did)
            passes += share <= 0.5 ? t.half[column]
                      : t.places == 2 ? full : t.half[column] + (share - 0.5) * 2.0 * (full - t.half[column]);
        }
        const int steps = 2 * ((k / 256 + t.kw - 1) / t.kw);
        const double us = t.base + passes * steps;
        if (us < best) {
            best = us;
            *tiling = i;
        }
    }
    // (fp32 activations: a launch that reads and converts them)
    return best + 2.5 + (double)rows * k * 6e-6 / 4.0;
}

int jl_launch_gemm_reg(jl_context *ctx, const jl_weight *const *weights, int count, const _Float16 *A,
                       const float *row_scale, const float *X, float *C, bool c_f16, int rows, int64_t ldo,
                       int64_t col_offset, int epilogue, int tiling) {
    const int type = weights[0]->type, k = (int)weights[0]->cols;
    const bool dual = epilogue == JL_SWIGLU;
    RegParams p{};
    p.nseg = dual ? 1 : count;
    int groups = 0, col = 0;
    for (int i = 0; i < p.nseg; i++) {
        p.w[i] = weights[i]->blocks;
        p.seg_rows[i] = (int)weights[i]->rows;
        p.seg_group_begin[i] = groups;
        p.seg_col_begin[i] = col;
        groups += ((int)weights[i]->rows + kGroup - 1) / kGroup;
        col += (int)weights[i]->rows;
    }
    p.seg_group_begin[p.nseg] = groups;
    p.w_up = dual ? weights[1]->blocks : nullptr;
    p.A = A;
    p.row_scale = row_scale;
    p.X = X;
    p.C = C;
    p.c_f16 = c_f16 ? 1 : 0;
    p.rows = rows;
    p.k = k;
    p.ldo = ldo;
    p.col_offset = col_offset;
    p.epilogue = epilogue;
    p.row_bytes = k / jl_block_elems(type) * jl_block_bytes(type);
    if (tiling < 0 || tiling >= kTilingCount) return jl_fail(JL_ERR_INVALID, "jl_gemm: no such tiling");
    tiles_of(kTilings[tiling], rows, groups, dual, &p.ntiles, &p.mtiles);
    switch (type) {
        case JL_Q8_0: return launch_tiling<JL_Q8_0, 0>(ctx, p, tiling);
        case JL_Q4_0: return launch_tiling<JL_Q4_0, 0>(ctx, p, tiling);
        case JL_Q4_K: return launch_tiling<JL_Q4_K, 0>(ctx, p, tiling);
        case JL_Q6_K: return launch_tiling<JL_Q6_K, 0>(ctx, p, tiling);
        default: return jl_fail(JL_ERR_UNSUPPORTED, "jl_gemm: no kernel for a ggml type %d weight", type);
    }
}
