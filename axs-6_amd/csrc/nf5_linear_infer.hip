// The quantized linear without gradients (gfx950), fake-quantize of the weight
// inside the contraction:
//   Y[M, N] = FQ(X)[M, K] . FQ(W)[N, K]^T + bias, block 32, K a multiple of 32.
//
// The training forward packs W to fp16 in a launch of its own and keeps it
// for the backward; without a backward that is a read, a write and a second
// read of the weight for one use.  Here a workgroup owns all rows of X (up
// to 256) and 128 rows of W, so a weight value is read from HBM and quantized
// once, and goes to LDS as the 16-bit MFMA operand:
//   * X is quantized first by a launch of its own (it is small);
//   * per 64-wide K step, X's slab comes by LDS-DMA (three slabs, two steps
//     ahead) and W's raw values into registers, two steps ahead.  In step s a
//     wave looks its share of step s + 1 up in the tables, runs the MFMAs of step
//     s over those reads' latency and writes the quantized values to the other
//     of two W slabs; one barrier per step.  Loads past the range go to an
//     empty buffer resource (zeros, no traffic), so every step issues the same
//     count and the waits are exact;
//   * few output tiles leave CUs idle: K is split over workgroups, which write
//     f32 partial tiles, as they lie in the registers, that a second launch
//     adds in order.
// What bounds it: at few rows the FQ of the weight (about 9 VALU operations and
// a table read a value) beside its stream; at 256 rows the step's parts, which
// the barrier keeps in phase: timing-only builds of 256 x 4096 x 11008 bf16 (61
// us for this kernel then) take 27 us with the weight's loads alone, 36 with
// X's too, 42 with the FQ as well, 49 with the MFMAs instead, and 18 with none
// of them.  Measured and not kept there: four steps of weight values in
// flight (the same), waves of two roles, X loads and MFMAs against W loads and
// FQ (80 against 72 us for the call), the FQ between the MFMAs by scheduling
// groups and K ranges started at different steps (each 1-4 us longer).
// Operands: 16-bit types contract their own FQ values (bf16 or f16 MFMA, exact
// operands).  f32 values take 11-bit fp16 magnitudes +-lut with the block's
// 2^e1 applied to the block's product in f32 -- one 16x16x32 MFMA is one block
// -- against X packed as in the training forward: the same operand rounding.
// The sums carry the blocks' own scales while those lie in [2^kRefLow,
// 2^kRefHigh], where no sum overflows or loses digits whatever X's scale.  A
// workgroup that meets a block outside runs its range a second time with each
// row's scales relative to its largest (the training forward packs every row so),
// and the epilogue puts that exponent back: the loop proper carries no state for
// it, the blocks outside already leave the short sequence.
#include "nf5_device.h"

#include "gemm_tile.h"

namespace axs6 {
namespace {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kIN = 128;                 // rows of W per workgroup
constexpr int kIK = 64;                  // K step: two NF5 blocks
constexpr int kIThreads = 512;
constexpr int kBfTab = 1 + 6 * 128;      // bf16 magnitudes in the block's six upper binades, and below
// f32: block scales are stored as 2^(e1 - 15) and X's rows are packed up to 2^15,
// so a partial sum is the product's own size, not 2^15 over it
constexpr int kScaleDown = 15;
// Block exponents whose products need no reference: a block's product is under
// 2^20 times its scale 2^(e1 - 15), so a sum of 2^25 blocks under 2^(90 + 5 + 25),
// and at 2^(-80 - 15) an X value 2^30 under its row's largest still leaves a
// normal product.  The magnitudes that have them:
constexpr int kRefLow = -80, kRefHigh = 90;
constexpr uint32_t kRefLowBits = (uint32_t)(kExpBias + kRefLow - 1) << 23;
constexpr uint32_t kRefHighBits = (uint32_t)(kExpBias + kRefHigh) << 23;
constexpr int kOob = 0x7ffffff0;         // a buffer offset past every operand (they stay under 2 GiB)

struct InferK {
    const void* x; int ldx;              // FQ(X) as MFMA operand: fp16 (f32 input) or the 16-bit type
    const void* w; const int32_t* sx;    // sx: X's row shifts (f32 input)
    const void* bias; int bias_dtype; void* out; float* partial;
    int* again; int* refs;               // f32, K split: a second pass was run [split][tile], its exponents [..][kIN]
    int M, N, K, dtype;
    int steps;                           // K steps per workgroup
    int tiles_n, splits;
    const float* lut; const uint8_t* band;
};

struct InferTables {
    float lut[kLutSize];
    uint32_t band[kBandSize / 4];
    uint16_t mag[kLutSize];              // f32, f16: the LUT in fp16; bf16: kBfTab magnitudes
};

// The bf16 table.  A bf16 block's e1 is its largest exponent field E - 126 (no
// bf16 value lies in the log2 band under a power of two), and n = |x| 2^-e1 has
// the bits of |x| with the exponent field moved, so the level is a function of
// bits(|x|) - ((E - 5) << 7): entry 1 + j holds n = 2^-6 (1 + ..) up from j = 0,
// entry 0 everything below 2^-6, whose indices (< 16) all give the lowest level.
__device__ __forceinline__ void build_bf16_table(uint16_t* mag, const float* lut_s, int tid) {
    for (int j = tid; j < kBfTab; j += kIThreads) {
        const float n = j ? __uint_as_float((uint32_t)((121 << 7) + j - 1) << 16) : 0.0f;
        mag[j] = f32_to_bf16_rne(lut_s[(int)(n * 1023.0f)]);
    }
}

__device__ __forceinline__ uint32_t pk(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ u16x2 unpk(uint32_t v) { return __builtin_bit_cast(u16x2, v); }

// FQ of 8 consecutive values of a row (a block is a DPP quad of lanes) to the
// MFMA operand's 16 bytes, in two halves: `look` finds the block's exponent and
// issues the table reads, `finish` puts the values together -- so that a step's
// MFMAs run over the reads' latency.  look is free of branches; a wave with a
// block the short sequence does not cover (NaN, inf, tiny, within 255 ulps
// under a power of two, or outside what the 16-bit type's exponent addition
// covers) says so, and finish redoes it from the raw values.
template <int DT>
struct FqLook {
    uint32_t v[8];       // table values
    int e1;
    bool special;        // wave-uniform
    bool zeros;          // wave-uniform (f32): some value is +-0
};

template <int DT>
__device__ __forceinline__ void look(const u32x4* raw, const InferTables& t, FqLook<DT>& q) {
    if constexpr (DT == AXS6_BF16) {
        const uint32_t w[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w};
        u16x2 a[4];                                   // 2 |bits|: the sign shifted out, two bytes per step
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = unpk(w[i]) << 1;
        const u16x2 mx = __builtin_elementwise_max(__builtin_elementwise_max(a[0], a[1]),
                                                   __builtin_elementwise_max(a[2], a[3]));
        const uint32_t m = group_umax<4>(mx.x > mx.y ? mx.x : mx.y);
        const uint32_t E = m >> 8;
        q.special = __builtin_amdgcn_ballot_w64(m != 0 && (E < 27 || E >= 254)) != 0;
        q.e1 = (int)E - 126;
        // E >= 27 or a special wave; clamped for the read of a special one
        const uint32_t base = E >= 27 ? ((E - 5) << 8) - 2 : 0xffffu;
        const u16x2 b2 = {(uint16_t)base, (uint16_t)base};
        const char* tab = reinterpret_cast<const char*>(t.mag);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t j = pk(__builtin_elementwise_sub_sat(a[i], b2));
            q.v[2 * i] = *reinterpret_cast<const uint16_t*>(tab + (j & 0xffffu));
            q.v[2 * i + 1] = *reinterpret_cast<const uint16_t*>(tab + (j >> 16));
        }
    } else if constexpr (DT == AXS6_F16) {
        const uint32_t w[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w};
        u16x2 a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = unpk(w[i] & 0x7fff7fffu);
        const u16x2 mx = __builtin_elementwise_max(__builtin_elementwise_max(a[0], a[1]),
                                                   __builtin_elementwise_max(a[2], a[3]));
        const uint32_t m = group_umax<4>(mx.x > mx.y ? mx.x : mx.y);
        const int e1 = (int)(m >> 10) - 14;
        const bool sp = m != 0 && (e1 < -6 || e1 > 15);
        q.special = __builtin_amdgcn_ballot_w64(sp) != 0;
        q.e1 = m ? e1 : 0;
        const float c = sp ? 0.0f : __builtin_amdgcn_ldexpf(1023.0f, -q.e1);   // 0: index 0, in the table
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
            const f16x2 f = __builtin_bit_cast(f16x2, a[i]);
            q.v[2 * i] = t.mag[(uint32_t)((float)f.x * c)];
            q.v[2 * i + 1] = t.mag[(uint32_t)((float)f.y * c)];
        }
    } else {
        float f[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f[4 * h] = __uint_as_float(raw[h].x); f[4 * h + 1] = __uint_as_float(raw[h].y);
            f[4 * h + 2] = __uint_as_float(raw[h].z); f[4 * h + 3] = __uint_as_float(raw[h].w);
        }
        float amx = __builtin_elementwise_maximum(__builtin_fabsf(f[0]), __builtin_fabsf(f[1]));
        float amn = __builtin_elementwise_minimum(__builtin_fabsf(f[0]), __builtin_fabsf(f[1]));
#pragma unroll
        for (int e = 2; e < 8; ++e) {
            amx = __builtin_elementwise_maximum(amx, __builtin_fabsf(f[e]));
            amn = __builtin_elementwise_minimum(amn, __builtin_fabsf(f[e]));
        }
        const uint32_t m = group_umax<4>(__float_as_uint(amx));
        const int e1 = (int)(m >> 23) - 126;
        // the log2 bands are under 256 values wide
        const bool band = (m & 0x7fffffu) > 0x7fff00u;
        const bool sp = m != 0u && (m < kRefLowBits || m >= kRefHighBits || band);
        q.special = __builtin_amdgcn_ballot_w64(sp) != 0;
        q.zeros = __builtin_amdgcn_ballot_w64(__float_as_uint(amn) == 0u) != 0;
        q.e1 = m ? e1 : 0;
        // a special block reads index 0 (its values past the type times 0 are NaN, which converts to 0)
        const float c = sp ? 0.0f : __builtin_amdgcn_ldexpf(1023.0f, -q.e1);
#pragma unroll
        for (int e = 0; e < 8; ++e) q.v[e] = t.mag[(uint32_t)(__builtin_fabsf(f[e]) * c)];
    }
}

template <int DT>
__device__ __forceinline__ u32x4 finish(const u32x4* raw, const FqLook<DT>& q, float* scale) {
    uint32_t r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = q.v[2 * i] | (q.v[2 * i + 1] << 16);
    if constexpr (DT == AXS6_F32) {
        const uint32_t w[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[1].x, raw[1].y, raw[1].z, raw[1].w};
        *scale = __builtin_amdgcn_ldexpf(1.0f, q.e1 - kScaleDown);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // FQ(+-0) = 0 (its sign is of no consequence to a sum); the two values' signs
            if (q.zeros) r[i] &= ((w[2 * i] << 1) ? 0xffffu : 0u) | ((w[2 * i + 1] << 1) ? 0xffff0000u : 0u);
            r[i] |= __builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], 0x07060302u) & 0x80008000u;
        }
    } else {
        const uint32_t w[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w};
        // 2^e1: an addition to the (normal) table value's exponent field
        const uint32_t ex = (uint32_t)q.e1 << (DT == AXS6_BF16 ? 7 : 10);
        const u16x2 e2 = {(uint16_t)ex, (uint16_t)ex}, one = {1, 1};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // +0 where the value is +-0: 2 |bits| is at least 2 elsewhere
            const u16x2 nz = (u16x2)(0) - __builtin_elementwise_min(unpk(w[i]) << 1, one);
            r[i] = (pk(unpk(r[i]) + e2) | (w[i] & 0x80008000u)) & pk(nz);
        }
    }
    u32x4 out;
    out.x = r[0]; out.y = r[1]; out.z = r[2]; out.w = r[3];
    return out;
}

// The same 8 values by the general sequence (a wave whose look was special).
// f32: the scale is taken down by `down`, and *outside set where the block's
// exponent lies outside [kRefLow, kRefHigh].
template <int DT>
__device__ __forceinline__ u32x4 fq_general(const u32x4* raw, const InferTables& t, int down, float* scale,
                                            int* outside) {
    const uint8_t* band_s = reinterpret_cast<const uint8_t*>(t.band);
    float f[8];
    if constexpr (DT == AXS6_F32) {
        Elem<DT>::unpack(raw[0], f);
        Elem<DT>::unpack(raw[1], f + 4);
    } else {
        Elem<DT>::unpack(raw[0], f);
    }
    uint32_t m = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t ab = __float_as_uint(f[e]) & 0x7fffffffu;
        m = m > ab ? m : ab;
    }
    const FqScale s = fq_scale_general(group_umax<4>(m), band_s);
    if constexpr (DT != AXS6_F32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = fq_value(f[e], s, t.lut, false, 0.0f);
        return Elem<DT>::pack(f);
    } else {
        // the FQ value (a tiny block's is rounded to f32's subnormals) over 2^e1;
        // NaN and infinite scales give the operand's NaN and inf themselves
        uint32_t r[4];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = fq_value(f[e], s, t.lut, false, 0.0f);
            const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)__builtin_amdgcn_ldexpf(v, -s.e1));
            r[e >> 1] = e & 1 ? r[e >> 1] | (h << 16) : h;
        }
        const bool nonfinite = s.nan_block || s.inf_scale;
        *scale = nonfinite ? 1.0f : __builtin_amdgcn_ldexpf(1.0f, s.e1 - down);
        if (!nonfinite && !s.zero && (s.e1 < kRefLow || s.e1 > kRefHigh)) *outside = 1;
        u32x4 out;
        out.x = r[0]; out.y = r[1]; out.z = r[2]; out.w = r[3];
        return out;
    }
}

template <int DT>
__device__ __forceinline__ f32x4m mfma_elem(u32x4 a, u32x4 b, f32x4m c) {
    if constexpr (DT == AXS6_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
}

constexpr int kXSlabs = 3;
// Waves per SIMD that an instance's registers are kept to; a workgroup is two.
constexpr int infer_waves(int dtype, int bm) { return bm >= 128 || (dtype == AXS6_F32 && bm == 64) ? 2 : 4; }

constexpr size_t infer_lds(int BM) {
    return (size_t)kXSlabs * BM * kIK * 2 + 2 * kIN * kIK * 2 + 2 * 2 * kIN * sizeof(float);
}

// lgkmcnt(0) alone, then a bare barrier: __syncthreads() would also drain the
// loads in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
}

// The exponent that a weight row's scales are taken relative to, from the bits
// of its largest magnitude: 0 inside the window, else its largest block's (at
// most 127: a block that scales to inf or NaN is its row's result whatever the
// others sum to).
__device__ __forceinline__ int row_ref(uint32_t m) {
    if (m == 0u || (m >= kRefLowBits && m < kRefHighBits)) return 0;
    return m >= 0x7f000000u ? 127 : m >= 0x00800000u ? (int)(m >> 23) - 126 : 31 - __clz((int)m) - 148;
}

// Four consecutive outputs of a row, from column col: 2^sh v + bias.
__device__ __forceinline__ void finish_store(const InferK& k, int row, int col, const int (&sh)[4],
                                             const float (&v)[4]) {
    if (col >= k.N) return;
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        o[r] = __builtin_amdgcn_ldexpf(v[r], sh[r]) +
               (k.bias && col + r < k.N ? load_elem(k.bias, k.bias_dtype, col + r) : 0.0f);
    const int es = k.dtype == AXS6_F32 ? 4 : 2;
    store4(k.out, k.N, k.N, k.dtype, row, col, o, k.N % 4 == 0 && (uintptr_t)k.out % (4 * es) == 0);
}

// A wave's blocks of the output tile: TM x TN 16x16 blocks, W's
// rows as the MFMA's A operand, so a lane holds four consecutive output
// columns (rows 4 fq .. of a block) of output row fr.
template <int DT, int TM, int TN>
struct InferTile {
    f32x4m acc[TN][TM];
    int m, n;            // first row and column inside the workgroup's tile
    __device__ void clear() {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[j][i] = f32x4m{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // block b (0, 1) of a step
    __device__ __forceinline__ void multiply(const char* xb, const char* wb, const float* sc_b, int b, int fr, int fq) {
        u32x4 xf[TM], wf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
            xf[i] = *reinterpret_cast<const u32x4*>(xb + swz<kIK>(m + i * 16 + fr, b * 4 + fq));
#pragma unroll
        for (int j = 0; j < TN; ++j)
            wf[j] = *reinterpret_cast<const u32x4*>(wb + swz<kIK>(n + j * 16 + fr, b * 4 + fq));
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (DT == AXS6_F32) {
                const f32x4m sc = *reinterpret_cast<const f32x4m*>(sc_b + b * kIN + n + j * 16 + 4 * fq);
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const f32x4m p = mfma_elem<DT>(wf[j], xf[i], f32x4m{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[j][i][r] = __builtin_fmaf(p[r], sc[r], acc[j][i][r]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[j][i] = mfma_elem<DT>(wf[j], xf[i], acc[j][i]);
            }
        }
    }
    // The tile's values, finished to the output or (K split) as they lie in the
    // registers: one contiguous KiB per store.  Partial tiles written by rows (64
    // bytes of 16 rows per store) made this 8 us of 256 x 4096 x 11008.
    // ref: the rows' exponents after a second pass, else null.
    __device__ __forceinline__ void store(const InferK& k, int n0, float* part, const int* ref, int fr, int fq) const {
        constexpr bool SCALED = DT == AXS6_F32;
        if (k.splits > 1) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) *reinterpret_cast<f32x4m*>(part + (j * TM + i) * 256) = acc[j][i];
            return;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = m + i * 16 + fr;
            if (row >= k.M) continue;
            const int sx = SCALED ? kScaleDown + k.sx[row] : 0;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float v[4] = {acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]};
                int sh[4] = {sx, sx, sx, sx};
                if (SCALED && ref) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) sh[r] += ref[n + j * 16 + 4 * fq + r];
                }
                finish_store(k, row, n0 + n + j * 16 + 4 * fq, sh, v);
            }
        }
    }
};

// Adds the K splits' partial tiles in order (InferTile::store's layout) and
// finishes them.  A workgroup takes 16 rows x 64 columns of a tile, a wave four
// of the rows, so that its stores cover whole rows of 64.
template <bool SCALED, int BM, int MW, int NW>
__global__ __launch_bounds__(256) void infer_reduce_kernel(InferK k) {
    constexpr int TM = BM / (16 * MW), TN = kIN / (16 * NW), PARTS = BM / 16 * 2;
    const int part = (int)blockIdx.x % PARTS, tile = (int)blockIdx.x / PARTS;
    const int ib = part >> 1, jb = (part & 1) * 4 + (threadIdx.x >> 2 & 3);
    const int r = threadIdx.x >> 4, cq = threadIdx.x & 3;
    const int row = ib * 16 + r;
    const int col = tile * kIN + jb * 16 + 4 * cq;
    if (row >= k.M || col >= k.N) return;
    const int wave = ib / TM * NW + jb / TN;
    const float* p = k.partial + (int64_t)tile * (BM * kIN) +
                     ((wave * TN + jb % TN) * TM + ib % TM) * 256 + (cq * 16 + r) * 4;
    const int64_t stride = (int64_t)k.tiles_n * (BM * kIN);
    const int sx = SCALED ? k.sx[row] + kScaleDown : 0;
    int sh[4] = {sx, sx, sx, sx};
    int again = 0;
    f32x4m v = *reinterpret_cast<const f32x4m*>(p);
    if constexpr (SCALED) again = k.again[tile];
#pragma unroll 4
    for (int z = 1; z < k.splits; ++z) {
        v += *reinterpret_cast<const f32x4m*>(p + z * stride);
        if constexpr (SCALED) again |= k.again[z * k.tiles_n + tile];
    }
    if (SCALED && again != 0) {
        // parts with exponents of their own: summed relative to the largest of
        // those of parts that are not 0
        int ref[4], top[4] = {INT_MIN, INT_MIN, INT_MIN, INT_MIN};
        v = f32x4m{0.0f, 0.0f, 0.0f, 0.0f};
        for (int pass = 0; pass < 2; ++pass) {
            for (int z = 0; z < k.splits; ++z) {
                const f32x4m pz = *reinterpret_cast<const f32x4m*>(p + z * stride);
                const bool own = k.again[z * k.tiles_n + tile] != 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    ref[r] = own ? k.refs[(z * k.tiles_n + tile) * kIN + jb * 16 + 4 * cq + r] : 0;
                    if (pz[r] == 0.0f) continue;
                    if (pass == 0) top[r] = ref[r] > top[r] ? ref[r] : top[r];
                    else v[r] += __builtin_amdgcn_ldexpf(pz[r], ref[r] - top[r]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) sh[r] += top[r] == INT_MIN ? 0 : top[r];
    }
    const float f[4] = {v[0], v[1], v[2], v[3]};
    finish_store(k, row, col, sh, f);
}

// MW x NW waves over the BM x 128 tile.
template <int DT, int BM, int MW, int NW>
__global__ __launch_bounds__(kIThreads, infer_waves(DT, BM)) void infer_gemm_kernel(InferK k) {
#if defined(__HIP_DEVICE_COMPILE__)
    static_assert(MW * NW == 8, "eight waves");
    constexpr int TM = BM / (16 * MW), TN = kIN / (16 * NW);
    constexpr bool SCALED = DT == AXS6_F32;
    constexpr int ES = DT == AXS6_F32 ? 4 : 2;
    constexpr int RV = ES * 8 / 16;                  // 16-byte vectors per 8 weight values
    constexpr int XSLAB = BM * kIK * 2, WSLAB = kIN * kIK * 2;
    constexpr int XINST = BM / 8;                    // 1 KiB DMA instructions per X slab
    constexpr int XI = XINST >= 8 ? XINST / 8 : 1;   // per (issuing) wave
    constexpr int WI = 2 * RV;
    constexpr int D = 2;                             // K steps of raw weight values in flight
    extern __shared__ __align__(16) char smem[];
    __shared__ InferTables tab;
    __shared__ int ref_s[SCALED ? kIN : 1], again_s;   // f32: the second pass' row exponents; that one is needed
    char* const xs = smem;
    char* const wsl = smem + kXSlabs * XSLAB;
    float* const scl = reinterpret_cast<float*>(wsl + 2 * WSLAB);   // [slab][block][row]

    const int split = (int)blockIdx.x % k.splits, tile = (int)blockIdx.x / k.splits, n0 = tile * kIN;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    const int all = (k.K + kIK - 1) / kIK;           // K steps of the whole contraction
    const int s0 = split * k.steps;
    const int T = all - s0 < k.steps ? all - s0 : k.steps;
    // the last step's second block when K ends after its first
    const int tail = k.K % kIK ? all - 1 : INT_MAX;
    // the tables' loads go first; they are awaited before the loads behind them
    float4 lutv = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t bandv = 0;
    if (tid < kLutSize / 4) lutv = reinterpret_cast<const float4*>(k.lut)[tid];
    if (tid < kBandSize / 4) bandv = reinterpret_cast<const uint32_t*>(k.band)[tid];

    // X: slab row group 8 (wave + 8 i); a lane fetches the chunk whose swizzled
    // slot it fills.  W: chunk tid % 8 of rows tid / 8 and tid / 8 + 64.
    const int xbytes = (int)((int64_t)k.M * k.ldx * 2), wbytes = (int)((int64_t)k.N * k.K * ES);
    int xoff[XI], woff[2];
    bool xhi[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int row = (wave + 8 * i) * 8 + lane / 8;
        const int chunk = (lane % 8) ^ swz_key<kIK>(row);
        xoff[i] = row < k.M ? row * k.ldx * 2 + chunk * 16 : kOob;
        xhi[i] = chunk >= 4;
    }
    const int wrow = tid >> 3, wchunk = tid & 7;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int row = n0 + wrow + 64 * c;
        woff[c] = row < k.N ? (int)(((int64_t)row * k.K + wchunk * 8) * ES) : kOob;
    }
    auto issue_x = [&](int s) {
        if (XINST < 8 && wave >= XINST) return;
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc((void*)k.x, 0, s < T ? xbytes : 0, kBufferConfig);
        const int ks = s0 + s, so = s < T ? ks * kIK * 2 : 0;
        char* slab = xs + (s % kXSlabs) * XSLAB;
#pragma unroll
        for (int i = 0; i < XI; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                r, (__attribute__((address_space(3))) void*)(slab + (wave + 8 * i) * 1024), 16,
                !SCALED && ks == tail && xhi[i] ? kOob : xoff[i], so, 0, 0);
    };
    auto issue_w = [&](int s, u32x4 (&o)[2][RV]) {
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc((void*)k.w, 0, s < T ? wbytes : 0, kBufferConfig);
        const int ks = s0 + s, so = s < T ? ks * kIK * ES : 0;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int off = ks == tail && wchunk >= 4 ? kOob : woff[c];
#pragma unroll
            for (int v = 0; v < RV; ++v)
                o[c][v] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * v, so, 0));
        }
    };
    FqLook<DT> q[2];
    u32x4 val[2];
    float scale[2];
    auto look_w = [&](const u32x4 (&o)[2][RV]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) look<DT>(o[c], tab, q[c]);
    };
    auto finish_w = [&](const u32x4 (&o)[2][RV]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) val[c] = finish<DT>(o[c], q[c], &scale[c]);
    };
    auto store_w = [&](int s, const u32x4 (&o)[2][RV]) {
        char* slab = wsl + (s & 1) * WSLAB;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int row = wrow + 64 * c;
            if (q[c].special) val[c] = fq_general<DT>(o[c], tab, kScaleDown, &scale[c], &again_s);
            *reinterpret_cast<u32x4*>(slab + swz<kIK>(row, wchunk)) = val[c];
            if constexpr (SCALED) {
                if ((wchunk & 3) == 0) scl[((s & 1) * 2 + (wchunk >> 2)) * kIN + row] = scale[c];
            }
        }
    };
    u32x4 raw[D][2][RV];
#pragma unroll
    for (int s = 0; s < kXSlabs - 1; ++s) issue_x(s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D; ++d) issue_w(d, raw[d]);
    InferTile<DT, TM, TN> t;
    t.m = wave / NW * TM * 16;
    t.n = wave % NW * TN * 16;
    t.clear();
    if (tid < kLutSize / 4) {
        reinterpret_cast<float4*>(tab.lut)[tid] = lutv;
        if constexpr (DT != AXS6_BF16) {
            const float f[4] = {lutv.x, lutv.y, lutv.z, lutv.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) tab.mag[4 * tid + e] = __builtin_bit_cast(uint16_t, (_Float16)f[e]);
        }
    }
    if (tid < kBandSize / 4) tab.band[tid] = bandv;
    if (SCALED && tid == 0) again_s = 0;
    lds_barrier();
    if constexpr (DT == AXS6_BF16) {
        build_bf16_table(tab.mag, tab.lut, tid);
        lds_barrier();
    }
    look_w(raw[0]);
    finish_w(raw[0]);
    store_w(0, raw[0]);
    // D steps per iteration, so that the ring's slots are compile-time.  No
    // load sits under a branch: the compiler's waits would see two histories
    // and wait for the whole ring.
    for (int s = 0;; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (s + d >= T) goto summed;
            // slab s + d has landed once only the W issues after it, and the
            // slab between them, are outstanding
            wait_vmcnt<XI + 2 * WI>();
            lds_barrier();
            issue_x(s + d + kXSlabs - 1);
            __builtin_amdgcn_sched_barrier(0);
            issue_w(s + d + D, raw[d]);
            const char* xb = xs + ((s + d) % kXSlabs) * XSLAB;
            const char* wb = wsl + (d & 1) * WSLAB;
            const float* sb = scl + (d & 1) * 2 * kIN;
            look_w(raw[(d + 1) % D]);
            t.multiply(xb, wb, sb, 0, fr, fq);
            finish_w(raw[(d + 1) % D]);
            t.multiply(xb, wb, sb, 1, fr, fq);
            store_w(s + d + 1, raw[(d + 1) % D]);
        }
    }
summed:
    // the thread's place again: kept across the loop it costs the f32 32-row
    // instance, at its register limit, a spill
    const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), et = wave * 64 + el;
    const int efr = el & 15, efq = el >> 4;
    bool again = false;
    if constexpr (SCALED) {
        lds_barrier();
        again = __builtin_amdgcn_readfirstlane(again_s) != 0;
        if (again) {
            // the largest magnitude of each row's range (a row is 8 lanes' chunks)
            uint32_t top[2] = {0u, 0u};
            for (int s = 0; s < T; ++s) {
                issue_w(s, raw[0]);
#pragma unroll
                for (int i = 0; i < 8 * RV; ++i) {
                    const uint32_t ab = raw[0][i / (4 * RV)][i / 4 % RV][i % 4] & 0x7fffffffu;
                    uint32_t& m = top[i / (4 * RV)];
                    m = m > ab ? m : ab;
                }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int ref = row_ref(group_umax<8>(top[c]));
                if (et % 8 == 0) ref_s[et / 8 + 64 * c] = ref;
            }
            t.clear();
            for (int s = 0; s < T; ++s) {
                // nothing in flight into the slabs, nobody still reading them
                wait_vmcnt<0>();
                lds_barrier();
                issue_x(s);
                issue_w(s, raw[0]);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int row = et / 8 + 64 * c, chunk = et % 8;
                    const u32x4 v = fq_general<DT>(raw[0][c], tab, kScaleDown + ref_s[row], &scale[c], &again_s);
                    *reinterpret_cast<u32x4*>(wsl + swz<kIK>(row, chunk)) = v;
                    if (chunk % 4 == 0) scl[chunk / 4 * kIN + row] = scale[c];
                }
                wait_vmcnt<0>();
                lds_barrier();
                t.multiply(xs + (s % kXSlabs) * XSLAB, wsl, scl, 0, efr, efq);
                t.multiply(xs + (s % kXSlabs) * XSLAB, wsl, scl, 1, efr, efq);
            }
        }
        if (k.splits > 1) {
            const int part = split * k.tiles_n + tile;
            if (et == 0) k.again[part] = again ? 1 : 0;
            if (again && et < kIN) k.refs[part * kIN + et] = ref_s[et];
        }
    }
    t.store(k, n0,
            k.partial + (int64_t)(split * k.tiles_n + tile) * (BM * kIN) + wave * (TM * TN * 256) + el * 4,
            again ? ref_s : nullptr, efr, efq);
#endif
}

template <int DT, int BM, int MW, int NW>
int run_infer(const InferK& k, hipStream_t st) {
    const size_t lds = infer_lds(BM);
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void*)infer_gemm_kernel<DT, BM, MW, NW>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        attr_set = true;
    }
    infer_gemm_kernel<DT, BM, MW, NW><<<(unsigned)(k.tiles_n * k.splits), kIThreads, lds, st>>>(k);
    if (k.splits > 1) infer_reduce_kernel<DT == AXS6_F32, BM, MW, NW><<<(unsigned)(k.tiles_n * (BM / 8)), 256, 0, st>>>(k);
    return check_launch("infer_gemm");
}

template <int DT>
int run_infer_dt(const InferK& k, int bm, hipStream_t st) {
    switch (bm) {
        case 32: return run_infer<DT, 32, 1, 8>(k, st);
        case 64: return run_infer<DT, 64, 2, 4>(k, st);
        case 128: return run_infer<DT, 128, 2, 4>(k, st);
        default:
            if constexpr (DT != AXS6_F32) return run_infer<DT, 256, 4, 2>(k, st);
            return fail(AXS6_ERR_UNSUPPORTED, "infer_gemm: row tile");   // infer_plan gives f32 at most 128
    }
}

// Row tile, K split and workspace of a shape.
struct InferPlan { int bm, steps, splits; size_t xq, sx, again, refs, partial, total; };

// Where this form is the faster one.  The packed path's cost is the weight's
// (a read, a write and a read back), this one's grows with the rows: the FQ of
// a weight value costs its wave as much as 8 (f32: more) MFMA columns, and past
// 256 rows (f32: 128) it is repeated.  Measured, three or more weights in turn,
// us, packed path / this one:
//            M x K x N          bf16          f32
//     16 x 4096 x 11008   67.8 / 35.9    71.3 / 48.9
//     64 x 4096 x 4096    42.4 / 22.5    46.8 / 29.8
//    128 x 4096 x 4096    43.5 / 27.8    47.6 / 33.5
//    256 x 4096 x 4096    43.0 / 34.8    48.0 / 50.8
//    256 x 4096 x 11008   75.5 / 61.3    84.0 / 124.7
//    256 x 11008 x 4096  104.8 / 55.3   111.7 / 103.7
//    512 x 4096 x 4096    44.8 / 47.4    49.4 / 82.2
//     64 x 2048 x 2048         -         26.6 / 22.3
//    128 x 2048 x 2048         -         26.2 / 27.8
//    128 x 1024 x 1024    17.3 / 17.4    17.7 / 19.5
//     16 x 512 x 11008         -         16.6 / 19.2
// One and two rows come here where FQ(X) is past the streamed form's LDS (one
// row of 12288 values, two of 6144): 2 x 11008 x 4096 bf16 100.8 / 39.9, 1 x 14336 x
// 4096 f32 140.2 / 67.4.
// A K off 32 and blocks of 8 and 16 stay with the packed path: 64 x 4096 x 4096
// f32 29.7 here, 46.6 there in blocks of 16 and 55.7 at K 4100.
// part_n: the rows of one of the weights that make up W, whose plan it takes (N:
// W is one weight).
bool infer_plan(int64_t M, int64_t N, int64_t K, int64_t part_n, int dtype, InferPlan* p) {
    const bool f32 = dtype == AXS6_F32;
    const int64_t most = part_n * K >= (int64_t)1 << 23 ? (f32 ? 128 : 256) : (f32 ? 64 : 128);
    if (M < 1 || M > most || K < 1024 || part_n * K < (int64_t)1 << 22) return false;
    // 32-bit buffer offsets
    if (N * K * (f32 ? 4 : 2) >= (int64_t)kOob || M * (K + kGemmK) * 2 >= (int64_t)kOob) return false;
    p->bm = M <= 32 ? 32 : M <= 64 ? 64 : M <= 128 ? 128 : 256;
    const int64_t tiles = (N + kIN - 1) / kIN, part_tiles = (part_n + kIN - 1) / kIN;
    const int64_t steps = (K + kIK - 1) / kIK;
    // K splits: rounds of workgroups times the steps of each, the fill of its
    // pipeline (about 4 steps) and the partial sums' traffic (about 1 step per split).
    // The slots are the workgroups that fit the CUs: counted as 512 where one
    // fits a CU (f32 of 64 rows), twice the splits ran in two rounds: 64 x 11008 x
    // 4096 71 us against 53, 48 x 4096 x 6144 44 against 34.5.
    const int64_t slots = 256 * infer_waves(dtype, p->bm) / 2;
    int64_t s = 1, best = INT64_MAX;
    for (int64_t c = 1; c <= 16 && c <= steps / 4 + 1; ++c) {
        const int64_t cost = ((part_tiles * c + slots - 1) / slots) * (((steps + c - 1) / c) + 4) + (c > 1 ? 2 + c : 0);
        if (cost < best) { best = cost; s = c; }
    }
    p->steps = (int)((steps + s - 1) / s);
    p->splits = (int)((steps + p->steps - 1) / p->steps);
    size_t off = 0;
    auto take = [&](size_t b) { const size_t o = off; off = (off + b + 255) / 256 * 256; return o; };
    const int64_t Kp = pad_to(K, kGemmK);
    p->xq = take((size_t)M * (dtype == AXS6_F32 ? Kp : K) * 2);
    p->sx = take((size_t)M * sizeof(int32_t));
    const size_t parts = f32 && p->splits > 1 ? (size_t)p->splits * tiles : 0;
    p->again = parts ? take(parts * sizeof(int)) : 0;
    p->refs = parts ? take(parts * kIN * sizeof(int)) : 0;
    p->partial = p->splits > 1 ? take((size_t)p->splits * tiles * p->bm * kIN * sizeof(float)) : 0;
    p->total = off;
    return true;
}

}  // namespace
}  // namespace axs6

using namespace axs6;

extern "C" int64_t axs6_nf5_linear_infer_stacked_workspace(int64_t M, int64_t N, int64_t K, int64_t part_n,
                                                           int32_t dtype, int32_t block_size) {
    if (!valid_dtype(dtype) || block_size != 32 || M <= 0 || N <= 0 || K <= 0 || K % 32 != 0 || M > (1 << 30) ||
        N > (1 << 30) || K > (1 << 30) || part_n <= 0 || part_n > N)
        return -1;
    // the streamed form's waves per row follow the weight's size
    if (infer_rows_fit(M, N, K)) return part_n == N ? 0 : -1;
    InferPlan p;
    return infer_plan(M, N, K, part_n, dtype, &p) ? (int64_t)p.total : -1;
}

extern "C" int64_t axs6_nf5_linear_infer_workspace(int64_t M, int64_t N, int64_t K, int32_t dtype,
                                                   int32_t block_size) {
    return axs6_nf5_linear_infer_stacked_workspace(M, N, K, N, dtype, block_size);
}

extern "C" int axs6_nf5_linear_infer(const void* x, const void* w, const void* bias, int32_t bias_dtype, void* y,
                                     int32_t dtype, int64_t M, int64_t N, int64_t K, int32_t block_size,
                                     int32_t quantize_input, void* workspace, int64_t workspace_bytes, void* stream) {
    return axs6_nf5_linear_infer_stacked(x, w, bias, bias_dtype, y, dtype, M, N, K, N, block_size, quantize_input,
                                         workspace, workspace_bytes, stream);
}

extern "C" int axs6_nf5_linear_infer_stacked(const void* x, const void* w, const void* bias, int32_t bias_dtype,
                                             void* y, int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t part_n,
                                             int32_t block_size, int32_t quantize_input, void* workspace,
                                             int64_t workspace_bytes, void* stream) {
    const char* fn = "axs6_nf5_linear_infer";
    if (!valid_dtype(dtype) || (bias && !valid_dtype(bias_dtype)))
        return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: unknown dtype code %d", fn, valid_dtype(dtype) ? bias_dtype : dtype);
    if (block_size != 32)
        return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: block_size must be 32 (got %d)", fn, block_size);
    if (M < 0 || N < 0 || K < 0) return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: negative dimension", fn);
    if (M == 0 || N == 0) return AXS6_OK;
    const int64_t need = axs6_nf5_linear_infer_stacked_workspace(M, N, K, part_n, dtype, block_size);
    if (need < 0) return fail(AXS6_ERR_UNSUPPORTED, "%s: no inference form for this shape (use the forward)", fn);
    if (!x || !w || !y) return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: null pointer", fn);
    if ((uintptr_t)x % 16 || (uintptr_t)w % 16)
        return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: x and w must be 16-byte aligned", fn);
    if (need && (!workspace || workspace_bytes < need || (uintptr_t)workspace % 16))
        return fail(AXS6_ERR_INVALID_ARGUMENT, "%s: workspace of %lld bytes (16-byte aligned) required", fn,
                    (long long)need);
    DeviceTables t;
    int rc = device_tables(&t);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const bool qx = quantize_input != 0;
    if (infer_rows_fit(M, N, K)) return launch_infer_rows(x, w, bias, bias_dtype, y, dtype, M, N, K, qx, t, st);

    InferPlan p;
    infer_plan(M, N, K, part_n, dtype, &p);
    char* ws = (char*)workspace;
    InferK k{};
    k.w = w; k.bias = bias; k.bias_dtype = bias_dtype; k.out = y; k.dtype = dtype;
    k.M = (int)M; k.N = (int)N; k.K = (int)K;
    k.steps = p.steps; k.splits = p.splits;
    k.tiles_n = (int)((N + kIN - 1) / kIN);
    k.partial = (float*)(ws + p.partial);
    k.lut = t.lut; k.band = t.band;
    k.x = ws + p.xq;
    if (dtype == AXS6_F32) {
        const int64_t Kp = pad_to(K, kGemmK);
        k.ldx = (int)Kp;
        k.sx = (const int32_t*)(ws + p.sx);
        if (p.splits > 1) {
            k.again = (int*)(ws + p.again);
            k.refs = (int*)(ws + p.refs);
        }
        const PackRowsArgs px{x, dtype, M, K, 32, qx, false, 0, 0, nullptr, nullptr, (_Float16*)(ws + p.xq), Kp, Kp,
                              (int32_t*)(ws + p.sx), nullptr, nullptr, nullptr};
        rc = launch_pack_rows(px, t, st);
    } else {
        k.ldx = (int)K;
        if (qx) rc = axs6_nf5_fake_quantize(x, ws + p.xq, dtype, M, K, 32, 0, 0, 0, nullptr, stream);
        else k.x = x;
    }
    if (rc) return rc;
    return dtype == AXS6_F32 ? run_infer_dt<AXS6_F32>(k, p.bm, st)
           : dtype == AXS6_BF16 ? run_infer_dt<AXS6_BF16>(k, p.bm, st) : run_infer_dt<AXS6_F16>(k, p.bm, st);
}
