// Prefill GEMM over the tile-packed GGUF bank copy for gfx950: Y[m, n] (fp32) =
// sum_k X[m, k] W[n, k] for the kadan encodings Q4_K, Q8_0 and Q6_K.
//
// The reference runs prefill chunks by decoding a packed tile to fp32 and calling
// cublasSgemm (IW/src/cuda/h3_compute.cu:2201-2218,2451, project<float> :1780-2530; IW =
// services/hikari/inference_worker), so its product is the fp32 product of exactly
// decoded weights (kadan::gguf::decode, IW/include/kadan/gguf_quantization.hpp:631-762).
// Here the weights stay packed in HBM and are dequantised in registers to fp16 MFMA
// operands; the activations are fp16 after an exact power-of-two scale per token (so
// no value overflows fp16 and none goes subnormal); products accumulate in fp32 on
// v_mfma_f32_32x32x16_f16 and the scale is undone in the epilogue.  Roundings: the
// activation once to fp16; the weight once (Q8_0: fp16(d * q); Q4_K: fp16(q * fp16(d *
// sc) - fp16(dmin * m)); Q6_K: fp16((q - 32) * fp16(d * sc))).
//
// Kernels:
//   stage_kernel<ENC>  one workgroup per token row: the row's power-of-two scale, and the
//                      row as fp16 in the order the weight lanes consume each 256-value
//                      group (the permutation depends on the format's packed lane image)
//   stream_gemm_kernel<ENC, PAIR>  short chunks and grouped (MoE) layers: 64-token tiles,
//                      the weights of two groups in flight
//   gemm_kernel<ENC, W, TB>  128 tokens (TB = 4; TB = 3: 96) x 256 weight rows per
//                      workgroup, W = 4 wavefronts each owning two 32-row weight operands
//                      (W = 8: one) and all the tokens; weights go from HBM straight
//                      into operand registers (16-byte loads of the packed lane images,
//                      issued one group ahead) and are dequantised there; activations
//                      are staged into swizzled LDS by buffer->LDS DMA; the fp32 output
//                      tile leaves through LDS as whole rows.
#include "kdq_common.hpp"

#include <algorithm>

namespace kdq {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int PM = 128;                      // tokens per workgroup tile (4 blocks of 32)
constexpr int NB = 2;                        // 32-row weight operands per wavefront
constexpr int kTiles = 8 * NB;               // 16-row packed tiles per workgroup
constexpr int kStageRow = 512;               // LDS bytes per token of one staged group
constexpr int kDmaRows = 1024 / kStageRow;   // token rows per 64-lane 16-byte DMA
constexpr int kOutPitch = kTiles * 16 * 4 + 16;  // fp32 output row in LDS (+16: banks)
constexpr int kStreamTM = int(kGroupedTileRows);  // tokens per tile of the streaming kernel
// LDS of a workgroup of TB 32-token blocks: two activation stages, reused for the output
template <int TB> constexpr size_t kLds =
    32 * TB * std::max(size_t(kOutPitch), 2 * size_t(kStageRow));

typedef __attribute__((address_space(3))) void lds_void;

// ------------------------------------------------------------------ formats
//
// Lane (r, h) of a 32-row weight operand (MFMA lane r + 32h: weight row r, K values
// 8h..8h+7 of each 16-value sub-step) reads, for group chunk G = 2j + h (j = 0, 1), the
// packed lane position l = 16G + r % 16 of tile r / 16.  Sub-step s = 8j + 4p + u (p,
// u as each format names them) gives the lane 8 values of chunk G; value(s, h, e) is the
// group index (0..255) of operand element e, which the staging kernel uses to place the
// activations.  Packed units (kdq_gguf_pack): Q4_K 2304 B = code pieces 0, 1 (bytes
// 16p..16p+15 of sub-block pair G), 16-byte row headers at 2048 + 16 (r % 16); Q8_0 4352
// B = pieces 2c + hh (bytes 16hh..16hh+15 of block 2G + c), scale dwords at 4096 + 4l
// (d of blocks 2G, 2G+1); Q6_K 3360 B = ql pieces 0, 1 (bytes 32G + 16p..), the qh bit
// pairs in piece 2 (dword m: position 8m + i in the high nibble of byte i, 8m + 4 + i in
// its low nibble, block-0 bits | block-1 bits << 2), scale dwords at 3072 + 4l (the
// chunk's four int8 scales), row d at 3328 + 4 (slot / 2).
template <int ENC> struct GemmFormat;

template <> struct GemmFormat<KDQ_Q4_K> {
    static constexpr int unit = 2304, loads = 5;  // per operand and group
    struct Regs {
        u32x4 code[2][2];
        u32x4 head;
    };
    // operand element e of sub-step s: low nibbles of code bytes 16p + 4u + {0, 2, 1, 3}
    // (block 2G), then the high nibbles of the same bytes (block 2G + 1)
    __host__ __device__ static unsigned value(unsigned s, unsigned h, unsigned e) {
        const unsigned G = 2 * (s / 8) + h, p = (s / 4) % 2, u = s % 4;
        const unsigned ord[4] = {0, 2, 1, 3};
        return 64 * G + (e >= 4 ? 32 : 0) + 16 * p + 4 * u + ord[e % 4];
    }
};

template <> struct GemmFormat<KDQ_Q8_0> {
    static constexpr int unit = 4352, loads = 10;
    struct Regs {
        u32x4 code[2][4];
        unsigned scale[2];
    };
    // s = 8j + 4c + 2hh + v: bytes 16hh + 8v .. +7 of block 2G + c, in order
    __host__ __device__ static unsigned value(unsigned s, unsigned h, unsigned e) {
        const unsigned G = 2 * (s / 8) + h, c = (s / 4) % 2, hh = (s / 2) % 2, v = s % 2;
        return 64 * G + 32 * c + 16 * hh + 8 * v + e;
    }
};

template <> struct GemmFormat<KDQ_Q6_K> {
    static constexpr int unit = 3360, loads = 9;
    struct Regs {
        u32x4 code[2][2];
        u32x4 qh[2];
        unsigned scale[2];
        unsigned d;
    };
    // s = 8j + 4p + u: ql bytes 16p + 4u + {0..3} of chunk G; their low nibbles are
    // super-block positions 128(G/2) + 32(G%2) + t (t = 16p + 4u + i), the high nibbles
    // the same + 64
    __host__ __device__ static unsigned value(unsigned s, unsigned h, unsigned e) {
        const unsigned G = 2 * (s / 8) + h, p = (s / 4) % 2, u = s % 4;
        return 128 * (G / 2) + 32 * (G % 2) + (e >= 4 ? 64 : 0) + 16 * p + 4 * u + e % 4;
    }
};

__device__ __forceinline__ f16x2 pair(float v) {
    const _Float16 h = _Float16(v);
    return f16x2{h, h};
}

__device__ __forceinline__ f16x2 as_f16x2(unsigned v) {
    return __builtin_bit_cast(f16x2, v);
}

// fp16 value as fp32 (exact), of the low or high half of a dword
__device__ __forceinline__ float half_lo(unsigned v) {
    return float(__builtin_bit_cast(_Float16, uint16_t(v & 0xffffu)));
}
__device__ __forceinline__ float half_hi(unsigned v) {
    return float(__builtin_bit_cast(_Float16, uint16_t(v >> 16)));
}

// Per-group operand scales of one lane (computed once per group from its registers).
template <int ENC> struct Scales;

// Q4_K: for the lane's blocks 4j + 2h + b (b = 0, 1): fp16(d * sc) and fp16(-dmin * m)
template <> struct Scales<KDQ_Q4_K> {
    f16x2 dsc[2][2], ndm[2][2];
    __device__ __forceinline__ void prepare(const GemmFormat<KDQ_Q4_K>::Regs& g, unsigned h,
                                            unsigned& flags) {
        const float d = half_lo(g.head.x), dmin = half_hi(g.head.x);
        const unsigned s[3] = {g.head.y, g.head.z, g.head.w};  // scale bytes 0..11
        auto byte = [&](unsigned i) { return (s[i / 4] >> (8 * (i % 4))) & 255u; };
        if (!isfinite(d) || !isfinite(dmin))
            flags |= 1u;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const unsigned k = 4 * j + 2 * h + b;  // block of the super-block
                unsigned sc, m;
                if (k < 4) {
                    sc = byte(k) & 63u;
                    m = byte(k + 4) & 63u;
                } else {
                    sc = (byte(k + 4) & 15u) | ((byte(k - 4) >> 6) << 4);
                    m = (byte(k + 4) >> 4) | ((byte(k) >> 6) << 4);
                }
                const float a = d * float(sc), c = dmin * float(m);
                if (15.f * fabsf(a) + fabsf(c) > 65504.f)
                    flags |= 2u;  // a weight past the fp16 range
                dsc[j][b] = pair(a);
                ndm[j][b] = pair(-c);
            }
    }
};

// Q8_0: d of blocks 2G + c
template <> struct Scales<KDQ_Q8_0> {
    f16x2 d[2][2];
    __device__ __forceinline__ void prepare(const GemmFormat<KDQ_Q8_0>::Regs& g, unsigned,
                                            unsigned& flags) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const unsigned sc = g.scale[j];
            const float d0 = half_lo(sc), d1 = half_hi(sc);
            if (!isfinite(d0) || !isfinite(d1))
                flags |= 1u;
            if (128.f * fmaxf(fabsf(d0), fabsf(d1)) > 65504.f)
                flags |= 2u;
            d[j][0] = as_f16x2(__builtin_amdgcn_perm(sc, sc, 0x01000100u));
            d[j][1] = as_f16x2(__builtin_amdgcn_perm(sc, sc, 0x03020302u));
        }
    }
};

// Q6_K: fp16(d * sc) of the four 16-value scales the lane's chunk uses, per j
template <> struct Scales<KDQ_Q6_K> {
    f16x2 dsc[2][4];
    __device__ __forceinline__ void prepare(const GemmFormat<KDQ_Q6_K>::Regs& g, unsigned r,
                                            unsigned& flags) {
        const float d = (r % 2) ? half_hi(g.d) : half_lo(g.d);
        if (!isfinite(d))
            flags |= 1u;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = d * float(int8_t((g.scale[j] >> (8 * i)) & 255u));
                if (32.f * fabsf(a) > 65504.f)
                    flags |= 2u;
                dsc[j][i] = pair(a);
            }
    }
};

// The 8 fp16 weights of sub-step s (operand element order of GemmFormat::value).
template <int ENC>
__device__ __forceinline__ f16x8 dequant(const typename GemmFormat<ENC>::Regs& g,
                                         const Scales<ENC>& sc, int s, unsigned magic);

template <>
__device__ __forceinline__ f16x8 dequant<KDQ_Q4_K>(const GemmFormat<KDQ_Q4_K>::Regs& g,
                                                   const Scales<KDQ_Q4_K>& sc, int s,
                                                   unsigned magic) {
    const int j = s / 8, p = (s / 4) % 2, u = s % 4;
    const unsigned w = g.code[j][p][u], w8 = w >> 8;
    const f16x2 k1024 = as_f16x2(0x64006400u);      // 1024
    const f16x2 sixteenth = as_f16x2(0x2c002c00u);  // 1/16
    const f16x2 m64 = as_f16x2(0xd400d400u);        // -64
    // 1024 + q (low nibbles) or 1024 + 16 q (high), then exactly q
    const f16x2 q0 = as_f16x2((w & 0x000f000fu) | magic) - k1024;
    const f16x2 q1 = as_f16x2((w8 & 0x000f000fu) | magic) - k1024;
    const f16x2 q2 = __builtin_elementwise_fma(as_f16x2((w & 0x00f000f0u) | magic), sixteenth, m64);
    const f16x2 q3 = __builtin_elementwise_fma(as_f16x2((w8 & 0x00f000f0u) | magic), sixteenth, m64);
    const f16x2 r0 = __builtin_elementwise_fma(q0, sc.dsc[j][0], sc.ndm[j][0]);
    const f16x2 r1 = __builtin_elementwise_fma(q1, sc.dsc[j][0], sc.ndm[j][0]);
    const f16x2 r2 = __builtin_elementwise_fma(q2, sc.dsc[j][1], sc.ndm[j][1]);
    const f16x2 r3 = __builtin_elementwise_fma(q3, sc.dsc[j][1], sc.ndm[j][1]);
    return f16x8{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
}

template <>
__device__ __forceinline__ f16x8 dequant<KDQ_Q8_0>(const GemmFormat<KDQ_Q8_0>::Regs& g,
                                                   const Scales<KDQ_Q8_0>& sc, int s, unsigned) {
    const int j = s / 8, c = (s / 4) % 2, hh = (s / 2) % 2, v = s % 2;
    const u32x4 piece = g.code[j][2 * c + hh];
    const unsigned w0 = v ? piece.z : piece.x, w1 = v ? piece.w : piece.y;
    const f16x2 bias = as_f16x2(0x64806480u);  // 1152
    // (b ^ 0x80) in the mantissa of 1024: 1152 + q exactly, then q
    auto two = [&](unsigned w, unsigned sel) {
        return as_f16x2(__builtin_amdgcn_perm(0u, w, sel) ^ 0x64806480u) - bias;
    };
    const f16x2 d = sc.d[j][c];
    const f16x2 r0 = two(w0, 0x0c010c00u) * d, r1 = two(w0, 0x0c030c02u) * d;
    const f16x2 r2 = two(w1, 0x0c010c00u) * d, r3 = two(w1, 0x0c030c02u) * d;
    return f16x8{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
}

template <>
__device__ __forceinline__ f16x8 dequant<KDQ_Q6_K>(const GemmFormat<KDQ_Q6_K>::Regs& g,
                                                   const Scales<KDQ_Q6_K>& sc, int s,
                                                   unsigned magic) {
    const int j = s / 8, p = (s / 4) % 2, u = s % 4;
    const unsigned ql = g.code[j][p][u];
    const u32x4 qh = g.qh[j];
    const unsigned m = 2 * p + u / 2;
    const unsigned qd = m == 0 ? qh.x : m == 1 ? qh.y : m == 2 ? qh.z : qh.w;
    const unsigned qn = (u % 2 ? qd : qd >> 4) & 0x0f0f0f0fu;
    const unsigned lo = (ql & 0x0f0f0f0fu) | ((qn & 0x03030303u) << 4);  // block-0 codes
    const unsigned hi = ((ql >> 4) & 0x0f0f0f0fu) | ((qn & 0x0c0c0c0cu) << 2);
    const f16x2 k1056 = as_f16x2(0x64206420u);  // 1024 + 32
    auto two = [&](unsigned w, unsigned sel) {
        return as_f16x2(__builtin_amdgcn_perm(0u, w, sel) | magic) - k1056;  // q - 32
    };
    const f16x2 a = sc.dsc[j][p], b = sc.dsc[j][2 + p];
    const f16x2 r0 = two(lo, 0x0c010c00u) * a, r1 = two(lo, 0x0c030c02u) * a;
    const f16x2 r2 = two(hi, 0x0c010c00u) * b, r3 = two(hi, 0x0c030c02u) * b;
    return f16x8{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
}

// Weight load i (0 .. loads - 1) of one operand's group into its registers, from p + the
// item's place in the unit: `p` is the operand's lane address in the group (the tile's
// unit, plus lane_code(r, h) bytes).
__device__ __forceinline__ unsigned lane_code(unsigned r, unsigned h) {
    return 16 * (16 * h + r % 16);
}
template <int ENC>
__device__ __forceinline__ void load_item(const uint8_t* p, unsigned h, unsigned r,
                                          typename GemmFormat<ENC>::Regs& g, int i) {
    const unsigned lane_bytes = lane_code(r, h);  // already in `p`
    if constexpr (ENC == KDQ_Q4_K) {
        if (i < 4)
            g.code[i / 2][i % 2] = load16(p + 1024 * (i % 2) + 512 * (i / 2));
        else
            g.head = load16(p + 2048 + 16 * (r % 16) - lane_bytes);
    } else if constexpr (ENC == KDQ_Q8_0) {
        if (i < 8)
            g.code[i / 4][i % 4] = load16(p + 1024 * (i % 4) + 512 * (i / 4));
        else
            g.scale[i - 8] = load4(p + 4096 + 128 * (i - 8) + 4 * (16 * h + r % 16) - lane_bytes);
    } else {
        if (i < 4)
            g.code[i / 2][i % 2] = load16(p + 1024 * (i % 2) + 512 * (i / 2));
        else if (i < 6)
            g.qh[i - 4] = load16(p + 2048 + 512 * (i - 4));
        else if (i < 8)
            g.scale[i - 6] = load4(p + 3072 + 128 * (i - 6) + 4 * (16 * h + r % 16) - lane_bytes);
        else
            g.d = load4(p + 3328 + 4 * ((r % 16) / 2) - lane_bytes);
    }
}

// The sub-step after which load i's registers hold nothing that the group still needs (the
// dequantisation of sub-step s runs one sub-step before it; scales are read out first).
template <int ENC> constexpr int free_at(int i) {
    if (ENC == KDQ_Q4_K)
        return i < 4 ? 4 * i + 3 : 0;
    if (ENC == KDQ_Q8_0)
        return i < 8 ? 2 * i + 1 : 0;
    return i < 4 ? 4 * i + 3 : i < 6 ? 8 * (i - 4) + 7 : 0;
}

// The GEMM's scale checks over a whole packed matrix, without the product: 32 threads
// per (16-row tile, 256-value group), lane (r = s, h) of the GEMM's operand lanes for row
// slot s, each loading that lane's registers as the GEMM does and running the same
// Scales::prepare, so a matrix this finds clean never raises a flag in the GEMM.
template <int ENC>
__global__ __launch_bounds__(256) void check_kernel(const uint8_t* __restrict__ w,
                                                    unsigned groups, size_t units,
                                                    unsigned* __restrict__ flags) {
    using F = GemmFormat<ENC>;
    const size_t id = size_t(blockIdx.x) * 256 + threadIdx.x;
    const size_t unit = id / 32;
    if (unit >= units)
        return;
    const unsigned s = threadIdx.x % 16, h = (threadIdx.x / 16) % 2;
    const uint8_t* base = w + unit * F::unit + 16 * (16 * h + s);
    typename F::Regs g;
#pragma unroll
    for (int i = 0; i < F::loads; ++i)
        load_item<ENC>(base, h, s, g, i);
    unsigned f = 0;
    Scales<ENC> sc;
    sc.prepare(g, ENC == KDQ_Q6_K ? s : h, f);
    if (f)
        atomicOr(flags, f);
    (void)groups;
}

// ------------------------------------------------------------------ staging

// Row t of x (fp32, k values): its scale sigma = 2^e with max|x| / sigma in [2^14, 2^15)
// (1 for an all-zero row), and fp16(x / sigma) permuted per 256-value group: logical
// 16-byte chunk q = 16j + 8h + 4p + u of a group holds operand elements 0..7 of sub-step
// s = 8j + 4p + u for lane half h.  One workgroup per row; the row passes
// through LDS.  With `slot_of` (rows are positions of a grouped layer), rows from *used on
// and rows with slot_of[t] < 0 are not staged.
template <int ENC, int THREADS>
__global__ __launch_bounds__(THREADS) void stage_kernel(const float* __restrict__ x, unsigned k,
                                                    uint16_t* __restrict__ xs,
                                                    float* __restrict__ sigma,
                                                    const int32_t* __restrict__ slot_of,
                                                    const unsigned* __restrict__ used) {
    extern __shared__ __align__(16) float row[];
    __shared__ float wave_max[THREADS / 64];
    const unsigned t = blockIdx.x;
    if (slot_of && (t >= *used || slot_of[t] < 0))
        return;
    const float* src = x + size_t(t) * k;
    float amax = 0.f;
    for (unsigned i = threadIdx.x; i < k / 4; i += THREADS) {
        const float4 v = reinterpret_cast<const float4*>(src)[i];
        reinterpret_cast<float4*>(row)[i] = v;
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        if (!(isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w)))
            amax = INFINITY;
    }
    amax = wave_max_nonneg(amax);
    if (threadIdx.x % 64 == 0)
        wave_max[threadIdx.x / 64] = amax;
    __syncthreads();
    amax = wave_max[0];
#pragma unroll
    for (int v = 1; v < THREADS / 64; ++v)
        amax = fmaxf(amax, wave_max[v]);
    // exponent of amax (normal or subnormal), scale 2^(e - 14)
    int e = 0;
    float scale = 1.f, inv = 1.f;
    if (isfinite(amax) && amax >= 0x1p-100f) {  // (smaller rows: their fp16 values are 0)
        (void)frexpf(amax, &e);  // amax in [2^(e-1), 2^e)
        scale = ldexpf(1.f, e - 15);
        inv = ldexpf(1.f, 15 - e);
    } else if (!isfinite(amax)) {
        scale = __builtin_nanf("");  // a non-finite input poisons its row
    }
    if (threadIdx.x == 0)
        sigma[t] = scale;
    uint16_t* dst = xs + size_t(t) * k;
    for (unsigned c = threadIdx.x; c < k / 8; c += THREADS) {
        const unsigned g = c / 32, q = c % 32;
        const unsigned h = (q / 8) % 2, s = 8 * (q / 16) + 4 * ((q / 4) % 2) + q % 4;
        unsigned words[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = row[256 * g + GemmFormat<ENC>::value(s, h, 2 * i)] * inv;
            const float b = row[256 * g + GemmFormat<ENC>::value(s, h, 2 * i + 1)] * inv;
            words[i] = unsigned(__builtin_bit_cast(uint16_t, _Float16(a))) |
                       unsigned(__builtin_bit_cast(uint16_t, _Float16(b))) << 16;
        }
        *reinterpret_cast<uint4*>(dst + 8 * size_t(c)) =
            make_uint4(words[0], words[1], words[2], words[3]);
    }
}

// ------------------------------------------------------------------- GEMM

// The staged rows from `xs` on, for the DMAs into LDS.  These go out as buffer loads: the
// compiler takes a global load to LDS for a flat access, whose return order it does not
// trust, and would wait for every load and LDS read in flight wherever it needs one.
__device__ __forceinline__ auto activation_resource(const uint16_t* xs) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(xs), 0, int(0xffffffffu),
                                             0x00027000);
}

// Workgroup tile: 32 TB tokens (96 or 128, launch_gemm) x 256 weight rows (16 packed
// tiles); wavefront w owns tiles 4w .. 4w + 3 as two 32-row operands.  K runs over
// 256-value groups; each group's tokens x 512 bytes of permuted activations are staged into
// LDS by 16-byte DMA (double-buffered, one group ahead), chunk q of token t at t*512 + 16*(q ^ (t % 16)),
// and the next group's weight registers load during the current group's sub-steps.
// `xs` has rows up to the next multiple of 128 tokens (rows past m are computed, never
// stored).  *status |= 1 for a non-finite weight scale, |= 2 when a dequantised weight
// could pass the fp16 range (the caller then takes another path).
//
// K slices (narrow products, too few tiles for the compute units): workgroup slice `ks`
// runs groups [ks * per, (ks + 1) * per) and writes its fp32 tile to part[ks] (m x n);
// reduce_kernel then sums the slices in order.
//
template <int ENC, int W, int TB>
__global__ __launch_bounds__(W * 64, 1) void gemm_kernel(
    const uint16_t* __restrict__ xs, const float* __restrict__ sigma,
    const uint8_t* __restrict__ w, unsigned m, unsigned n, unsigned k, unsigned slices,
    unsigned per, float* __restrict__ y, float* __restrict__ part,
    unsigned* __restrict__ status) {
    using F = GemmFormat<ENC>;
    using Regs = typename F::Regs;
    extern __shared__ __align__(16) uint8_t lds[];
    // W wavefronts of NBW 32-row operands each (8 operands, 256 rows, per workgroup), TB
    // token blocks of 32
    constexpr int TM = 32 * TB, NBW = 8 / W;
    constexpr int DMAS = TM / kDmaRows / W;  // DMA instructions per wavefront per group
    constexpr int SB = TM * kStageRow;       // bytes of one activation stage
    constexpr int TILES = kTiles;            // 16-row output tiles per workgroup

    const unsigned groups = k / 256, wtiles = (n + 15) / 16;
    const unsigned m_tiles = (m + TM - 1) / TM, n_tiles = (wtiles + TILES - 1) / TILES;
    // XCD-aware order: the M tiles of one weight tile (and K slice) run together on one
    // XCD (L2).
    const unsigned id = blockIdx.x, xcd = id % 8, local = id / 8;
    const unsigned per_xcd = (m_tiles * n_tiles * slices + 7) / 8;
    const unsigned linear = xcd * per_xcd + local;
    if (local >= per_xcd || linear >= m_tiles * n_tiles * slices)
        return;
    const unsigned n_tile = linear / (m_tiles * slices);
    const unsigned slice = (linear / m_tiles) % slices, m0 = (linear % m_tiles) * TM;
    // slices = ceil(groups / per), so every slice has at least one group
    const unsigned g_begin = slice * per, g_end = min(groups, g_begin + per);
    float* __restrict__ dst_base = slices > 1 ? part + size_t(slice) * m * n : y;

    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const unsigned lane = threadIdx.x % 64;
    const unsigned r = lane % 32, h = lane / 32;
    const size_t row_pitch = size_t(k) * 2;

    // operand c = tiles tile0 + 2c (rows 0-15) and tile0 + 2c + 1 (rows 16-31); tiles
    // past the end load the last tile, and their results are never stored
    const unsigned tile0 = n_tile * TILES + wave * 2 * NBW;
    const uint8_t* base[NBW];
#pragma unroll
    for (int c = 0; c < NBW; ++c)
        base[c] = w + size_t(min(tile0 + 2 * c + r / 16, wtiles - 1)) * groups * F::unit +
                  lane_code(r, h);
    auto load_weight = [&](unsigned g, Regs* rg, int i) {
        load_item<ENC>(base[i / F::loads] + size_t(g) * F::unit, h, r, rg[i / F::loads],
                       i % F::loads);
    };

    // DMA: instruction J = W j + wave covers tokens 2J, 2J + 1 of the tile; lane L fills LDS
    // chunk L % 32 of token 2J + L / 32 from logical chunk (L % 32) ^ (token % 16).  The
    // wavefronts take turns, so that a wavefront's tokens repeat every 8 / W of its
    // instructions, 16 tokens on, and so does the swizzle.
    constexpr int kTurn = 8 / W;
    unsigned xlane[kTurn];
#pragma unroll
    for (int jm = 0; jm < kTurn; ++jm) {
        const unsigned tok = kDmaRows * (W * jm + wave) + lane / 32;
        xlane[jm] = unsigned(tok * row_pitch) + 16 * ((lane % 32) ^ tok);
    }
    const auto x_rsrc = activation_resource(xs + size_t(m0) * k);
    auto stage_one = [&](unsigned g, unsigned buf, int j) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            x_rsrc, (lds_void*)(lds + buf * SB + (W * j + wave) * 1024), 16,
            int(xlane[j % kTurn]),
            int(g * 512 + unsigned(j / kTurn) * (16 * unsigned(row_pitch))), 0, 0);
    };
    constexpr int kLoads = DMAS + F::loads * NBW, kPerStep = 4;
    static_assert(kLoads <= 16 * kPerStep, "the loads must fit the group's sub-steps");
    auto issue = [&](int s, unsigned g, unsigned buf, Regs* rg) {
#pragma unroll
        for (int i = kPerStep * s; i < kPerStep * (s + 1) && i < kLoads; ++i) {
            if (i < DMAS)
                stage_one(g, buf, i);
            else
                load_weight(g, rg, i - DMAS);
        }
    };
    auto issue_all = [&](unsigned g, unsigned buf, Regs* rg) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            if (i < DMAS)
                stage_one(g, buf, i);
            else
                load_weight(g, rg, i - DMAS);
        }
    };

    f32x16 acc[NBW][TB];
#pragma unroll
    for (int c = 0; c < NBW; ++c)
#pragma unroll
        for (int b = 0; b < TB; ++b)
            acc[c][b] = f32x16{};

    unsigned flags = 0;
    unsigned magic = 0x64006400u;  // kept in a VGPR: the mask-and-or takes one SGPR only
    asm volatile("" : "+v"(magic));
    // 16 sub-steps per group, software-pipelined by one sub-step: while the TB * NBW MFMAs
    // of sub-step s run, the activation operands of s + 1 are read from LDS and its
    // weights dequantised; one MFMA, then up to four VALU ops / one LDS read / one load.
    auto compute = [&](unsigned buf, const Regs* rg, unsigned next_g, unsigned next_buf,
                       Regs* next_rg) {
        const uint8_t* a = lds + buf * SB + r * kStageRow;
        auto read_x = [&](int s, f16x8* xf) {
            const unsigned q = 16 * (s / 8) + 8 * h + 4 * ((s / 4) % 2) + s % 4;
#pragma unroll
            for (int b = 0; b < TB; ++b)
                xf[b] = *reinterpret_cast<const f16x8*>(a + b * 32 * kStageRow +
                                                         16 * (q ^ (r % 16)));
        };
        Scales<ENC> sc[NBW];
#pragma unroll
        for (int c = 0; c < NBW; ++c)
            sc[c].prepare(rg[c], ENC == KDQ_Q6_K ? r : h, flags);
        f16x8 xf[2][TB], wf[2][NBW];
        read_x(0, xf[0]);
#pragma unroll
        for (int c = 0; c < NBW; ++c)
            wf[0][c] = dequant<ENC>(rg[c], sc[c], 0, magic);
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            __builtin_amdgcn_sched_barrier(0);
            issue(s, next_g, next_buf, next_rg);
            if (s + 1 < 16) {
                read_x(s + 1, xf[(s + 1) % 2]);
#pragma unroll
                for (int c = 0; c < NBW; ++c)
                    wf[(s + 1) % 2][c] = dequant<ENC>(rg[c], sc[c], s + 1, magic);
            }
#pragma unroll
            for (int c = 0; c < NBW; ++c)
#pragma unroll
                for (int b = 0; b < TB; ++b) {
                    acc[c][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[s % 2][c], xf[s % 2][b],
                                                                       acc[c][b], 0, 0, 0);
                    if constexpr (NBW == 1)  // the MFMAs stay in their sub-step (else the
                        asm volatile("" : "+v"(acc[c][b]));  // compiler sinks them all)
                }
#pragma unroll
            for (int q = 0; q < TB * NBW; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 32 / (TB * NBW), 0);  // VALU
                if (q < TB)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
                if (q < kPerStep)
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one global load
            }
        }
    };

    // Ping-pong over group pairs: group g in buffer 0 / registers ra, g + 1 in buffer 1 /
    // rb; each compute issues the other buffer's loads.  After the last pair the prefetch
    // reloads the last group (consumed only when the group count is odd).
    Regs ra[NBW], rb[NBW];
    const unsigned last = g_end - 1;
    issue_all(g_begin, 0, ra);
    unsigned g = g_begin;
    for (; g + 1 < g_end; g += 2) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        compute(0, ra, g + 1, 1, rb);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        compute(1, rb, min(g + 2, last), 0, ra);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA outlives the workgroup
    if (g < g_end) {  // odd group count: the last group sits in buffer 0 / ra
        __syncthreads();
        compute(0, ra, last, 1, rb);  // its prefetch reloads the last group (never used)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    // Output tile through LDS (free after the K loop): D of operand c, token block b holds
    // token 32b + r and weight rows 8(v / 4) + 4h + v % 4 of the operand's 32; scaled
    // back by the token's sigma, written as [token][row] fp32, then stored as whole rows.
    float sig[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        const unsigned tok = m0 + 32 * b + r;
        sig[b] = tok < m ? sigma[tok] : 1.f;
    }
    __syncthreads();  // every wavefront is done reading the activation stages
#pragma unroll
    for (int c = 0; c < NBW; ++c)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const unsigned row = (wave * NBW + c) * 32 + 8 * q + 4 * h;
                *reinterpret_cast<float4*>(lds + (32 * b + r) * kOutPitch + 4 * row) =
                    make_float4(acc[c][b][4 * q] * sig[b], acc[c][b][4 * q + 1] * sig[b],
                                acc[c][b][4 * q + 2] * sig[b], acc[c][b][4 * q + 3] * sig[b]);
            }
    __syncthreads();
    const unsigned f0 = n_tile * TILES * 16;       // first weight row of the tile
    constexpr int kChunks = TILES * 16 * 4 / 16;  // 16-byte chunks per token row
    for (unsigned e = threadIdx.x; e < TM * kChunks; e += W * 64) {
        const unsigned t = e / kChunks, ch = e % kChunks, tok = m0 + t, f = f0 + 4 * ch;
        if (tok >= m || f >= n)
            continue;
        const float4 v = *reinterpret_cast<const float4*>(lds + t * kOutPitch + 16 * ch);
        float* dst = dst_base + size_t(tok) * n + f;
        if (f + 3 < n && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
            *reinterpret_cast<float4*>(dst) = v;
        } else {
            const float vals[4] = {v.x, v.y, v.z, v.w};
            for (unsigned j = 0; j < 4 && f + j < n; ++j)
                dst[j] = vals[j];
        }
    }
    if (status) {
        unsigned all = flags;
        for (int o = 32; o > 0; o >>= 1)
            all |= __shfl_xor(all, o, 64);
        if (lane == 0 && all)
            atomicOr(status, all);
    }
}

// The weight-streaming form, for few tokens per weight matrix (grouped MoE layers, short
// chunks): 64 tokens per workgroup of four wavefronts, each with NBW 32-row weight operands
// (stream_operands: as many as leave room for two workgroups per compute unit).  What bounds it is the wait for the weights: a
// workgroup has few groups (8 of a 2048-value row), each multiplied in a fraction of the
// time its bytes take to arrive.  So a group's registers are reloaded with the group
// after the next as soon as each is read out (free_at), which keeps between one and two
// groups per wavefront in flight in two groups' registers, and a group ends by waiting only
// for its activation DMA, which goes out first (the counted wait below).  Past the last
// group the loads go on, so that the count stays the same: the DMAs to one address, the
// weights to group 0 of the operand's first tile, up to two groups' worth that nothing reads
// (with those to one address per wavefront too, 720 dense calls took 0.998 of the time, the
// short ones as well).  (Before, the next group's loads were spread over a group and waited for at its
// end, most of their latency showing; at 4096 slots over 128 experts, Q4_K gate / up 2048 ->
// 768: 90 -> 68 us, the 226 MB of weights at 3.3 TB/s; Q6_K down 768 -> 2048: 72 -> 58.)
// Only the tile's live tokens cost anything: the DMA of a dead one repeats token 0's lines,
// and a tile of at most 32 live tokens runs one 32-token block.
//
// Dense form: token t of tile m0 is staged row m0 + t, K slices as in gemm_kernel.
// Grouped (MoE) form, `tile_expert` given: token tile t multiplies the weights of expert
// tile_expert[t] of a stack of packed experts `expert_bytes` apart; tiles whose entry is
// negative are skipped (the whole workgroup returns before any barrier).  Position p holds
// slot slot_of[p] (negative: dead; a tile's live positions come first), whose staged row is
// slot / topk, or p itself when topk is 0.
//
// PAIR: a workgroup takes the same output rows of two matrices stored alike, `w` (gate) and
// `w2` (up), and the epilogue writes silu(gate) * up (the reference's silu, on the
// scaled-back fp32 values): one staging of x and no SwiGLU pass, the same bits as the two
// products and the pass.  With two operands a wavefront holds both matrices' rows (128 per
// workgroup); with one, wavefronts 0 and 1 hold the gate's and 2 and 3 the up's (64), which
// meet in LDS.
template <int ENC> constexpr int stream_operands = ENC == KDQ_Q4_K ? 2 : 1;
constexpr int kStreamWaves = 4;
template <int ENC, bool PAIR> constexpr int stream_tiles =
    2 * kStreamWaves * stream_operands<ENC> / (PAIR ? 2 : 1);
// fp32 output row of the tile in LDS (+16: banks), and a workgroup's LDS
template <int ENC> constexpr int kStreamOutPitch =
    kStreamWaves * stream_operands<ENC> * 32 * 4 + 16;
template <int ENC> constexpr size_t kStreamLds =
    std::max(size_t(kStreamTM) * kStreamOutPitch<ENC>, 2 * size_t(kStreamTM) * kStageRow);

template <int ENC, bool PAIR>
__global__ __launch_bounds__(kStreamWaves * 64, 2) void stream_gemm_kernel(
    const uint16_t* __restrict__ xs, const float* __restrict__ sigma,
    const uint8_t* __restrict__ w, unsigned m, unsigned n, unsigned k, unsigned slices,
    unsigned per, float* __restrict__ y, float* __restrict__ part, unsigned* __restrict__ status,
    const int32_t* __restrict__ tile_expert, size_t expert_bytes, const uint8_t* __restrict__ w2,
    const int32_t* __restrict__ slot_of, unsigned topk, const unsigned* __restrict__ used) {
    using F = GemmFormat<ENC>;
    using Regs = typename F::Regs;
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int TM = kStreamTM, W = kStreamWaves, NBW = stream_operands<ENC>;
    constexpr int SB = TM * kStageRow;  // bytes of one activation stage
    constexpr int TILES = stream_tiles<ENC, PAIR>;  // 16-row output tiles per workgroup
    constexpr int kOutPitch = kStreamOutPitch<ENC>;
    constexpr int kWeightLoads = F::loads * NBW;       // per wavefront and group

    const unsigned groups = k / 256, wtiles = (n + 15) / 16;
    // (grouped: the used token tiles only, so that every XCD gets the same share of them)
    const unsigned m_tiles = used ? max(*used / TM, 1u) : (m + TM - 1) / TM;
    const unsigned n_tiles = (wtiles + TILES - 1) / TILES;
    // XCD-aware order: the M tiles of one weight tile (and K slice) run together on one XCD
    const unsigned id = blockIdx.x, xcd = id % 8, local = id / 8;
    const unsigned per_xcd = (m_tiles * n_tiles * slices + 7) / 8;
    const unsigned linear = xcd * per_xcd + local;
    if (local >= per_xcd || linear >= m_tiles * n_tiles * slices)
        return;
    const unsigned n_tile = linear / (m_tiles * slices);
    const unsigned slice = (linear / m_tiles) % slices, m0 = (linear % m_tiles) * TM;
    if (tile_expert) {
        const int e = tile_expert[m0 / TM];
        if (e < 0)
            return;
        w += size_t(e) * expert_bytes;
        if constexpr (PAIR)
            w2 += size_t(e) * expert_bytes;
    }
    const unsigned g_begin = slice * per, g_end = min(groups, g_begin + per);
    float* __restrict__ dst_base = slices > 1 ? part + size_t(slice) * m * n : y;

    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const unsigned lane = threadIdx.x % 64;
    const unsigned r = lane % 32, h = lane / 32;
    const unsigned row_pitch = k * 2;
    // live tokens of the tile (at least one), and lane t's: the staged row of token t
    unsigned live = min(m - m0, unsigned(TM)), row_of_lane = m0 + lane;
    if (slot_of) {
        const int slot = slot_of[m0 + lane];
        live = __popcll(__ballot(slot >= 0));
        if (topk)
            row_of_lane = unsigned(max(slot, 0)) / topk;
    }
    auto staged_row = [&](unsigned t) {  // by the whole wavefront; dead tokens: token 0's
        return unsigned(__shfl(int(row_of_lane), int(t < live ? t : 0), 64));
    };

    // an operand is two packed tiles (rows 0-15, rows 16-31); tiles past the end load the
    // last tile, and their results are never stored.  ubase: the uniform
    // address of the first one in group 0; lane_at: the lane's bytes from there.
    const uint8_t* ubase[NBW];
    unsigned lane_at[NBW];
#pragma unroll
    for (int c = 0; c < NBW; ++c) {
        const unsigned operand = PAIR ? (NBW == 2 ? wave : wave % (W / 2)) : wave * NBW + c;
        const bool second = PAIR && (NBW == 2 ? c == 1 : wave >= W / 2);
        const unsigned first = min(n_tile * TILES + 2 * operand, wtiles - 1);
        ubase[c] = (second ? w2 : w) + size_t(first) * groups * F::unit;
        lane_at[c] = (min(n_tile * TILES + 2 * operand + r / 16, wtiles - 1) - first) * groups *
                         F::unit +
                     lane_code(r, h);
    }

    const auto x_rsrc = activation_resource(xs);

    unsigned flags = 0;
    unsigned magic = 0x64006400u;  // kept in a VGPR: the mask-and-or takes one SGPR only
    asm volatile("" : "+v"(magic));

    auto run = [&]<int TB>() {
        constexpr int DMAS = 32 * TB / kDmaRows / W;  // DMA instructions per wavefront and group
        static_assert(DMAS <= 8, "the DMAs of a group go out in two sub-steps");
        // instruction J = wave * DMAS + j covers tokens 2J, 2J + 1 of the tile; lane L fills
        // LDS chunk L % 32 of token 2J + L / 32 from logical chunk (L % 32) ^ (token % 16)
        unsigned xlane[DMAS];
#pragma unroll
        for (int j = 0; j < DMAS; ++j) {
            const unsigned tok = 2 * (wave * DMAS + j) + lane / 32;
            xlane[j] = staged_row(tok) * row_pitch +
                       (tok < live ? 16 * ((lane % 32) ^ (tok % 16)) : 0u);
        }
        auto stage_x = [&](unsigned g, unsigned buf, int j0, int j1) {
            const bool more = g < g_end;
            const int from = more ? int(g * 512) : 0;
#pragma unroll
            for (int j = j0; j < j1; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    x_rsrc, (lds_void*)(lds + buf * SB + (wave * DMAS + j) * 1024), 16,
                    more ? int(xlane[j]) : 0, from, 0, 0);
        };
        struct Source {
            const uint8_t* base[NBW];
            unsigned at[NBW];
        };
        auto source = [&](unsigned g) {
            Source s;
            const bool more = g < g_end;
#pragma unroll
            for (int c = 0; c < NBW; ++c) {
                s.base[c] = ubase[c] + (more ? size_t(g) * F::unit : 0);
                s.at[c] = more ? lane_at[c] : lane_code(r, h);
            }
            return s;
        };
        f32x16 acc[NBW][TB];
#pragma unroll
        for (int c = 0; c < NBW; ++c)
#pragma unroll
            for (int b = 0; b < TB; ++b)
                acc[c][b] = f32x16{};

        // group g from stage `buf` and registers rg: the DMAs of g + 1 into the other stage
        // first, then rg's reloads (group g + 2)
        auto compute = [&](unsigned g, unsigned buf, Regs* rg) {
            const uint8_t* a = lds + buf * SB + r * kStageRow;
            auto read_x = [&](int s, f16x8* xf) {
                const unsigned q = 16 * (s / 8) + 8 * h + 4 * ((s / 4) % 2) + s % 4;
#pragma unroll
                for (int b = 0; b < TB; ++b)
                    xf[b] = *reinterpret_cast<const f16x8*>(a + b * 32 * kStageRow +
                                                             16 * (q ^ (r % 16)));
            };
            Scales<ENC> sc[NBW];
#pragma unroll
            for (int c = 0; c < NBW; ++c)
                sc[c].prepare(rg[c], ENC == KDQ_Q6_K ? r : h, flags);
            const Source next = source(g + 2);
            f16x8 xf[2][TB], wf[2][NBW];
            read_x(0, xf[0]);
#pragma unroll
            for (int c = 0; c < NBW; ++c)
                wf[0][c] = dequant<ENC>(rg[c], sc[c], 0, magic);
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                __builtin_amdgcn_sched_barrier(0);
                if (s < 2)
                    stage_x(g + 1, buf ^ 1u, s * (DMAS / 2), s ? DMAS : DMAS / 2);
#pragma unroll
                for (int c = 0; c < NBW; ++c)
#pragma unroll
                    for (int i = 0; i < F::loads; ++i)
                        if (s == (free_at<ENC>(i) < 2 ? 2 : free_at<ENC>(i)))
                            load_item<ENC>(next.base[c] + next.at[c], h, r, rg[c], i);
                if (s + 1 < 16) {
                    read_x(s + 1, xf[(s + 1) % 2]);
#pragma unroll
                    for (int c = 0; c < NBW; ++c)
                        wf[(s + 1) % 2][c] = dequant<ENC>(rg[c], sc[c], s + 1, magic);
                }
#pragma unroll
                for (int c = 0; c < NBW; ++c)
#pragma unroll
                    for (int b = 0; b < TB; ++b) {
                        acc[c][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            wf[s % 2][c], xf[s % 2][b], acc[c][b], 0, 0, 0);
                        if constexpr (NBW == 1)  // the MFMAs stay in their sub-step (else the
                            asm volatile("" : "+v"(acc[c][b]));  // compiler sinks them all)
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // every load but the newest group's weights has arrived (so the DMAs have), for every
        // wavefront
        auto arrive = [&]() {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kWeightLoads) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        static_assert(kWeightLoads < 64, "vmcnt holds six bits");
        Regs ra[NBW], rb[NBW];
        auto load_all = [&](unsigned g, Regs* rg) {
            const Source s = source(g);
#pragma unroll
            for (int c = 0; c < NBW; ++c)
#pragma unroll
                for (int i = 0; i < F::loads; ++i)
                    load_item<ENC>(s.base[c] + s.at[c], h, r, rg[c], i);
        };
        stage_x(g_begin, 0, 0, DMAS);
        __builtin_amdgcn_sched_barrier(0);
        load_all(g_begin, ra);
        __builtin_amdgcn_sched_barrier(0);
        load_all(g_begin + 1, rb);
        __builtin_amdgcn_sched_barrier(0);
        unsigned g = g_begin;
        for (; g + 1 < g_end; g += 2) {
            arrive();
            compute(g, 0, ra);
            arrive();
            compute(g + 1, 1, rb);
        }
        if (g < g_end) {  // odd group count
            arrive();
            compute(g, 0, ra);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA outlives the workgroup

        // Output tile through LDS (free after the K loop), scaled back by the token's sigma,
        // as [token][row] fp32: D of operand c, token block b holds token 32b + r and weight
        // rows 8(v / 4) + 4h + v % 4 of the operand's 32.
        float sig[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b)
            sig[b] = sigma[staged_row(32 * b + r)];
        __syncthreads();  // every wavefront is done reading the activation stages
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float* out = reinterpret_cast<float*>(lds + (32 * b + r) * kOutPitch);
                if constexpr (PAIR && NBW == 2) {
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        v[i] = silu_of(acc[0][b][4 * q + i] * sig[b]) *
                               (acc[1][b][4 * q + i] * sig[b]);
                    *reinterpret_cast<float4*>(out + wave * 32 + 8 * q + 4 * h) =
                        make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int c = 0; c < NBW; ++c)
                        *reinterpret_cast<float4*>(out + (wave * NBW + c) * 32 + 8 * q + 4 * h) =
                            make_float4(acc[c][b][4 * q] * sig[b], acc[c][b][4 * q + 1] * sig[b],
                                        acc[c][b][4 * q + 2] * sig[b],
                                        acc[c][b][4 * q + 3] * sig[b]);
                }
            }
        __syncthreads();
    };
    if (live <= 32)
        run.template operator()<1>();
    else
        run.template operator()<2>();

    const unsigned f0 = n_tile * TILES * 16;       // first weight row of the tile
    constexpr unsigned kChunks = TILES * 16 * 4 / 16;  // 16-byte chunks per token row
    for (unsigned e = threadIdx.x; e < live * kChunks; e += W * 64) {
        const unsigned t = e / kChunks, ch = e % kChunks, f = f0 + 4 * ch;
        if (f >= n)
            continue;
        float4 v = *reinterpret_cast<const float4*>(lds + t * kOutPitch + 16 * ch);
        if constexpr (PAIR && NBW == 1) {
            const float4 u =
                *reinterpret_cast<const float4*>(lds + t * kOutPitch + 16 * (kChunks + ch));
            v = make_float4(silu_of(v.x) * u.x, silu_of(v.y) * u.y, silu_of(v.z) * u.z,
                            silu_of(v.w) * u.w);
        }
        float* dst = dst_base + size_t(m0 + t) * n + f;
        if (f + 3 < n && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
            *reinterpret_cast<float4*>(dst) = v;
        } else {
            const float vals[4] = {v.x, v.y, v.z, v.w};
            for (unsigned j = 0; j < 4 && f + j < n; ++j)
                dst[j] = vals[j];
        }
    }
    if (status) {
        unsigned all = flags;
        for (int o = 32; o > 0; o >>= 1)
            all |= __shfl_xor(all, o, 64);
        if (lane == 0 && all)
            atomicOr(status, all);
    }
}

// y[i] = sum of the K slices' partials part[s][i] in slice order (4 values per thread).
__global__ __launch_bounds__(256) void reduce_kernel(const float* __restrict__ part,
                                                     size_t count, unsigned slices,
                                                     float* __restrict__ y) {
    const size_t i = (size_t(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= count)
        return;
    if (i + 4 <= count && (count % 4) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
        float4 acc = *reinterpret_cast<const float4*>(part + i);
        for (unsigned s = 1; s < slices; ++s) {
            const float4 v = *reinterpret_cast<const float4*>(part + size_t(s) * count + i);
            acc = make_float4(acc.x + v.x, acc.y + v.y, acc.z + v.z, acc.w + v.w);
        }
        *reinterpret_cast<float4*>(y + i) = acc;
    } else {
        for (size_t j = i; j < i + 4 && j < count; ++j) {
            float acc = part[j];
            for (unsigned s = 1; s < slices; ++s)
                acc += part[size_t(s) * count + j];
            y[j] = acc;
        }
    }
}

// K slices: enough workgroups for the compute units when the output tiles are few, each
// slice at least 2 groups (512 values) deep.
// Returns the groups per slice; the slice count is ceil(groups / per) (no empty slice).
unsigned gemm_slice_depth(size_t m, size_t n, size_t k) {
    const size_t groups = k / 256;
    const size_t tiles = ((m + PM - 1) / PM) * (((n + 15) / 16 + kTiles - 1) / kTiles);
    const size_t units = compute_units();
    if (tiles * 3 >= units * 2)
        return unsigned(groups);
    size_t ks = std::max<size_t>(1, units / tiles);
    ks = std::min(ks, std::max<size_t>(1, groups / 2));
    return unsigned((groups + ks - 1) / ks);
}

// Wavefronts per GEMM workgroup: 8 with one 32-row operand each where two operands per
// wavefront do not fit the registers (Q6_K spilled 240 bytes per lane: 4096->14336 at 512
// tokens 125 -> 83 us with 8), else 4 (Q4_K and Q8_0 measured 2-4 % slower with 8).
template <int ENC> constexpr int gemm_waves = ENC == KDQ_Q6_K ? 8 : 4;

// Dense calls of up to this many rows run on the streaming kernel, one 64-token tile: 64 x
// 4096 -> 14336 Q8_0 31.5 us against 36.4 in a 128-token tile, 16 x 4096 -> 4096 Q6_K 15.7
// against 20.2.  Two such tiles read the weights twice: 128 x 4096 -> 14336 Q4_K 39.6 us
// against 38.5, 77 x 14336 -> 4096 Q6_K 47.9 against 42.0.
constexpr size_t kStreamRows = 64;

template <int ENC>
int configure() {
    static bool configured = false;  // one attribute call per instantiation
    if (!configured) {
        constexpr int W = gemm_waves<ENC>;
        const auto few = stage_kernel<ENC, 256>;
        const auto many = stage_kernel<ENC, 1024>;
        for (const void* f : {reinterpret_cast<const void*>(few),
                              reinterpret_cast<const void*>(many)})
            KDQ_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        128 * 1024));
        KDQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<ENC, W, 3>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds<3>)));
        KDQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<ENC, W, 4>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds<4>)));
        for (const void* f : {reinterpret_cast<const void*>(&stream_gemm_kernel<ENC, false>),
                              reinterpret_cast<const void*>(&stream_gemm_kernel<ENC, true>)})
            KDQ_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        int(kStreamLds<ENC>)));
        configured = true;
    }
    return KDQ_OK;
}

// Stages `rows` rows of k values: 1024 threads a row where each has a whole 16-byte load or
// more (4096 values), else 256, which would loop: 77 rows of 14336 8.0 -> 4.3 us, 512 of 4096
// 7.2 -> 6.2.
template <int ENC>
int launch_stage(const float* x, size_t rows, size_t k, uint16_t* xs, float* sigma,
                 const int32_t* slot_of, const unsigned* used, hipStream_t st) {
    const bool wide = k >= 4096;
    auto kernel = wide ? stage_kernel<ENC, 1024> : stage_kernel<ENC, 256>;
    hipLaunchKernelGGL(kernel, dim3(unsigned(rows)), dim3(wide ? 1024 : 256), k * 4, st, x,
                       unsigned(k), xs, sigma, slot_of, used);
    KDQ_HIP(hipGetLastError());
    return KDQ_OK;
}

// One launch of the streaming kernel over m rows (64-token tiles); `up` given: the paired
// form.
template <int ENC>
int launch_stream(const uint16_t* xs, const float* sigma, const void* packed, const void* up,
                  size_t m, size_t n, size_t k, unsigned slices, unsigned per, float* y,
                  float* part, unsigned* status, const int32_t* tile_expert, size_t expert_bytes,
                  const int32_t* slot_of, unsigned topk, const unsigned* used, hipStream_t st) {
    const size_t per_tile = up ? stream_tiles<ENC, true> : stream_tiles<ENC, false>;
    const size_t tiles =
        (m + kStreamTM - 1) / kStreamTM * (((n + 15) / 16 + per_tile - 1) / per_tile) * slices;
    auto kernel = up ? stream_gemm_kernel<ENC, true> : stream_gemm_kernel<ENC, false>;
    hipLaunchKernelGGL(kernel, dim3(unsigned((tiles + 7) / 8 * 8)), dim3(kStreamWaves * 64),
                       kStreamLds<ENC>, st, xs, sigma, static_cast<const uint8_t*>(packed),
                       unsigned(m), unsigned(n), unsigned(k), slices, per, y, part, status,
                       tile_expert, expert_bytes, static_cast<const uint8_t*>(up), slot_of, topk,
                       used);
    KDQ_HIP(hipGetLastError());
    return KDQ_OK;
}

// Grouped form: the rows of x staged (topk > 0: each token once; topk == 0: the live
// positions), then one launch over the token tiles.
template <int ENC>
int launch_grouped(const void* packed, const void* up, size_t expert_bytes,
                   const int32_t* tile_expert, size_t n, size_t k, const float* x, size_t x_rows,
                   const int32_t* inv, unsigned topk, const unsigned* used, size_t positions,
                   float* y, unsigned* status, uint16_t* xs, float* sigma, hipStream_t st) {
    int rc;
    if ((rc = configure<ENC>()))
        return rc;
    if ((rc = launch_stage<ENC>(x, x_rows, k, xs, sigma, topk ? nullptr : inv, used, st)))
        return rc;
    return launch_stream<ENC>(xs, sigma, packed, up, positions, n, k, 1u, unsigned(k / 256), y,
                              nullptr, status, tile_expert, expert_bytes, inv, topk, used, st);
}

// How one dense call runs: on 64-token tiles of the streaming kernel or 128-token tiles, and
// its K slices (groups per slice; the count is ceil(groups / per)).
struct GemmPlan {
    bool stream;
    unsigned per, slices;
};

GemmPlan gemm_plan(int encoding, size_t m, size_t n, size_t k) {
    GemmPlan p;
    p.stream = m <= kStreamRows;
    const size_t groups = k / 256;
    if (p.stream) {
        const size_t wt = encoding == KDQ_Q4_K ? stream_tiles<KDQ_Q4_K, false>
                                               : stream_tiles<KDQ_Q8_0, false>;
        const size_t tiles = (m + kStreamTM - 1) / kStreamTM * (((n + 15) / 16 + wt - 1) / wt);
        // K slices of two groups or more, as many as there are places for; none where their
        // partials, written and read back, cost more than the idle places: a tile has two
        // places and K is not very deep (64 x 1280 -> 65536 Q4_K 34.4 us in two slices, 23.2
        // in one; 9 x 14336 -> 28672 Q6_K 82.0 and 92.7), or fewer than eight and K is short
        // (64 x 768 -> 28672 Q6_K 22.3 and 13.0)
        const size_t places = std::max<size_t>(1, 2 * compute_units() / tiles);
        const bool whole = (places < 3 && groups < 32) || (places < 8 && groups <= 4);
        const size_t ks = whole ? 1 : places;
        p.per = unsigned((groups + ks - 1) / ks);
        p.per = unsigned(std::min<size_t>(groups, std::max<size_t>(p.per, 2)));
    } else {
        p.per = gemm_slice_depth(m, n, k);
    }
    p.slices = unsigned((groups + p.per - 1) / p.per);
    return p;
}

// Scratch of one dense GEMM call: x staged as fp16 rows padded to whole token tiles, the
// row scales, and the K slices' partials (none with one slice).
struct GemmScratch {
    size_t xs, sigma, part, total;
};

GemmScratch gemm_scratch(int encoding, size_t m, size_t n, size_t k) {
    const size_t m_pad = (m + PM - 1) / PM * PM;
    const unsigned slices = gemm_plan(encoding, m, n, k).slices;
    GemmScratch g;
    g.xs = (m_pad * k * 2 + 255) & ~size_t(255);
    g.sigma = (m * 4 + 255) & ~size_t(255);
    g.part = slices > 1 ? (size_t(slices) * m * n * 4 + 255) & ~size_t(255) : 0;
    g.total = g.xs + g.sigma + g.part;
    return g;
}

template <int ENC>
int launch_gemm(const float* x, const uint8_t* packed, size_t m, size_t n, size_t k, float* y,
                unsigned* status, uint8_t* scratch, hipStream_t st) {
    int rc;
    const GemmPlan plan = gemm_plan(ENC, m, n, k);
    const unsigned per = plan.per, slices = plan.slices;
    const GemmScratch g = gemm_scratch(ENC, m, n, k);
    auto* xs = reinterpret_cast<uint16_t*>(scratch);
    auto* sigma = reinterpret_cast<float*>(scratch + g.xs);
    auto* part = slices > 1 ? reinterpret_cast<float*>(scratch + g.xs + g.sigma) : nullptr;
    if ((rc = configure<ENC>()))
        return rc;
    if ((rc = launch_stage<ENC>(x, m, k, xs, sigma, nullptr, nullptr, st)))
        return rc;
    if (plan.stream) {
        if ((rc = launch_stream<ENC>(xs, sigma, packed, nullptr, m, n, k, slices, per, y, part,
                                     status, nullptr, 0, nullptr, 0u, nullptr, st)))
            return rc;
    } else {
        constexpr int W = gemm_waves<ENC>;
        const size_t tiles = (m + PM - 1) / PM * (((n + 15) / 16 + kTiles - 1) / kTiles) * slices;
        // Tiles of three 32-token blocks where no more of them are needed than of four (up to 96
        // rows, 129 to 192, 257 to 288): they multiply less padding for the same reads of the
        // weights.  Four blocks and three, Q6_K / Q4_K / Q8_0: 77 x 14336 -> 4096 34.2 -> 32.8,
        // 33.5 -> 30.5, 37.4 -> 34.1 us; 150 x 4096 -> 14336 47 -> 44.5, 42.0 -> 37.9, 46.2 ->
        // 41.2; 288 (Q8_0 270) x 4096 -> 14336 64.6 -> 61.9, 55.3 -> 47.3, 59.6 -> 53.5.
        const bool three = (m + 95) / 96 == (m + PM - 1) / PM;
        auto kernel = three ? gemm_kernel<ENC, W, 3> : gemm_kernel<ENC, W, 4>;
        hipLaunchKernelGGL(kernel, dim3(unsigned((tiles + 7) / 8 * 8)), dim3(W * 64),
                           three ? kLds<3> : kLds<4>, st,
                           xs, sigma, packed, unsigned(m), unsigned(n), unsigned(k), slices, per,
                           y, part, status);
        KDQ_HIP(hipGetLastError());
    }
    if (slices > 1) {
        const size_t count = m * n;
        hipLaunchKernelGGL(reduce_kernel, dim3(unsigned((count / 4 + 256) / 256)), dim3(256), 0,
                           st, part, count, slices, y);
        KDQ_HIP(hipGetLastError());
    }
    return KDQ_OK;
}

}  // namespace

int gemm_check(int encoding, const void* packed, size_t n, size_t k, unsigned* flags,
               hipStream_t st) {
    const size_t units = (n + 15) / 16 * (k / 256);
    const dim3 grid(unsigned((units * 32 + 255) / 256));
    auto* w = static_cast<const uint8_t*>(packed);
    switch (encoding) {
    case KDQ_Q4_K:
        hipLaunchKernelGGL(check_kernel<KDQ_Q4_K>, grid, dim3(256), 0, st, w, unsigned(k / 256),
                           units, flags);
        break;
    case KDQ_Q8_0:
        hipLaunchKernelGGL(check_kernel<KDQ_Q8_0>, grid, dim3(256), 0, st, w, unsigned(k / 256),
                           units, flags);
        break;
    case KDQ_Q6_K:
        hipLaunchKernelGGL(check_kernel<KDQ_Q6_K>, grid, dim3(256), 0, st, w, unsigned(k / 256),
                           units, flags);
        break;
    default:
        return KDQ_ERR_UNSUPPORTED;
    }
    KDQ_HIP(hipGetLastError());
    return KDQ_OK;
}

size_t dense_gemm_scratch(int encoding, size_t m, size_t n, size_t k) {
    return gemm_scratch(encoding, m, n, k).total;
}

int dense_gemm(int encoding, const void* packed, size_t n, size_t k, const float* x, size_t m,
               float* y, unsigned* status, void* scratch, hipStream_t st) {
    auto* w = static_cast<const uint8_t*>(packed);
    auto* sc = static_cast<uint8_t*>(scratch);
    switch (encoding) {
    case KDQ_Q4_K:
        return launch_gemm<KDQ_Q4_K>(x, w, m, n, k, y, status, sc, st);
    case KDQ_Q8_0:
        return launch_gemm<KDQ_Q8_0>(x, w, m, n, k, y, status, sc, st);
    case KDQ_Q6_K:
        return launch_gemm<KDQ_Q6_K>(x, w, m, n, k, y, status, sc, st);
    default:
        return KDQ_ERR_UNSUPPORTED;
    }
}

int dense_gemm_pair(int encoding, const void* gate, const void* up, size_t n, size_t k,
                    const float* x, size_t m, float* y, unsigned* status, void* scratch,
                    hipStream_t st) {
    if (!grouped_gemm_takes(encoding, k))
        return KDQ_ERR_UNSUPPORTED;
    auto* sc = static_cast<uint8_t*>(scratch);
    const GemmScratch g = gemm_scratch(encoding, m, n, k);
    auto launch = [&]<int ENC>() -> int {
        int rc;
        if ((rc = configure<ENC>()))
            return rc;
        auto* xs = reinterpret_cast<uint16_t*>(sc);
        auto* sigma = reinterpret_cast<float*>(sc + g.xs);
        if ((rc = launch_stage<ENC>(x, m, k, xs, sigma, nullptr, nullptr, st)))
            return rc;
        return launch_stream<ENC>(xs, sigma, gate, up, m, n, k, 1u, unsigned(k / 256), y, nullptr,
                                  status, nullptr, 0, nullptr, 0u, nullptr, st);
    };
    return encoding == KDQ_Q4_K   ? launch.template operator()<KDQ_Q4_K>()
           : encoding == KDQ_Q8_0 ? launch.template operator()<KDQ_Q8_0>()
                                  : launch.template operator()<KDQ_Q6_K>();
}

bool grouped_gemm_takes(int encoding, size_t k) {
    return (encoding == KDQ_Q4_K || encoding == KDQ_Q8_0 || encoding == KDQ_Q6_K) &&
           k % 256 == 0 && k <= 32768;
}

int grouped_gemm(int encoding, const void* packed, size_t expert_bytes,
                 const int32_t* tile_expert, size_t n, size_t k, const float* x, size_t x_rows,
                 const int32_t* inv, unsigned topk, const unsigned* used, size_t positions,
                 float* y, unsigned* status, uint16_t* xs, float* sigma, hipStream_t st,
                 const void* up) {
    if (!grouped_gemm_takes(encoding, k) || positions % kStreamTM)
        return KDQ_ERR_UNSUPPORTED;
    auto launch = [&](auto go) {
        return go(packed, up, expert_bytes, tile_expert, n, k, x, x_rows, inv, topk, used,
                  positions, y, status, xs, sigma, st);
    };
    return encoding == KDQ_Q4_K   ? launch(launch_grouped<KDQ_Q4_K>)
           : encoding == KDQ_Q8_0 ? launch(launch_grouped<KDQ_Q8_0>)
                                  : launch(launch_grouped<KDQ_Q6_K>);
}

}  // namespace kdq

using namespace kdq;

extern "C" int kdq_gemm_packed(int encoding, const void* packed, size_t n, size_t k,
                               const float* x, size_t m, float* y, unsigned* status,
                               void* stream) {
    if (!packed || !x || !y || !m || !n || !k)
        return KDQ_ERR_ARGUMENT;
    if (encoding != KDQ_Q4_K && encoding != KDQ_Q8_0 && encoding != KDQ_Q6_K)
        return KDQ_ERR_UNSUPPORTED;
    if (k % 256 || k > 32768 || m > 0xffffffu || n > 0xffffffu)
        return KDQ_ERR_SHAPE;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(packed) % 16 ||
        reinterpret_cast<uintptr_t>(y) % 4)
        return KDQ_ERR_ALIGNMENT;
    const size_t packed_bytes = kdq_gguf_packed_bytes(encoding, k, n);
    if (overlaps(y, m * n * 4, x, m * k * 4) || overlaps(y, m * n * 4, packed, packed_bytes))
        return KDQ_ERR_ALIAS;
    int rc;
    void* scratch = workspace(dense_gemm_scratch(encoding, m, n, k), &rc);
    if (rc)
        return rc;
    return dense_gemm(encoding, packed, n, k, x, m, y, status, scratch,
                      static_cast<hipStream_t>(stream));
}

extern "C" int kdq_gguf_gemm_check(int encoding, const void* packed, size_t n, size_t k,
                                   unsigned* flags, void* stream) {
    if (!packed || !flags || !n || !k)
        return KDQ_ERR_ARGUMENT;
    if (encoding != KDQ_Q4_K && encoding != KDQ_Q8_0 && encoding != KDQ_Q6_K)
        return KDQ_ERR_UNSUPPORTED;
    if (k % 256 || k > 32768 || n > 0xffffffu)
        return KDQ_ERR_SHAPE;
    if (reinterpret_cast<uintptr_t>(packed) % 16 || reinterpret_cast<uintptr_t>(flags) % 4)
        return KDQ_ERR_ALIGNMENT;
    return gemm_check(encoding, packed, n, k, flags, static_cast<hipStream_t>(stream));
}
