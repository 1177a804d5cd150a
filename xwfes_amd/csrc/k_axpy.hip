// k_axpy.hip -- the column-axpy form y[m, j] += sum_i h[m, i] * W[i, j]
// (matmul_down_axpy, src/cpu_backend.cpp:60-75) on MFMA over the tensor as it
// is stored: n_in rows of N columns, blocks along the columns, no re-tiled
// copy, any h.
//
// Along the contraction i every row carries its own block scale, so the scale
// goes into the activation operand: A = h[m, i] * d[i, block], formed in fp32
// and split into three bf16 limbs by truncation (8 + 8 + 8 bits: the split is
// exact and needs no range assumption), B = the block's integers, exact in
// bf16 (q - 8, q or q - 32: at most 8 bits).  Three MFMAs per product; every
// product is exact and the only rounding is that of the fp32 sums.
//   Q4_0  d (q - 8)         Q8_0  d q            one A per 32 columns
//   Q6_K  d (sc (q - 32))                         one A per 256 columns: the
//         integers (at most 4096) as two bf16 limbs, nearest and rest, five
//         MFMAs (third limb x rest, 2^-26 of the product, is left out); with
//         d sc in A, one per 16 columns, the splits took three quarters of
//         the time
//   Q4_K  (d sc) (q - c) - (dmin m - c d sc)      one A per 32 columns; the min
//         term is a product of its own, h (3 limbs) x its 3 limbs, with the
//         four 32-column sub-blocks as B columns; c is the integer nearest to
//         dmin m / (d sc) (q4k_c), so that neither sum is larger than the
//         weights call for (a fixed c = 8 left a zero weight as the difference
//         of two terms)
//
// The MFMA wants 8 contraction values (rows) of one column in a lane, the
// tensor has a row's columns side by side.  A wave loads 8 rows x 4 or 8
// bytes per lane, transposes bytes in registers (v_perm) and passes the
// columns through its own LDS slots ([tile][kq][column] x 8 bytes, columns
// XOR-swizzled by the tile: no bank conflict either way); no barrier until
// the end.  A workgroup's 8 waves take a 128-column group's 32-row slices in
// turn and are added in LDS in wave order; splits over the rows leave
// partials for the next kernel.
//
// What bounds it: up to 16 tokens the arrival of the weights and the byte
// work (about 100 VALU instructions per 32 x 32 weights), above that the limb
// splits (52 VALU per 32 x 32 weights and 16 tokens; Q6_K an eighth of that) and
// MFMAs.
// Measured, one launch (before: the generic kernel, or Q6_K's 8-token chunks):
// Q4_0 14336 x 4096, 24 tokens 2013 -> 29.7 us; Q6_K, 256 tokens 531 -> 141 us
// (213 TFLOP/s; 219 with d sc in A and two workgroups a CU assumed by the
// split rule); up to 8 tokens of Q8_0 / Q4_0 go to k_axpy_few below.  Error
// against 64 bits 0.5e-7 to 1.5e-7 (1408 to 14336 rows; Q6_K, 64 tokens of 14336
// rows 2.0e-7) where the fp32 sums of the generic kernel had 1.6e-7 to 5.7e-7:
// the waves and the splits are added in 64 bits.
#include <algorithm>

#include "ftx_internal.h"
#include "mm_dev.h"
#include "quant_dev.h"

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int AX_WAVES = 8;
constexpr int AX_COLS = 128;  // columns per workgroup

struct AxArgs {
    const uint8_t* W;
    int64_t row_bytes, n_in, N;
    const float* h;
    int64_t ldh;
    int M;
    int ntt;               // token tiles of 16 MS
    int slices_per_split;  // 32-row slices
    float* out;            // partials [split][M][ldo], or y with accum
    int64_t ldo, split_stride;
    int accum;
};

// loads of any alignment (the hardware takes them as they come)
struct __attribute__((packed)) u32u { uint32_t v; };
struct __attribute__((packed)) u64u { uint32_t v[2]; };
struct __attribute__((packed)) u16u { uint16_t v; };
struct __attribute__((packed)) u128u { uint32_t v[4]; };
struct __attribute__((packed, aligned(4))) f4u { float v[4]; };

// rows r0..r3 of four bytes -> columns c[0..3], byte e = row e
__device__ __forceinline__ void tr4(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t* c) {
    const uint32_t a = perm(r1, r0, 0x05010400u), b = perm(r1, r0, 0x07030602u);
    const uint32_t d = perm(r3, r2, 0x05010400u), e = perm(r3, r2, 0x07030602u);
    c[0] = perm(d, a, 0x05040100u);
    c[1] = perm(d, a, 0x07060302u);
    c[2] = perm(e, b, 0x05040100u);
    c[3] = perm(e, b, 0x07060302u);
}

// The scales (Q4_K: the activations) enter times 2^24, undone on the sums: the
// limbs of products h d down to the smallest normal number stay clear of the
// subnormal range, which the MFMA does not keep (third limbs of 1e-30, second
// limbs of 1e-34 were lost).  Products that this takes out of the fp32 range
// are formed again (ax_redo).
constexpr float AX_UP = 16777216.f, AX_DOWN = 1.f / 16777216.f;

template <int DT>
struct AxCfg {
    // LDS tiles of 16 columns x 32 rows (nibble types hold two in one)
    static constexpr int TILES = (DT == FTX_Q8_0 || DT == FTX_Q6_K) ? 8 : 4;
    static constexpr int SWZ = DT == FTX_Q8_0 ? 7 : 3;
    // scales per row: blocks, Q4_K's scales then mins, Q6_K's 16-column
    // integer scales then d
    static constexpr int NSC = DT == FTX_Q6_K ? 9 : (DT == FTX_Q4_K ? 8 : 4);
    // Q4_K: 128 - c of every row and sub-block, a byte each, after the scales
    static constexpr int CEN = DT == FTX_Q4_K ? 128 : 0;
    static constexpr int WORDS = (DT == FTX_Q8_0 || DT == FTX_Q6_K) ? 2 : 1;  // per lane and row
};

// a wave's raw operands of one slice: 8 rows of the lane's bytes, and the
// scale fields of row 8 kq + c % 8 (c = lane % 16)
template <int DT>
struct AxRaw {
    uint32_t w[8][AxCfg<DT>::WORDS];
    uint32_t s[DT == FTX_Q4_K ? 4 : 2];
};

// rows i0 .. i1 - 1 of token m and column col, product by product: for sums
// that do not come out finite (an infinite or NaN operand breaks the limbs,
// and h d may leave the fp32 range where h (d q) does not)
__device__ float ax_redo(const AxArgs& a, int dt, int m, int64_t col, int64_t i0, int64_t i1) {
    const float* hr = a.h + (int64_t)m * a.ldh;
    float v = 0.f;
    for (int64_t i = i0; i < i1; ++i) {
        float q[8], x = 0.f;
        dq8(a.W + i * a.row_bytes, dt, col & ~(int64_t)7, a.N, q);
#pragma unroll
        for (int e = 0; e < 8; ++e) x = (int)(col & 7) == e ? q[e] : x;
        v += hr[i] * x;
    }
    return v;
}

template <int DT, int MS>
__global__ void __launch_bounds__(64 * AX_WAVES)
    __attribute__((amdgpu_waves_per_eu(MS == 1 ? 4 : 2, MS == 1 ? 4 : 2))) k_axpy(AxArgs a) {
    using C = AxCfg<DT>;
    // per wave: columns, then scales; at the end the waves' sums of one
    // 16-token tile
    constexpr int WB = C::TILES * 512 + C::NSC * 128 + C::CEN;
    __shared__ __attribute__((aligned(16))) uint8_t lds[65536];
    static_assert(WB * AX_WAVES <= 65536, "");
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, kq = lane >> 4;
    const int64_t j0 = (int64_t)(blockIdx.x / (unsigned)a.ntt) * AX_COLS;  // first column
    const int m0 = (int)(blockIdx.x % (unsigned)a.ntt) * 16 * MS;
    const int ks = blockIdx.z;
    const int64_t nsl = (a.n_in + 31) / 32;
    const int64_t I0 = (int64_t)ks * a.slices_per_split;
    const int64_t I1 = min(I0 + (int64_t)a.slices_per_split, nsl);
    // The MFMA rounds its sums down (toward minus infinity): odd waves form
    // theirs negated, so that the shares cancel in the waves' sum
    const float sgn = (w & 1) ? -1.f : 1.f;
    uint2* cols = (uint2*)(lds + w * WB);
    float* scl = (float*)(lds + w * WB + C::TILES * 512);  // [NSC][kq][8]
    uint8_t* cen = (uint8_t*)(scl + C::NSC * 32);          // Q4_K: [4][kq][8]

    // the lane's byte offset in a row and its scale fields' (blocks past the
    // row's end read the last one; their columns are not stored)
    int64_t off, soff[2] = {0, 0}, doff = 0;
    if constexpr (DT == FTX_Q4_0 || DT == FTX_Q8_0) {
        constexpr int bb = DT == FTX_Q4_0 ? 18 : 34;
        const int64_t nb = a.N / 32, b0 = j0 / 32;
        off = min(b0 + c / 4, nb - 1) * bb + 2 + (c % 4) * (bb - 2) / 4;
        soff[0] = min(b0 + c / 8, nb - 1) * bb;
        soff[1] = min(b0 + 2 + c / 8, nb - 1) * bb;
    } else if constexpr (DT == FTX_Q4_K) {
        const int64_t sb = j0 / 256;
        off = sb * 144 + 16 + 64 * ((j0 / 128) & 1) + 4 * c;
        soff[0] = sb * 144;
    } else {  // planar Q6_K rows (quant_dev.h)
        const int64_t sb = j0 / 256, nsb = a.N / 256, half = (j0 / 128) & 1;
        off = sb * 128 + 64 * (c >> 3) + 32 * half + 4 * (c & 7);
        soff[0] = nsb * 128 + sb * 64 + 32 * (c >> 3) + 16 * half + 4 * (c & 3);  // QH
        soff[1] = nsb * 192 + sb * 16 + 8 * half + 4 * (c >> 3);                   // 4 scales
        doff = nsb * 208 + sb * 2;
    }
    auto load = [&](AxRaw<DT>& o, int64_t I) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint8_t* r = a.W + min(32 * I + 8 * kq + e, a.n_in - 1) * a.row_bytes;
            if constexpr (DT == FTX_Q8_0) {
                const u64u v = *(const u64u*)(r + off);
                o.w[e][0] = v.v[0];
                o.w[e][1] = v.v[1];
            } else {
                o.w[e][0] = ((const u32u*)(r + off))->v;
                if constexpr (DT == FTX_Q6_K) o.w[e][1] = ((const u32u*)(r + soff[0]))->v;
            }
        }
        const uint8_t* r = a.W + min(32 * I + 8 * kq + (c & 7), a.n_in - 1) * a.row_bytes;
        if constexpr (DT == FTX_Q4_K) {
            const u128u v = *(const u128u*)(r + soff[0]);
#pragma unroll
            for (int i = 0; i < 4; ++i) o.s[i] = v.v[i];
        } else if constexpr (DT == FTX_Q6_K) {
            o.s[0] = ((const u32u*)(r + soff[1]))->v;
            o.s[1] = ((const u16u*)(r + doff))->v;
        } else {
            o.s[0] = ((const u16u*)(r + soff[0]))->v;
            o.s[1] = ((const u16u*)(r + soff[1]))->v;
        }
    };
    // the columns of tile n into its slots: row octet kq, column col
    auto slot = [&](int n, int col) { return (n * 4 + kq) * 16 + (col ^ (n & C::SWZ)); };
    auto put = [&](const AxRaw<DT>& o) {
        uint32_t lo[4], hi[4];
        if constexpr (DT == FTX_Q8_0) {
#pragma unroll
            for (int hw = 0; hw < 2; ++hw) {
                tr4(o.w[0][hw], o.w[1][hw], o.w[2][hw], o.w[3][hw], lo);
                tr4(o.w[4][hw], o.w[5][hw], o.w[6][hw], o.w[7][hw], hi);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    cols[slot(c >> 1, 8 * (c & 1) + 4 * hw + i)] = uint2{lo[i], hi[i]};
            }
        } else if constexpr (DT == FTX_Q6_K) {
            // ql byte of element 32 k + l (k = a, and 2 + a in its high
            // nibble), l = 16 b + 8 g + t; the two high bits from the qh byte
            const int g = c >> 3, av = (c >> 2) & 1, b = (c >> 1) & 1, t = 4 * (c & 1);
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
                uint32_t q[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    q[e] = minus4(((o.w[e][0] >> (4 * k2)) & 0x0F0F0F0Fu) |
                                      (((o.w[e][1] >> (4 * k2 + 2 * av)) & 0x03030303u) << 4), 32);
                tr4(q[0], q[1], q[2], q[3], lo);
                tr4(q[4], q[5], q[6], q[7], hi);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    cols[slot(2 * (2 * k2 + av) + b, 8 * g + t + i)] = uint2{lo[i], hi[i]};
            }
        } else {
            tr4(o.w[0][0], o.w[1][0], o.w[2][0], o.w[3][0], lo);
            tr4(o.w[4][0], o.w[5][0], o.w[6][0], o.w[7][0], hi);
#pragma unroll
            for (int i = 0; i < 4; ++i) cols[slot(c >> 2, 4 * (c & 3) + i)] = uint2{lo[i], hi[i]};
        }
        // scales of row 8 kq + c % 8
        const int at = kq * 8 + (c & 7), hf = c >> 3;
        if constexpr (DT == FTX_Q4_K) {
            const float d = sgn * h2f((uint16_t)(o.s[0] & 0xFFFF)), dmin = sgn * h2f((uint16_t)(o.s[0] >> 16));
            // sub-blocks 4 h .. 4 h + 3 of the row's super-block; this lane
            // takes two of them
            const bool up = ((j0 / 128) & 1) != 0;
            const uint32_t sc = up ? (o.s[3] & 0x0F0F0F0Fu) | ((o.s[1] >> 2) & 0x30303030u)
                                   : o.s[1] & 0x3F3F3F3Fu;
            const uint32_t mn = up ? ((o.s[3] >> 4) & 0x0F0F0F0Fu) | ((o.s[2] >> 2) & 0x30303030u)
                                   : o.s[2] & 0x3F3F3F3Fu;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int sh = 16 * hf + 8 * i;
                const float ds = d * (float)((sc >> sh) & 0xFF);
                scl[(2 * hf + i) * 32 + at] = ds;
                const float dm = dmin * (float)((mn >> sh) & 0xFF), ctr = q4k_c(ds, dm);
                scl[(4 + 2 * hf + i) * 32 + at] = q4k_g(ds, dm, ctr);
                cen[(2 * hf + i) * 32 + at] = (uint8_t)(128.f - ctr);
            }
        } else if constexpr (DT == FTX_Q6_K) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                scl[(4 * hf + i) * 32 + at] = (float)(int8_t)(o.s[0] >> (8 * i));
            scl[8 * 32 + at] = sgn * AX_UP * h2f((uint16_t)o.s[1]);  // (both halves the same value)
        } else {
            scl[hf * 32 + at] = sgn * AX_UP * h2f((uint16_t)o.s[0]);
            scl[(2 + hf) * 32 + at] = sgn * AX_UP * h2f((uint16_t)o.s[1]);
        }
    };
    // h of the lane's token (past M: the last one's, never stored) in each
    // 16-token tile, rows 8 kq .. + 7 of the slice (zero past n_in)
    auto load_h = [&](float (&hv)[MS][8], int64_t I) {
        const float* hrow[MS];
        int cc = c;  // (formed anew per slice: held, the pointers spill)
        asm("" : "+v"(cc));
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
            hrow[ms] = a.h + (int64_t)min(m0 + 16 * ms + cc, a.M - 1) * a.ldh;
        const int64_t i = 32 * I + 8 * kq;
        if (32 * I + 32 <= a.n_in) {  // uniform
#pragma unroll
            for (int ms = 0; ms < MS; ++ms) {
                const f4u u = *(const f4u*)(hrow[ms] + i), v = *(const f4u*)(hrow[ms] + i + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hv[ms][e] = u.v[e];
                    hv[ms][4 + e] = v.v[e];
                }
            }
        } else {
#pragma unroll
            for (int ms = 0; ms < MS; ++ms)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = hrow[ms][min(i + e, a.n_in - 1)];
                    hv[ms][e] = i + e < a.n_in ? v : 0.f;
                }
        }
        if constexpr (DT == FTX_Q4_K)
#pragma unroll
            for (int ms = 0; ms < MS; ++ms)
#pragma unroll
                for (int e = 0; e < 8; ++e) hv[ms][e] *= AX_UP;
    };
    // (two tiles, whose registers allow it: the first limbs' products in a
    // sum of their own, so that a slice rounds that once and not three times: 24
    // tokens of 14336 rows of Q4_0 / Q6_K 1.4e-7 / 2.0e-7 -> 0.6e-7 / 1.0e-7
    // against 64 bits, at the same time)
    constexpr bool LO = MS == 2;
    v4f acc[8][MS], acl[LO ? 8 : 1][LO ? MS : 1], accm[DT == FTX_Q4_K ? MS : 1];
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
            acc[n][ms] = v4f{0.f, 0.f, 0.f, 0.f};
            if constexpr (LO) acl[n][ms] = v4f{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
    for (int ms = 0; ms < (DT == FTX_Q4_K ? MS : 1); ++ms) accm[ms] = v4f{0.f, 0.f, 0.f, 0.f};
    auto low = [&](int n, int ms) -> v4f& {
        if constexpr (LO) return acl[n][ms];
        else return acc[n][ms];
    };
    auto mfma3 = [&](const v8bf* l, const v8bf& b, int n, int ms) {
        low(n, ms) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[2], b, low(n, ms), 0, 0, 0);
        low(n, ms) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[1], b, low(n, ms), 0, 0, 0);
        acc[n][ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[0], b, acc[n][ms], 0, 0, 0);
    };
    auto scales8 = [&](int s, int q, float* d) {
        const float4 u = *(const float4*)&scl[s * 32 + q * 8], v = *(const float4*)&scl[s * 32 + q * 8 + 4];
        d[0] = u.x; d[1] = u.y; d[2] = u.z; d[3] = u.w;
        d[4] = v.x; d[5] = v.y; d[6] = v.z; d[7] = v.w;
    };

    if (I0 + w < I1) {
        AxRaw<DT> raw;
        float hv[MS][8];
        load(raw, I0 + w);
        for (int64_t I = I0 + w; I < I1; I += AX_WAVES) {
            load_h(hv, I);
            put(raw);
            // (the last slice's load is its own again: no branch between the
            // loads and the waits)
            load(raw, min(I + AX_WAVES, I1 - 1));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if constexpr (DT == FTX_Q4_K) {
                // B column b < 4: dmin m - c d sc of sub-block b
                float dm[8];
                scales8(4 + (c & 3), kq, dm);
#pragma unroll
                for (int e = 0; e < 8; ++e) dm[e] = c < 4 ? dm[e] : 0.f;
                v8bf bm[3];
                split3(dm, bm);
#pragma unroll
                for (int ms = 0; ms < MS; ++ms) {
                    v8bf l[3];
                    split3(hv[ms], l);
#pragma unroll
                    for (int p = 2; p >= 0; --p)
#pragma unroll
                        for (int q = p; q >= 0; --q)
                            accm[ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[q], bm[p - q], accm[ms], 0, 0, 0);
                }
            }
            if constexpr (DT == FTX_Q6_K) {
                float d[8];
                scales8(8, kq, d);
                v8bf l[MS][3];
#pragma unroll
                for (int ms = 0; ms < MS; ++ms) {
                    float t[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) t[e] = hv[ms][e] * d[e];
                    split3(t, l[ms]);
                }
#pragma unroll
                for (int n = 0; n < 8; ++n) {  // 16 columns
                    const uint2 v = cols[slot(n, c)];
                    float t[8];
                    scales8(n, kq, t);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        t[e] *= (float)(int8_t)((e < 4 ? v.x : v.y) >> (8 * (e & 3)));
                    v8bf bw[2];
                    split2(t, bw);
#pragma unroll
                    for (int ms = 0; ms < MS; ++ms) {
                        low(n, ms) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[ms][1], bw[1], low(n, ms), 0, 0, 0);
                        low(n, ms) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l[ms][0], bw[1], low(n, ms), 0, 0, 0);
                        mfma3(l[ms], bw[0], n, ms);
                    }
                }
            }
            if constexpr (DT != FTX_Q6_K) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {  // 32 columns
                v8bf bw[2];
                if constexpr (DT == FTX_Q4_0) {
                    const uint2 v = cols[slot(b, c)];
#pragma unroll
                    for (int p = 0; p < 2; ++p)
                        bw[p] = sbytes(minus4((v.x >> (4 * p)) & 0x0F0F0F0Fu, 8),
                                       minus4((v.y >> (4 * p)) & 0x0F0F0F0Fu, 8));
                } else if constexpr (DT == FTX_Q4_K) {
                    const uint2 cb = *(const uint2*)&cen[b * 32 + kq * 8];  // of the 8 rows
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint2 v = cols[slot(2 * (b >> 1) + p, c)];
                        bw[p] = sbytes((((v.x >> (4 * (b & 1))) & 0x0F0F0F0Fu) + cb.x) ^ 0x80808080u,
                                       (((v.y >> (4 * (b & 1))) & 0x0F0F0F0Fu) + cb.y) ^ 0x80808080u);
                    }
                } else {  // Q8_0
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint2 v = cols[slot(2 * b + p, c)];
                        bw[p] = sbytes(v.x, v.y);
                    }
                }
                float d[8];
                scales8(b, kq, d);
#pragma unroll
                for (int ms = 0; ms < MS; ++ms) {
                    v8bf l[3];
                    float t[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) t[e] = hv[ms][e] * d[e];
                    split3(t, l);
#pragma unroll
                    for (int p = 0; p < 2; ++p) mfma3(l, bw[p], 2 * b + p, ms);
                }
            }
            }
            // (the reads above before the next slice's writes)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    if constexpr (LO)
#pragma unroll
        for (int n = 0; n < 8; ++n)
#pragma unroll
            for (int ms = 0; ms < MS; ++ms) acc[n][ms] += acl[n][ms];
    if constexpr (DT == FTX_Q4_K) {
        // the min sums: lane (c, kq) of tile n holds tokens 4 kq + r; those of
        // sub-block n / 2 are in lane 16 kq + n / 2
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = __shfl(accm[ms][r], 16 * kq + b, 64);
                    acc[2 * b][ms][r] -= v;
                    acc[2 * b + 1][ms][r] -= v;
                }
    }
    // wave w adds the eight waves' sums of tile w, in wave order, and writes
    // them: columns 32 (w / 2) + .. of the group
    v4f* red = (v4f*)lds;  // [wave][tile][lane]
    const int64_t col = j0 + 32 * (w >> 1) + (DT == FTX_Q4_0 ? 2 * c + (w & 1) : 16 * (w & 1) + c);
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
        __syncthreads();
#pragma unroll
        for (int n = 0; n < 8; ++n) red[(w * 8 + n) * 64 + lane] = acc[n][ms];
        __syncthreads();
        v4d s = {0., 0., 0., 0.};
#pragma unroll
        for (int k = 0; k < AX_WAVES; ++k) {
            const v4d v = __builtin_convertvector(red[(k * 8 + w) * 64 + lane], v4d);
            s = (k & 1) ? s - v : s + v;
        }
        if (col >= a.N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * ms + 4 * kq + r;
            if (m >= a.M) continue;
            float v = (float)s[r] * AX_DOWN;
            if (!is_finite(v)) v = ax_redo(a, DT, m, col, 32 * I0, min(32 * I1, a.n_in));
            float* p = a.out + (int64_t)ks * a.split_stride + (int64_t)m * a.ldo + col;
            *p = a.accum ? *p + v : v;
        }
    }
}

// ---------------------------------------------------------------- few tokens
//
// Up to 8 tokens of Q8_0 / Q4_0: with so few rows of A in use the MFMA form
// spends its time on limbs and transposes, while the products themselves are
// few.  Here a lane owns 8 neighbouring columns and walks rows: y[m][j] +=
// (h[m][i] d) q, one multiplication per row and token for h d, a conversion
// and M multiply-adds per weight, all fp32.  A wave covers 512 columns of a
// contiguous run of rows (one load of 512 or 256 contiguous quant bytes a
// row), four rows in flight ahead of the four computed; h comes through
// scalar loads.  The 8 waves of a workgroup are added in LDS in wave order.
// Measured, one token: Q8_0 14336 x 4096 25.6 (k_axpy) -> 15.6 us (4.0 TB/s)
// with a sum of the partials of 4.4 us (6.2 before); Q4_0 1408 x 512 5.8 -> 4.1.
constexpr int AF_WAVES = 8, AF_ROWS = 4;

template <int DT, int MC>
__global__ void __launch_bounds__(64 * AF_WAVES) k_axpy_few(AxArgs a) {
    constexpr int QW = DT == FTX_Q8_0 ? 2 : 1, BB = DT == FTX_Q8_0 ? 34 : 18;
    __shared__ __attribute__((aligned(16))) float red[AF_WAVES][512];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t j0 = (int64_t)blockIdx.x * 512;
    const int ks = blockIdx.z;
    // (columns past the row's end read its last block and are not stored)
    const int64_t blk = min(j0 / 32 + lane / 4, a.N / 32 - 1);
    const uint32_t soff = (uint32_t)(blk * BB), qoff = soff + 2 + (lane & 3) * 4 * QW;
    // (slices_per_split counts rows here, an eighth of them per wave)
    const int64_t i0 = (int64_t)ks * a.slices_per_split, i1 = min(i0 + (int64_t)a.slices_per_split, a.n_in);
    const int64_t per = (i1 - i0 + AF_WAVES - 1) / AF_WAVES;
    const int64_t r0 = i0 + w * per, r1 = min(r0 + per, i1);
    float acc[MC][8];
#pragma unroll
    for (int m = 0; m < MC; ++m)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[m][e] = 0.f;
    struct Rows {
        uint32_t q[AF_ROWS][QW], d[AF_ROWS];
    } cur, nxt;
    auto load = [&](Rows& o, int64_t r) {
#pragma unroll
        for (int u = 0; u < AF_ROWS; ++u) {
            const uint8_t* p = a.W + min(r + u, a.n_in - 1) * a.row_bytes;  // uniform
            o.d[u] = ((const u16u*)(p + soff))->v;
            if constexpr (DT == FTX_Q8_0) {
                const u64u v = *(const u64u*)(p + qoff);
                o.q[u][0] = v.v[0];
                o.q[u][1] = v.v[1];
            } else {
                o.q[u][0] = ((const u32u*)(p + qoff))->v;
            }
        }
    };
    auto row = [&](const Rows& o, int u, int64_t r) {
        float q[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            q[e] = DT == FTX_Q8_0 ? (float)(int8_t)(o.q[u][e / 4 % QW] >> (8 * (e & 3)))
                                  : (float)((int)((o.q[u][0] >> (4 * e)) & 15u) - 8);
        const float d = AX_UP * h2f((uint16_t)o.d[u]);
#pragma unroll
        for (int m = 0; m < MC; ++m) {
            const float t = a.h[(int64_t)min(m, a.M - 1) * a.ldh + r] * d;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[m][e] = fmaf(t, q[e], acc[m][e]);
        }
    };
    if (r0 < r1) {
        load(cur, r0);
        int64_t r = r0;
        for (; r + AF_ROWS <= r1; r += AF_ROWS) {
            load(nxt, r + AF_ROWS);
#pragma unroll
            for (int u = 0; u < AF_ROWS; ++u) row(cur, u, r + u);
            cur = nxt;
        }
#pragma unroll
        for (int u = 0; u < AF_ROWS; ++u)
            if (r + u < r1) row(cur, u, r + u);  // uniform
    }
#pragma unroll
    for (int m = 0; m < MC; ++m) {
        if (m >= a.M) break;  // uniform
        if (m) __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *(float4*)&red[w][8 * lane + 4 * h] =
                float4{acc[m][4 * h], acc[m][4 * h + 1], acc[m][4 * h + 2], acc[m][4 * h + 3]};
        __syncthreads();
        float s = red[0][tid];
#pragma unroll
        for (int k = 1; k < AF_WAVES; ++k) s += red[k][tid];
        s *= AX_DOWN;
        if (j0 + tid < a.N) {
            if (!is_finite(s)) s = ax_redo(a, DT, m, j0 + tid, i0, i1);
            float* p = a.out + (int64_t)ks * a.split_stride + (int64_t)m * a.ldo + j0 + tid;
            *p = a.accum ? *p + s : s;
        }
    }
}

// y[m][n] += sum_s part[s][m][n] of few rows: 64 columns per workgroup, its
// four waves a quarter of the splits each (four partial sums, added in order)
__global__ void __launch_bounds__(256) k_axpy_sum(const float* __restrict__ part, int S, int64_t stride,
                                                  int64_t N, float* __restrict__ y, int64_t ldy) {
    __shared__ float red[4][64];
    const int c = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t n = (int64_t)blockIdx.x * 64 + c, m = blockIdx.y;
    const float* p = part + m * N + min(n, N - 1);
    const int per = (S + 3) / 4, s0 = w * per, s1 = min(s0 + per, S);
    float v = 0.f;
    for (int s = s0; s < s1; s += 8) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = p[(int64_t)min(s + u, S - 1) * stride];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += s + u < s1 ? t[u] : 0.f;
    }
    red[w][c] = v;
    __syncthreads();
    if (w == 0 && n < N) y[m * ldy + n] += ((red[0][c] + red[1][c]) + red[2][c]) + red[3][c];
}

}  // namespace

// whole blocks along a row (the K types have 256-column blocks)
bool axpy_supported(int dt, int64_t N) {
    return N > 0 && (((dt == FTX_Q4_0 || dt == FTX_Q8_0) && N % 32 == 0) ||
                     ((dt == FTX_Q4_K || dt == FTX_Q6_K) && N % 256 == 0));
}

// splits of the few-token kernel: workgroups of 512 columns, 8 waves each;
// about 512 of them, at least 64 rows (8 a wave) per split, within `cap`
static bool axpy_few(int dt, int64_t M) { return M <= 8 && (dt == FTX_Q8_0 || dt == FTX_Q4_0); }
static int axpy_few_splits(int64_t M, int64_t n_in, int64_t N, size_t cap) {
    const int64_t wg = (N + 511) / 512;
    int64_t S = std::min(std::max<int64_t>(512 / wg, 1), std::max<int64_t>(n_in / 64, 1));
    while (S > 1 && (size_t)(S * M * N) > cap) --S;
    return (int)S;
}
// 16-token tiles per workgroup, and splits over the rows: one-tile workgroups run
// two to a CU, those of two and four tiles (164 to 256 VGPRs) one, in rounds, each
// as long as its waves' slices (every eighth of the split's) plus about two
// slices of start and reduction; the fewest slice times, the fewest splits on
// ties, within `cap` partial floats (one split writes y itself).  (Two to a CU
// assumed for two tiles as well: twice the splits in two rounds, 24 tokens of
// Q4_0 14336 x 4096 79 us a call against 70 us, 4096 x 4096 60 against 53.)
static int axpy_ms(int64_t M) { return M <= 16 ? 1 : (M <= 32 ? 2 : 4); }
static int axpy_splits(int64_t M, int64_t n_in, int64_t N, size_t cap, int cu_count) {
    const int ms = axpy_ms(M);
    const int64_t wg = (N + AX_COLS - 1) / AX_COLS * ((M + 16 * ms - 1) / (16 * ms));
    const int64_t nsl = (n_in + 31) / 32, slots = (ms == 1 ? 2 : 1) * (cu_count > 0 ? cu_count : 256);
    int best = 1;
    int64_t best_cost = -1;
    for (int64_t S = 1; S <= 32 && S <= nsl; ++S) {
        // (the reduce has a grid row per token)
        if (S > 1 && ((size_t)(S * M * N) > cap || M > 65535)) break;
        const int64_t per = (nsl + S - 1) / S;
        const int64_t cost = (wg * S + slots - 1) / slots * ((per + AX_WAVES - 1) / AX_WAVES + 2);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = (int)S;
        }
    }
    return best;
}

size_t axpy_part_floats(int dt, int64_t M, int64_t n_in, int64_t N, size_t cap, int cu_count) {
    const int S = M <= 0 ? 1 : (axpy_few(dt, M) ? axpy_few_splits(M, n_in, N, cap)
                                                 : axpy_splits(M, n_in, N, cap, cu_count));
    return S > 1 ? (size_t)S * (size_t)(M * N) : 0;
}

hipError_t launch_axpy(hipStream_t st, const uint8_t* W, int dt, int64_t row_bytes, int64_t n_in,
                       int64_t N, const float* h, int64_t ldh, int64_t M, float* y, int64_t ldy,
                       float* part, size_t part_floats, int cu_count, MmPend* pend) {
    if (pend) *pend = MmPend{};
    if (M <= 0 || n_in <= 0) return hipSuccess;
    if (!axpy_supported(dt, N)) return hipErrorInvalidValue;
    const bool few = axpy_few(dt, M);
    int S = few ? axpy_few_splits(M, n_in, N, part ? part_floats : 0)
                : axpy_splits(M, n_in, N, part ? part_floats : 0, cu_count);
    // rows (few) or 32-row slices
    const int64_t nsl = few ? n_in : (n_in + 31) / 32;
    AxArgs a{};
    a.W = W;
    a.row_bytes = row_bytes;
    a.n_in = n_in;
    a.N = N;
    a.h = h;
    a.ldh = ldh;
    a.M = (int)M;
    const int ms = axpy_ms(M);
    a.ntt = (int)((M + 16 * ms - 1) / (16 * ms));
    a.slices_per_split = (int)((nsl + S - 1) / S);
    S = (int)((nsl + a.slices_per_split - 1) / a.slices_per_split);
    a.out = S > 1 ? part : y;
    a.ldo = S > 1 ? N : ldy;
    a.split_stride = S > 1 ? M * N : 0;
    a.accum = S == 1;
    using K_t = void (*)(AxArgs);
    if (few) {
        static const K_t fk[2][4] = {
            {k_axpy_few<FTX_Q8_0, 1>, k_axpy_few<FTX_Q8_0, 2>, k_axpy_few<FTX_Q8_0, 4>, k_axpy_few<FTX_Q8_0, 8>},
            {k_axpy_few<FTX_Q4_0, 1>, k_axpy_few<FTX_Q4_0, 2>, k_axpy_few<FTX_Q4_0, 4>, k_axpy_few<FTX_Q4_0, 8>}};
        ktimed_launch(fk[dt == FTX_Q4_0][M == 1 ? 0 : (M == 2 ? 1 : (M <= 4 ? 2 : 3))],
                      dim3((unsigned)((N + 511) / 512), 1, (unsigned)S), dim3(64 * AF_WAVES), 0, st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || S == 1) return e;
        // (many small partials: added here, not left in *pend)
        hipLaunchKernelGGL(k_axpy_sum, dim3((unsigned)((N + 63) / 64), (unsigned)M), dim3(256), 0, st, part,
                           S, M * N, N, y, ldy);
        return hipGetLastError();
    }
    static const K_t kerns[4][3] = {
        {k_axpy<FTX_Q4_0, 1>, k_axpy<FTX_Q4_0, 2>, k_axpy<FTX_Q4_0, 4>},
        {k_axpy<FTX_Q8_0, 1>, k_axpy<FTX_Q8_0, 2>, k_axpy<FTX_Q8_0, 4>},
        {k_axpy<FTX_Q4_K, 1>, k_axpy<FTX_Q4_K, 2>, k_axpy<FTX_Q4_K, 4>},
        {k_axpy<FTX_Q6_K, 1>, k_axpy<FTX_Q6_K, 2>, k_axpy<FTX_Q6_K, 4>}};
    const int di = dt == FTX_Q4_0 ? 0 : (dt == FTX_Q8_0 ? 1 : (dt == FTX_Q4_K ? 2 : 3));
    const dim3 grid((unsigned)((N + AX_COLS - 1) / AX_COLS * a.ntt), 1, (unsigned)S);
    ktimed_launch(kerns[di][ms == 4 ? 2 : ms - 1], grid, dim3(64 * AX_WAVES), 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || S == 1) return e;
    MmPend p;
    p.part = part;
    p.split_stride = M * N;
    p.ldp = N;
    p.S = S;
    p.N = N;
    p.accum = 1;
    if (pend) {
        *pend = p;  // added into y by the next kernel that reads it
        return hipSuccess;
    }
    return launch_mm_fold(st, p, M, y, ldy, 1);
}
