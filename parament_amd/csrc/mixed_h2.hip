// Mixed-precision slice kernel on scaled fp16 two-way split products (gfx950 fp16 matrix cores, the
// slice Hamiltonian and the first-order term in FP64), with the lowest levels of the pairwise product
// tree fused in, for tau Hnorm <= 1.  Every FP32 operand of a product is held as
//
//     x = (h0 + h1) / S,   h0 = fp16(S x),  h1 = fp16(S x - h0),   S = 2^14
//
// fp16 keeps 11 significant bits, so the two parts carry 22 bits (the difference S x - h0 is
// exact in FP32), and a product is the sum h0 h0' + h0 h1' + h1 h0' (+ h1 h1' when FULL = 4) of
// fp16 products accumulated in FP32: three (four) matrix-core products per FP32-accurate product
// instead of the six of the bf16 three-way split (mixed.hip), and two operand planes instead of three.
// The scale keeps the operands in fp16's range: an entry is at most the spectral norm of its matrix,
// which for Z = -i tau X, its powers and the combinations formed here is below 2 while ||tau X||_2 <= 1
// (for controls of modulus <= 1, ||tau X||_2 <= tau Hnorm <= 1 here), and the tree nodes |E| = |U - I| <= 2
// for unitary slices, so S x stays below 2^15 < 65504 (overflow needs an entry of 4).  An entry whose low part falls
// below fp16's normal range loses at most 2^-25 / S = 2^-39 in absolute terms.  The 22-bit
// products' rounding grows with ||tau X||_2 (controls well above 1 in modulus): see the precision
// modes in parament.h.  Every tile is held multiplied by S (exact), so that its planes are written
// without a multiply; the accumulated products carry S^2.
//
// Layout.  A lane's four accumulator elements are consecutive rows of one column, so planes are stored
// column by column (8 bytes per plane and lane); a product M1 M2 reads M2's columns as the second operand
// and M1's rows as the first, through the LDS transpose read (ds_read_b64_tr_b16), so no plane is ever written
// in 2-byte pieces.  Four plane sets are used as two pairs, one pair per product in turn, so a product
// needs one barrier: the one between its operands' stores and its reads.  What bounds the kernel is vector
// issue and latency (one work-group of eight waves per CU at D = 64); this layout and the three-product scheme
// took 32,767 dim-64 slices from 1.42 to 1.05 ms, and 10,006 slices of dim 45 (Horner's rule, M = 5) from 456
// to 335 us.
#include "kernels.hpp"

#include <type_traits>

namespace pa {

namespace {

typedef float f32x4h __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr float kScale = 16384.0f;                       // S = 2^14
constexpr float kInvScale = 1.0f / 16384.0f;

// Wave tiles of 16 x 32 (two 16x16 blocks sharing each A fragment), as in mixed.hip.
// Dims pad to 32 or 64 (h2_padded_dim).
template <int D> struct HShape {
    static constexpr int TN = 2;
    static constexpr int WR = D / 16;
    static constexpr int WC = D / 32;
    static constexpr int G = WR * WC;
    static constexpr int PL = D * D;
    // unpadded rows of 16-byte chunks, permuted so that a wave's 8- and 16-byte accesses spread over the banks
    static __device__ __forceinline__ int off(int row, int col) {
        if constexpr (D == 64) return row * D + ((((col >> 3) ^ row) & 7) << 3) + (col & 7);
        else return row * D + (((col >> 3) ^ ((row >> 2) & 2)) << 3) + (col & 7);
    }
};

// The two fp16 parts of values held scaled by S (round to nearest even).  one holds 1.0 where the
// compiler cannot see it, so that s - h0 becomes one mixed-precision FMA (s * one - h0, rounded to fp16) instead of a
// conversion, a subtraction and a conversion.
__device__ __forceinline__ void split2s(float s0, float s1, float one, f16x2& h0, f16x2& h1) {
    h0[0] = (_Float16)s0;
    h0[1] = (_Float16)s1;
    h1[0] = (_Float16)__builtin_fmaf(s0, one, -(float)h0[0]);
    h1[1] = (_Float16)__builtin_fmaf(s1, one, -(float)h0[1]);
}
__device__ __forceinline__ int hrow(int row0, int v) { return row0 + 4 * ((threadIdx.x & 63) >> 4) + v; }
__device__ __forceinline__ int hcol(int col0, int n) { return col0 + 16 * n + (threadIdx.x & 15); }

template <int TN> struct HTile {
    f32x4h re[TN], im[TN];
};

__device__ __forceinline__ f16x8 tr_pair(const _Float16* a, const _Float16* b) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const f16x4 x = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)a));
    const f16x4 y = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)b));
    return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
}

// -v, one XOR per pair (the compiler's negation of a half vector is three instructions per pair)
__device__ __forceinline__ f16x8 hneg(f16x8 v) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(f16x8, __builtin_bit_cast(u32x4, v) ^ 0x80008000u);
}

// The wave's tile of S^2 M1 M2: planes P1 of M1 and P2 of M2 (by columns), plane 2 * part + {0: re, 1: im}.  NP = 1: h0 h0' only (relative error ~2^-11); 3: with the
// two cross terms (~2^-21); 4: all four products.  Im Im' goes into the same accumulator as Re Re' with a
// negated operand: the matrix cores' accumulation rounds with a bias that the signs then cancel (summed
// apart and subtracted, the dim-64 chain's propagator drifted 3.4e-6 from unitary instead of 1e-7).
template <int D, int NP>
__device__ __forceinline__ void wave_cgemm_h2(const _Float16* P1, const _Float16* P2, int row0, int col0,
                                              HTile<HShape<D>::TN>& c) {
    constexpr int PL = HShape<D>::PL, TN = HShape<D>::TN;
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) { c.re[n][v] = 0.f; c.im[n][v] = 0.f; }
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
        // M1[row0 + r][k], k = 32 ks + 8 kq + 0 .. 7: 16 lanes transpose four rows of 16 at a time
        const int a0 = HShape<D>::off(32 * ks + 8 * kq + (r >> 2), row0 + 4 * (r & 3));
        const int a1 = HShape<D>::off(32 * ks + 8 * kq + 4 + (r >> 2), row0 + 4 * (r & 3));
        f16x8 Ar[2], Ai[2], An[2];
#pragma unroll
        for (int p = 0; p < (NP == 1 ? 1 : 2); ++p) {
            Ar[p] = tr_pair(P1 + (2 * p) * PL + a0, P1 + (2 * p) * PL + a1);
            Ai[p] = tr_pair(P1 + (2 * p + 1) * PL + a0, P1 + (2 * p + 1) * PL + a1);
            An[p] = hneg(Ai[p]);
        }
#pragma unroll
        for (int q = 0; q < (NP == 1 ? 1 : 2); ++q) {
            f16x8 Br[TN], Bi[TN];
#pragma unroll
            for (int n = 0; n < TN; ++n) {
                const int kb = HShape<D>::off(col0 + 16 * n + r, 32 * ks + 8 * kq);
                Br[n] = *reinterpret_cast<const f16x8*>(P2 + (2 * q) * PL + kb);
                Bi[n] = *reinterpret_cast<const f16x8*>(P2 + (2 * q + 1) * PL + kb);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const bool use = (p == 0 && q == 0) || (NP >= 3 && p + q == 1) || (NP == 4 && p == 1 && q == 1);
                if (!use) continue;
                // the tile's accumulators in turn, so that a product does not wait for the one before
#pragma unroll
                for (int n = 0; n < TN; ++n) {
                    c.re[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ar[p], Br[n], c.re[n], 0, 0, 0);
                    c.im[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ar[p], Bi[n], c.im[n], 0, 0, 0);
                }
#pragma unroll
                for (int n = 0; n < TN; ++n) {
                    c.re[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(An[p], Bi[n], c.re[n], 0, 0, 0);
                    c.im[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ai[p], Br[n], c.im[n], 0, 0, 0);
                }
            }
        }
    }
}

// The NL leading fp16 parts of four elements adjacent in a column (one accumulator block of a lane, scaled
// by S) of the real (c = 0) or imaginary (c = 1) plane.
template <int D, int NL>
__device__ __forceinline__ void store4_h2(const f32x4h& x, int c, _Float16* P, int at, float one) {
    constexpr int PL = HShape<D>::PL;
    f16x2 lo0, lo1, hi0, hi1;
    split2s(x[0], x[1], one, lo0, lo1);
    split2s(x[2], x[3], one, hi0, hi1);
    *reinterpret_cast<f16x4*>(P + c * PL + at) = f16x4{lo0[0], lo0[1], hi0[0], hi0[1]};
    if (NL > 1) *reinterpret_cast<f16x4*>(P + (2 + c) * PL + at) = f16x4{lo1[0], lo1[1], hi1[0], hi1[1]};
}
template <int D, int NL = 2>
__device__ __forceinline__ void write_h2(const HTile<HShape<D>::TN>& b, _Float16* P, int row0, int col0, float one) {
#pragma unroll
    for (int n = 0; n < HShape<D>::TN; ++n) {
        const int at = HShape<D>::off(hcol(col0, n), hrow(row0, 0));
        store4_h2<D, NL>(b.re[n], 0, P, at, one);
        store4_h2<D, NL>(b.im[n], 1, P, at, one);
    }
}

struct RawCoefH {
    double2 c0, c1, c2;
};
__device__ __forceinline__ RawCoefH coef_load_h(const Controls<double>& q, int t, int j) {
    RawCoefH r;
    if (q.mode == QUAD_NONE) { r.c0 = sample(q, t, j); r.c1 = r.c2 = mk<double>(0, 0); }
    else if (q.mode == QUAD_MIDPOINT) { r.c0 = sample(q, t, j); r.c1 = sample(q, t, j + 1); r.c2 = mk<double>(0, 0); }
    else { r.c0 = sample(q, t, 2 * j); r.c1 = sample(q, t, 2 * j + 1); r.c2 = sample(q, t, 2 * j + 2); }
    return r;
}
__device__ __forceinline__ double2 coef_finish_h(const Controls<double>& q, const RawCoefH& r) {
    if (q.mode == QUAD_NONE) return r.c0;
    if (q.mode == QUAD_MIDPOINT) {
        const double2 s = cadd(r.c0, r.c1);
        return mk<double>(0.5 * s.x, 0.5 * s.y);
    }
    const double2 s = cadd(cadd(r.c0, mk<double>(4.0 * r.c1.x, 4.0 * r.c1.y)), r.c2);
    const double sixth = 1.0 / 6.0;
    return mk<double>(s.x * sixth, s.y * sixth);
}

}  // namespace

// E = U - I of a slice as a polynomial in Z = -i tau X with real coefficients a.zc (power_real /
// poly_scheme in host.cpp), tau Hnorm <= 1.  SCHEME 8: degree 8 on three products (see poly_slice_tile,
// fused_device.hpp); 0: any degree M by Horner's rule in Z2 = Z Z,
//   E = c_0' I + c_1 Z + c_2 Z2 + Z2 (c_3 Z + Z2 (c_4 I + c_5 Z + Z2 (..)))   (c_0' = c_0 - 1),
// (M + 1) / 2 products, the inner ones at the part count the host chose (a.ps_levels: 0 = the leading
// products only, otherwise FULL).  The terms in Z are exact to FP64: Z is kept as an FP32 value and its
// residual, and E is rounded once.  a.ops holds the operators padded with zeros to D x D, so that every load is
// unconditional and its address a fixed offset (masked loads at dims below D spilled 100 registers); the
// padding stays isolated from the d x d block in every product.
//
// Tree fold: the work-group's 2^F slices run one after another (a loop, so the slice code is
// emitted once); after slice p, the carry chain over the levels l (unrolled, so every pending
// node sits in fixed registers) combines with the pending earlier sibling pend[l] while bit l of
// p is set, and otherwise parks the node in pend[l].  Slices past N are zero nodes, which the
// combine returns unchanged bit for bit (the reference's odd carry).
// Node w of the problem a: its 2^F slices and their product.  cur: first plane set of the pair the next product's operands go to
// (kept by the caller from one problem to the next: waves may still read the other pair).
//
// CHECK: values beyond fp16's range are met (controls of any modulus, slices far from unitary).  They become
// infinities in their product and reach the node as these or as NaNs, so a node that is not finite is not stored and
// the result is false.  F32: the node with FP32 products instead (S = 1, two plane pairs of FP32, a barrier on
// either side of a product), for such nodes.
template <int D, int F, int FULL, int SCHEME, bool CHECK = false, bool F32 = false>
__device__ __forceinline__ bool h2_node(const MixedArgs& a, _Float16* planes, double2* coef, int& cur, int w) {
    constexpr float S = F32 ? 1.0f : kScale, inv = 1.0f / S;
    constexpr int G = HShape<D>::G, PL = HShape<D>::PL, WC = HShape<D>::WC;
    constexpr int TN = HShape<D>::TN;
    constexpr int NB = 1 << F;
    typedef HTile<TN> Tile;
    const int tid = threadIdx.x, wave = tid >> 6;
    const int row0 = 16 * (wave / WC), col0 = 16 * TN * (wave % WC);
    constexpr int DD = D * D;
    const int d = a.d, dd = d * d, M = a.M;
    const bool prefetch = !a.ctl.magnus && a.ncoef <= 64 * G;
    bool coef_ready = false;
    // diagonal positions of the wave's tile (fixed for the launch)
    bool dg[TN][4];
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) dg[n][v] = hrow(row0, v) == hcol(col0, n);

    float one = 1.0f;   // opaque to the compiler (split2s)
    asm volatile("" : "+v"(one));
    auto set = [&](int k) { return planes + cur + 4 * PL * k; };
    constexpr int SF = D + 2, PF = D * SF;
    static_assert(4 * PF * sizeof(float) <= 16 * PL * sizeof(_Float16), "the FP32 planes fit in the others' place");
    float* fp = reinterpret_cast<float*>(planes);
    // operand k = 0, 1 of the next product; lead: its leading part is enough
    auto put = [&](const Tile& t, int k, auto lead) {
        if constexpr (F32) {
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int at = 2 * k * PF + hrow(row0, v) * SF + hcol(col0, n);
                    fp[at] = t.re[n][v]; fp[PF + at] = t.im[n][v];
                }
        } else {
            write_h2<D, decltype(lead)::value ? 1 : 2>(t, set(k), row0, col0, one);
        }
    };
    // the product of operands k1 and k2, after a barrier; the next one's may be put at once
    auto product = [&](int k1, int k2, Tile& c, auto lead) {
        if constexpr (F32) {
            CTile<float, 1, TN> t;
            wave_cgemm<float, 1, TN, D, SF, SF>(fp + 2 * k1 * PF, fp + (2 * k1 + 1) * PF, fp + 2 * k2 * PF,
                                                fp + (2 * k2 + 1) * PF, row0, col0, t);
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) { c.re[n][v] = t.re[0][n][v]; c.im[n][v] = t.im[0][n][v]; }
            __syncthreads();
        } else {
            wave_cgemm_h2<D, decltype(lead)::value ? 1 : FULL>(set(k1), set(k2), row0, col0, c);
            cur = 8 * PL - cur;
        }
    };
    constexpr std::false_type full{};
    constexpr std::true_type lead{};
    // the assembly forms S Z = -i tau S H0 + sum_t (-i tau S c'_t) O_t: coef[] holds -i tau S c'_t
    const double ts = a.ctl.tau * (double)S;
    auto scaled = [&](double2 c) { return mk<double>(c.y * ts, -c.x * ts); };
    auto slice = [&](int j, int jn, Tile& e) __attribute__((always_inline)) {
        if (!coef_ready) {
            for (int t = tid; t < a.ncoef; t += 64 * G) coef[t] = scaled(slice_coefficient(a.ctl, t, j));
            __syncthreads();
        }
        Tile z, zl;   // Z in FP32, and what that leaves of the FP64 value
#pragma unroll
        for (int n = 0; n < TN; ++n) {
            const double2* ops = a.ops + hrow(row0, 0) * D + hcol(col0, n);
            double2 x[4];
            if (a.ncoef <= 3) {
                // every operator element of the block requested before any arithmetic (one load
                // latency): an operator slot past ncoef reads H0's element again and is weighted by zero
                double2 h[4], o[3][4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    h[v] = ops[v * D];
#pragma unroll
                    for (int q = 0; q < 3; ++q) o[q][v] = ops[(q < a.ncoef ? (q + 1) * DD : 0) + v * D];
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) x[v] = mk<double>(h[v].y * ts, -h[v].x * ts);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const double2 cc = (q < a.ncoef) ? coef[q] : mk<double>(0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        x[v].x = __builtin_fma(cc.x, o[q][v].x, x[v].x);
                        x[v].x = __builtin_fma(-cc.y, o[q][v].y, x[v].x);
                        x[v].y = __builtin_fma(cc.x, o[q][v].y, x[v].y);
                        x[v].y = __builtin_fma(cc.y, o[q][v].x, x[v].y);
                    }
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) x[v] = mk<double>(ops[v * D].y * ts, -ops[v * D].x * ts);
                for (int t = 0; t < a.ncoef; ++t) {
                    ops += DD;
                    double2 o[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) o[v] = ops[v * D];
                    const double2 cc = coef[t];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {   // x += cc o, four FMAs
                        x[v].x = __builtin_fma(cc.x, o[v].x, x[v].x);
                        x[v].x = __builtin_fma(-cc.y, o[v].y, x[v].x);
                        x[v].y = __builtin_fma(cc.x, o[v].y, x[v].y);
                        x[v].y = __builtin_fma(cc.y, o[v].x, x[v].y);
                    }
                }
            }
            // the empty asm statement keeps the compiler from merging the roundings to FP32 and to fp16
            // into a double -> half conversion, which has no instruction and is emulated
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float yr = (float)x[v].x, yi = (float)x[v].y;
                asm volatile("" : "+v"(yr), "+v"(yi));
                z.re[n][v] = yr; z.im[n][v] = yi;
                zl.re[n][v] = (float)(x[v].x - (double)yr); zl.im[n][v] = (float)(x[v].y - (double)yi);
            }
        }
        put(z, 0, full);
        __syncthreads();
        const bool pre = prefetch && jn >= 0 && jn < a.N;
        RawCoefH raw;
        if (pre && tid < a.ncoef) raw = coef_load_h(a.ctl, tid, jn);
        Tile z2, p, acc;
        product(0, 0, acc, full);   // Z Z
        auto unscale = [&](Tile& t) {
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) { t.re[n][v] = acc.re[n][v] * inv; t.im[n][v] = acc.im[n][v] * inv; }
        };
        unscale(z2);
        auto publish = [&]() {   // the operands stored above become readable
            if (pre && tid < a.ncoef) coef[tid] = scaled(coef_finish_h(a.ctl, raw));
            __syncthreads();
        };
        Tile rest;   // E - Z without the last product
        if constexpr (SCHEME == 8) {
            const float q3 = a.zc[3], q4 = a.zc[4], q5 = a.zc[5], q6 = a.zc[6], q7 = a.zc[7], q8 = a.zc[8], q2 = a.zc[2];
            Tile t;
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    t.re[n][v] = __builtin_fmaf(q3, z2.re[n][v], z.re[n][v]);
                    t.im[n][v] = __builtin_fmaf(q3, z2.im[n][v], z.im[n][v]);
                }
            put(z2, 0, full);
            put(t, 1, full);
            publish();
            product(0, 1, acc, full);   // P = Z2 (Z + q3 Z2)
            unscale(p);
            Tile u;
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    u.re[n][v] = __builtin_fmaf(q4, p.re[n][v], z2.re[n][v]);
                    u.im[n][v] = __builtin_fmaf(q4, p.im[n][v], z2.im[n][v]);
                    t.re[n][v] = __builtin_fmaf(q6, p.re[n][v], __builtin_fmaf(q5, z2.re[n][v], z.re[n][v]));
                    t.im[n][v] = __builtin_fmaf(q6, p.im[n][v], __builtin_fmaf(q5, z2.im[n][v], z.im[n][v]));
                    rest.re[n][v] = __builtin_fmaf(q8, p.re[n][v], __builtin_fmaf(q7, p.re[n][v], __builtin_fmaf(q2, z2.re[n][v], 0.5f * z2.re[n][v])));
                    rest.im[n][v] = __builtin_fmaf(q8, p.im[n][v], __builtin_fmaf(q7, p.im[n][v], __builtin_fmaf(q2, z2.im[n][v], 0.5f * z2.im[n][v])));
                }
            put(u, 0, full);
            put(t, 1, full);
            __syncthreads();
            product(0, 1, acc, full);
            const float zw = F32 ? a.zw * kScale : a.zw;
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    rest.re[n][v] = __builtin_fmaf(zw, acc.re[n][v], rest.re[n][v]);
                    rest.im[n][v] = __builtin_fmaf(zw, acc.im[n][v], rest.im[n][v]);
                }
        } else {
            // Q_j = c_2j I + c_2j+1 Z + Z2 Q_j+1 for j = J .. 1, without c_2 I in Q_1; each Q_j's planes go
            // beside a copy of Z2's, so that both operands of a product lie in its pair
            const int J = (M - 1) / 2;
            auto lead_only = [&](int jj) { return !CHECK && !F32 && jj >= 1 && ((a.ps_levels >> (2 * jj)) & 3) == 0; };
            Tile q;
            for (int jj = J; jj >= 1; --jj) {
                const float cd = jj > 1 ? a.zc[2 * jj] * S : 0.f, cz = a.zc[2 * jj + 1], cl = jj == 1 ? a.zw : 0.f;
#pragma unroll
                for (int n = 0; n < TN; ++n)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float br = jj < J ? acc.re[n][v] * inv : 0.f;
                        const float bi = jj < J ? acc.im[n][v] * inv : 0.f;
                        q.re[n][v] = __builtin_fmaf(cl, z.re[n][v], __builtin_fmaf(cz, z.re[n][v], br + (dg[n][v] ? cd : 0.f)));
                        q.im[n][v] = __builtin_fmaf(cl, z.im[n][v], __builtin_fmaf(cz, z.im[n][v], bi));
                    }
                if (lead_only(jj - 1)) {
                    put(z2, 0, lead);
                    put(q, 1, lead);
                } else {
                    put(z2, 0, full);
                    put(q, 1, full);
                }
                if (jj == J) publish();
                else __syncthreads();
                if (lead_only(jj - 1)) product(0, 1, acc, lead);
                else product(0, 1, acc, full);
            }
            const float q2 = a.zc[2];
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    rest.re[n][v] = __builtin_fmaf(q2, z2.re[n][v], __builtin_fmaf(0.5f, z2.re[n][v], acc.re[n][v] * inv));
                    rest.im[n][v] = __builtin_fmaf(q2, z2.im[n][v], __builtin_fmaf(0.5f, z2.im[n][v], acc.im[n][v] * inv));
                }
        }
        coef_ready = pre;
        // E = c_0' I + Z + (c_1 - 1) Z + rest, Z = z + zl: what is added to z is below z in size, and the
        // sum is rounded once
        const float e0 = a.zc[0] * S, e1 = a.zc[1];
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float lr = zl.re[n][v] + (dg[n][v] ? e0 : 0.f), li = zl.im[n][v];
                e.re[n][v] = z.re[n][v] + (rest.re[n][v] + __builtin_fmaf(e1, z.re[n][v], lr));
                e.im[n][v] = z.im[n][v] + (rest.im[n][v] + __builtin_fmaf(e1, z.im[n][v], li));
            }
    };

    // A := A + B + A B for the later node A and the earlier node B (in place; both held scaled by S)
    auto combine = [&](Tile& A, const Tile& B) __attribute__((always_inline)) {
        put(A, 0, full);
        put(B, 1, full);
        __syncthreads();
        Tile acc;
        product(0, 1, acc, full);
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                A.re[n][v] = __builtin_fmaf(acc.re[n][v], inv, A.re[n][v] + B.re[n][v]);
                A.im[n][v] = __builtin_fmaf(acc.im[n][v], inv, A.im[n][v] + B.im[n][v]);
            }
    };

    Tile pend[F > 0 ? F : 1];
#pragma unroll 1
    for (int p = 0; p < NB; ++p) {
        const int j = w * NB + p;
        Tile e;
        if (j < a.N) {   // uniform
            slice(j, p + 1 < NB ? j + 1 : -1, e);
        } else {
#pragma unroll
            for (int n = 0; n < TN; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) { e.re[n][v] = 0.f; e.im[n][v] = 0.f; }
        }
        bool carry = true;
#pragma unroll
        for (int l = 0; l < F; ++l) {
            if (carry) {
                if ((p >> l) & 1) {
                    combine(e, pend[l]);
                } else {
                    pend[l] = e;
                    carry = false;
                }
            }
        }
        if (carry) {   // p = 2^F - 1: e is the block's node
            if constexpr (CHECK) {
                bool lost = false;
#pragma unroll
                for (int n = 0; n < TN; ++n)
#pragma unroll
                    for (int v = 0; v < 4; ++v) lost |= !(fabsf(e.re[n][v]) + fabsf(e.im[n][v]) < INFINITY);
                if (__syncthreads_or(lost)) return false;
            }
            float2* out = a.out + (size_t)w * dd;
#pragma unroll
            for (int n = 0; n < TN; ++n) {
                const int i = hrow(row0, 0), k = hcol(col0, n);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (i + v < d && k < d)
                        out[(i + v) * d + k] = make_float2(e.re[n][v] * inv, e.im[n][v] * inv);
            }
        }
    }
    return true;
}

template <int D, int F, int FULL, int SCHEME>
__global__ __launch_bounds__(64 * HShape<D>::G, 2) void cheb_h2_kernel(MixedArgs a) {
    // plane sets 0, 1 (one pair) and 2, 3 (the other)
    __shared__ __attribute__((aligned(16))) _Float16 planes[16 * HShape<D>::PL];
    __shared__ double2 coef[kMaxCoeffs];
    int cur = 0;
    h2_node<D, F, FULL, SCHEME>(a, planes, coef, cur, (int)blockIdx.x);
}

// Nodes of many problems (an ensemble's dim class): task (i, w) is node w of inst[i], whose arguments stay
// in memory and are read as scalars.  A node whose values leave fp16's range is formed again in FP32 products; those on
// leading parts only, which rest on controls of modulus 1, are not used.  16 systems of dims 33-64 with
// 1,000-4,000 slices take 1.41 ms with it against 2.42 ms on the FP32 slice kernel and its two lowest tree levels.
template <int D, int F, int FULL, int SCHEME>
__global__ __launch_bounds__(64 * HShape<D>::G, 2) void ens_h2_kernel(const MixedArgs* __restrict__ inst,
                                                                     const int2* __restrict__ tasks, int ntasks) {
    __shared__ __attribute__((aligned(16))) _Float16 planes[16 * HShape<D>::PL];
    __shared__ double2 coef[kMaxCoeffs];
    int cur = 0;
    for (int t = blockIdx.x; t < ntasks; t += gridDim.x) {
        const int2 tk = tasks[t];
        if (!h2_node<D, F, FULL, SCHEME, true>(inst[tk.x], planes, coef, cur, tk.y))
            h2_node<D, F, FULL, SCHEME, false, true>(inst[tk.x], planes, coef, cur, tk.y);
    }
}

__global__ __launch_bounds__(256) void pad_kernel(const double2* __restrict__ in, int count, int d, int D,
                                                  double2* __restrict__ out) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x, DD = (long)D * D;
    if (e >= count * DD) return;
    const long t = e / DD, i = (e % DD) / D, k = e % D;
    out[e] = (i < d && k < d) ? in[(t * d + i) * d + k] : mk<double>(0, 0);
}

// count d x d matrices -> h2_padded_dim(d)^2 each, zeros outside
hipError_t launch_pad(const double2* in, int count, int d, double2* out, hipStream_t st) {
    const int D = h2_padded_dim(d);
    const long total = (long)count * D * D;
    hipLaunchKernelGGL(pad_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, in, count, d, D, out);
    return hipGetLastError();
}

// fp16 two-way split form of the mixed slice kernel (tau Hnorm' <= 1); full = 3 or 4 products per
// FP32-accurate product.
hipError_t launch_cheb_h2(const MixedArgs& a, int full, hipStream_t st) {
    if (a.d <= 0 || a.d > 64 || a.N <= 0 || a.M < 3 || a.M >= kMaxCheb || a.ncoef > kMaxCoeffs || !a.ps ||
        (full != 3 && full != 4) || (a.scheme != 0 && a.scheme != 8))
        return hipErrorInvalidValue;
    const int F = mixed_fused_levels(a.N);
    const int grid = (a.N + (1 << F) - 1) >> F;
    auto go = [&](auto kern, int g) { hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * g), 0, st, a); };
#define PA_H2_GO(DD, FL, SC)                                                         \
    switch (F) {                                                                     \
        case 3: go(cheb_h2_kernel<DD, 3, FL, SC>, HShape<DD>::G); break;             \
        case 2: go(cheb_h2_kernel<DD, 2, FL, SC>, HShape<DD>::G); break;             \
        case 1: go(cheb_h2_kernel<DD, 1, FL, SC>, HShape<DD>::G); break;             \
        default: go(cheb_h2_kernel<DD, 0, FL, SC>, HShape<DD>::G); break;            \
    }
#define PA_H2_D(DD)                                                                  \
    if (a.scheme == 8) { if (full == 3) { PA_H2_GO(DD, 3, 8) } else { PA_H2_GO(DD, 4, 8) } } \
    else { if (full == 3) { PA_H2_GO(DD, 3, 0) } else { PA_H2_GO(DD, 4, 0) } }
    if (a.d <= 32) { PA_H2_D(32) } else { PA_H2_D(64) }
#undef PA_H2_D
#undef PA_H2_GO
    return hipGetLastError();
}

// ntasks nodes of 2^F slices each of problems of dims up to D (32 or 64), all of one scheme
hipError_t launch_ens_h2(int D, int F, int full, int scheme, const MixedArgs* inst, const int2* tasks, int ntasks,
                         hipStream_t st) {
    if ((D != 32 && D != 64) || F < 0 || F > 3 || (full != 3 && full != 4) || (scheme != 0 && scheme != 8))
        return hipErrorInvalidValue;
    if (ntasks <= 0) return hipSuccess;
    auto go = [&](auto kern, int g) { hipLaunchKernelGGL(kern, dim3(ntasks), dim3(64 * g), 0, st, inst, tasks, ntasks); };
#define PA_H2_GO(DD, FL, SC)                                                         \
    switch (F) {                                                                     \
        case 3: go(ens_h2_kernel<DD, 3, FL, SC>, HShape<DD>::G); break;              \
        case 2: go(ens_h2_kernel<DD, 2, FL, SC>, HShape<DD>::G); break;              \
        case 1: go(ens_h2_kernel<DD, 1, FL, SC>, HShape<DD>::G); break;              \
        default: go(ens_h2_kernel<DD, 0, FL, SC>, HShape<DD>::G); break;             \
    }
#define PA_H2_D(DD)                                                                  \
    if (scheme == 8) { if (full == 3) { PA_H2_GO(DD, 3, 8) } else { PA_H2_GO(DD, 4, 8) } } \
    else { if (full == 3) { PA_H2_GO(DD, 3, 0) } else { PA_H2_GO(DD, 4, 0) } }
    if (D == 32) { PA_H2_D(32) } else { PA_H2_D(64) }
#undef PA_H2_D
#undef PA_H2_GO
    return hipGetLastError();
}

}  // namespace pa
