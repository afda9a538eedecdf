// Slices and the lowest tree levels of dims up to 8, on the 4x4 block matrix-core instructions.
//
// A 16x16 matrix-core tile holds at most two 8x8 slices and computes four times their products' work
// (sixteen times at dims up to 4).  The 4x4 forms have no such padding: v_mfma_f32_4x4x1_16b multiplies
// sixteen 4x4 blocks, four 8x8 (or sixteen 4x4) slices a wave, and v_mfma_f64_4x4x4_4b four blocks, one
// 8x8 (or four 4x4) slices a wave.
//
// A work-group of W waves forms W NS nodes (NS slices side by side per wave), each the product of 2^F
// consecutive slices that the wave runs one after another, and reduces them to one node in LDS; pairing, odd
// carry (zero nodes past N) and deviation form E = U - I are the tree kernels'.  Up to 16 NS slices are a
// single launch.  What bounds it at length is the matrix cores and LDS reads, at 4,096 slices the latency of a
// wave's chain of products.  Against padded 16x16 tiles with a separate tree (per call): a million
// slices of dim 8, M = 3, complex64 711 -> 242 us; of dim 4, M = 5, complex64 567 -> 95 us; of dim 8, M = 5,
// complex128 1951 -> 501 us; 4,096 slices of dim 8, complex128 32.8 -> 19.6 us.
#include "kernels.hpp"

namespace pa {

namespace {

template <class R, int NE> struct TinyTile { R re[NE], im[NE]; };

// Lane layout of NS matrices padded to BD x BD (BD = 4, 8) and their copies in LDS (SL elements each).
template <class R, int BD> struct Tiny;

// Complex64: lane l is column l % 4 of 4x4 block (l / 4), its four elements the block's rows.  In LDS by
// columns: a tile is stored, and the second operand read, in 16-byte pieces; COL spreads the columns over
// the banks.
template <int BD> struct Tiny<float, BD> {
    static constexpr int NB = BD / 4, NS = 16 / (NB * NB), NE = 4;
    static constexpr int COL = BD == 8 ? 10 : 4, SL = BD * COL + (BD == 8 ? 0 : 2);
    typedef TinyTile<float, NE> Tile;
    int q, bi, i, col;
    __device__ __forceinline__ Tiny() {
        const int l = threadIdx.x & 63, b = l >> 2;
        q = b / (NB * NB); bi = (b % (NB * NB)) / NB; i = l & 3; col = 4 * (b % NB) + i;
    }
    __device__ __forceinline__ int row(int e) const { return 4 * bi + e; }
    __device__ __forceinline__ void store(float2* m, const Tile& t) const {
        float4* p = reinterpret_cast<float4*>(m + col * COL + 4 * bi);
        p[0] = make_float4(t.re[0], t.im[0], t.re[1], t.im[1]);
        p[1] = make_float4(t.re[2], t.im[2], t.re[3], t.im[3]);
    }
    __device__ __forceinline__ Tile load(const float2* m) const {
        const float4* p = reinterpret_cast<const float4*>(m + col * COL + 4 * bi);
        const float4 x = p[0], y = p[1];
        return Tile{{x.x, x.z, y.x, y.z}, {x.y, x.w, y.y, y.w}};
    }
    __device__ __forceinline__ Tile mul(const float2* A, const float2* B) const {
        f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
        float2 a[BD], b[BD];
#pragma unroll
        for (int k = 0; k < BD; ++k) a[k] = A[k * COL + 4 * bi + i];
#pragma unroll
        for (int k = 0; k < BD; k += 2) {
            const float4 v = *reinterpret_cast<const float4*>(B + col * COL + k);
            b[k] = make_float2(v.x, v.y); b[k + 1] = make_float2(v.z, v.w);
        }
#pragma unroll
        for (int k = 0; k < BD; ++k) {
            re = __builtin_amdgcn_mfma_f32_4x4x1f32(a[k].x, b[k].x, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f32_4x4x1f32(a[k].x, b[k].y, im, 0, 0, 0);
            re = __builtin_amdgcn_mfma_f32_4x4x1f32(-a[k].y, b[k].y, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f32_4x4x1f32(a[k].y, b[k].x, im, 0, 0, 0);
        }
        return Tile{{re[0], re[1], re[2], re[3]}, {im[0], im[1], im[2], im[3]}};
    }
};

// Complex128: lane l holds element (l / 16, l % 4) of 4x4 block (l / 4) % 4; operands as the first
// operand's element (l % 4, l / 16) and the second's (l / 16, l % 4).  In LDS by rows.
template <int BD> struct Tiny<double, BD> {
    static constexpr int NB = BD / 4, NS = 4 / (NB * NB), NE = 1;
    static constexpr int ROW = BD == 8 ? 9 : 4, SL = BD * ROW + (BD == 8 ? 0 : 1);
    typedef TinyTile<double, NE> Tile;
    int q, bi, i, t, col;
    __device__ __forceinline__ Tiny() {
        const int l = threadIdx.x & 63, b = (l >> 2) & 3;
        q = b / (NB * NB); bi = (b % (NB * NB)) / NB; i = l & 3; t = l >> 4; col = 4 * (b % NB) + i;
    }
    __device__ __forceinline__ int row(int) const { return 4 * bi + t; }
    __device__ __forceinline__ void store(double2* m, const Tile& x) const {
        m[row(0) * ROW + col] = mk<double>(x.re[0], x.im[0]);
    }
    __device__ __forceinline__ Tile load(const double2* m) const {
        const double2 v = m[row(0) * ROW + col];
        return Tile{{v.x}, {v.y}};
    }
    __device__ __forceinline__ Tile mul(const double2* A, const double2* B) const {
        double re = 0.0, im = 0.0;
        double2 a[NB], b[NB];
#pragma unroll
        for (int s = 0; s < NB; ++s) {
            a[s] = A[(4 * bi + i) * ROW + 4 * s + t];
            b[s] = B[(4 * s + t) * ROW + col];
        }
#pragma unroll
        for (int s = 0; s < NB; ++s) {
            re = __builtin_amdgcn_mfma_f64_4x4x4f64(a[s].x, b[s].x, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f64_4x4x4f64(a[s].x, b[s].y, im, 0, 0, 0);
            re = __builtin_amdgcn_mfma_f64_4x4x4f64(-a[s].y, b[s].y, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f64_4x4x4f64(a[s].y, b[s].x, im, 0, 0, 0);
        }
        return Tile{{re}, {im}};
    }
};

// Orders a wave's own LDS stores before its later loads (the LDS serves a wave's accesses in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

constexpr int kTinyFold = 5;   // most tree levels a wave folds one slice after another

// NC: operators after H0 held in registers for the launch (0: any number, from LDS, with each coefficient
// evaluated by one lane and handed to its slice's lanes through LDS; evaluated by every lane, 64 of them took 87 us at
// 4,096 slices of dim 5, complex128, and 47 so).  SCHEME 0: the
// recurrence; 8, 12: poly_slice_tile's schemes (complex128).
template <class R, int BD, int NC, int SCHEME>
__global__ __launch_bounds__(1024) void tiny_kernel(ChebArgs<R> a, int F, int final_level) {
    typedef Tiny<R, BD> T;
    typedef typename T::Tile Tile;
    typedef cplx<R> C;
    constexpr int NE = T::NE, NS = T::NS, SL = T::SL;
    extern __shared__ __attribute__((aligned(16))) unsigned char tiny_lds[];
    C* lds = reinterpret_cast<C*>(tiny_lds);
    const T L;
    const int W = blockDim.x >> 6, wave = threadIdx.x >> 6, d = a.d, dd = d * d;
    // per wave: NS matrices as first operands, NS as second ones; then (NC = 0) the operators and, per wave, 64
    // coefficients
    C* const s0 = lds + (size_t)wave * 2 * NS * SL + L.q * SL;
    C* const s1 = s0 + NS * SL;
    C* const ops = lds + (size_t)W * 2 * NS * SL;
    bool in[NE], dg[NE];
    int at[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        in[e] = L.row(e) < d && L.col < d;
        dg[e] = L.row(e) == L.col;
        at[e] = in[e] ? L.row(e) * d + L.col : 0;
    }
    C h0[NE], hk[NC > 0 ? NC : 1][NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        h0[e] = in[e] ? a.ops[at[e]] : mk<R>(0, 0);
#pragma unroll
        for (int t = 0; t < NC; ++t) hk[t][e] = in[e] ? a.ops[(t + 1) * dd + at[e]] : mk<R>(0, 0);
    }
    if constexpr (NC == 0) {
        for (int e = threadIdx.x; e < a.ncoef * dd; e += blockDim.x) ops[e] = a.ops[dd + e];
        __syncthreads();
    }
    const int nd = (blockIdx.x * W + wave) * NS + L.q;   // this lane's node
    const long j0 = (long)nd << F;
    auto each = [&](auto f) {
#pragma unroll
        for (int e = 0; e < NE; ++e) f(e);
    };
    auto product = [&](const Tile& x, const Tile& y) {
        wave_order();
        L.store(s0, x);
        L.store(s1, y);
        wave_order();
        return L.mul(s0, s1);
    };
    C next[NC > 0 ? NC : 1];
    auto prefetch = [&](long j) {
#pragma unroll
        for (int t = 0; t < NC; ++t)
            next[t] = j < a.N ? slice_coefficient(a.ctl, t, a.j0 + (int)j) : mk<R>(0, 0);
    };
    prefetch(j0);
    // NC = 0: lane l evaluates coefficients PER r + l % PER, r = 0, 1, .., of the wave's node l / PER
    constexpr int PER = 64 / NS;
    const int lane = threadIdx.x & 63, mine = lane % PER;
    const long jm = (long)((blockIdx.x * W + wave) * NS + lane / PER) << F;
    const int live = (int)min(max(a.N - jm, 0l), 1l << F);   // slices of that node
    C* const cf = ops + a.ncoef * dd + wave * 64;
    auto evaluate = [&](int t, int p) {
        return t < a.ncoef && p < live ? slice_coefficient(a.ctl, t, a.j0 + (int)jm + p) : mk<R>(0, 0);
    };
    C ahead = mk<R>(0, 0);
    if constexpr (NC == 0) ahead = evaluate(mine, 0);
    Tile pend[kTinyFold], e;
#pragma unroll 1
    for (int p = 0; p < (1 << F); ++p) {
        const long j = j0 + p;
        C x[NE];
        each([&](int k) { x[k] = h0[k]; });
        if constexpr (NC > 0) {
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const C c = next[t];
                each([&](int k) { x[k] = cadd(x[k], cmul(c, hk[t][k])); });
            }
            if (p + 1 < (1 << F)) prefetch(j + 1);
        } else {
            for (int t0 = 0; t0 < a.ncoef; t0 += PER) {
                wave_order();
                cf[lane] = ahead;
                wave_order();
                const bool more = t0 + PER < a.ncoef;
                ahead = evaluate(more ? t0 + PER + mine : mine, more ? p : p + 1);
                const int cnt = min(PER, a.ncoef - t0);
                for (int t = 0; t < cnt; ++t) {
                    const C c = cf[L.q * PER + t];
                    each([&](int k) {
                        if (in[k]) x[k] = cadd(x[k], cmul(c, ops[(t0 + t) * dd + at[k]]));
                    });
                }
            }
        }
        if constexpr (SCHEME == 0) {
            // b_M = a_M I, b_{M-1} = s a_M X + a_{M-1} I; b_k = s X b_{k+1} - b_{k+2} + a_k I; E = s X b_1 - 2 b_2
            // + (a_0 - 1) I
            Tile X, b1, b2;
            const C saM = mk<R>(a.s * a.are[a.M], a.s * a.aim[a.M]);
            each([&](int k) {
                X.re[k] = x[k].x; X.im[k] = x[k].y;
                b2.re[k] = dg[k] ? a.are[a.M] : R(0); b2.im[k] = dg[k] ? a.aim[a.M] : R(0);
                const C y = cmul(saM, x[k]);
                b1.re[k] = y.x + (dg[k] ? a.are[a.M - 1] : R(0));
                b1.im[k] = y.y + (dg[k] ? a.aim[a.M - 1] : R(0));
            });
            wave_order();
            L.store(s0, X);
            for (int m = a.M - 2; m >= 0; --m) {
                wave_order();
                L.store(s1, b1);
                wave_order();
                const Tile acc = L.mul(s0, s1);
                const R beta = m == 0 ? R(-2) : R(-1), ar = a.are[m], ai = a.aim[m];
                each([&](int k) {
                    const R nr = a.s * acc.re[k] + beta * b2.re[k] + (dg[k] ? ar : R(0));
                    const R ni = a.s * acc.im[k] + beta * b2.im[k] + (dg[k] ? ai : R(0));
                    b2.re[k] = b1.re[k]; b2.im[k] = b1.im[k];
                    b1.re[k] = nr; b1.im[k] = ni;
                });
            }
            e = b1;
        } else {
            const R* q = a.pc;
            const R tau = a.ctl.tau;
            Tile z, z2, y, u;
            each([&](int k) { z.re[k] = tau * x[k].y; z.im[k] = -tau * x[k].x; });
            z2 = product(z, z);
            if constexpr (SCHEME == 8) {
                each([&](int k) { y.re[k] = z.re[k] + q[3] * z2.re[k]; y.im[k] = z.im[k] + q[3] * z2.im[k]; });
                const Tile P = product(z2, y);
                each([&](int k) {
                    u.re[k] = z2.re[k] + q[4] * P.re[k]; u.im[k] = z2.im[k] + q[4] * P.im[k];
                    y.re[k] = z.re[k] + q[5] * z2.re[k] + q[6] * P.re[k];
                    y.im[k] = z.im[k] + q[5] * z2.im[k] + q[6] * P.im[k];
                    e.re[k] = q[7] * P.re[k] + q[2] * z2.re[k] + q[1] * z.re[k] + (dg[k] ? q[0] : R(0));
                    e.im[k] = q[7] * P.im[k] + q[2] * z2.im[k] + q[1] * z.im[k];
                });
                const Tile acc = product(u, y);
                each([&](int k) { e.re[k] += q[8] * acc.re[k]; e.im[k] += q[8] * acc.im[k]; });
            } else {
                const Tile z3 = product(z, z2);
                each([&](int k) {
                    y.re[k] = z.re[k] + q[4] * z2.re[k] + q[5] * z3.re[k];
                    y.im[k] = z.im[k] + q[4] * z2.im[k] + q[5] * z3.im[k];
                });
                const Tile P = product(y, y);
                each([&](int k) {
                    u.re[k] = P.re[k] + q[6] * z.re[k] + q[7] * z2.re[k] + q[8] * z3.re[k];
                    u.im[k] = P.im[k] + q[6] * z.im[k] + q[7] * z2.im[k] + q[8] * z3.im[k];
                    y.re[k] = z.re[k] + q[9] * z2.re[k] + q[10] * z3.re[k] + q[11] * P.re[k];
                    y.im[k] = z.im[k] + q[9] * z2.im[k] + q[10] * z3.im[k] + q[11] * P.im[k];
                    e.re[k] = q[12] * P.re[k] + q[3] * z3.re[k] + q[2] * z2.re[k] + q[1] * z.re[k] + (dg[k] ? q[0] : R(0));
                    e.im[k] = q[12] * P.im[k] + q[3] * z3.im[k] + q[2] * z2.im[k] + q[1] * z.im[k];
                });
                const Tile acc = product(u, y);
                each([&](int k) { e.re[k] += q[13] * acc.re[k]; e.im[k] += q[13] * acc.im[k]; });
            }
        }
        each([&](int k) {
            if (j >= a.N || !in[k]) { e.re[k] = R(0); e.im[k] = R(0); }
        });
        // binary counter over the levels (unrolled: every pending node in fixed registers)
        bool carry = true;
#pragma unroll
        for (int l = 0; l < kTinyFold; ++l) {
            if (carry && l < F) {
                if ((p >> l) & 1) {
                    const Tile acc = product(e, pend[l]);
                    each([&](int k) {
                        e.re[k] = acc.re[k] + (e.re[k] + pend[l].re[k]);
                        e.im[k] = acc.im[k] + (e.im[k] + pend[l].im[k]);
                    });
                } else {
                    pend[l] = e;
                    carry = false;
                }
            }
        }
    }
    // the work-group's W NS nodes: node i of a level at first-operand place i 2^level
    wave_order();
    L.store(s0, e);
    __syncthreads();
    const int n = W * NS;
    auto place = [&](int i) { return lds + (size_t)(i / NS) * 2 * NS * SL + (i % NS) * SL; };
    for (int lev = 0; (1 << lev) < n; ++lev) {
        const int cnt = n >> (lev + 1);
        if (wave * NS < cnt) {   // uniform
            const int t = min(wave * NS + L.q, cnt - 1);
            const C* A = place((2 * t + 1) << lev);
            C* B = place((2 * t) << lev);
            const Tile x = L.load(A), y = L.load(B), acc = L.mul(A, B);
            each([&](int k) {
                e.re[k] = acc.re[k] + (x.re[k] + y.re[k]);
                e.im[k] = acc.im[k] + (x.im[k] + y.im[k]);
            });
            wave_order();
            if (wave * NS + L.q < cnt) L.store(B, e);
        }
        __syncthreads();
    }
    if (wave == 0 && L.q == 0) {
        C* out = a.out + (size_t)blockIdx.x * dd;
        each([&](int k) {
            if (in[k]) out[at[k]] = mk<R>(e.re[k] + (final_level && dg[k] ? R(1) : R(0)), e.im[k]);
        });
    }
}

template <class R> constexpr int tiny_slices(int d) {   // slices per wave
    return sizeof(R) == 4 ? (d <= 4 ? 16 : 4) : (d <= 4 ? 4 : 1);
}

struct TinyPlan { int waves, fold, nodes; };
// Work-groups of 16 waves (fewer when one work-group holds all slices).  Folding a level halves the
// nodes left for the tree launches and doubles a wave's serial work: none while at most 64 nodes are left (one
// further launch), then as many as keep 512 work-groups.
template <class R> TinyPlan tiny_plan(int N, int d) {
    const int ns = tiny_slices<R>(d);
    TinyPlan p{16, 0, 1};
    if (N <= 16 * ns) {
        p.waves = 1;
        while (p.waves * ns < N) p.waves *= 2;
        return p;
    }
    auto groups = [&](int f) { return (int)(((long)N + ((long)16 * ns << f) - 1) / ((long)16 * ns << f)); };
    while (p.fold < 2 && groups(p.fold) > 64) ++p.fold;
    if (groups(p.fold) > 64) {
        p.fold = 0;
        while (p.fold < kTinyFold && groups(p.fold) > 512) ++p.fold;
    }
    p.nodes = groups(p.fold);
    return p;
}

}  // namespace

bool tiny_supported(int d, int ncoef) { return d >= 1 && d <= 8 && ncoef >= 1 && ncoef <= 64; }

template <class R> int tiny_nodes(int N, int d) { return tiny_plan<R>(N, d).nodes; }
template int tiny_nodes<float>(int, int);
template int tiny_nodes<double>(int, int);

template <class R> hipError_t launch_tiny(const ChebArgs<R>& a, hipStream_t st) {
    if (!tiny_supported(a.d, a.ncoef) || a.N <= 0 || a.M < 3 || a.M >= kMaxCheb || (a.pdeg && a.pdeg != 8 && a.pdeg != 12) ||
        (sizeof(R) == 4 && a.pdeg))
        return hipErrorInvalidValue;
    const TinyPlan p = tiny_plan<R>(a.N, a.d);
    const int nc = a.ncoef <= 3 ? a.ncoef : 0;
    auto go = [&](auto kern, int ns, int sl) {
        const size_t lds = ((size_t)p.waves * 2 * ns * sl + (nc ? 0 : (size_t)a.ncoef * a.d * a.d + 64 * p.waves)) * sizeof(cplx<R>);
        hipLaunchKernelGGL(kern, dim3(p.nodes), dim3(64 * p.waves), lds, st, a, p.fold, p.nodes == 1 ? 1 : 0);
    };
#define PA_TINY(BD, SC)                                                                     \
    {                                                                                       \
        constexpr int NS = Tiny<R, BD>::NS, SL = Tiny<R, BD>::SL;                           \
        switch (nc) {                                                                       \
            case 1: go(tiny_kernel<R, BD, 1, SC>, NS, SL); break;                           \
            case 2: go(tiny_kernel<R, BD, 2, SC>, NS, SL); break;                           \
            case 3: go(tiny_kernel<R, BD, 3, SC>, NS, SL); break;                           \
            default: go(tiny_kernel<R, BD, 0, SC>, NS, SL); break;                          \
        }                                                                                   \
    }
    if constexpr (sizeof(R) == 8) {
        if (a.pdeg == 8) { if (a.d <= 4) PA_TINY(4, 8) else PA_TINY(8, 8) return hipGetLastError(); }
        if (a.pdeg == 12) { if (a.d <= 4) PA_TINY(4, 12) else PA_TINY(8, 12) return hipGetLastError(); }
    }
    if (a.d <= 4) PA_TINY(4, 0) else PA_TINY(8, 0)
#undef PA_TINY
    return hipGetLastError();
}
template hipError_t launch_tiny<float>(const ChebArgs<float>&, hipStream_t);
template hipError_t launch_tiny<double>(const ChebArgs<double>&, hipStream_t);

}  // namespace pa
