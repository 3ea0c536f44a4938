// Workgroup FFTs with every size known at compile time, for kernels that the
// library compiles at run time (hipRTC) for the transform lengths of a handle
// that the register kernels do not cover: lengths with odd factors (2064 = 2^4
// 3 43 for a centre offset at N0 = 2048) and short ones (rows below 256 points,
// columns below 256).
//
// A self-sorting Stockham FFT of NL lines.  Each stage reads its inputs into
// registers, transforms them, and writes them to the next stage's slots of
// the same LDS buffer (the compute sits between the reads and a barrier, so
// one buffer is enough and two to four blocks share a CU).  The first stage
// reads through a caller's functor and the last one writes through another
// one, so loads from HBM, the product with the kernel spectrum and stores to
// HBM cost no LDS pass of their own.
//
// Radices up to 24 without a prime factor above 13 run one butterfly per lane
// in registers (composites as coprime products of small closed forms, without
// twiddles; 7, 11 and 13 by conjugate pairs; larger ones would spill); a length
// costs about the same VALU work per point in each stage whatever its radix, so
// the host picks few stages of large radix.  A prime factor R >= 17 is a
// product with the R x R DFT matrix and runs on the matrix cores
// (mfma_stage): in registers it would cost ~R / 2 fused multiply-adds per
// point plus as many LDS reads of its weights, which bounded these passes
// before (columns of 4128 = 43 96: 4.71 ms per 32 slices).
#pragma once
#include "fft_lds.hpp"

namespace lpct {

template <int... Rs>
struct Radices {};

// cos and sin of 2 pi k / n at compile time: Taylor series of the residual
// angle (|x| <= pi / 4) in double
constexpr double ct_sin(double x) {
    double t = x, s = x;
    for (int i = 1; i < 10; ++i) {
        t *= -x * x / ((2 * i) * (2 * i + 1));
        s += t;
    }
    return s;
}
constexpr double ct_cos(double x) {
    double t = 1, s = 1;
    for (int i = 1; i < 11; ++i) {
        t *= -x * x / ((2 * i - 1) * (2 * i));
        s += t;
    }
    return s;
}
constexpr double ct_turn(int k, int n, bool cosine) {
    k %= n;
    const int qd = (4 * k + n / 2) / n;                                       // nearest quarter turn
    const double x = (4 * k - qd * n) * (1.57079632679489661923 / n);         // the rest of the angle
    switch ((cosine ? qd : qd + 3) & 3) {   // sin a = cos(a - quarter turn)
        case 0: return ct_cos(x);
        case 1: return -ct_sin(x);
        case 2: return -ct_cos(x);
        default: return ct_sin(x);
    }
}
template <int R>
struct Turn {
    float c[R], s[R];
    constexpr Turn() : c(), s() {
        for (int k = 0; k < R; ++k) {
            c[k] = (float)ct_turn(k, R, true);
            s[k] = (float)ct_turn(k, R, false);
        }
    }
};

constexpr int largest_prime(int n) {
    int p = 1;
    for (int q = 2; q <= n; ++q)
        while (n % q == 0) { p = q; n /= q; }
    return p;
}
// the first factor of a composite register radix: coprime to the other one
// unless the radix is a prime power
constexpr int split_of(int R) {
    return R == 9 ? 3 : R % 13 == 0 ? 13 : R % 11 == 0 ? 11 : R % 7 == 0 ? 7 : R % 5 == 0 ? 5 : R % 9 == 0 ? 9
           : R % 8 == 0 ? 8 : R % 4 == 0 ? 4 : R % 3 == 0 ? 3 : 2;
}
// the multiple of B below A B that is 1 mod A (A, B coprime)
constexpr int idempotent(int A, int B) {
    int e = B;
    while (e % A != 1) e += B;
    return e;
}
// a stage on the matrix cores
constexpr bool on_mfma(int R) { return R >= 17 && largest_prime(R) == R; }

// odd prime R by conjugate pairs: y_p = A_p + i B_p, y_{R-p} = A_p - i B_p
template <int R>
__device__ __forceinline__ void dft_odd(float2* v, int dir) {
    constexpr int hR = (R - 1) / 2;
    constexpr Turn<R> w{};
    float2 s[hR], d[hR], sum = v[0];
#pragma unroll
    for (int q = 0; q < hR; ++q) {
        s[q] = cadd(v[q + 1], v[R - 1 - q]);
        d[q] = csub(v[q + 1], v[R - 1 - q]);
        sum = cadd(sum, s[q]);
    }
    const float2 x0 = v[0];
    v[0] = sum;
#pragma unroll
    for (int p = 1; p <= hR; ++p) {
        float2 A = x0, B = make_float2(0.f, 0.f);
#pragma unroll
        for (int q = 1; q <= hR; ++q) {
            const float c = w.c[(p * q) % R], sn = w.s[(p * q) % R];
            A.x = fmaf(s[q - 1].x, c, A.x);
            A.y = fmaf(s[q - 1].y, c, A.y);
            B.x = fmaf(d[q - 1].x, sn, B.x);
            B.y = fmaf(d[q - 1].y, sn, B.y);
        }
        const float2 iB = rot90(B, dir);
        v[p] = cadd(A, iB);
        v[R - p] = csub(A, iB);
    }
}

// length-R DFT in registers, natural order in and out
template <int R>
__device__ __forceinline__ void dft(float2* v, int dir) {
    if constexpr (R == 1) {
    } else if constexpr (R == 2 || R == 3 || R == 4 || R == 5 || R == 8) {
        dft_small<R>(v, dir);
    } else if constexpr (R == 16) {
        dft16(v, dir);
    } else if constexpr (largest_prime(R) == R) {
        dft_odd<R>(v, dir);
    } else {
        constexpr int A = split_of(R), B = R / A;
        float2 a[B][A];
        if constexpr (A % B != 0) {
            // R = A B, coprime: with input B n1 + A n2 and output k1 mod A, k2 mod
            // B it is A-point DFTs over n1 and B-point DFTs over n2, without
            // twiddles (those of 10 and 20, rounded, have mean gains of 5e-9 and
            // 8e-9, which add up over the passes)
            constexpr int eA = idempotent(A, B), eB = idempotent(B, A);
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
                for (int n1 = 0; n1 < A; ++n1) a[n2][n1] = v[(B * n1 + A * n2) % R];
                dft<A>(a[n2], dir);
            }
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) {
                float2 t[B];
#pragma unroll
                for (int n2 = 0; n2 < B; ++n2) t[n2] = a[n2][k1];
                dft<B>(t, dir);
#pragma unroll
                for (int k2 = 0; k2 < B; ++k2) v[(eA * k1 + eB * k2) % R] = t[k2];
            }
        } else {
            // 9 = 3 3: DFTs over elements 3 apart, twiddles, DFTs
            constexpr Turn<R> w{};
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
                for (int n1 = 0; n1 < A; ++n1) a[n2][n1] = v[n1 * B + n2];
                dft<A>(a[n2], dir);
#pragma unroll
                for (int k1 = 1; k1 < A; ++k1)
                    if (n2 > 0) {
                        const float c = w.c[n2 * k1], s = w.s[n2 * k1];
                        a[n2][k1] = cmul(a[n2][k1], make_float2(c, dir < 0 ? -s : s));
                    }
            }
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) {
                float2 t[B];
#pragma unroll
                for (int n2 = 0; n2 < B; ++n2) t[n2] = a[n2][k1];
                dft<B>(t, dir);
#pragma unroll
                for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
            }
        }
    }
}

// Block barrier that waits for this wave's LDS traffic only: loads from and
// stores to HBM keep running across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS slot of element x of a line whose plan starts with radix R0: a first
// radix that is odd spreads its writes (stride R0) over all banks by itself;
// after an even one a pad slot follows every 16 elements.
template <int R0>
__device__ __forceinline__ int slot(int x) {
    return (R0 & 1) ? x : x + (x >> 4);
}
template <int R0>
constexpr int slots(int n) {
    return (R0 & 1) ? n : n + (n >> 4) + 1;
}

// What the last stage does to its outputs: load(x) fetches the operand of
// output x (issued ahead of the butterfly), apply(value, operand).
template <class Load, class Apply>
struct Post {
    static constexpr bool active = true;
    Load load;
    Apply apply;
};
template <class Load, class Apply>
__device__ __forceinline__ Post<Load, Apply> make_post(Load l, Apply a) {
    return Post<Load, Apply>{l, a};
}
struct NoPost {
    static constexpr bool active = false;
};
// Where a stage reads: get(line, x) fetches, fix(line, x, value) is applied
// once the loads of the stage are on their way (masks: a select beside its
// load would wait for it).
template <class Get, class Fix>
struct Source {
    Get get;
    Fix fix;
};
template <class Get, class Fix>
__device__ __forceinline__ Source<Get, Fix> make_source(Get g, Fix f) {
    return Source<Get, Fix>{g, f};
}

// Every load above is issued before anything below: the scheduler otherwise
// sinks each load to its use to save registers and pays its latency there
// (first version of these stages: 70 % of the wave cycles waiting).
__device__ __forceinline__ void issue_loads() { __builtin_amdgcn_sched_barrier(0); }

// The powers w^q, q < R, of a butterfly's twiddle from few table reads: w .. w^m
// and w^b at steps of 2 m + 1 (the last one at R - 1), every other one the product
// of a w^b with w^d or its conjugate, d <= m.  As many reads as for w, w^2, w^4, ..
// up to radix 13 (one more above), whose products of up to four factors round
// worse: with these powers and the twiddle-free radices above, fwd and adj at 38
// lengths from 96 to 2000 are on average 0.94 as far from float64, in the same time.
template <int R>
struct Powers {
    static constexpr int steps(int m) { return R - 1 > m ? (R - 1 - m + 2 * m) / (2 * m + 1) : 0; }
    static constexpr int pick() {
        int m = 1;
        for (int k = 2; k < 4; ++k)
            if (k + steps(k) < m + steps(m)) m = k;
        return m;
    }
    static constexpr int m = pick(), count = R > 1 ? m + steps(m) : 1;
    // nearest power that is read, and the slot of a power that is
    static constexpr int base(int q) { return q <= m ? q : (q + m) / (2 * m + 1) * (2 * m + 1) < R ? (q + m) / (2 * m + 1) * (2 * m + 1) : R - 1; }
    static constexpr int slot(int q) { return q <= m ? q - 1 : m + (q + m) / (2 * m + 1) - 1; }
};

// One register stage of radix R (Ns = product of the radices before it) over
// NL lines of M points: in (a Source) gives the inputs, the post operation on the
// outputs, then a barrier (every read of the block is done), then
// out(line, element, item, output, value) for the block's butterflies; items
// are tid, tid + NT, ...  MID: the barrier is needed (some wave may still
// read what out overwrites).
template <int M, int NL, int NT, int Ns, int R, bool MID, class In, class P, class Out>
__device__ __forceinline__ void reg_stage(In in, P post, Out out, const float2* __restrict__ tw, int dir, int tid) {
    constexpr int nbf = M / R, total = NL * nbf, NI = (total + NT - 1) / NT;
    constexpr int tstep = M / (Ns * R);
    using W = Powers<R>;
    float2 v[NI][R], wl[NI][W::count];
    auto item = [&](int c) { return (c + 1) * NT <= total ? tid + c * NT : min(tid + c * NT, total - 1); };
#pragma unroll
    for (int c = 0; c < NI; ++c) {
        const int t = item(c), b = NL == 1 ? 0 : t / nbf, i = t - b * nbf;
        if (Ns > 1) {
#pragma unroll
            for (int q = 1; q < R; ++q)
                if (W::base(q) == q) wl[c][W::slot(q)] = tw[(i % Ns) * tstep * q];
        }
#pragma unroll
        for (int q = 0; q < R; ++q) v[c][q] = in.get(b, i + q * nbf);
    }
    issue_loads();
#pragma unroll
    for (int c = 0; c < NI; ++c) {
        const int t = item(c), b = NL == 1 ? 0 : t / nbf, i = t - b * nbf, k = Ns == 1 ? 0 : i % Ns;
        float2 g[P::active ? R : 1];
        if constexpr (P::active) {
#pragma unroll
            for (int q = 0; q < R; ++q) g[q] = post.load((i - k) * R + k + q * Ns);
            issue_loads();
        }
#pragma unroll
        for (int q = 0; q < R; ++q) v[c][q] = in.fix(b, i + q * nbf, v[c][q]);
        if (Ns > 1) {
#pragma unroll
            for (int q = 1; q < R; ++q) {
                float2 w = wl[c][W::slot(q)];
                const int d = q - W::base(q);
                if (d != 0) w = d > 0 ? cmul(w, wl[c][d - 1]) : cmul(w, cconj(wl[c][-d - 1]));
                v[c][q] = cmul(v[c][q], dir < 0 ? w : cconj(w));
            }
        }
        dft<R>(v[c], dir);
        if constexpr (P::active) {
#pragma unroll
            for (int q = 0; q < R; ++q) v[c][q] = post.apply(v[c][q], g[q]);
        }
    }
    if (MID) lds_barrier();
#pragma unroll
    for (int c = 0; c < NI; ++c) {
        // lanes past the last butterfly repeat it (same values to the same
        // places): a guard here would draw their loads and arithmetic behind
        // the barrier
        const int t = item(c), b = NL == 1 ? 0 : t / nbf, i = t - b * nbf, k = Ns == 1 ? 0 : i % Ns;
        const int dst = (i - k) * R + k;
#pragma unroll
        for (int q = 0; q < R; ++q) out(b, dst + q * Ns, c, q, v[c][q]);
    }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Tiling of a prime radix R over NT threads: the butterflies of the block
// (columns) in tiles of 16, the outputs p = 0 .. (R-1)/2 in MT tiles of 16,
// the terms q = 0 .. (R-1)/2 in KS steps of 4.  A wave's unit is one column
// tile and MTC output tiles; MTC balances the waves against reading the
// inputs once per unit, with at most 64 accumulators where a choice has that
// few.  KC steps' loads travel together, a chunk ahead of the products, as
// far as REGS registers allow (a spill costs more than any latency: 3.0
// against 2.2 ms for the forward rows of N = 2064).
template <int R, int NBF, int NT, int REGS>
struct Mfma {
    static constexpr int hR = (R - 1) / 2, MT = (hR + 16) / 16, KS = (hR + 4) / 4;
    static constexpr int NTL = (NBF + 15) / 16, NW = NT / 64;
    static constexpr int units(int mtc) { return NTL * ((MT + mtc - 1) / mtc); }
    static constexpr int rounds(int mtc) { return (units(mtc) + NW - 1) / NW; }
    static constexpr int cost(int mtc) {
        return rounds(mtc) * (mtc * 128 + 64) * (mtc * rounds(mtc) > 4 ? 2 : 1);
    }
    static constexpr int pick() {
        int best = 1;
        for (int m = 2; m <= MT && m <= 4; ++m)
            if (cost(m) <= cost(best)) best = m;
        return best;
    }
    static constexpr int MTC = pick(), MCH = (MT + MTC - 1) / MTC, U = units(MTC), JU = rounds(MTC);
    static constexpr int chunk() {
        const int room = REGS - 48 - 16 * JU * MTC, each = 8 + 4 * MTC, most = 2;
        return room / each < 1 ? 1 : room / each < most ? room / each : most;
    }
    static constexpr int KC = chunk(), NCH = (KS + KC - 1) / KC;
    static constexpr int size = MT * KS * 128;   // floats of the weight table
};

// One stage of prime radix R on the matrix cores.  With s_q = x_q + x_{R-q},
// d_q = x_q - x_{R-q} (s_0 = x_0, d_0 = 0) and t = 2 pi p q / R,
//   A_p = sum_q s_q cos t,  B_p = sum_q d_q sin t,  y_p = A_p -+ i B_p,
//   y_{R-p} = A_p +- i B_p   (upper signs forward),
// i.e. four real products (cos, sin) x (re, im) of [p][q] weights with the
// [q][butterfly] inputs: v_mfma_f32_16x16x4_f32, full FP32, each input read
// once per unit and the weights one float per lane and step.  wgt: per
// (output tile, step) 64 cosines then 64 sines in lane order, zero outside
// the matrix (built on the host).  The loads run one chunk of steps ahead of
// the products.
template <int M, int NL, int NT, int REGS, int Ns, int R, bool MID, class In, class Out>
__device__ __forceinline__ void mfma_stage(In in, Out out, const float2* __restrict__ tw,
                                           const float* __restrict__ wgt, int dir, int tid) {
    constexpr int nbf = M / R, total = NL * nbf;
    using T = Mfma<R, total, NT, REGS>;
    constexpr int tstep = M / (Ns * R), ST = T::JU * T::NCH;
    constexpr bool one_w = T::MCH == 1 && T::NCH == 1;   // every unit uses the same weights
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = lane >> 4;
    f32x4 acc[T::JU][T::MTC][4];
    struct Chunk {
        float2 xa[T::KC], xb[T::KC], ta[Ns > 1 ? T::KC : 1], tb[Ns > 1 ? T::KC : 1];
        float wc[T::MTC][T::KC], ws[T::MTC][T::KC];
    } cur, nxt;
    // unit of step st (the last round's spare waves repeat the last unit)
    auto unit = [&](int st) { return min(wave + (st / T::NCH) * T::NW, T::U - 1); };
    auto load_w = [&](int st, Chunk& c) {
        const int m0 = unit(st) / T::NTL * T::MTC;
#pragma unroll
        for (int m = 0; m < T::MTC; ++m)
#pragma unroll
            for (int e = 0; e < T::KC; ++e) {
                // a chunk or tile past the matrix repeats valid weights; its products are not used
                const int ks = min((st % T::NCH) * T::KC + e, T::KS - 1);
                const float* w = wgt + ((size_t)min(m0 + m, T::MT - 1) * T::KS + ks) * 128 + lane;
                c.wc[m][e] = w[0];
                c.ws[m][e] = w[64];
            }
    };
    // term q of step ks in this lane, and R - q.  Terms past (R-1)/2 meet zero
    // weights: any valid element will do
    auto term = [&](int ks) { return ks * 4 + 3 > T::hR ? min(ks * 4 + kg, T::hR) : ks * 4 + kg; };
    auto mirror = [&](int ks, int q) { return ks == 0 && q == 0 ? 0 : R - q; };
    auto load_x = [&](int st, Chunk& c) {
        const int t = min((unit(st) % T::NTL) * 16 + (lane & 15), total - 1);
        const int b = NL == 1 ? 0 : t / nbf, i = t - b * nbf, k = Ns == 1 ? 0 : i % Ns;
#pragma unroll
        for (int e = 0; e < T::KC; ++e) {
            const int ks = (st % T::NCH) * T::KC + e, q = term(ks), qc = mirror(ks, q);
            c.xa[e] = in.get(b, i + q * nbf);
            c.xb[e] = in.get(b, i + qc * nbf);
            if (Ns > 1) {
                c.ta[e] = tw[q * k * tstep];
                c.tb[e] = tw[qc * k * tstep];
            }
        }
    };
    load_w(0, cur);
    load_x(0, cur);
#pragma unroll
    for (int st = 0; st < ST; ++st) {
        const int j = st / T::NCH, ch = st % T::NCH;
        if (st + 1 < ST) {
            if (!one_w) load_w(st + 1, nxt);
            load_x(st + 1, nxt);
        }
        issue_loads();
        const int t = min((unit(st) % T::NTL) * 16 + (lane & 15), total - 1);
        const int b = NL == 1 ? 0 : t / nbf, i = t - b * nbf;
        if (ch == 0) {
#pragma unroll
            for (int m = 0; m < T::MTC; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[j][m][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int e = 0; e < T::KC; ++e) {
            if (ch * T::KC + e >= T::KS) break;
            const int q = term(ch * T::KC + e), qc = mirror(ch * T::KC + e, q);
            float2 xa = in.fix(b, i + q * nbf, cur.xa[e]), xb = in.fix(b, i + qc * nbf, cur.xb[e]);
            if (Ns > 1) {
                xa = cmul(xa, dir < 0 ? cur.ta[e] : cconj(cur.ta[e]));
                xb = cmul(xb, dir < 0 ? cur.tb[e] : cconj(cur.tb[e]));
            }
            const float2 d = csub(xa, xb);
            float2 s = cadd(xa, xb);
            // q = 0: s = x_0 (its cosine weight is 1, its sine weight 0)
            if (ch * T::KC + e == 0 && kg == 0) s = xa;
#pragma unroll
            for (int m = 0; m < T::MTC; ++m) {
                acc[j][m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.wc[m][e], s.x, acc[j][m][0], 0, 0, 0);
                acc[j][m][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.wc[m][e], s.y, acc[j][m][1], 0, 0, 0);
                acc[j][m][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.ws[m][e], d.x, acc[j][m][2], 0, 0, 0);
                acc[j][m][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.ws[m][e], d.y, acc[j][m][3], 0, 0, 0);
            }
        }
        if (st + 1 < ST) {
#pragma unroll
            for (int e = 0; e < T::KC; ++e) {
                cur.xa[e] = nxt.xa[e];
                cur.xb[e] = nxt.xb[e];
                if (Ns > 1) {
                    cur.ta[e] = nxt.ta[e];
                    cur.tb[e] = nxt.tb[e];
                }
#pragma unroll
                for (int m = 0; m < T::MTC; ++m)
                    if (!one_w) {
                        cur.wc[m][e] = nxt.wc[m][e];
                        cur.ws[m][e] = nxt.ws[m][e];
                    }
            }
        }
    }
    if (MID) lds_barrier();
    const float sg = dir < 0 ? 1.f : -1.f;
#pragma unroll
    for (int j = 0; j < T::JU; ++j) {
        const int u = unit(j * T::NCH), m0 = (u / T::NTL) * T::MTC;
        const int t = min((u % T::NTL) * 16 + (lane & 15), total - 1);
        const int b = NL == 1 ? 0 : t / nbf, i = t - b * nbf;
        const int k = Ns == 1 ? 0 : i % Ns;
        const int dst = (i - k) * R + k;
#pragma unroll
        for (int m = 0; m < T::MTC; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // lane group kg holds outputs 4 kg .. 4 kg + 3 of the tile
                const int p = (m0 + m) * 16 + kg * 4 + e;
                if (p > T::hR) continue;
                const float2 A = make_float2(acc[j][m][0][e], acc[j][m][1][e]);
                const float2 iB = make_float2(sg * acc[j][m][3][e], -sg * acc[j][m][2][e]);
                out(b, dst + p * Ns, 0, 0, cadd(A, iB));
                // (p = 0: B is zero, the same value again)
                out(b, dst + (p == 0 ? 0 : R - p) * Ns, 0, 0, csub(A, iB));
            }
    }
}

// The stages of a plan: the first reads through `first`, the last writes
// through `last`, the others use buf (line stride LS slots).  Before the last
// stage's `last` runs every lane has passed a barrier behind its reads when
// MIDL is set (last writes to buf); a first stage that reads from HBM and a
// stage that reads buf are both followed by a barrier before buf is written.
template <int M, int NL, int LS, int NT, int REGS, int R0, int Ns, bool FIRST, bool MIDL, class First, class P, class Last, int R,
          int... Rest>
__device__ __forceinline__ void run(float2* buf, First first, P post, Last last, const float2* __restrict__ tw,
                                    const float* __restrict__ wgt, int dir, int tid, Radices<R, Rest...>) {
    constexpr bool end = sizeof...(Rest) == 0;
    auto in = make_source(
        [&](int b, int x) {
            if constexpr (FIRST) return first.get(b, x);
            else return buf[b * LS + slot<R0>(x)];
        },
        [&](int b, int x, float2 v) {
            if constexpr (FIRST) return first.fix(b, x, v);
            else return v;
        });
    auto out = [&](int b, int x, int c, int q, float2 v) {
        if constexpr (end) last(b, x, c, q, v);
        else buf[b * LS + slot<R0>(x)] = v;
    };
    constexpr bool MID = !end || MIDL;
    if constexpr (on_mfma(R)) {
        static_assert(!end, "a register stage comes last");
        mfma_stage<M, NL, NT, REGS, Ns, R, MID>(in, out, tw, wgt, dir, tid);
        wgt += Mfma<R, 1, 64, 128>::size;
    } else {
        if constexpr (end) reg_stage<M, NL, NT, Ns, R, MID>(in, post, out, tw, dir, tid);
        else reg_stage<M, NL, NT, Ns, R, MID>(in, NoPost{}, out, tw, dir, tid);
    }
    if constexpr (!end) {
        lds_barrier();
        run<M, NL, LS, NT, REGS, R0, Ns * R, false, MIDL>(buf, first, post, last, tw, wgt, dir, tid, Radices<Rest...>{});
    }
}

// FFT of NL lines of M points (dir = -1 forward, +1 inverse, unnormalised).
// first (a Source) gives the input (from HBM, or from buf: every read of buf
// happens before the first write).  post (Post or NoPost) is applied to the
// outputs ahead of the last barrier;
// last(line, x, item, output, value) takes the result; (item, output)
// enumerate a thread's outputs; REGS: registers per lane.  Ends without a barrier behind `last`.
template <int M, int NL, int LS, int NT, int REGS, bool MIDL, class First, class P, class Last, int R0, int... Rest>
__device__ __forceinline__ void fft(float2* buf, First first, P post, Last last, const float2* __restrict__ tw,
                                    const float* __restrict__ wgt, int dir, int tid, Radices<R0, Rest...> r) {
    run<M, NL, LS, NT, REGS, R0, 1, true, MIDL>(buf, first, post, last, tw, wgt, dir, tid, r);
}

}  // namespace lpct
