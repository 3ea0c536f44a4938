// Row and column passes of the log-polar convolution, and the filtered
// sinogram rows, with every size a compile-time constant, instantiated at run
// time (hipRTC) for the lengths of a handle that the radix-16 register
// kernels do not cover.  Same data layout as k_rows_fwd, k_cols, k_rows_inv
// and k_sino_rows_pair of kernels.hip; the FFTs are those of fft_ct.hpp: the
// first stage of each reads its input (from HBM in the forward transforms),
// the last one applies the kernel spectrum or stores to HBM.
//
// Grids are one-dimensional and XCD-aware: neighbouring row blocks share the
// 128-byte lines of the transposed half spectra, the slice groups and spans
// of one column its kernel spectrum, so each run behind one L2.
#pragma once
#include "kernels.hpp"
#include "fft_ct.hpp"

namespace lpct {

template <class T>
__device__ __forceinline__ T ld_at(const T* base, unsigned off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}
template <class T>
__device__ __forceinline__ void st_at(T* base, unsigned off, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off) = v;
}

// logical index of hardware block b of n: each of the 8 XCDs (b mod 8) takes
// a contiguous range
__device__ __forceinline__ int xcd_block(int b, int n) {
    const int q = n / 8, r = n - q * 8, x = b % 8;
    return x * q + min(x, r) + b / 8;
}

__device__ __forceinline__ float2 fzval(const float2* __restrict__ fz, int i, int conj) {
    float2 v = fz[i];
    return conj ? make_float2(v.x, -v.y) : v;
}

// An opaque zero, produced inside a loop: index arithmetic and table reads
// that depend on it are redone per pass of the loop instead of being held in
// registers across it.
__device__ __forceinline__ int opaque_zero() {
    int z;
    asm volatile("s_mov_b32 %0, 0" : "=s"(z));
    return z;
}

template <int... Rs>
struct Plan;
template <int R0, int... Rest>
struct Plan<R0, Rest...> {
    static constexpr int first = R0;
    static constexpr int last = [] {
        int r = R0;
        ((r = Rest), ...);
        return r;
    }();
};

// Column pass (k_cols): FFT along rho of one theta-frequency column of S, the
// kernel-spectrum product (column 0 packs the theta-DC and Nyquist columns),
// inverse FFT.  One column per block and slice; grid h x 3 x slice groups.
// VAR bit 1: index arithmetic redone per slice.
template <int M, int NT, int WPE, int VAR, int... Rs>
__global__ void __launch_bounds__(NT, WPE) k_cols_ct(lpk::RowPass rp, const float2* __restrict__ twM,
                                                     const float2* __restrict__ fzT) {
    constexpr int R0 = Plan<Rs...>::first, RL = Plan<Rs...>::last, nbl = M / RL, NI = (nbl + NT - 1) / NT;
    static_assert(NI * RL <= 32, "a thread's outputs are masked by one word");
    // (rounded up to whole 1 KB load-to-LDS chunks)
    __shared__ __align__(16) float2 buf[(slots<R0>(M) + 127) / 128 * 128];
    const int h = rp.h;
    const int nzg = (rp.nz + rp.zgroup - 1) / rp.zgroup;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int zg = lb % nzg, fs = lb / nzg, span = fs % 3, f = fs / 3;
    const int z0 = zg * rp.zgroup, z1 = min(z0 + rp.zgroup, rp.nz);
    const float2* fz = fzT + (size_t)f * M;
    const float2* fzh = fzT + (size_t)h * M;
    const int2 ir = rp.in_rows ? rp.in_rows[span] : make_int2(0, M);
    // the rows that are stored, of this thread's outputs i + q nbl
    unsigned smask = 0xffffffffu;
    if (rp.out_rows) {
        const unsigned char* om = rp.out_rows + (size_t)span * M;
        smask = 0;
#pragma unroll
        for (int c = 0; c < NI; ++c)
#pragma unroll
            for (int q = 0; q < RL; ++q)
                smask |= om[min((int)threadIdx.x + c * NT, nbl - 1) + q * nbl] ? 1u << (c * RL + q) : 0u;
    }
    for (int z = z0; z < z1; ++z) {
        float2* col = rp.S + (((size_t)span * rp.nz + z) * h + f) * (size_t)M;
        const int tid = (int)threadIdx.x + ((VAR & 2) ? opaque_zero() : 0);
        // rows without data are zeros
        auto mask = [&](int, int i, float2 v) {
            const bool ok = i >= ir.x && i < ir.y;
            return make_float2(ok ? v.x : 0.f, ok ? v.y : 0.f);
        };
        auto reload = make_source([&](int, int i) { return buf[slot<R0>(i)]; }, [](int, int, float2 v) { return v; });
        auto product = make_post([&](int x) { return ld_at(fz, (unsigned)x * 8u); },
                                 [&](float2 v, float2 w) {
                                     w.y = rp.conj ? -w.y : w.y;
                                     return cmul(v, f == 0 ? make_float2(1.f, 0.f) : w);
                                 });
        auto keep = [&](int, int x, int, int, float2 v) { buf[slot<R0>(x)] = v; };
        if constexpr (on_mfma(R0)) {
            // a matrix-core stage reads an input once per unit, so the column
            // goes to LDS first: 16 bytes a lane straight into buf (its first
            // radix is odd: no padding), one wait for all of it
            const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
            lds_barrier();   // the previous slice's last stage has read buf
            for (int c = wave * 128; c < M; c += NT * 2) {
                const int i = max(min(c + lane * 2, (ir.y - 2) & ~1), 0);
                __builtin_amdgcn_global_load_lds(col + i, buf + c, 16, 0, 0);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            auto staged = make_source([&](int, int i) { return buf[slot<R0>(i)]; }, mask);
            fft<M, 1, M, NT, 512 / WPE, true>(buf, staged, product, keep, twM, rp.wodd, -1, tid, Radices<Rs...>{});
        } else {
            auto load = make_source([&](int, int i) { return ld_at(col, (unsigned)max(min(i, ir.y - 1), ir.x) * 8u); }, mask);
            fft<M, 1, M, NT, 512 / WPE, true>(buf, load, product, keep, twM, rp.wodd, -1, tid, Radices<Rs...>{});
        }
        lds_barrier();
        if (f == 0) {
            for (int k = tid; k <= M / 2; k += NT) {
                const int km = k == 0 ? 0 : M - k;
                const float2 A = buf[slot<R0>(k)], Bc = cconj(buf[slot<R0>(km)]);
                const float2 D = make_float2(0.5f * (A.x + Bc.x), 0.5f * (A.y + Bc.y));
                const float2 E = make_float2(0.5f * (A.x - Bc.x), 0.5f * (A.y - Bc.y));
                const float2 Q = make_float2(E.y, -E.x);  // E / i
                const float2 yk = cadd(cmul(D, fzval(fz, k, rp.conj)), rot90(cmul(Q, fzval(fzh, k, rp.conj)), 1));
                const float2 ykm =
                    cadd(cmul(cconj(D), fzval(fz, km, rp.conj)), rot90(cmul(cconj(Q), fzval(fzh, km, rp.conj)), 1));
                buf[slot<R0>(k)] = yk;
                if (km != k) buf[slot<R0>(km)] = ykm;
            }
            lds_barrier();
        }
        auto store = [&](int, int x, int c, int q, float2 v) {
            if (smask & (1u << (c * RL + q))) st_at(col, (unsigned)x * 8u, v);
        };
        // (its own index: the table reads of the forward transform are not held
        // in registers until the inverse needs them again)
        const int tid2 = (int)threadIdx.x + ((VAR & 2) ? opaque_zero() : 0);
        fft<M, 1, M, NT, 512 / WPE, false>(buf, reload, NoPost{}, store, twM, rp.wodd, +1, tid2, Radices<Rs...>{});
    }
}

// Row pass, forward (k_rows_fwd): R log-polar rows of one span, real FFT of
// length 2H along theta (complex FFT of length H, then the R2C step on the
// way out), half spectra stored transposed into S.  LS: slots between rows
// in LDS, = 32 / R (mod 32) so that the transposed reads, R rows x 32 / R
// frequencies per half wave, fall on distinct banks.  Grid Nrho / R x slice
// groups x 3.
template <int H, int R, int LS, int NT, int WPE, int OPQ, int... Rs>
__global__ void __launch_bounds__(NT, WPE) k_rows_fwd_ct(lpk::RowPass rp, const float* __restrict__ F,
                                                    const int2* __restrict__ range) {
    constexpr int R0 = Plan<Rs...>::first, Nt = 2 * H;
    __shared__ float2 buf[R * (LS > slots<R0>(H) ? LS : slots<R0>(H))];
    __shared__ int2 rng_s[R];
    __shared__ float2 twn_s[H / 2 + 1];   // W_2H^k of the R2C step
    const int Nr = rp.Nrho;
    const int nrb = Nr / R, nzg = (rp.nz + rp.zgroup - 1) / rp.zgroup;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int row0 = (lb % nrb) * R, span = lb / (nrb * nzg);
    const int z0 = ((lb / nrb) % nzg) * rp.zgroup;
    const int z1 = min(z0 + rp.zgroup, rp.nz);
    if (rp.in_rows) {
        // no data in these rows: the column pass reads them as zeros
        const int2 ir = rp.in_rows[span];
        if (row0 + R <= ir.x || row0 >= ir.y) return;
    }
    if (threadIdx.x < R) rng_s[threadIdx.x] = range ? range[(size_t)span * Nr + row0 + threadIdx.x] : make_int2(0, Nt);
    for (int k = threadIdx.x; k <= H / 2; k += NT) twn_s[k] = rp.twN[k];
    __syncthreads();
    for (int z = z0; z < z1; ++z) {
        const float* Fz = F + (((size_t)span * rp.nz + z) * Nr + row0) * (size_t)Nt;
        const int tid = (int)threadIdx.x + (OPQ ? opaque_zero() : 0);
        // the rows to LDS, NT / R lanes each: unconditional loads at an index
        // clamped into the row's sampled range (its lines are loaded anyway),
        // zeros outside it
        {
            constexpr int TR = NT / R, NL = (H + TR - 1) / TR, U = NL <= 18 ? NL : 16;
            const int r = min(tid / TR, R - 1), l = tid - r * TR;   // (lanes past R TR repeat values of the last row)
            const int2 lr = rng_s[r];
            const int tlo = min(max(lr.x & ~1, 0), Nt - 2), thi = max(tlo, min((lr.y - 1) & ~1, Nt - 2));
            const unsigned row = (unsigned)(r * Nt);
            for (int c0 = 0; c0 < NL; c0 += U) {
                float2 v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int th = 2 * min(l + (c0 + u) * TR, H - 1);
                    v[u] = ld_at(reinterpret_cast<const float2*>(Fz), (row + (unsigned)min(max(th, tlo), thi)) * 4u);
                }
                issue_loads();
                if (c0 == 0) lds_barrier();   // the previous slice's rows have been stored
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int e = min(l + (c0 + u) * TR, H - 1), th = 2 * e;
                    v[u].x = (th >= lr.x && th < lr.y) ? v[u].x : 0.f;
                    v[u].y = (th + 1 >= lr.x && th + 1 < lr.y) ? v[u].y : 0.f;
                    buf[r * LS + slot<R0>(e)] = v[u];
                }
            }
        }
        lds_barrier();
        auto reload =
            make_source([&](int r, int x) { return buf[r * LS + slot<R0>(x)]; }, [](int, int, float2 v) { return v; });
        auto keep = [&](int r, int x, int, int, float2 v) { buf[r * LS + slot<R0>(x)] = v; };
        fft<H, R, LS, NT, 512 / WPE, true>(buf, reload, NoPost{}, keep, rp.twh, rp.wodd, -1, tid, Radices<Rs...>{});
        lds_barrier();
        // R2C step of the pairs (k, H - k) and the transposed store, rows
        // fastest: segments of R x 8 bytes
        float2* out = rp.S + ((size_t)span * rp.nz + z) * H * (size_t)Nr + row0;
        constexpr int np = H / 2 + 1;
#pragma unroll 4
        for (int t = tid; t < R * np; t += NT) {
            const int k = t / R, r = t - k * R, kk = H - k;
            const float2 A = buf[r * LS + slot<R0>(k)], Bc = cconj(buf[r * LS + slot<R0>(k == 0 ? 0 : kk)]);
            const float2 E = make_float2(0.5f * (A.x + Bc.x), 0.5f * (A.y + Bc.y));
            const float2 D = make_float2(0.5f * (A.x - Bc.x), 0.5f * (A.y - Bc.y));
            const float2 WO = cmul(twn_s[k], make_float2(D.y, -D.x));
            float2 x = cadd(E, WO);
            if (k == 0) x = make_float2(A.x + A.y, A.x - A.y);
            st_at(out, (unsigned)(k * Nr + r) * 8u, x);
            if (k != 0 && kk != k) st_at(out, (unsigned)(kk * Nr + r) * 8u, cconj(csub(E, WO)));
        }
    }
}

// Row pass, inverse (k_rows_inv): C2R along theta for R rows, writing the
// theta columns the output gather reads.
template <int H, int R, int LS, int NT, int WPE, int OPQ, int... Rs>
__global__ void __launch_bounds__(NT, WPE) k_rows_inv_ct(lpk::RowPass rp, float* __restrict__ G,
                                                    const int2* __restrict__ wrange) {
    constexpr int R0 = Plan<Rs...>::first, Nt = 2 * H;
    __shared__ float2 buf[R * (LS > slots<R0>(H) ? LS : slots<R0>(H))];
    __shared__ int2 wr_s[R];
    __shared__ float2 twn_s[H / 2 + 1];
    const int Nr = rp.Nrho;
    const int nrb = Nr / R, nzg = (rp.nz + rp.zgroup - 1) / rp.zgroup;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int row0 = (lb % nrb) * R, span = lb / (nrb * nzg);
    const int z0 = ((lb / nrb) % nzg) * rp.zgroup;
    const int z1 = min(z0 + rp.zgroup, rp.nz);
    int some = 0;
    if (threadIdx.x < R) {
        const int2 w = wrange ? wrange[(size_t)span * Nr + row0 + threadIdx.x] : make_int2(0, Nt);
        wr_s[threadIdx.x] = w;
        some = w.x < w.y;
    }
    some = __syncthreads_or(some);
    // no row of the block is read later (the column pass stored none of them)
    if (rp.out_rows && !some) return;
    for (int k = threadIdx.x; k <= H / 2; k += NT) twn_s[k] = rp.twN[k];   // (read behind a barrier)
    for (int z = z0; z < z1; ++z) {
        const float2* in = rp.S + ((size_t)span * rp.nz + z) * H * (size_t)Nr + row0;
        const int tid = (int)threadIdx.x + (OPQ ? opaque_zero() : 0);
        constexpr int np = H / 2 + 1, items = R * np, NL = (items + NT - 1) / NT, U = NL <= 10 ? NL : 8;
        for (int base = 0; base < items; base += U * NT) {   // uniform over the block
            const int t0 = base + tid;
            float2 P[U], Q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = min(t0 + u * NT, items - 1);
                const int k = t / R, r = t - k * R;
                P[u] = ld_at(in, (unsigned)(k * Nr + r) * 8u);
                Q[u] = ld_at(in, (unsigned)((k == 0 ? 0 : H - k) * Nr + r) * 8u);
            }
            issue_loads();
            if (base == 0) lds_barrier();   // the previous slice's last stage has read the rows
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = t0 + u * NT;
                if (t >= items) break;
                const int k = t / R, r = t - k * R, kk = H - k;
                const float2 S = cadd(P[u], cconj(Q[u])), D = csub(P[u], cconj(Q[u])), w = twn_s[k];
                float2 x = cadd(S, cmul(make_float2(w.y, w.x), D));
                if (k == 0) x = make_float2(P[u].x + P[u].y, P[u].x - P[u].y);
                buf[r * LS + slot<R0>(k)] = x;
                if (k != 0 && kk != k)
                    buf[r * LS + slot<R0>(kk)] =
                        cadd(cconj(S), cmul(make_float2(w.y, -w.x), cconj(make_float2(-D.x, -D.y))));
            }
        }
        lds_barrier();
        auto reload =
            make_source([&](int r, int x) { return buf[r * LS + slot<R0>(x)]; }, [](int, int, float2 v) { return v; });
        float* out = G + (((size_t)span * rp.nz + z) * Nr + row0) * (size_t)Nt;
        auto store = [&](int r, int e, int, int, float2 v) {
            const int2 wr = wr_s[r];
            if (2 * e + 1 >= wr.x && 2 * e < wr.y) st_at(reinterpret_cast<float2*>(out), (unsigned)(r * Nt + 2 * e) * 4u, v);
        };
        fft<H, R, LS, NT, 512 / WPE, false>(buf, reload, NoPost{}, store, rp.twh, rp.wodd, +1, tid, Radices<Rs...>{});
    }
}

// Filtered sinogram rows (k_sino_rows_pair): two kept angles per block, the
// FBP filter as one complex FFT pair of length M = 2N of x0 + i x1 (the
// filter spectrum is real and even), then both lines' prefilters side by
// side.  The filtered lines and the prefilter's scratch take the FFT
// buffer's place in LDS.  Grid
// ((P0 + 1) / 2, nz), NT threads.
template <int N, int NT, int WPE, int... Rs>
__global__ void __launch_bounds__(NT, WPE) k_sino_rows_pair_ct(const float* __restrict__ R, float* __restrict__ Rc,
                                                               lpk::SinoPrep sp, int cubic) {
    constexpr int M = 2 * N, R0 = Plan<Rs...>::first;
    __shared__ float2 buf[slots<R0>(M)];
    float* line = reinterpret_cast<float*>(buf);   // [2][N] lines, then [2][N] scratch
    float* tmp = line + 2 * N;
    const int a0 = 2 * blockIdx.x, z = blockIdx.y, tid = threadIdx.x;
    const int nrow = min(2, sp.P0 - a0);
    for (int u = 0; u < (cubic ? 0 : nrow); ++u)
        for (int j = 1; j < sp.os; ++j) {
            float* dz = Rc + ((size_t)z * sp.P + (size_t)(a0 + u) * sp.os + j) * N;
            for (int x = tid; x < N; x += NT) dz[x] = 0.f;
        }
    const float* src0 = R + ((size_t)z * sp.P0 + a0) * sp.N0;
    const float* src1 = R + ((size_t)z * sp.P0 + min(a0 + 1, sp.P0 - 1)) * sp.N0;
    auto row = [&](int x) {
        const unsigned xs = (unsigned)min(max(x - sp.lb, 0), sp.N0 - 1) * 4u;
        return make_float2(ld_at(src0, xs), ld_at(src1, xs));
    };
    auto pad = [&](int, int x, float2 v) { return make_float2(x < N ? v.x : 0.f, x < N && nrow > 1 ? v.y : 0.f); };
    auto reload = make_source([&](int, int x) { return buf[slot<R0>(x)]; }, [](int, int, float2 v) { return v; });
    auto response = make_post([&](int x) { return make_float2(sp.H2[x <= N ? x : M - x], 0.f); },
                              [](float2 v, float2 w) { return make_float2(v.x * w.x, v.y * w.x); });
    auto keep = [&](int, int x, int, int, float2 v) { buf[slot<R0>(x)] = v; };
    if constexpr (on_mfma(R0)) {
        // (a matrix-core stage reads an input once per unit)
        constexpr int U = 8;
        for (int x0 = tid; x0 < M; x0 += U * NT) {
            float2 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = row(min(x0 + u * NT, M - 1));
            issue_loads();
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int x = min(x0 + u * NT, M - 1);
                buf[slot<R0>(x)] = pad(0, x, v[u]);
            }
        }
        lds_barrier();
        fft<M, 1, M, NT, 512 / WPE, true>(buf, reload, response, keep, sp.tw2Nc, sp.wodd, -1, tid, Radices<Rs...>{});
    } else {
        auto load = make_source([&](int, int x) { return row(x); }, pad);
        fft<M, 1, M, NT, 512 / WPE, true>(buf, load, response, keep, sp.tw2Nc, sp.wodd, -1, tid, Radices<Rs...>{});
    }
    lds_barrier();
    auto lines = [&](int, int x, int, int, float2 v) {
        if (x < N) {
            line[x] = v.x;
            line[N + x] = v.y;
        }
    };
    fft<M, 1, M, NT, 512 / WPE, true>(buf, reload, NoPost{}, lines, sp.tw2Nc, sp.wodd, +1, tid + opaque_zero(), Radices<Rs...>{});
    __syncthreads();
    // the two lines' prefilters run side by side on the two halves of the block
    constexpr int half = NT / 2;
    const int u = tid < half ? 0 : 1;
    if (cubic) lpk::iir_line_lds(line + u * N, tmp + u * N, N, tid - u * half, half);
    for (int v = 0; v < nrow; ++v) {
        float* dst = Rc + ((size_t)z * sp.P + (size_t)(a0 + v) * sp.os) * N;
        for (int x = tid; x < N; x += NT) dst[x] = line[v * N + x];
    }
}

}  // namespace lpct
