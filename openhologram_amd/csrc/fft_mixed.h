// fft_mixed.h -- LDS-resident Stockham FFT for lengths N = 2^a 3^b 5^c on
// gfx950 (the SLM grids that are not powers of two, e.g. 11520 x 2160).
//
// A line of N complex64 values is transformed by NT threads, stage by stage
// over a compile-time radix plan (plan(N): the few large radices that cost
// least, e.g. 1920 = 16 x 15 x 8).  A stage of radix R after radices of product
// Ns has N/R butterflies; butterfly j reads j + r N/R (r < R), multiplies by
// exp(SIGN i 2 pi r k/(Ns R)), k = j mod Ns, does the R-point DFT in registers
// and writes (j - k) R + k + r Ns (self-sorting, output in natural order).
// Each thread keeps all of its butterflies' inputs in registers across the
// stage's barrier, so stages work in place.  line() takes and leaves the line
// in LDS (natural order, fft::pad16 indexing); line_ends() takes the first
// stage's inputs and leaves the last stage's outputs in registers, so that
// the line passes through LDS only between stages.  Twiddles come from a
// per-length table (oph_twiddles_mixed) laid out as the power-of-two
// engine's: stage s >= 1 holds tws[(r-1) Ns + k] = exp(-2 pi i k r/(Ns R)),
// stages concatenated.
#pragma once

#include "fft_engine.h"

namespace fft {

// 3-point DFT: X1,2 = x0 - (x1 + x2)/2 +- SIGN i (sqrt 3/2)(x1 - x2)
template <int SIGN>
struct Dft<3, SIGN> {
    __device__ static void run(float2* v) {
        constexpr float h = 0.86602540378443865f;
        const float2 t1 = cadd(v[1], v[2]);
        const float2 t2 = make_float2(fmaf(-0.5f, t1.x, v[0].x), fmaf(-0.5f, t1.y, v[0].y));
        const float2 d = csub(v[1], v[2]);
        const float2 t3 = mul_si<SIGN>(make_float2(h * d.x, h * d.y));
        v[0] = cadd(v[0], t1);
        v[1] = cadd(t2, t3);
        v[2] = csub(t2, t3);
    }
};

// 5-point DFT with c_k = cos(2 pi k/5), s_k = sin(2 pi k/5):
//   X0 = x0 + a1 + a2 (a1 = x1 + x4, a2 = x2 + x3, b1 = x1 - x4, b2 = x2 - x3)
//   X1,4 = x0 + c1 a1 + c2 a2 +- SIGN i (s1 b1 + s2 b2)
//   X2,3 = x0 + c2 a1 + c1 a2 +- SIGN i (s2 b1 - s1 b2)
template <int SIGN>
struct Dft<5, SIGN> {
    __device__ static void run(float2* v) {
        constexpr float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
        constexpr float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
        const float2 a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]);
        const float2 a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
        const float2 m1 = make_float2(v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y);
        const float2 m2 = make_float2(v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y);
        const float2 n1 = mul_si<SIGN>(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y));
        const float2 n2 = mul_si<SIGN>(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y));
        v[0] = make_float2(v[0].x + a1.x + a2.x, v[0].y + a1.y + a2.y);
        v[1] = cadd(m1, n1);
        v[4] = csub(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
    }
};

// N = A B with A and B coprime, without twiddles: input (B n1 + A n2) mod N is
// element (n1, n2) of an A x B transform, whose output (k1, k2) is the k with
// k mod A = k1 and k mod B = k2 (n k/N = n1 k/A + n2 k/B up to whole numbers).
template <int A, int B, int SIGN>
struct DftCoprime {
    static constexpr int crt(int k1, int k2) {
        int k = k1;
        while (k % B != k2) k += A;
        return k;
    }
    __device__ static void run(float2* v) {
        float2 x[B][A], y[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) x[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
            Dft<A, SIGN>::run(x[n2]);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) y[n2] = x[n2][k1];
            Dft<B, SIGN>::run(y);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[crt(k1, k2)] = y[k2];
        }
    }
};
template <int SIGN>
struct Dft<6, SIGN> : DftCoprime<2, 3, SIGN> {};
template <int SIGN>
struct Dft<10, SIGN> : DftCoprime<2, 5, SIGN> {};
template <int SIGN>
struct Dft<12, SIGN> : DftCoprime<4, 3, SIGN> {};
template <int SIGN>
struct Dft<15, SIGN> : DftCoprime<3, 5, SIGN> {};

// 9 = 3 x 3: X[k1 + 3 k2] = sum_{n2} W3^{n2 k2} W9^{n2 k1} sum_{n1} W3^{n1 k1} x[3 n1 + n2]
template <int SIGN>
struct Dft<9, SIGN> {
    __device__ static void run(float2* v) {
        constexpr float c1 = 0.76604444311897804f, s1 = 0.64278760968653933f;   // 2 pi/9
        constexpr float c2 = 0.17364817766693035f, s2 = 0.98480775301220806f;   // 4 pi/9
        constexpr float c4 = -0.93969262078590838f, s4 = 0.34202014332566873f;  // 8 pi/9
        float2 x[3][3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < 3; ++n1) x[n2][n1] = v[3 * n1 + n2];
            Dft<3, SIGN>::run(x[n2]);
        }
        x[1][1] = cmul(x[1][1], make_float2(c1, SIGN * s1));
        x[1][2] = cmul(x[1][2], make_float2(c2, SIGN * s2));
        x[2][1] = cmul(x[2][1], make_float2(c2, SIGN * s2));
        x[2][2] = cmul(x[2][2], make_float2(c4, SIGN * s4));
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            float2 y[3] = {x[0][k1], x[1][k1], x[2][k1]};
            Dft<3, SIGN>::run(y);
#pragma unroll
            for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = y[k2];
        }
    }
};

}  // namespace fft

namespace fftm {

struct Plan {
    int n;       // number of stages (-1: N has a prime factor other than 2, 3, 5)
    int r[24];   // radices in order
};

// Threads per line: a radix-16 stage's butterfly count rounded up to whole
// waves, at most
// 512 (a longer line keeps more elements per thread, but 8 waves of up to
// 256 registers each, where 12 would be held to 168).
__host__ __device__ constexpr int threads(int N) {
    const int t = ((N + 15) / 16 + 63) / 64 * 64;
    return t < 512 ? t : 512;
}
// Cost of a radix-R stage of an N-point line to a thread: its butterflies'
// instructions, twiddles and LDS accesses, and the stage's barriers.
__host__ __device__ constexpr int stage_cost(int N, int R, bool first) {
    const int ops = R == 16 ? 190 : R == 15 ? 220 : R == 12 ? 140 : R == 10 ? 124 : R == 9 ? 120 : R == 8 ? 76
                  : R == 6 ? 60 : R == 5 ? 48 : R == 4 ? 24 : R == 3 ? 22 : 8;
    const int per = (N / R + threads(N) - 1) / threads(N);
    return per * (ops + (first ? 0 : 8 * (R - 1)) + 16 * R) + 60;
}

// The radices in falling order whose stages together cost least.
struct Search {
    int cost;
    Plan best;
};
__host__ __device__ constexpr void search(int N, int rest, int max_radix, const Plan& path, int cost, Search& s) {
    if (rest == 1) {
        if (cost < s.cost) {
            s.cost = cost;
            s.best = path;
        }
        return;
    }
    for (int R = max_radix; R >= 2; --R) {
        if (rest % R || (R > 6 && (R < 8 || R == 11 || R == 13 || R == 14))) continue;
        Plan next = path;
        next.r[next.n++] = R;
        search(N, rest / R, R, next, cost + stage_cost(N, R, path.n == 0), s);
    }
}
__host__ __device__ constexpr Plan plan(int N) {
    int rest = N;
    for (int f = 2; f <= 5; ++f)
        while (f != 4 && rest > 1 && rest % f == 0) rest /= f;
    Search s{1 << 30, {-1, {}}};
    if (rest == 1 && N > 1) search(N, N, 16, Plan{0, {}}, 0, s);
    return s.best;
}
template <int N>
constexpr Plan PLAN = plan(N);   // (searched once per length)

// Elements per thread when a thread owns t + m NT, m < ept(N).
__host__ __device__ constexpr int ept(int N) { return (N + threads(N) - 1) / threads(N); }

// Marks every element of w (but w[0]) as needed at this point, after all
// of them were loaded: the loads are issued as one batch and waited for
// once (left to itself the compiler orders load, wait, use per element).
template <int R>
__device__ __forceinline__ void batch_ready(float2 (&w)[R]) {
#pragma unroll
    for (int r = 1; r < R; ++r) asm volatile("" : "+v"(w[r].x), "+v"(w[r].y));
}

// One stage of radix R (Ns = product of the earlier radices) by NT threads;
// tws is the stage's table (unused for Ns = 1).  Starts and ends with the
// line complete in LDS (a barrier separates its reads from its writes and
// ends it).
template <int N, int R, int NS, int NT, int SIGN>
__device__ __forceinline__ void stage(float2* buf, const float2* __restrict__ tws, int t) {
    constexpr int NB = N / R;
    constexpr int PER = (NB + NT - 1) / NT;
    float2 v[PER][R];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int j = t + p * NT;
        if (PER * NT == NB || j < NB) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[p][r] = buf[fft::pad16(j + r * NB)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int j = t + p * NT;
        if (PER * NT == NB || j < NB) {
            const int k = j % NS;
            if constexpr (NS > 1) {
                // the butterfly's R - 1 twiddles are all requested before the
                // first is used: one wait for the batch, not one per load
                float2 w[R];
#pragma unroll
                for (int r = 1; r < R; ++r) w[r] = tws[(r - 1) * NS + k];
                batch_ready(w);
#pragma unroll
                for (int r = 1; r < R; ++r) v[p][r] = SIGN < 0 ? fft::cmul(v[p][r], w[r]) : fft::cmulc(v[p][r], w[r]);
            }
            fft::Dft<R, SIGN>::run(v[p]);
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[fft::pad16(base + r * NS)] = v[p][r];
        }
    }
    __syncthreads();
}

template <int N, int NT, int SIGN, int S, int NS, int OFF>
__device__ __forceinline__ void line_from(float2* buf, const float2* __restrict__ tw, int t) {
    if constexpr (S < PLAN<N>.n) {
        constexpr int R = PLAN<N>.r[S];
        stage<N, R, NS, NT, SIGN>(buf, tw + OFF, t);
        line_from<N, NT, SIGN, S + 1, NS * R, OFF + (NS > 1 ? (R - 1) * NS : 0)>(buf, tw, t);
    }
}

// Full transform of one LDS line (natural order in and out) by threads
// t < NT of the workgroup; every thread of the workgroup must call it (the
// stages hold barriers).  Caller syncs before (line loaded).
template <int N, int NT, int SIGN>
__device__ __forceinline__ void line(float2* buf, const float2* __restrict__ tw, int t) {
    static_assert(PLAN<N>.n > 0, "length must be 2^a 3^b 5^c");
    line_from<N, NT, SIGN, 0, 1, 0>(buf, tw, t);
}

// ---- register-ended lines ----
// The first stage's butterfly t + p NT has the inputs (t + p NT) + r NB0, the
// last stage's the outputs (t + p NT) + r NBL: per thread PER0 x R0 and PERL x
// RL elements, of which those of butterflies beyond NB0 (NBL) do not exist.
template <int N>
struct Ends {
    static constexpr int NT = threads(N), LAST = PLAN<N>.n - 1;
    static_assert(PLAN<N>.n >= 2, "two stages at least");
    static constexpr int R0 = PLAN<N>.r[0], NB0 = N / R0, PER0 = (NB0 + NT - 1) / NT;
    static constexpr int RL = PLAN<N>.r[LAST], NBL = N / RL, PERL = (NBL + NT - 1) / NT;
};

// Stages S .. n - 2, in LDS
template <int N, int SIGN, int S, int NS, int OFF>
__device__ __forceinline__ void mid_stages(float2* buf, const float2* __restrict__ tw, int t) {
    if constexpr (S < Ends<N>::LAST) {
        constexpr int R = PLAN<N>.r[S];
        stage<N, R, NS, Ends<N>::NT, SIGN>(buf, tw + OFF, t);
        mid_stages<N, SIGN, S + 1, NS * R, OFF + (R - 1) * NS>(buf, tw, t);
    }
}
template <int N>
constexpr int last_offset() {
    int off = 0, ns = PLAN<N>.r[0];
    for (int s = 1; s < PLAN<N>.n - 1; ++s) {
        off += (PLAN<N>.r[s] - 1) * ns;
        ns *= PLAN<N>.r[s];
    }
    return off;
}

// Full transform of a line from vi (first stage's inputs) to vo (last stage's
// outputs).  The caller syncs before the line is written again (other threads
// may still read the last stage's inputs); every thread of the workgroup calls
// it.
template <int N, int SIGN>
__device__ __forceinline__ void line_ends(float2 (&vi)[Ends<N>::PER0][Ends<N>::R0],
                                          float2 (&vo)[Ends<N>::PERL][Ends<N>::RL], float2* buf,
                                          const float2* __restrict__ tw, int t) {
    using E = Ends<N>;
#pragma unroll
    for (int p = 0; p < E::PER0; ++p) {
        const int j = t + p * E::NT;
        if (E::PER0 * E::NT == E::NB0 || j < E::NB0) {
            fft::Dft<E::R0, SIGN>::run(vi[p]);
#pragma unroll
            for (int r = 0; r < E::R0; ++r) buf[fft::pad16(j * E::R0 + r)] = vi[p][r];
        }
    }
    __syncthreads();
    mid_stages<N, SIGN, 1, E::R0, 0>(buf, tw, t);
    const float2* tl = tw + last_offset<N>();
#pragma unroll
    for (int p = 0; p < E::PERL; ++p) {
        const int j = t + p * E::NT;
        if (E::PERL * E::NT == E::NBL || j < E::NBL) {
            float2 w[E::RL];
#pragma unroll
            for (int r = 1; r < E::RL; ++r) w[r] = tl[(r - 1) * E::NBL + j];
#pragma unroll
            for (int r = 0; r < E::RL; ++r) vo[p][r] = buf[fft::pad16(j + r * E::NBL)];
            batch_ready(w);
#pragma unroll
            for (int r = 1; r < E::RL; ++r) vo[p][r] = SIGN < 0 ? fft::cmul(vo[p][r], w[r]) : fft::cmulc(vo[p][r], w[r]);
            fft::Dft<E::RL, SIGN>::run(vo[p]);
        }
    }
}

// LDS elements of a padded line
__host__ __device__ constexpr int padded_len(int N) { return N + N / 16 + 1; }

}  // namespace fftm

// Device twiddle table of the mixed-radix plan of length N (layout above,
// FP64-computed, rounded to float), cached per length in the context.
// Returns nullptr on failure (error recorded).
const float2* oph_twiddles_mixed(oph_ctx* ctx, int N);
