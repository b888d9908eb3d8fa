// LDS-resident mixed-radix Stockham inverse FFT for gfx950.
//
// One transform of compile-time length N is held in a padded LDS array and
// processed by NT threads (a "group"); several groups of one workgroup may
// transform independent arrays in lock-step (every stage ends in a workgroup
// barrier).  Each stage loads R elements per butterfly into registers,
// applies the stage twiddles, runs an in-register radix-R butterfly and
// writes back in Stockham (self-sorting) order, so no bit-reversal pass is
// needed.  Twiddles come from a per-plan table generated on the host in FP64
// and rounded once to FP32.
//
// Direction: inverse (unnormalised), X[k] = sum_j x[j] exp(+2 pi i j k / N),
// the direction of the reference's cuFFT call (FIPkernels.cu:679, :741).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

namespace fip {

// ---------------------------------------------------------------- complex ops
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// a * (+i)
__device__ __forceinline__ float2 cmul_i(float2 a) { return make_float2(-a.y, a.x); }
// a * (-i)
__device__ __forceinline__ float2 cmul_mi(float2 a) { return make_float2(a.y, -a.x); }
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }

// LDS padding: one float2 of padding every 32 elements breaks the
// power-of-two strides of the early Stockham stages across banks.
__host__ __device__ constexpr int lds_pad(int i) { return i + (i >> 5); }
__host__ __device__ constexpr int lds_len(int n) { return n + (n >> 5) + 1; }

// ---------------------------------------------------------- radix butterflies
// In-register inverse DFTs of size R: v[s] <- sum_r v[r] exp(+2 pi i r s / R).
template <int R> struct Bfly;

template <> struct Bfly<2> {
    static __device__ __forceinline__ void run(float2* v)
    {
        float2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};

template <> struct Bfly<3> {
    static __device__ __forceinline__ void run(float2* v)
    {
        const float s3 = 0.866025403784438646763723170752936183f;   // sqrt(3)/2
        float2 t = cadd(v[1], v[2]);
        float2 u = csub(v[1], v[2]);
        float2 a = v[0];
        v[0] = cadd(a, t);
        float2 m = make_float2(a.x - 0.5f * t.x, a.y - 0.5f * t.y);
        float2 iu = cmul_i(cscale(u, s3));
        v[1] = cadd(m, iu);
        v[2] = csub(m, iu);
    }
};

template <> struct Bfly<4> {
    static __device__ __forceinline__ void run(float2* v)
    {
        float2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
        float2 c = cadd(v[1], v[3]), d = cmul_i(csub(v[1], v[3]));
        v[0] = cadd(a, c);
        v[2] = csub(a, c);
        v[1] = cadd(b, d);
        v[3] = csub(b, d);
    }
};

template <> struct Bfly<8> {
    static __device__ __forceinline__ void run(float2* v)
    {
        const float r = 0.707106781186547524400844362104849039f;
        float2 e[4] = {v[0], v[2], v[4], v[6]};
        float2 o[4] = {v[1], v[3], v[5], v[7]};
        Bfly<4>::run(e);
        Bfly<4>::run(o);
        // o[k] *= exp(+2 pi i k / 8)
        float2 o1 = make_float2(r * (o[1].x - o[1].y), r * (o[1].x + o[1].y));
        float2 o2 = cmul_i(o[2]);
        float2 o3 = make_float2(-r * (o[3].x + o[3].y), r * (o[3].x - o[3].y));
        v[0] = cadd(e[0], o[0]);
        v[4] = csub(e[0], o[0]);
        v[1] = cadd(e[1], o1);
        v[5] = csub(e[1], o1);
        v[2] = cadd(e[2], o2);
        v[6] = csub(e[2], o2);
        v[3] = cadd(e[3], o3);
        v[7] = csub(e[3], o3);
    }
};

// Compile-time sine and cosine (Taylor series in FP64; |x| <= pi) for the
// constant rotations inside composite butterflies.
constexpr double kPiD = 3.14159265358979323846264338327950288;
constexpr double ct_sin(double x)
{
    double term = x, sum = x;
    for (int n = 1; n < 24; ++n) {
        term *= -x * x / ((2.0 * n) * (2.0 * n + 1.0));
        sum += term;
    }
    return sum;
}
constexpr double ct_cos(double x)
{
    double term = 1.0, sum = 1.0;
    for (int n = 1; n < 24; ++n) {
        term *= -x * x / ((2.0 * n - 1.0) * (2.0 * n));
        sum += term;
    }
    return sum;
}

// a * exp(+2 pi i K / R) with the angle reduced to (-pi, pi]; quarter turns
// are exact sign swaps, odd eighth turns take two multiplies.
template <int R, int K>
__device__ __forceinline__ float2 rot(float2 a)
{
    constexpr int k = ((K % R) + R) % R;
    if constexpr (k == 0) {
        return a;
    } else if constexpr (4 * k == R) {
        return cmul_i(a);
    } else if constexpr (2 * k == R) {
        return make_float2(-a.x, -a.y);
    } else if constexpr (4 * k == 3 * R) {
        return cmul_mi(a);
    } else {
        constexpr int kr = (2 * k > R) ? k - R : k;
        constexpr double ang = 2.0 * kPiD * (double)kr / (double)R;
        if constexpr ((8 * k) % R == 0) {
            constexpr float r = 0.707106781186547524400844362104849039f;
            constexpr float cs = ct_cos(ang) > 0.0 ? 1.0f : -1.0f;
            constexpr float ss = ct_sin(ang) > 0.0 ? 1.0f : -1.0f;
            return make_float2(r * (cs * a.x - ss * a.y), r * (ss * a.x + cs * a.y));
        } else {
            constexpr float c = (float)ct_cos(ang), s = (float)ct_sin(ang);
            return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
        }
    }
}

// Compile-time loop: f(std::integral_constant<int, i>) for i = 0..N-1.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Sums and differences whose operands may be known zeros (ZA, ZB): the
// compiler keeps x + 0 for the sign of zero, so a pruned transform leaves
// them out itself.
template <bool ZA, bool ZB> __device__ __forceinline__ float2 cadd_z(float2 a, float2 b)
{
    if constexpr (ZB) return a;
    else if constexpr (ZA) return b;
    else return cadd(a, b);
}
template <bool ZA, bool ZB> __device__ __forceinline__ float2 csub_z(float2 a, float2 b)
{
    if constexpr (ZB) return a;
    else if constexpr (ZA) return make_float2(-b.x, -b.y);
    else return csub(a, b);
}
// Radix 4 with the inputs whose bit is set in MASK; the others are zeros.
template <unsigned MASK>
__device__ __forceinline__ void bfly4_masked(float2* v)
{
    constexpr bool z0 = !(MASK & 1u), z1 = !(MASK & 2u), z2 = !(MASK & 4u), z3 = !(MASK & 8u);
    const float2 a = cadd_z<z0, z2>(v[0], v[2]), b = csub_z<z0, z2>(v[0], v[2]);
    const float2 c = cadd_z<z1, z3>(v[1], v[3]), d = cmul_i(csub_z<z1, z3>(v[1], v[3]));
    constexpr bool za = z0 && z2, zc = z1 && z3;
    v[0] = cadd_z<za, zc>(a, c);
    v[2] = csub_z<za, zc>(a, c);
    v[1] = cadd_z<za, zc>(b, d);
    v[3] = csub_z<za, zc>(b, d);
}

// Inputs 0..LO-1 and R-HI..R-1 of a radix-R butterfly, as a bit mask (every
// bit where that is all of them).
template <int R, int LO, int HI>
constexpr unsigned band_mask()
{
    if (LO + HI >= R) return 0xffffffffu;
    const unsigned all = R >= 32 ? 0xffffffffu : ((1u << R) - 1u);
    return (((1u << LO) - 1u) | ~((1u << (R - HI)) - 1u)) & all;
}

// Composite radix R = A * B in registers (Cooley-Tukey): input r = B r1 + r2,
// output s = s1 + A s2; A-point DFTs over r1, rotation by
// exp(+2 pi i r2 s1 / R), then B-point DFTs over r2.  With A = 4, inputs
// whose bit is clear in MASK are taken as zeros and not read.
template <int A, int B>
struct BflyAB {
    // Inputs from fetch(std::integral_constant<int, r>).  Radix 32 holds 64
    // registers of data: its inputs are fetched and its DFTs formed a few at a
    // time, or the schedule spills at 80 registers (and a kernel that needs
    // scratch memory starts 6 us late).
    template <unsigned MASK, class F>
    static __device__ __forceinline__ void run_from(float2* v, const F& fetch)
    {
        constexpr int R = A * B;
        static_assert(A == 4 || MASK == 0xffffffffu, "pruned inputs need 4-point DFTs first");
        float2 x[B][A];
        auto get = [&](auto r2) {
            static_for<A>([&](auto r1) {
                constexpr int r = B * decltype(r1)::value + decltype(r2)::value;
                if constexpr ((MASK >> r) & 1u) x[r2][r1] = fetch(std::integral_constant<int, r>{});
            });
        };
        constexpr int AHEAD = R == 32 ? 4 : B;   // DFTs' inputs in flight
        static_for<AHEAD>(get);
        static_for<B>([&](auto r2) {
            constexpr int q = decltype(r2)::value;
            if constexpr (R == 32) __builtin_amdgcn_sched_barrier(0);
            if constexpr (A == 4 && MASK != 0xffffffffu) {
                constexpr unsigned m = ((MASK >> q) & 1u) | (((MASK >> (B + q)) & 1u) << 1) |
                                       (((MASK >> (2 * B + q)) & 1u) << 2) | (((MASK >> (3 * B + q)) & 1u) << 3);
                bfly4_masked<m>(x[r2]);
            } else {
                Bfly<A>::run(x[r2]);
            }
            static_for<A>([&](auto s1) { x[r2][s1] = rot<R, decltype(r2)::value * decltype(s1)::value>(x[r2][s1]); });
            if constexpr (q + AHEAD < B) get(std::integral_constant<int, q + AHEAD>{});
        });
        static_for<A>([&](auto s1) {
            float2 y[B];
            static_for<B>([&](auto r2) { y[r2] = x[r2][s1]; });
            if constexpr (R == 32) __builtin_amdgcn_sched_barrier(0);
            Bfly<B>::run(y);
            static_for<B>([&](auto s2) { v[s1 + A * s2] = y[s2]; });
        });
    }
    template <unsigned MASK = 0xffffffffu>
    static __device__ __forceinline__ void run(float2* v)
    {
        run_from<MASK>(v, [&](auto r) { return v[decltype(r)::value]; });
    }
};
template <> struct Bfly<6> : BflyAB<2, 3> {};
template <> struct Bfly<12> : BflyAB<4, 3> {};
template <> struct Bfly<16> : BflyAB<4, 4> {};
template <> struct Bfly<24> : BflyAB<8, 3> {};
template <> struct Bfly<32> : BflyAB<4, 8> {};

// Butterfly of radix R with zero inputs outside MASK, where the radix has a
// pruned form (4-point DFTs first); the others read every input.
constexpr bool bfly_prunes(int R) { return R == 12 || R == 16 || R == 32; }
constexpr bool bfly_fetches(int R) { return R == 32; }
template <int R, unsigned MASK>
__device__ __forceinline__ void bfly_masked(float2* v)
{
    static_assert(bfly_prunes(R) || MASK == 0xffffffffu, "no pruned form of this radix");
    if constexpr (bfly_prunes(R))
        Bfly<R>::template run<MASK>(v);
    else
        Bfly<R>::run(v);
}

// ----------------------------------------------------------------- FFT plans
// Radix lists for N = 3 * 2^k.  The host twiddle generator walks the same
// list (make_stage_twiddles), so the two stay consistent by construction.  From
// N = 1536 on, a transform gets N/12 threads (12 points per thread): more
// waves per workgroup hide the LDS and barrier latency of each stage.  Each
// stage is one LDS round trip and two barriers, so these lengths take the
// fewest stages that keep a butterfly's registers within occupancy: radix 16
// and 12 in registers (three stages for 384 to 6144, four for 12288) measured
// 3-13% faster than radix 8/4/3/2 lists of five or six stages, and 6144 as
// 32, 16, 12 takes the column kernel from 82 to 76 us and the row pass from 88 to
// 85 at 4096^2 against 16, 16, 2, 12 (one LDS round trip less; the radix-32 stage
// fills three of the eight waves, which the CU's other workgroups cover).  Every
// list ends in radix 12: the last stage's outputs then lie N/12 apart, so a crop
// to the central two thirds is four whole outputs dropped per butterfly, and the
// kept ones leave from registers.
template <int NT, int... Rs>
struct PlanDef {
    static constexpr int nt = NT;
    static constexpr int nstages = sizeof...(Rs);
    static constexpr int radix[sizeof...(Rs)] = {Rs...};
};
template <int N> struct FftPlan;
#define FIP_PLAN(N_, NT_, ...)                                 \
    template <> struct FftPlan<N_> : PlanDef<NT_, __VA_ARGS__> { \
        static constexpr int n = N_;                           \
    }
FIP_PLAN(48, 64, 4, 12);
FIP_PLAN(96, 64, 8, 12);
FIP_PLAN(192, 64, 16, 12);
FIP_PLAN(384, 64, 8, 4, 12);
FIP_PLAN(768, 64, 16, 4, 12);
FIP_PLAN(1536, 128, 16, 8, 12);
FIP_PLAN(3072, 256, 16, 16, 12);
FIP_PLAN(6144, 512, 32, 16, 12);
FIP_PLAN(12288, 1024, 16, 16, 4, 12);
#undef FIP_PLAN

// Padded LDS offsets of the R elements of a butterfly relative to the padded
// index of its first element, when they are compile-time constants (so the
// LDS instructions carry them as immediates):
//  - loads j + r*NB with NB % 32 == 0: r * (NB + NB/32);
//  - stores base + r*Ns, base = (j/Ns)*Ns*R + (j%Ns): if Ns*R divides 32,
//    base % 32 + r*Ns < 32 and the offset is r*Ns; if Ns % 32 == 0, or Ns
//    divides 32 and 32 divides Ns*R, base % 32 < Ns and the offset is
//    r*Ns + (r*Ns)/32.
template <int NB> struct LoadOff {
    static constexpr bool ok = (NB % 32) == 0;
    static constexpr __host__ __device__ int at(int r) { return r * (NB + NB / 32); }
};
template <int Ns, int R> struct StoreOff {
    static constexpr bool small = (32 % (Ns * R)) == 0;
    static constexpr bool big = (Ns % 32 == 0) || ((32 % Ns) == 0 && ((Ns * R) % 32) == 0);
    static constexpr bool ok = small || big;
    static constexpr __host__ __device__ int at(int r) { return small ? r * Ns : r * Ns + ((r * Ns) >> 5); }
};

// Input j + r N/R of a butterfly from the padded LDS array buf.
template <int N, int R>
__device__ __forceinline__ float2 lds_input(const float2* buf, int j, int r)
{
    constexpr int NB = N / R;
    if constexpr (LoadOff<NB>::ok) return (buf + lds_pad(j))[LoadOff<NB>::at(r)];
    return buf[lds_pad(j + r * NB)];
}

// One Stockham stage of radix R with Ns = product of earlier radices.
// tw points at this stage's twiddles laid out [r-1][k], k < Ns.  Threads
// t >= NT of a larger workgroup (whole waves, NT a multiple of 64) take no
// butterfly but reach the barriers.
//
// The first stage's inputs come from load(j, r) = x[j + r N/R], and the last
// stage's outputs go to store(j, v): X[j + r N/R] = v[r] (there Ns = N/R,
// so j is the output index's low part); every other exchange goes through buf.
// LoadLds / StoreLds say whether load reads or store writes LDS that this
// transform (or its caller's data in the same memory) uses, which needs a
// barrier between the reads and the writes.  MASK: the first stage's inputs
// that can be non-zero (the others are not loaded).  A store with a
// prefetch(t) member has it called ahead of the last stage (one butterfly per
// thread there).
template <class P, int S, int Ns, int TwOff, bool LoadLds, bool StoreLds, unsigned MASK, class Load, class Store>
__device__ __forceinline__ void fft_stage(float2* __restrict__ buf, const float2* __restrict__ tw, int t,
                                          Load& load, Store& store)
{
    constexpr int N = P::n, NT = P::nt, R = P::radix[S];
    constexpr bool first = S == 0, last = S + 1 == P::nstages;
    constexpr int NB = N / R;                    // butterflies in this stage
    constexpr int BPT = (NB + NT - 1) / NT;      // butterflies per thread
    // The two barriers around the exchange of in-place data.
    constexpr bool mid = (!first || LoadLds) && (!last || StoreLds), end = !last || StoreLds;
    auto body = [&](auto ALL) {
        constexpr bool all = decltype(ALL)::value;   // every thread here has all its butterflies
        float2 v[BPT][R];
        // Twiddles do not depend on the data: issue their (L1/L2-resident)
        // loads before the LDS loads and the barrier so their latency is
        // hidden; likewise what store needs.
        if constexpr (last && requires { store.prefetch(t); }) store.prefetch(t);
        float2 w[BPT][R > 1 ? R - 1 : 1];
        if (Ns > 1) {
#pragma unroll
            for (int b = 0; b < BPT; ++b) {
                const int j = t + b * NT;
                const int k = (all || j < NB) ? j % Ns : 0;
#pragma unroll
                for (int r = 1; r < R; ++r) w[b][r - 1] = (tw + TwOff)[(r - 1) * Ns + k];
            }
        }
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const int j = t + b * NT;
            if (all || (t < NT && j < NB)) {
                if constexpr (first && bfly_fetches(R)) {
                    Bfly<R>::template run_from<MASK>(
                        v[b], [&](auto r) { return load(j, decltype(r)::value); });
                } else if constexpr (first) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if ((MASK >> r) & 1u) v[b][r] = load(j, r);
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r) v[b][r] = lds_input<N, R>(buf, j, r);
                }
            }
        }
        if constexpr (mid) __syncthreads();
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const int j = t + b * NT;
            if (all || (t < NT && j < NB)) {
                const int k = j % Ns;
                if (Ns > 1) {
#pragma unroll
                    for (int r = 1; r < R; ++r) v[b][r] = cmul(v[b][r], w[b][r - 1]);
                }
                if constexpr (!(first && bfly_fetches(R))) bfly_masked<R, first ? MASK : 0xffffffffu>(v[b]);
                if constexpr (last) {
                    store(j, v[b]);
                } else {
                    const int base = (j / Ns) * Ns * R + k;
                    if constexpr (StoreOff<Ns, R>::ok) {
                        float2* p = buf + lds_pad(base);
#pragma unroll
                        for (int r = 0; r < R; ++r) p[StoreOff<Ns, R>::at(r)] = v[b][r];
                    } else {
#pragma unroll
                        for (int r = 0; r < R; ++r) buf[lds_pad(base + r * Ns)] = v[b][r];
                    }
                }
            }
        }
        if constexpr (end) __syncthreads();
    };
    // Where the butterflies fill whole waves, the waves without one only take
    // the barriers (a wave-uniform branch: every wave of the workgroup reaches
    // each barrier once), so no register is merged across the branch.
    constexpr bool exact = (NB % NT) == 0;
    if constexpr (exact) {
        if (__builtin_amdgcn_readfirstlane(t) < NT) {
            body(std::true_type{});
        } else {
            if constexpr (mid) __syncthreads();
            if constexpr (end) __syncthreads();
        }
    } else if constexpr (BPT == 1 && NB % 64 == 0) {
        if (__builtin_amdgcn_readfirstlane(t) < NB) {
            body(std::true_type{});
        } else {
            if constexpr (mid) __syncthreads();
            if constexpr (end) __syncthreads();
        }
    } else {
        body(std::false_type{});
    }
    if constexpr (!last)
        fft_stage<P, S + 1, Ns * R, TwOff + (Ns > 1 ? (R - 1) * Ns : 0), LoadLds, StoreLds, MASK>(buf, tw, t, load,
                                                                                                  store);
}

// Inverse FFT of length N between load and store (see fft_stage) with buf
// (lds_len(N) entries) for the exchanges.
template <int N, bool LoadLds, bool StoreLds, unsigned MASK = 0xffffffffu, class Load, class Store>
__device__ __forceinline__ void fft_inverse_io(float2* buf, const float2* __restrict__ tw, int t, Load&& load,
                                               Store&& store)
{
    fft_stage<FftPlan<N>, 0, 1, 0, LoadLds, StoreLds, MASK>(buf, tw, t, load, store);
}

// Inverse FFT of the N-point padded LDS array buf.  Caller must have a
// workgroup barrier between filling buf and this call; on return the result
// is in buf (natural order) and visible to the whole workgroup.
template <int N>
__device__ __forceinline__ void fft_inverse(float2* buf, const float2* __restrict__ tw, int t)
{
    using P = FftPlan<N>;
    constexpr int R0 = P::radix[0], R1 = P::radix[P::nstages - 1];
    fft_inverse_io<N, true, true>(
        buf, tw, t,
        [&](int j, int r) { return lds_input<N, R0>(buf, j, r); },
        [&](int j, const float2* v) {
#pragma unroll
            for (int r = 0; r < R1; ++r) buf[lds_pad(j + r * (N / R1))] = v[r];
        });
}

// Number of twiddle entries the plan of length N uses (N - 1).
__host__ __device__ constexpr int fft_twiddle_count(int n) { return n - 1; }

}  // namespace fip
