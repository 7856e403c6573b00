// fft_filter.hip -- FBP row filter on gfx950: edge-replicate pad, FFT,
// multiply by the (Hermitian) filter, inverse FFT, window store.
//
// One workgroup filters two sinogram rows at once -- the same angle of two
// consecutive slices: the padded rows u0, u1 (length n = npad) form
// z = u0 + i u1 in LDS; a mixed-radix Stockham FFT (radices 8, 4, 2, 3, 5, 7,
// 11, 13; twiddles from an FP64-built table) runs entirely in LDS with the
// butterfly inputs held in registers across one barrier per pass.  Because
// the filter H is Hermitian (H_{n-k} = conj H_k, the spectrum of a real
// kernel), conj(FFT(conj(Z H))) returns q0 + i q1, the two filtered rows.  H
// carries 1/(npad * pixel) (filters.cu:184-186); the store multiplies by
// dtheta_a * angular scale and writes only the bin window the backprojector
// reads, zeros outside [0, n), into the slice-interleaved layout
// [group][angle][bin][SB] (SB = 4 for FP32 rows, 8 for FP16 rows).
//
// Twelve sizes, 512, 640, 768, 1024 and 1536, 2048, 2560, 3072, 4096, 5120, 6144, 8192
// bins, run k_filter_dif instead: forward passes that leave the spectrum permuted, H
// in that order, and the same passes back.
//
// Padded sizes with a prime factor > 5 or n > 16384 run the same circular
// convolution q[m] = sum_j g[(m - j) mod n] u[j], g = IDFT(H) (built on the host
// in FP64), in FP64: by transforms (k_filter_conv) or, for short rows and for
// rows past its transforms' length, as that sum (k_filter_direct).
//
// Reference behaviour restated: paddR2R (padding.cu:140-178), filterFBP /
// convolution_R2C_C2R_1D / fbp_filtering_R2C2R (filters.cu:33-51,68-87,163-190),
// Filter::apply (filters.cu:395-438).
#include "raft_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace raft {

namespace {

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 mul_mi(float2 a) { return make_float2(a.y, -a.x); } // * (-i)

// Twiddles W_n^m = exp(-2 pi i m / n), m < n <= 16384, from two small tables
// kept in LDS: W^m = hi[m >> 7] * lo[m & 127] (one FP32 product of two
// FP64-built values; error ~2 ulp).
struct Tw {
    const float2* lo; // [128]
    const float2* hi; // [n / 128 + 1]
    __device__ __forceinline__ float2 operator()(int m) const { return cmul(hi[m >> 7], lo[m & 127]); }
};

// LDS index with one complex of padding per 16: Stockham passes with small
// strides (Ns = 1, 8) would otherwise put consecutive lanes on the same banks.
__device__ __forceinline__ int pix(int e) { return e + (e >> 4); }
__host__ __device__ constexpr size_t lds_elems(int n) { return (size_t)n + (size_t)(n >> 4) + 1; }

// in-register forward DFTs of size R (W_R = exp(-2 pi i / R))
template <int R> struct Dft;

template <> struct Dft<2> {
    __device__ static void run(float2* v, const Tw&, int)
    {
        float2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};

template <> struct Dft<3> {
    __device__ static void run(float2* v, const Tw&, int)
    {
        const float c1 = -0.5f, s1 = 0.86602540378443864676f; // sin(2 pi/3)
        float2 a = v[0], b = v[1], c = v[2];
        float2 sp = cadd(b, c), sm = csub(b, c);
        float2 m = make_float2(a.x + c1 * sp.x, a.y + c1 * sp.y);
        // W = c1 - i s1 : y1 = m - i s1 sm, y2 = m + i s1 sm
        float2 t = make_float2(s1 * sm.y, -s1 * sm.x); // -i s1 sm
        v[0] = cadd(a, sp);
        v[1] = cadd(m, t);
        v[2] = csub(m, t);
    }
};

template <> struct Dft<4> {
    __device__ static void run(float2* v, const Tw&, int)
    {
        float2 a = v[0], b = v[1], c = v[2], d = v[3];
        float2 s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = mul_mi(csub(b, d));
        v[0] = cadd(s0, s2);
        v[1] = cadd(s1, s3);
        v[2] = csub(s0, s2);
        v[3] = csub(s1, s3);
    }
};

template <> struct Dft<8> {
    __device__ static void run(float2* v, const Tw&, int)
    {
        const float h = 0.70710678118654752440f;
        float2 e[4] = {v[0], v[2], v[4], v[6]};
        float2 o[4] = {v[1], v[3], v[5], v[7]};
        Dft<4>::run(e, Tw{}, 0);
        Dft<4>::run(o, Tw{}, 0);
        // o[k] *= W8^k
        float2 o1 = make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)); // * h(1 - i)
        float2 o2 = mul_mi(o[2]);
        float2 o3 = make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)); // * h(-1 - i)
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

// odd prime radices: direct sum with W_R^m = W_n^(m n / R)
template <int R> struct DftGeneric {
    __device__ static void run(float2* v, const Tw& tw, int n)
    {
        float2 in[R];
#pragma unroll
        for (int q = 0; q < R; ++q) in[q] = v[q];
        const int st = n / R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float2 acc = in[0];
#pragma unroll
            for (int q = 1; q < R; ++q) acc = cadd(acc, cmul(in[q], tw(((q * r) % R) * st)));
            v[r] = acc;
        }
    }
};
template <> struct Dft<5> : DftGeneric<5> {};

// One Stockham pass (decimation in time, autosorting):
//   butterfly j (0 <= j < n/R), jm = j mod Ns:
//   in  x_r = z[j + r n/R] * W_{Ns R}^{jm r}   (W^{jm r} = (W^{jm})^r)
//   out z[(j - jm) R + jm + r Ns] = DFT_R(x)_r
// n / THREADS <= E, so a thread holds at most ceil(E/R) butterflies.
// Ns is a power of two for every pass before the first odd radix (radices
// are ordered 8, 4, 2 first), so jm is a mask there.
template <int R, int THREADS, int E>
__device__ __forceinline__ void fft_pass(float2* z, const Tw& tw, int n, int Ns, int twstep, unsigned nsm, int nss,
                                         int tid)
{
    constexpr int MAXB = (E + R - 1) / R;
    const int nb = n / R;
    const bool pow2 = (Ns & (Ns - 1)) == 0;
    // j mod Ns for j < nb: q = (j * nsm) >> nss equals j / Ns exactly (the host
    // picks nsm = ceil(2^nss / Ns) with 2^nss >= nb * Ns and checks every j),
    // in 24-bit full-rate multiplies instead of a 32-bit division
    auto jmod = [&](int j) __attribute__((always_inline)) {
        return pow2 ? (j & (Ns - 1)) : (int)((unsigned)j - __umul24(__umul24((unsigned)j, nsm) >> nss, (unsigned)Ns));
    };
    float2 v[MAXB][R];
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
        const int j = tid + b * THREADS;
        if (j < nb) {
            const int jm = jmod(j);
            // W^(r ts) = (W^ts)^r: one table twiddle per butterfly, the rest by
            // recurrence (at most R - 2 extra roundings)
            const float2 w1 = tw(jm * twstep);
            float2 w = w1;
            v[b][0] = z[pix(j)];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                v[b][r] = cmul(z[pix(j + r * nb)], w);
                if (r + 1 < R) w = cmul(w, w1);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MAXB; ++b) {
        const int j = tid + b * THREADS;
        if (j < nb) {
            Dft<R>::run(v[b], tw, n);
            const int jm = jmod(j);
            const int d = (j - jm) * R + jm;
#pragma unroll
            for (int r = 0; r < R; ++r) z[pix(d + r * Ns)] = v[b][r];
        }
    }
    __syncthreads();
}

// Waves per SIMD asked of the LDS FFT kernels: six keep them within 80 VGPRs, so
// that as many workgroups share a CU as their LDS allows (768 threads, n in
// (4096, 6144]: two instead of one; 384 threads: four instead of three) and one
// workgroup's barriers overlap the others' passes (shorter rows: their calls are
// mostly too small to fill the chip).  16 slices, n = 3072: the polar
// pass 0.51 -> 0.44 ms, the second inverse transform 0.37 -> 0.31.  The filter that
// takes one pair a workgroup spills 6 to 8 registers for it at 384 and 512 threads and
// runs as before (FP16 rows, 8 slices, 200 angles: n = 2400 209 us, 3600 369, 4050 412).
template <int THREADS> constexpr int fft_wpe() { return THREADS >= 384 && THREADS <= 768 ? 6 : 1; }

struct FftK {
    int n, nstages;
    int radix[24];
    // per stage: twiddle step n / (Ns R) and the exact-division pair for Ns
    int twstep[24];
    unsigned nsm[24];
    int nss[24];
};

template <int THREADS, int E>
__device__ void fft_run(float2* z, const Tw& tw, const FftK& p, int tid = threadIdx.x)
{
    int Ns = 1;
    for (int st = 0; st < p.nstages; ++st) {
        const int R = p.radix[st];
        const int ts = p.twstep[st], ss = p.nss[st];
        const unsigned sm = p.nsm[st];
        switch (R) {
        case 8: fft_pass<8, THREADS, E>(z, tw, p.n, Ns, ts, sm, ss, tid); break;
        case 4: fft_pass<4, THREADS, E>(z, tw, p.n, Ns, ts, sm, ss, tid); break;
        case 2: fft_pass<2, THREADS, E>(z, tw, p.n, Ns, ts, sm, ss, tid); break;
        case 3: fft_pass<3, THREADS, E>(z, tw, p.n, Ns, ts, sm, ss, tid); break;
        default: fft_pass<5, THREADS, E>(z, tw, p.n, Ns, ts, sm, ss, tid); break;
        }
        Ns *= R;
    }
}

struct FilterK {
    const float* tomo;
    void* q;
    const float2* H;
    const float2* tw; // [128 + n/128 + 1]: lo table then hi table
    const double* g; // direct-convolution kernel (FP64)
    const float* wa;
    int N, A, S, npad, L, tlo, W, none;
    int SB; // slices per interleaved group
    int split; // FP32: entries as three bf16 pieces, [3][W] 8-byte entries per row (the matrix backprojector's)
    int rg, ra; // row index of (group, angle): g rg + a ra
    float* rows; // k_filter_fft_entry_lds only: non-null -> windows to rows [S][A][W] instead of q
};

// block -> (group, angle, pair): rows (s0 = g*SB + 2*pair, a) and (s0 + 1, a)
struct PairIdx {
    int g, a, s0;
};
__device__ __forceinline__ PairIdx pair_index(const FilterK& k)
{
    const int pairs = k.SB / 2;
    PairIdx r;
    const int b = blockIdx.x;
    const int pr = b % pairs;
    const int ga = b / pairs;
    r.a = ga % k.A;
    r.g = ga / k.A;
    r.s0 = r.g * k.SB + 2 * pr;
    return r;
}

// padded rows of slices s0, s0+1 (missing slices read as zero) into z
template <int THREADS>
__device__ __forceinline__ void load_pair(const FilterK& k, const PairIdx& ix, float2* z)
{
    const bool v0 = ix.s0 < k.S, v1 = ix.s0 + 1 < k.S;
    const float* r0 = k.tomo + ((size_t)ix.s0 * k.A + ix.a) * k.N;
    const float* r1 = r0 + (size_t)k.A * k.N;
    for (int m = threadIdx.x; m < k.npad; m += THREADS) {
        int ii = m - k.L;
        ii = ii < 0 ? 0 : (ii > k.N - 1 ? k.N - 1 : ii);
        z[pix(m)] = make_float2(v0 ? r0[ii] : 0.0f, v1 ? r1[ii] : 0.0f);
    }
}

template <typename OT> struct Pair2;
template <> struct Pair2<float> {
    using T = float2;
    __device__ static __forceinline__ T make(float a, float b) { return make_float2(a, b); }
};
template <> struct Pair2<__half> {
    using T = __half2;
    __device__ static __forceinline__ T make(float a, float b) { return __floats2half2_rn(a, b); }
};

__device__ __forceinline__ size_t row_index(const FilterK& k, int g, int a)
{
    return (size_t)g * k.rg + (size_t)a * k.ra;
}

// entry w of (group, angle) row `ga`: four slices, as they are or in pieces
__device__ __forceinline__ void store_entry(const FilterK& k, size_t ga, int w, float4 v)
{
    if (k.split) {
        uint2 h, m, l;
        split4(v, h, m, l);
        uint2* d = static_cast<uint2*>(k.q) + ga * 3 * k.W + w;
        d[0] = h;
        d[k.W] = m;
        d[2 * (size_t)k.W] = l;
    } else {
        (static_cast<float4*>(k.q) + ga * k.W)[w] = v;
    }
}

// two slices of an entry in pieces: words `pr` of the three 8-byte entries
__device__ __forceinline__ void store_pair_split(const FilterK& k, const PairIdx& ix, int w, float v0, float v1)
{
    uint2 h, m, l;
    split4(make_float4(v0, v1, 0.0f, 0.0f), h, m, l);
    unsigned* d = static_cast<unsigned*>(k.q) + (row_index(k, ix.g, ix.a) * 3 * k.W + w) * 2 + (ix.s0 - ix.g * 4) / 2;
    d[0] = h.x;
    d[2 * (size_t)k.W] = m.x;
    d[4 * (size_t)k.W] = l.x;
}

// window store: bins [tlo, tlo + W) of both rows, times the angle weight
template <typename OT, int THREADS>
__device__ __forceinline__ void store_pair(const FilterK& k, const PairIdx& ix, const float2* z, float sign1)
{
    using P2 = typename Pair2<OT>::T;
    P2* dst = reinterpret_cast<P2*>(static_cast<OT*>(k.q) + (row_index(k, ix.g, ix.a) * k.W) * k.SB +
                                    (ix.s0 - ix.g * k.SB));
    const int stride = k.SB / 2; // in pairs
    const float wv = k.wa[ix.a];
    for (int w = threadIdx.x; w < k.W; w += THREADS) {
        const int T = k.tlo + w;
        float v0 = 0.0f, v1 = 0.0f;
        if (T >= 0 && T < k.npad) {
            const float2 zv = z[pix(T)];
            v0 = zv.x * wv;
            v1 = sign1 * zv.y * wv;
        }
        if (sizeof(OT) == 4 && k.split) store_pair_split(k, ix, w, v0, v1);
        else dst[(size_t)w * stride] = Pair2<OT>::make(v0, v1);
    }
}

template <typename OT, int THREADS, int E>
__global__ __launch_bounds__(THREADS, fft_wpe<THREADS>()) void k_filter_fft(FilterK a, FftK p)
{
    extern __shared__ float2 z[]; // [lds_elems(npad)] padded data, then the twiddle tables
    float2* tws = z + lds_elems(a.npad);
    const int ntw = 128 + a.npad / 128 + 1;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = a.tw[k];
    const Tw tw{tws, tws + 128};
    const PairIdx ix = pair_index(a);
    load_pair<THREADS>(a, ix, z);
    __syncthreads();
    if (a.none) {
        store_pair<OT, THREADS>(a, ix, z, 1.0f);
        return;
    }
    fft_run<THREADS, E>(z, tw, p);
    for (int k = threadIdx.x; k < a.npad; k += THREADS) {
        const float2 v = cmul(z[pix(k)], a.H[k]);
        z[pix(k)] = make_float2(v.x, -v.y);
    }
    __syncthreads();
    fft_run<THREADS, E>(z, tw, p);
    store_pair<OT, THREADS>(a, ix, z, -1.0f);
}

// Whole-entry form: one workgroup filters every slice pair of one (slice
// group, angle) in turn through the same LDS and stores full 16-byte entries
// of the interleaved rows (SB slices per bin), so no 64-byte line is written
// in halves by two workgroups.  The filtered window of the earlier pairs
// waits in registers: J window bins per thread (the host picks this form
// when W <= J * THREADS).  The arithmetic of each pair is that of
// k_filter_fft, so both forms store the same values.
template <typename OT, int THREADS, int E, int J>
__global__ __launch_bounds__(THREADS) void k_filter_fft_entry(FilterK a, FftK p)
{
    constexpr int SB = sizeof(OT) == 4 ? 4 : 8;
    constexpr int PAIRS = SB / 2;
    extern __shared__ float2 z[];
    float2* tws = z + lds_elems(a.npad);
    const int ntw = 128 + a.npad / 128 + 1;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = a.tw[k];
    const Tw tw{tws, tws + 128};
    const int ang = blockIdx.x % a.A, g = blockIdx.x / a.A;
    const float wv = a.wa[ang];
    const float sign1 = a.none ? 1.0f : -1.0f;
    float2 hold[PAIRS][J];
#pragma unroll
    for (int pr = 0; pr < PAIRS; ++pr) {
        const PairIdx ix{g, ang, g * SB + 2 * pr};
        __syncthreads(); // the twiddles are in; the previous pair's window reads are done
        load_pair<THREADS>(a, ix, z);
        __syncthreads();
        if (!a.none) {
            fft_run<THREADS, E>(z, tw, p);
            for (int k = threadIdx.x; k < a.npad; k += THREADS) {
                const float2 v = cmul(z[pix(k)], a.H[k]);
                z[pix(k)] = make_float2(v.x, -v.y);
            }
            __syncthreads();
            fft_run<THREADS, E>(z, tw, p);
        }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int T = a.tlo + (int)threadIdx.x + j * THREADS;
            float2 v = make_float2(0.0f, 0.0f);
            if ((int)threadIdx.x + j * THREADS < a.W && T >= 0 && T < a.npad) {
                const float2 zv = z[pix(T)];
                v = make_float2(zv.x * wv, sign1 * zv.y * wv);
            }
            hold[pr][j] = v;
        }
    }
    uint4* dst = reinterpret_cast<uint4*>(static_cast<OT*>(a.q)) + row_index(a, g, ang) * a.W;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int w = (int)threadIdx.x + j * THREADS;
        if (w >= a.W) continue;
        uint4 e;
        if constexpr (SB == 4) {
            store_entry(a, row_index(a, g, ang), w,
                        make_float4(hold[0][j].x, hold[0][j].y, hold[1][j].x, hold[1][j].y));
            continue;
        } else {
            unsigned u[PAIRS];
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                const __half2 h = __floats2half2_rn(hold[q][j].x, hold[q][j].y);
                u[q] = *reinterpret_cast<const unsigned*>(&h);
            }
            e = make_uint4(u[0], u[1], u[2], u[3]);
        }
        dst[w] = e;
    }
}

// Whole-entry form for FP32 rows with the first pair's filtered window kept
// in LDS (after the twiddle tables) instead of registers: without the held
// window and with the register budget of WPE waves per SIMD (80 VGPRs at 768
// threads), two workgroups fit a CU (twice 77 KB of LDS at n = 6144), so one
// workgroup's barriers overlap the other's passes.  The arithmetic of each
// pair is that of k_filter_fft, so the stored entries are the same bit for
// bit.
template <int THREADS, int E, int WPE, bool ROWS>
__global__ __launch_bounds__(THREADS, WPE) void k_filter_fft_entry_lds(FilterK a, FftK p)
{
    extern __shared__ float2 z[];
    float2* tws = z + lds_elems(a.npad);
    const int ntw = 128 + a.npad / 128 + 1;
    float2* win = tws + ntw; // [W]: pair 0's window
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = a.tw[k];
    const Tw tw{tws, tws + 128};
    const int ang = blockIdx.x % a.A, g = blockIdx.x / a.A;
    const float wv = a.wa[ang];
    const float sign1 = a.none ? 1.0f : -1.0f;
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
        const PairIdx ix{g, ang, g * 4 + 2 * pr};
        __syncthreads(); // the twiddles are in; the previous pair's window reads are done
        load_pair<THREADS>(a, ix, z);
        __syncthreads();
        if (!a.none) {
            fft_run<THREADS, E>(z, tw, p);
            for (int k = threadIdx.x; k < a.npad; k += THREADS) {
                const float2 v = cmul(z[pix(k)], a.H[k]);
                z[pix(k)] = make_float2(v.x, -v.y);
            }
            __syncthreads();
            fft_run<THREADS, E>(z, tw, p);
        }
        for (int w = threadIdx.x; w < a.W; w += THREADS) {
            const int T = a.tlo + w;
            float2 v = make_float2(0.0f, 0.0f);
            if (T >= 0 && T < a.npad) {
                const float2 zv = z[pix(T)];
                v = make_float2(zv.x * wv, sign1 * zv.y * wv);
            }
            if (pr == 0) {
                win[w] = v; // read back by the same thread
            } else if (ROWS) {
                // the group's four rows of this angle, each written by this
                // workgroup only and after all of them were read (in place
                // when rows is tomo)
                const float2 h = win[w];
                const int s0 = g * 4;
                const size_t ss = (size_t)a.A * a.W;
                float* r0 = a.rows + ((size_t)s0 * a.A + ang) * a.W + w;
                if (s0 < a.S) r0[0] = h.x;
                if (s0 + 1 < a.S) r0[ss] = h.y;
                if (s0 + 2 < a.S) r0[2 * ss] = v.x;
                if (s0 + 3 < a.S) r0[3 * ss] = v.y;
            } else {
                const float2 h = win[w];
                store_entry(a, row_index(a, g, ang), w, make_float4(h.x, h.y, v.x, v.y));
            }
        }
    }
}

// bin w of both rows, FP64 sums
template <typename OT>
__device__ __forceinline__ void store_sum(const FilterK& a, const PairIdx& ix, int w, double s0, double s1)
{
    const float wv = a.wa[ix.a];
    const float v0 = (float)s0 * wv, v1 = (float)s1 * wv;
    if (sizeof(OT) == 4 && a.split) {
        store_pair_split(a, ix, w, v0, v1);
    } else {
        using P2 = typename Pair2<OT>::T;
        P2* dst = reinterpret_cast<P2*>(static_cast<OT*>(a.q) + (row_index(a, ix.g, ix.a) * a.W) * a.SB +
                                        (ix.s0 - ix.g * a.SB));
        dst[(size_t)w * (a.SB / 2)] = Pair2<OT>::make(v0, v1);
    }
}

// direct circular convolution for sizes the LDS FFT does not cover:
// q[m] = sum_j g[(m - j) mod n] u[j], bins [w0, w1) of the pair in z
template <typename OT, int THREADS>
__device__ __forceinline__ void direct_window(const FilterK& a, const PairIdx& ix, const float2* z, int w0, int w1)
{
    for (int w = w0 + (int)threadIdx.x; w < w1; w += THREADS) {
        const int T = a.tlo + w;
        // FP64 kernel and sums: the kernel sums to ~0 (no DC), so n FP32
        // products would lose ~sqrt(n) ulps of a cancelling sum
        double s0 = 0.0, s1 = 0.0;
        if (T >= 0 && T < a.npad) {
            int d = T; // (T - j) mod n, j = 0..n-1
            for (int j = 0; j < a.npad; ++j) {
                const double gv = a.g[d];
                const float2 zj = z[pix(j)];
                s0 = fma(gv, (double)zj.x, s0);
                s1 = fma(gv, (double)zj.y, s1);
                d = (d == 0) ? a.npad - 1 : d - 1;
            }
        }
        store_sum<OT>(a, ix, w, s0, s1);
    }
}

template <typename OT>
__global__ __launch_bounds__(256) void k_filter_direct(FilterK a)
{
    extern __shared__ float2 z[]; // u0 + i u1; the filtered values go straight to the staged rows
    const PairIdx ix = pair_index(a);
    load_pair<256>(a, ix, z);
    __syncthreads();
    if (a.none) {
        store_pair<OT, 256>(a, ix, z, 1.0f);
        return;
    }
    direct_window<OT, 256>(a, ix, z, 0, a.W);
}

// ---- the same convolution by FP64 transforms (k_filter_conv) --------------
//
// q[T] = sum_{i < N} g[(T - L - i) mod n] r[i] + r[0] e0[T] + r[N - 1] e1[T]: the
// padding's constant runs are two tables of partial sums of g, the interior is a
// linear convolution of N samples.  A workgroup computes `chunk` outputs of two
// rows (one complex signal: the kernel is real) with transforms of
// len >= N + chunk - 1 in LDS: decimation in frequency forward, the product with
// the kernel's spectrum in the order that leaves, decimation in time back, so
// nothing is reordered.  Passes of radix 8 in registers, the first reads the
// rows, the last writes the bins; one complex of padding per 8 keeps the passes'
// strides off each other's banks.  FP64 throughout, like the direct form: an
// FP32 transform's rounding (1e-6) would be ten times this path's error.
//
// What bounds it: twiddles and spectrum from L2 (16 bytes each; three twiddles a
// butterfly, the others their products) and LDS passes.  21 slices of 901 x 1301
// padded to 2602 (len 4096): 0.36 ms, the direct sum 22.7 (n x window products a
// row); 8 of 300 x 2047 padded to 6141 (len 8192): 0.13 against 9.7.
constexpr int CV_THREADS = 512;
constexpr int CV_MAX_LEN = 8192; // 147 KB of LDS
constexpr int CV_MAX_CHUNKS = 16;
// Padded rows from here on, direct -> transforms, us for 19200 row pairs of an FBP:
// 43 rays padded to 129 160 -> 178, 47 to 141 169 -> 178, 51 to 153 187 -> 181, 67 to
// 201 452 -> 231; a longer row has more bins to sum, 65 to 130 233 -> 215 (few pairs are
// 1 to 2 us faster by transforms at all of these).
constexpr int CV_MIN_N = 136, CV_LEAST_N = 128, CV_LEAST_RAYS = 60;
// The low-pass keeps N bins of a row, a wave of the direct sum per 64: 57 rays padded to
// 171 108 -> 178 us, 69 to 138 160 -> 181, 77 to 154 182 -> 179, 67 to 201 230 -> 190.
constexpr int CV_LEAST_LOWPASS = 300; // waves times padded bins
// binary orders of magnitude between two rows from which each is summed by itself:
// below, the larger one's rounding stays 2^8 below an FP32 rounding of the smaller
constexpr unsigned CV_APART = 20;
typedef double d2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int cpix(int e) { return e + (e >> 3); }
__host__ __device__ constexpr size_t conv_lds(int len) { return sizeof(double) * 2 * ((size_t)len + (size_t)(len >> 3) + 1); }

struct ConvK {
    const d2* spec;     // [chunks][len], permuted as the forward passes leave it, 1 / len folded in
    const d2* tw;       // [len] exp(-2 pi i k / len)
    const double* edge; // [2][n]: e0, e1
    int len, chunk, first, count; // outputs per chunk; first chunk and chunks of this launch
    int passes, radix[8];
    unsigned rows; // (group, angle) pairs
};

template <typename V> __device__ __forceinline__ V zmul(V a, V b)
{
    return V{fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)};
}
template <typename V> __device__ __forceinline__ V zconj(V a) { return V{a.x, -a.y}; }
// a * -i (forward), a * i (inverse)
template <bool INV, typename V> __device__ __forceinline__ V zrot(V a) { return INV ? V{-a.y, a.x} : V{a.y, -a.x}; }

template <bool INV, typename V> __device__ __forceinline__ void zdft4(V& a, V& b, V& c, V& d)
{
    const V s = a + c, t = a - c, u = b + d, v = zrot<INV>(b - d);
    a = s + u; b = t + v; c = s - u; d = t - v;
}

// cos and sin of 2 pi m / R, by their series at compile time
constexpr double series(double x, bool sine)
{
    double term = sine ? x : 1.0, sum = term;
    for (int k = sine ? 1 : 0; k < 40; k += 2) {
        term *= -x * x / ((k + 1.0) * (k + 2.0));
        sum += term;
    }
    return sum;
}
template <int R> struct Roots {
    double c[R], s[R];
    constexpr Roots() : c(), s()
    {
        for (int m = 0; m < R; ++m) {
            const double x = 6.28318530717958647693 * (2 * m > R ? m - R : m) / R;
            c[m] = series(x, false);
            s[m] = series(x, true);
        }
    }
};

// DFT of v[0..R) in place, W = exp(-+ 2 pi i / R)
template <int R, bool INV, typename V> __device__ __forceinline__ void zdft(V (&v)[R])
{
    using E = decltype(v[0].x + v[0].x);
    if constexpr (R == 3) {
        const E h = (E)0.86602540378443864676; // sin 60 degrees
        const V s = v[1] + v[2], m = v[0] - (E)0.5 * s, r = zrot<INV>(h * (v[1] - v[2]));
        v[0] = v[0] + s; v[1] = m + r; v[2] = m - r;
    } else if constexpr (R == 2) {
        const V a = v[0], b = v[1];
        v[0] = a + b; v[1] = a - b;
    } else if constexpr (R == 4) {
        zdft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 5) {
        const E c1 = (E)0.30901699437494742410, c2 = (E)-0.80901699437494742410; // cos 72, cos 144 degrees
        const E s1 = (E)0.95105651629515357212, s2 = (E)0.58778525229247312917;  // their sines
        const V p1 = v[1] + v[4], p2 = v[2] + v[3], q1 = v[1] - v[4], q2 = v[2] - v[3];
        const V m1 = v[0] + c1 * p1 + c2 * p2, m2 = v[0] + c2 * p1 + c1 * p2;
        const V r1 = zrot<INV>(s1 * q1 + s2 * q2), r2 = zrot<INV>(s2 * q1 - s1 * q2);
        v[0] = v[0] + p1 + p2;
        v[1] = m1 + r1; v[4] = m1 - r1; v[2] = m2 + r2; v[3] = m2 - r2;
    } else if constexpr (R == 8) {
        const E h = (E)0.70710678118654752440; // sqrt(1/2)
        zdft4<INV>(v[0], v[2], v[4], v[6]);
        zdft4<INV>(v[1], v[3], v[5], v[7]);
        // odd part times W_8^k, k = 0..3 (in v[1], v[3], v[5], v[7])
        const V o1 = h * (v[3] + zrot<INV>(v[3])), o2 = zrot<INV>(v[5]), o3 = h * (zrot<INV>(v[7]) - v[7]);
        const V e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = e0 + o0; v[4] = e0 - o0;
        v[1] = e1 + o1; v[5] = e1 - o1;
        v[2] = e2 + o2; v[6] = e2 - o2;
        v[3] = e3 + o3; v[7] = e3 - o3;
    } else {
        // R = A B: A-point transforms over n1 of v[B n1 + n2], W_R^(n2 k1), B-point
        // transforms over n2
        static_assert(R == 6 || R == 10 || R == 12 || R == 16, "radix");
        constexpr int A = R == 6 ? 3 : (R == 10 ? 5 : 4), B = R / A;
        constexpr Roots<R> W;
        V t[B][A];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[B * n1 + n2];
            zdft<A, INV>(t[n2]);
#pragma unroll
            for (int k1 = 1; k1 < A; ++k1)
                if (n2 > 0) t[n2][k1] = zmul(t[n2][k1], V{(E)W.c[n2 * k1], (E)(INV ? W.s[n2 * k1] : -W.s[n2 * k1])});
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            V u[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) u[n2] = t[n2][k1];
            zdft<B, INV>(u);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = u[k2];
        }
    }
}
// v[q] *= W_len^(x q) (conjugate for the inverse): the powers of two from the
// table, the others their products
template <int R, bool INV, typename V> __device__ __forceinline__ void ztwiddle(V (&v)[R], const V* tw, int x)
{
    V w[R];
#pragma unroll
    for (int q = 1; q < R; ++q) {
        int top = 1;
        while (2 * top <= q) top *= 2;
        w[q] = q == top ? tw[q * x] : zmul(w[top], w[q - top]);
    }
#pragma unroll
    for (int q = 1; q < R; ++q) v[q] = zmul(v[q], INV ? zconj(w[q]) : w[q]);
}

// maximum over the wave, in lane 63
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
#define RAFT_DPP_MAX(CTRL) v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false))
    RAFT_DPP_MAX(0x111); // row_shr 1, 2, 4, 8: lane 15 of every row of 16
    RAFT_DPP_MAX(0x112);
    RAFT_DPP_MAX(0x114);
    RAFT_DPP_MAX(0x118);
    RAFT_DPP_MAX(0x142); // row_bcast 15, 31
    RAFT_DPP_MAX(0x143);
#undef RAFT_DPP_MAX
    return v;
}

// the first forward pass, from the rows; returns the bits of the largest magnitude read
// of each row (a NaN's lie above an infinity's)
template <int R>
__device__ __forceinline__ uint2 conv_first(const FilterK& a, const PairIdx& ix, const ConvK& c, d2* z)
{
    const bool h0 = ix.s0 < a.S, h1 = ix.s0 + 1 < a.S;
    const float* r0 = a.tomo + ((size_t)ix.s0 * a.A + ix.a) * a.N;
    const float* r1 = r0 + (size_t)a.A * a.N;
    const int M = c.len / R;
    uint2 m = make_uint2(0u, 0u);
    for (int j = threadIdx.x; j < M; j += CV_THREADS) {
        d2 v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const int i = j + t * M;
            const float x0 = h0 && i < a.N ? r0[i] : 0.0f, x1 = h1 && i < a.N ? r1[i] : 0.0f;
            m.x = max(m.x, __float_as_uint(x0) & 0x7fffffffu);
            m.y = max(m.y, __float_as_uint(x1) & 0x7fffffffu);
            v[t] = d2{(double)x0, (double)x1};
        }
        zdft<R, false>(v);
        ztwiddle<R, false>(v, c.tw, j);
#pragma unroll
        for (int t = 0; t < R; ++t) z[cpix(j + t * M)] = v[t];
    }
    return m;
}
// a pass over blocks of B elements
template <int R, bool INV> __device__ __forceinline__ void conv_pass(const ConvK& c, int B, d2* z)
{
    const int M = B / R, lm = 31 - __clz(M), step = c.len / B; // M is a power of two
    for (int b = threadIdx.x; b < c.len / R; b += CV_THREADS) {
        const int j = b & (M - 1), base = (b >> lm) * B + j;
        d2 v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) v[t] = z[cpix(base + t * M)];
        if (INV) ztwiddle<R, true>(v, c.tw, step * j);
        zdft<R, INV>(v);
        if (!INV) ztwiddle<R, false>(v, c.tw, step * j);
#pragma unroll
        for (int t = 0; t < R; ++t) z[cpix(base + t * M)] = v[t];
    }
}
// the last inverse pass, to the bins
template <typename OT, int R>
__device__ __forceinline__ void conv_last(const FilterK& a, const PairIdx& ix, const ConvK& c, int T0, uint2 m,
                                          const d2* z)
{
    const float* r0 = a.tomo + ((size_t)ix.s0 * a.A + ix.a) * a.N;
    const float* r1 = r0 + (size_t)a.A * a.N;
    const bool h0 = ix.s0 < a.S, h1 = ix.s0 + 1 < a.S;
    const double l0 = h0 ? r0[0] : 0.0f, l1 = h1 ? r1[0] : 0.0f;
    const double u0 = h0 ? r0[a.N - 1] : 0.0f, u1 = h1 ? r1[a.N - 1] : 0.0f;
    const int M = c.len / R;
    const int lo = max(T0, a.tlo), hi = min(min(T0 + c.chunk, a.npad), a.tlo + a.W); // this chunk's bins
    for (int j = threadIdx.x; j < M; j += CV_THREADS) {
        d2 v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) v[t] = z[cpix(j + t * M)];
        ztwiddle<R, true>(v, c.tw, j);
        zdft<R, true>(v);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const int T = T0 + j + t * M;
            if (T < lo || T >= hi) continue;
            const double e0 = c.edge[T], e1 = c.edge[a.npad + T];
            store_sum<OT>(a, ix, T - a.tlo, m.x ? fma(u0, e1, fma(l0, e0, v[t].x)) : 0.0,
                          m.y ? fma(u1, e1, fma(l1, e0, v[t].y)) : 0.0);
        }
    }
}

template <typename OT> __global__ __launch_bounds__(CV_THREADS, 4) void k_filter_conv(FilterK a, ConvK c)
{
    extern __shared__ __align__(16) char conv_smem[];
    d2* z = reinterpret_cast<d2*>(conv_smem);
    // the pairs and chunks of a row on one XCD (workgroups go to the 8 XCDs round
    // robin): their interleaved stores share cache lines
    const unsigned per = (unsigned)(a.SB / 2) * c.count;
    const unsigned ga = (blockIdx.x >> 3) / per * 8u + (blockIdx.x & 7u);
    if (ga >= c.rows) return;
    const unsigned sub = (blockIdx.x >> 3) % per;
    PairIdx ix;
    ix.a = (int)(ga % (unsigned)a.A);
    ix.g = (int)(ga / (unsigned)a.A);
    ix.s0 = ix.g * a.SB + 2 * (int)(sub / c.count);
    const int ch = c.first + (int)(sub % c.count);
    const int T0 = ch * c.chunk;
    // bins outside [0, n) are zero: the launch's first and last chunk clear them
    if (ch == c.first)
        for (int w = threadIdx.x; w < min(-a.tlo, a.W); w += CV_THREADS) store_sum<OT>(a, ix, w, 0.0, 0.0);
    if (ch == c.first + c.count - 1)
        for (int w = max(a.npad - a.tlo, 0) + (int)threadIdx.x; w < a.W; w += CV_THREADS)
            store_sum<OT>(a, ix, w, 0.0, 0.0);
    if (ix.s0 >= a.S) { // padding slices of the last group
        for (int T = max(T0, a.tlo) + (int)threadIdx.x; T < min(min(T0 + c.chunk, a.npad), a.tlo + a.W); T += CV_THREADS)
            store_sum<OT>(a, ix, T - a.tlo, 0.0, 0.0);
        return;
    }

    uint2 m;
    switch (c.radix[0]) {
    case 3: m = conv_first<3>(a, ix, c, z); break;
    case 4: m = conv_first<4>(a, ix, c, z); break;
    case 5: m = conv_first<5>(a, ix, c, z); break;
    default: m = conv_first<8>(a, ix, c, z); break;
    }
    // over the workgroup, through LDS of its own behind the transform (a static array
    // would not fit beside the longest rows the direct sum takes)
    uint2* part = reinterpret_cast<uint2*>(conv_smem + conv_lds(c.len));
    m.x = wave_max(m.x);
    m.y = wave_max(m.y);
    if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = m;
    __syncthreads();
    m = make_uint2(0u, 0u);
#pragma unroll
    for (int w = 0; w < CV_THREADS / 64; ++w) {
        m.x = max(m.x, part[w].x);
        m.y = max(m.y, part[w].y);
    }
    // The rows share the transform's rounding, 2^-52 of the larger one: a pair too far
    // apart takes the direct sum, and a row of zeros stays zero.
    const bool apart = m.x > 0u && m.y > 0u && max(m.x, m.y) - min(m.x, m.y) >= CV_APART << 23;
    if (max(m.x, m.y) >= 0x7f800000u || apart) {
        __syncthreads(); // `part` is read
        // a row that is not finite, or far larger, must not reach the other of the pair
        load_pair<CV_THREADS>(a, ix, reinterpret_cast<float2*>(z));
        __syncthreads();
        direct_window<OT, CV_THREADS>(a, ix, reinterpret_cast<const float2*>(z), max(T0 - a.tlo, 0),
                                      min(min(T0 + c.chunk, a.npad) - a.tlo, a.W));
        return;
    }
    int B = c.len / c.radix[0];
    int p = 1;
    for (; p < c.passes - 1; ++p) {
        if (c.radix[p] == 4) conv_pass<4, false>(c, B, z);
        else conv_pass<8, false>(c, B, z);
        B /= c.radix[p];
        __syncthreads();
    }
    // the last forward pass (radix 8, blocks of 8: no twiddles), the product and
    // the first inverse pass in registers
    const d2* spec = c.spec + (size_t)ch * c.len;
    for (int b = threadIdx.x; b < c.len / 8; b += CV_THREADS) {
        d2 v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = z[cpix(8 * b) + t];
        zdft<8, false>(v);
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = zmul(v[t], spec[8 * b + t]);
        zdft<8, true>(v);
#pragma unroll
        for (int t = 0; t < 8; ++t) z[cpix(8 * b) + t] = v[t];
    }
    __syncthreads();
    for (p = c.passes - 2; p > 0; --p) {
        B *= c.radix[p];
        if (c.radix[p] == 4) conv_pass<4, true>(c, B, z);
        else conv_pass<8, true>(c, B, z);
        __syncthreads();
    }
    switch (c.radix[0]) {
    case 3: conv_last<OT, 3>(a, ix, c, T0, m, z); break;
    case 4: conv_last<OT, 4>(a, ix, c, T0, m, z); break;
    case 5: conv_last<OT, 5>(a, ix, c, T0, m, z); break;
    default: conv_last<OT, 8>(a, ix, c, T0, m, z); break;
    }
}

template <typename OT> void launch_conv(const FilterK& k, const FilterArgs& a, hipStream_t st)
{
    const ConvPlan& p = a.conv;
    ConvK c;
    c.spec = static_cast<const d2*>(a.conv_spec);
    c.tw = static_cast<const d2*>(a.conv_tw);
    c.edge = a.conv_edge;
    c.len = p.len; c.chunk = p.chunk; c.passes = p.passes;
    std::copy(p.radix, p.radix + 8, c.radix);
    // chunks that hold bins of the window (one at least, for the zeros outside [0, n))
    const int lo = std::min(std::max(k.tlo, 0), k.npad - 1), hi = std::min(std::max(k.tlo + k.W, 1), k.npad);
    c.first = lo / p.chunk;
    c.count = std::max((hi - 1) / p.chunk - c.first + 1, 1);
    c.rows = (unsigned)((long long)((k.S + k.SB - 1) / k.SB) * k.A);
    const long long blocks = ((long long)c.rows + 7) / 8 * 8 * (k.SB / 2) * c.count;
    if (blocks > 0x7fffffffLL) fail(RAFT_EUNSUPPORTED, "too many sinogram rows for one filter launch");
    const size_t lds = std::max(conv_lds(p.len) + CV_THREADS / 64 * sizeof(uint2), sizeof(float2) * lds_elems(k.npad));
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_filter_conv<OT>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_filter_conv<OT>), dim3((unsigned)blocks), dim3(CV_THREADS), lds, st, k, c);
}

// ---- FP32 rows of 64 x 8, 10, 12, 16 and 512 x 3, 4, 5, 6, 8, 10, 12, 16 bins ----
// ---- (k_filter_dif) ----
//
// The same passes in FP32 for the padded row itself (the circular convolution):
// radix M0 from the sinogram, radix 8 in LDS down to blocks of 8, the product
// with H (in the order that leaves) inside the last one, and back; the bins leave
// from the registers of the last pass.  A workgroup takes two slice pairs of an
// angle in turn and stores 16 bytes (FP16: 8) per bin; the first pair's window
// waits in LDS.
//
// Why instead of the transforms in natural order (k_filter_fft*): LDS passes and
// barriers bound those, and this form has 6 reads and 6 writes of LDS a pair
// instead of 10 and 10 (n = 6144) and 12 barriers instead of about 24; its
// twiddles come from tables in the lanes' order (products of two-level tables
// before), so the rows' error is about half.  Filter time before -> now: 64 slices
// of 2048 x 2048, n = 6144, FP32 rows in pieces 2.83 -> 1.64 ms, FP16 4.04 -> 1.52;
// per row pair at n = 512 / 1024 / 2048 / 4096 / 6144 / 8192 3.5 / 7.2 / 13.7 / 27.5 /
// 40.5 / 87.7 -> 1.7 / 3.5 / 9.2 / 20.7 / 28.0 / 51.0 ns.
typedef float f2 __attribute__((ext_vector_type(2)));
template <int M0, int E8> struct Dif {
    static constexpr int M = E8 == 3 ? 512 : 64, LEN = M0 * M, TH = LEN / 8;
    // waves per SIMD of as many workgroups as the LDS holds
    static constexpr int WPE = TH > 768 ? 4 : (TH == 640 || (M0 == 16 && E8 == 2) ? 5 : 6); // the last: registers
    static constexpr int PAD = LEN + LEN / 8 + 2; // complex values before the window
};

// v[q] *= W^(j q) (conjugate for the inverse) of a pass whose blocks have R M
// elements, from its table [q][j < M] (neighbouring lanes, neighbouring
// entries).  Powers below ONE and the multiples of ONE come from it, the others
// are one product: the radix-8 passes take all seven (their tables stay in the
// L1 cache; with products the error of the filtered rows grows by a fifth).
template <int R, int M, bool INV, int ONE> __device__ __forceinline__ void dif_twiddle(f2 (&v)[R], const f2* tw, int j)
{
    f2 w[R];
#pragma unroll
    for (int q = 1; q < R; ++q)
        w[q] = q < ONE || q % ONE == 0 ? tw[q * M + j] : zmul(w[q / ONE * ONE], w[q % ONE]);
#pragma unroll
    for (int q = 1; q < R; ++q) v[q] = zmul(v[q], INV ? zconj(w[q]) : w[q]);
}

template <int LEN, int TH, int B, bool INV> __device__ __forceinline__ void dif_pass(f2* z, const f2* tw, int b)
{
    constexpr int M = B / 8;
    const int j = b & (M - 1), base = (b / M) * B + j; // one butterfly a thread
    f2 v[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = z[cpix(base + t * M)];
    if (INV) dif_twiddle<8, M, true, 8>(v, tw, j);
    zdft<8, INV>(v);
    if (!INV) dif_twiddle<8, M, false, 8>(v, tw, j);
#pragma unroll
    for (int t = 0; t < 8; ++t) z[cpix(base + t * M)] = v[t];
}

template <typename OT, int M0, int E8, bool ROWS>
__global__ __launch_bounds__((Dif<M0, E8>::TH), (Dif<M0, E8>::WPE)) void k_filter_dif(FilterK a, const f2* __restrict__ H,
                                                                                   const f2* __restrict__ tw, unsigned rows)
{
    using D = Dif<M0, E8>;
    constexpr int M = D::M, TH = D::TH, LEN = D::LEN;
    constexpr bool F32 = sizeof(OT) == 4;
    extern __shared__ __align__(16) char conv_smem[];
    f2* z = reinterpret_cast<f2*>(conv_smem);
    f2* win = z + D::PAD;                         // [W]: the first pair's window (FP16: packed)
    unsigned* winh = reinterpret_cast<unsigned*>(win);
    // the halves of an FP16 entry on one XCD (see k_filter_conv)
    constexpr unsigned per = F32 ? 1 : 2;
    const unsigned ga = (blockIdx.x >> 3) / per * 8u + (blockIdx.x & 7u);
    if (ga >= rows) return;
    const int ang = (int)(ga % (unsigned)a.A), g = (int)(ga / (unsigned)a.A);
    const int s0 = g * a.SB + 4 * (int)((blockIdx.x >> 3) % per); // first of the four slices
    const float wv = a.wa[ang];
    const size_t ri = row_index(a, g, ang);
    const size_t ss = (size_t)a.A * a.N;

    auto store = [&](int w, f2 lo, f2 hi) __attribute__((always_inline)) {
        if constexpr (ROWS) {
            // the group's four rows of this angle, each written by this workgroup
            // only and after all of them were read (in place when rows is tomo)
            float* r = a.rows + ((size_t)s0 * a.A + ang) * a.W + w;
            const size_t rs = (size_t)a.A * a.W;
            if (s0 < a.S) r[0] = lo.x;
            if (s0 + 1 < a.S) r[rs] = lo.y;
            if (s0 + 2 < a.S) r[2 * rs] = hi.x;
            if (s0 + 3 < a.S) r[3 * rs] = hi.y;
        } else if constexpr (F32) {
            store_entry(a, ri, w, make_float4(lo.x, lo.y, hi.x, hi.y));
        } else {
            const __half2 h0 = __floats2half2_rn(lo.x, lo.y), h1 = __floats2half2_rn(hi.x, hi.y);
            reinterpret_cast<uint2*>(a.q)[(ri * a.W + w) * 2 + (s0 - g * a.SB) / 4] =
                make_uint2(*reinterpret_cast<const unsigned*>(&h0), *reinterpret_cast<const unsigned*>(&h1));
        }
    };
    // bins outside [0, n) are zero
    for (int w = threadIdx.x; w < a.W; w += TH)
        if (a.tlo + w < 0 || a.tlo + w >= LEN) store(w, f2{0.0f, 0.0f}, f2{0.0f, 0.0f});

#pragma unroll 1
    for (int pr = 0; pr < 2; ++pr) {
        // opaque: what depends on it (twiddles, addresses) is formed where it is
        // used, not kept in registers across the pairs
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int sl = s0 + 2 * pr;
        const bool h0 = sl < a.S, h1 = sl + 1 < a.S; // missing slices are zero
        const float* r0 = a.tomo + ((size_t)sl * a.A + ang) * a.N;
        for (int j = tid; j < M; j += TH) {
            f2 v[M0];
#pragma unroll
            for (int t = 0; t < M0; ++t) {
                const int i = min(max(j + t * M - a.L, 0), a.N - 1);
                v[t] = f2{h0 ? r0[i] : 0.0f, h1 ? r0[ss + i] : 0.0f};
            }
            zdft<M0, false>(v);
            dif_twiddle<M0, M, false, 4>(v, tw, j);
#pragma unroll
            for (int t = 0; t < M0; ++t) z[cpix(j + t * M)] = v[t];
        }
        __syncthreads();
        if constexpr (E8 == 3) {
            dif_pass<LEN, TH, 512, false>(z, tw + LEN, tid);
            __syncthreads();
        }
        dif_pass<LEN, TH, 64, false>(z, tw + LEN + 512, tid);
        __syncthreads();
        {
            const int b = 8 * tid;
            f2 v[8], h[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) h[t] = H[b + t];
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = z[cpix(b) + t];
            zdft<8, false>(v);
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = zmul(v[t], h[t]);
            zdft<8, true>(v);
#pragma unroll
            for (int t = 0; t < 8; ++t) z[cpix(b) + t] = v[t];
        }
        __syncthreads();
        dif_pass<LEN, TH, 64, true>(z, tw + LEN + 512, tid);
        __syncthreads();
        if constexpr (E8 == 3) {
            dif_pass<LEN, TH, 512, true>(z, tw + LEN, tid);
            __syncthreads();
        }
        for (int j = tid; j < M; j += TH) {
            f2 v[M0];
#pragma unroll
            for (int t = 0; t < M0; ++t) v[t] = z[cpix(j + t * M)];
            dif_twiddle<M0, M, true, 4>(v, tw, j);
            zdft<M0, true>(v);
#pragma unroll
            for (int t = 0; t < M0; ++t) {
                const int w = j + t * M - a.tlo;
                if ((unsigned)w >= (unsigned)a.W) continue;
                const f2 x = v[t] * wv;
                if (pr == 0) {
                    // read back by the same thread
                    if constexpr (F32) {
                        win[w] = x;
                    } else {
                        const __half2 hx = __floats2half2_rn(x.x, x.y);
                        winh[w] = *reinterpret_cast<const unsigned*>(&hx);
                    }
                } else if constexpr (F32) {
                    store(w, win[w], x);
                } else {
                    const __half2 hx = __floats2half2_rn(x.x, x.y);
                    reinterpret_cast<uint2*>(a.q)[(ri * a.W + w) * 2 + (s0 - g * a.SB) / 4] =
                        make_uint2(winh[w], *reinterpret_cast<const unsigned*>(&hx));
                }
            }
        }
        if (pr == 0) __syncthreads(); // the row is read before the next overwrites it
    }
}

template <typename OT, int M0, int E8> bool launch_dif_t(const FilterK& k, const FilterArgs& a, hipStream_t st)
{
    using D = Dif<M0, E8>;
    const size_t lds = sizeof(float2) * D::PAD + (size_t)k.W * (sizeof(OT) == 4 ? 8 : 4);
    if (lds > 160 * 1024) return false;
    const unsigned rows = (unsigned)((long long)((k.S + k.SB - 1) / k.SB) * k.A);
    const long long blocks = ((long long)rows + 7) / 8 * 8 * (k.SB / 4);
    if (blocks > 0x7fffffffLL) return false;
    const f2* H = reinterpret_cast<const f2*>(a.dif_H);
    const f2* tw = reinterpret_cast<const f2*>(a.dif_tw);
    const bool direct = sizeof(OT) == 4 && k.rows;
    const void* fn = reinterpret_cast<const void*>(&k_filter_dif<OT, M0, E8, false>);
    if constexpr (sizeof(OT) == 4)
        if (direct) fn = reinterpret_cast<const void*>(&k_filter_dif<OT, M0, E8, true>);
    RAFT_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    FilterK kk = k;
    unsigned rr = rows;
    void* args[] = {&kk, &H, &tw, &rr};
    RAFT_HIP(hipLaunchKernel(fn, dim3((unsigned)blocks), dim3(D::TH), args, lds, st));
    return true;
}
// false: not a size of this form
template <typename OT> bool launch_dif(const FilterK& k, const FilterArgs& a, hipStream_t st)
{
    switch (k.npad) {
    case 512: return launch_dif_t<OT, 8, 2>(k, a, st);
    case 640: return launch_dif_t<OT, 10, 2>(k, a, st);
    case 768: return launch_dif_t<OT, 12, 2>(k, a, st);
    case 1024: return launch_dif_t<OT, 16, 2>(k, a, st);
    case 1536: return launch_dif_t<OT, 3, 3>(k, a, st);
    case 2048: return launch_dif_t<OT, 4, 3>(k, a, st);
    case 2560: return launch_dif_t<OT, 5, 3>(k, a, st);
    case 3072: return launch_dif_t<OT, 6, 3>(k, a, st);
    case 4096: return launch_dif_t<OT, 8, 3>(k, a, st);
    case 5120: return launch_dif_t<OT, 10, 3>(k, a, st);
    case 6144: return launch_dif_t<OT, 12, 3>(k, a, st);
    case 8192: return launch_dif_t<OT, 16, 3>(k, a, st);
    default: return false;
    }
}

template <typename OT, int THREADS, int E>
void launch_fft_t(const FilterK& k, const FftK& p, int blocks, size_t lds, hipStream_t st)
{
    // whole-entry form when the window fits 4 bins per thread (every padding
    // of 2 or more at the benchmark sizes); blocks = (groups x angles) x pairs
    if (k.W <= 4 * THREADS && !std::getenv("RAFT_FILTER_PAIRS")) {
        const void* fn = reinterpret_cast<const void*>(&k_filter_fft_entry<OT, THREADS, E, 4>);
        RAFT_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL((k_filter_fft_entry<OT, THREADS, E, 4>), dim3(blocks / (k.SB / 2)), dim3(THREADS), lds, st,
                           k, p);
        return;
    }
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_filter_fft<OT, THREADS, E>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_filter_fft<OT, THREADS, E>), dim3(blocks), dim3(THREADS), lds, st, k, p);
}

template <int THREADS, int WPE, bool ROWS>
void launch_fft_lds_entry_t(const FilterK& k, const FftK& p, int blocks, size_t lds, hipStream_t st)
{
    const void* fn = reinterpret_cast<const void*>(&k_filter_fft_entry_lds<THREADS, 8, WPE, ROWS>);
    RAFT_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_filter_fft_entry_lds<THREADS, 8, WPE, ROWS>), dim3(blocks / 2), dim3(THREADS), lds, st, k,
                       p);
}

// the rows form is its own instantiation, so the staged-row form's code is
// unchanged by it
template <int THREADS, int WPE>
void launch_fft_lds_entry(const FilterK& k, const FftK& p, int blocks, size_t lds, hipStream_t st)
{
    if (k.rows) launch_fft_lds_entry_t<THREADS, WPE, true>(k, p, blocks, lds, st);
    else launch_fft_lds_entry_t<THREADS, WPE, false>(k, p, blocks, lds, st);
}

// THREADS = the smallest of 64, 128, 192, 256, 384, 512, 768, 1024 that is
// >= n/8, with E = 8 elements per thread; n in (8192, 16384] runs 1024
// threads with E = 16
template <typename OT>
bool launch_fft(const FilterK& k, const FftK& p, int threads, int blocks, size_t lds, hipStream_t st)
{
    // FP32 rows, n in (2048, 6144]: the two-workgroup form when two of them
    // fit a CU's 160 KB of LDS (RAFT_FFT_FORM=regs keeps the window in
    // registers instead: one workgroup per CU at n = 6144)
    const char* fe = std::getenv("RAFT_FFT_FORM");
    const size_t lw = lds + sizeof(float2) * (size_t)k.W;
    if (sizeof(OT) == 4 && p.n > 2048 && p.n <= 6144 && 2 * lw <= 160 * 1024 && !(fe && fe[0] == 'r') &&
        !std::getenv("RAFT_FILTER_PAIRS")) {
        if (p.n <= 3072) launch_fft_lds_entry<384, 3>(k, p, blocks, lw, st);
        else launch_fft_lds_entry<768, 6>(k, p, blocks, lw, st);
        return k.rows != nullptr;
    }
    if (p.n > 8192) {
        launch_fft_t<OT, 1024, 16>(k, p, blocks, lds, st);
        return false;
    }
    switch (threads) {
    case 64: launch_fft_t<OT, 64, 8>(k, p, blocks, lds, st); break;
    case 128: launch_fft_t<OT, 128, 8>(k, p, blocks, lds, st); break;
    case 192: launch_fft_t<OT, 192, 8>(k, p, blocks, lds, st); break;
    case 256: launch_fft_t<OT, 256, 8>(k, p, blocks, lds, st); break;
    case 384: launch_fft_t<OT, 384, 8>(k, p, blocks, lds, st); break;
    case 512: launch_fft_t<OT, 512, 8>(k, p, blocks, lds, st); break;
    case 768: launch_fft_t<OT, 768, 8>(k, p, blocks, lds, st); break;
    default: launch_fft_t<OT, 1024, 8>(k, p, blocks, lds, st); break;
    }
    return false;
}

// ---------------------------------------------------------------------------
// FBP by the Backprojection Slice Theorem (bst.cu:22-140, 251-312): mirrored
// half-rows of the filtered, padded projections -> C2C FFT -> sigma weights ->
// polar-to-Cartesian gather on the frequency grid -> 2-D inverse FFT.
// ---------------------------------------------------------------------------
struct BstPolarK {
    const float* q; // filtered padded rows, interleaved [G][A][n][4]
    float2* polar;  // [S][2A][n/2]
    const float2* tw;
    int n, A, S;
};

// row r of slice sl: r < A -> q[sl][r][n/2 - 1 - idx], r >= A -> q[sl][r - A][n/2 + idx],
// idx < n/2, weight 4 (2 at idx 0), zeros for idx >= n/2; forward FFT; times
// sigma_k = 2 / (n max(min(k, n - k), 1/2)).  Both rows of an angle are real,
// so one complex FFT carries the two: z = left + i right, and with
// W_k = conj(Z_{(n - k) mod n}), LEFT_k = (Z_k + W_k) / 2, RIGHT_k = (Z_k - W_k) / 2i.
template <int THREADS, int E>
__global__ __launch_bounds__(THREADS, fft_wpe<THREADS>()) void k_bst_polar(BstPolarK a, FftK p)
{
    extern __shared__ float2 z[];
    float2* tws = z + lds_elems(a.n);
    const int ntw = 128 + a.n / 128 + 1;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = a.tw[k];
    const Tw tw{tws, tws + 128};
    const int sl = blockIdx.x / a.A, ang = blockIdx.x % a.A;
    const int center = a.n / 2;
    const float* row = a.q + ((size_t)(sl / 4) * a.A + ang) * a.n * 4 + (sl % 4);
    for (int idx = threadIdx.x; idx < a.n; idx += THREADS) {
        float vl = 0.0f, vr = 0.0f;
        if (idx < a.n / 2) {
            const float w = idx == 0 ? 2.0f : 4.0f;
            vl = row[(size_t)(center - 1 - idx) * 4] * w;
            vr = row[(size_t)(center + idx) * 4] * w;
        }
        z[pix(idx)] = make_float2(vl, vr);
    }
    __syncthreads();
    fft_run<THREADS, E>(z, tw, p);
    // only radii [0, n/2) are ever interpolated (irho + 1 < n/2 - 1 + 1): rows
    // of n/2 entries
    const int h = a.n / 2;
    float2* outl = a.polar + ((size_t)sl * 2 * a.A + ang) * h;
    float2* outr = outl + (size_t)a.A * h;
    for (int k = threadIdx.x; k < h; k += THREADS) {
        const float sig = 2.0f / ((float)a.n * fmaxf(fminf((float)k, (float)(a.n - k)), 0.5f));
        const float2 zk = z[pix(k)];
        const float2 zm = z[pix(k == 0 ? 0 : a.n - k)];
        const float hs = 0.5f * sig;
        outl[k] = make_float2((zk.x + zm.x) * hs, (zk.y - zm.y) * hs);
        outr[k] = make_float2((zk.y + zm.y) * hs, (zm.x - zk.x) * hs);
    }
}

// One polar transform of k_bst_filter_polar: FFT of z, then the two real
// transforms it carries, separated and times sigma, into row offset `row` of
// the first slice (pa) and, if present, of the second (pb)
template <int THREADS, int E>
__device__ __forceinline__ void bst_pair_rows(float2* z, const Tw& tw, const FftK& p, float2* pa, float2* pb,
                                              size_t row, int h, int n, bool two)
{
    fft_run<THREADS, E>(z, tw, p);
    for (int k = threadIdx.x; k < h; k += THREADS) {
        const float sig = 2.0f / ((float)n * fmaxf(fminf((float)k, (float)(n - k)), 0.5f));
        const float2 zk = z[pix(k)];
        const float2 zm = z[pix(k == 0 ? 0 : n - k)];
        const float hs = 0.5f * sig;
        pa[row + k] = make_float2((zk.x + zm.x) * hs, (zk.y - zm.y) * hs);
        if (two) pb[row + k] = make_float2((zk.y + zm.y) * hs, (zm.x - zk.x) * hs);
    }
    __syncthreads();
}

// Filter and polar FFTs in one pass (the default BST form): one workgroup =
// one slice pair (s0, s0 + 1) of one angle.  The pair's padded rows are
// filtered as k_filter_fft does (one complex FFT carries both real rows), and
// the filtered values q_a = Re z wv, q_b = sign Im z wv -- the values the
// staged rows would hold -- go straight into the polar transforms, so the
// filtered rows are never written.  The polar rows of both slices come from
// two complex FFTs: z1 = w (q_a + i q_b) over the left half-rows (mirrored)
// and z2 = w (q_a + i q_b) over the right half-rows; the two real transforms
// each carries are separated by Hermitian symmetry as in k_bst_polar (first
// slice: (Z_k + conj Z_-k) / 2, second: (Z_k - conj Z_-k) / 2i), times sigma.
// The right half-rows wait in LDS (rh, n/2 entries) while z1 is transformed.
template <int THREADS, int E>
__global__ __launch_bounds__(THREADS, fft_wpe<THREADS>()) void k_bst_filter_polar(FilterK a, BstPolarK b, FftK p)
{
    extern __shared__ float2 z[];
    const int n = a.npad;
    float2* tws = z + lds_elems(n);
    const int ntw = 128 + n / 128 + 1;
    float2* rh = tws + ntw;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = a.tw[k];
    const Tw tw{tws, tws + 128};
    const PairIdx ix = pair_index(a);
    // the second pair of a last group with one slice has no slice: it writes
    // nothing (uniform for the workgroup, before any barrier)
    if (ix.s0 >= a.S) return;
    load_pair<THREADS>(a, ix, z);
    __syncthreads();
    float sign1 = 1.0f;
    if (!a.none) {
        fft_run<THREADS, E>(z, tw, p);
        for (int k = threadIdx.x; k < n; k += THREADS) {
            const float2 v = cmul(z[pix(k)], a.H[k]);
            z[pix(k)] = make_float2(v.x, -v.y);
        }
        __syncthreads();
        fft_run<THREADS, E>(z, tw, p);
        sign1 = -1.0f;
    }
    const int c = n / 2, h = n / 2;
    const float wv = a.wa[ix.a];
    // mirrored left half-rows through registers back into z (zeros past h),
    // right half-rows into rh
    {
        constexpr int JL = (E + 1) / 2; // h <= E THREADS / 2
        float2 lv[JL];
#pragma unroll
        for (int j = 0; j < JL; ++j) {
            const int idx = threadIdx.x + j * THREADS;
            lv[j] = make_float2(0.0f, 0.0f);
            if (idx < h) {
                const float w = idx == 0 ? 2.0f : 4.0f;
                const float2 zl = z[pix(c - 1 - idx)], zr = z[pix(c + idx)];
                lv[j] = make_float2(zl.x * wv * w, sign1 * zl.y * wv * w);
                rh[idx] = make_float2(zr.x * wv * w, sign1 * zr.y * wv * w);
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < JL; ++j) {
            const int idx = threadIdx.x + j * THREADS;
            if (idx < h) z[pix(idx)] = lv[j];
        }
    }
    for (int idx = h + threadIdx.x; idx < n; idx += THREADS) z[pix(idx)] = make_float2(0.0f, 0.0f);
    __syncthreads();
    const bool two = ix.s0 + 1 < a.S;
    float2* pa = b.polar + (size_t)ix.s0 * 2 * b.A * h;
    float2* pb = pa + (size_t)2 * b.A * h;
    bst_pair_rows<THREADS, E>(z, tw, p, pa, pb, (size_t)ix.a * h, h, n, two);
    for (int idx = threadIdx.x; idx < n; idx += THREADS) z[pix(idx)] = idx < h ? rh[idx] : make_float2(0.0f, 0.0f);
    __syncthreads();
    bst_pair_rows<THREADS, E>(z, tw, p, pa, pb, (size_t)(b.A + ix.a) * h, h, n, two);
}

// unnormalised inverse C2C FFT of `rows` rows of length n, in place
template <int THREADS, int E>
__global__ __launch_bounds__(THREADS, fft_wpe<THREADS>()) void k_ifft_rows(float2* data, const float2* twg, FftK p)
{
    extern __shared__ float2 z[];
    const int n = p.n;
    float2* tws = z + lds_elems(n);
    const int ntw = 128 + n / 128 + 1;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = twg[k];
    const Tw tw{tws, tws + 128};
    float2* row = data + (size_t)blockIdx.x * n;
    for (int k = threadIdx.x; k < n; k += THREADS) {
        const float2 v = row[k];
        z[pix(k)] = make_float2(v.x, -v.y);
    }
    __syncthreads();
    fft_run<THREADS, E>(z, tw, p);
    for (int k = threadIdx.x; k < n; k += THREADS) {
        const float2 v = z[pix(k)];
        row[k] = make_float2(v.x, -v.y);
    }
}

// polar (2A rows x n/2 radii) -> Cartesian frequency grid s x s (bst.cu:63-99),
// index arithmetic in FP64; the reference's weights (tfrac, 1 - tfrac) with
// tfrac = iarc - angle are kept as they are
__global__ void k_bst_p2c(const float2* polar, float2* cart, int n, int A2, int s, int S)
{
    const long long total = (long long)S * s * s;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int tx = (int)(e % s), ty = (int)((e / s) % s);
        const long long sl = e / ((long long)s * s);
        const int posx = tx - s / 2, posy = ty - s / 2;
        const double rho = (double)n * hypot((double)posx, (double)posy) / (double)s;
        const double angle = (double)A2 * (0.5 * atan2((double)posy, (double)posx) / M_PI + 0.5);
        const long long irho = (long long)rho;
        int iarc = (int)angle;
        float2 val = make_float2(0.0f, 0.0f);
        if (irho < n / 2 - 1) {
            const float pfrac = (float)(rho - (double)irho);
            const float tfrac = (float)((double)iarc - angle);
            iarc = iarc % A2;
            const int uarc = (iarc + 1) % A2;
            const int h = n / 2; // polar rows hold radii [0, n/2)
            const float2* P = polar + sl * (long long)A2 * h;
            const float2 a0 = P[(size_t)iarc * h + irho], a1 = P[(size_t)iarc * h + irho + 1];
            const float2 b0 = P[(size_t)uarc * h + irho], b1 = P[(size_t)uarc * h + irho + 1];
            const float2 i0 = make_float2(a0.x * (1.0f - pfrac) + a1.x * pfrac, a0.y * (1.0f - pfrac) + a1.y * pfrac);
            const float2 i1 = make_float2(b0.x * (1.0f - pfrac) + b1.x * pfrac, b0.y * (1.0f - pfrac) + b1.y * pfrac);
            val = make_float2(i0.x * tfrac + i1.x * (1.0f - tfrac), i0.y * tfrac + i1.y * (1.0f - tfrac));
        }
        const float sg = ((tx & 1) == (ty & 1)) ? 1.0f : -1.0f; // 4 (tx%2 - 1/2)(ty%2 - 1/2)
        cart[(sl * s + (ty + s / 2) % s) * (long long)s + (tx + s / 2) % s] = make_float2(val.x * sg, val.y * sg);
    }
}

// Fused form of k_bst_p2c and the inverse FFT of the grid rows (k_ifft_rows):
// one workgroup per destination row tyd of the shifted frequency grid and
// group of up to BST_SPB slices.  The FP64 polar coordinates of the row's
// cells do not depend on the slice and are computed once; for each slice the
// interpolated cells go straight into LDS, the row is inverse-transformed
// there (conjugate, forward FFT, conjugate), and only the N columns
// [L, L + N) the crop keeps are written, as rows of out [S][s][N].  The grid
// is never written to HBM.  The expressions are those of the two unfused
// kernels, so the values are the same bit for bit.
// Waiting for the gathers and between the passes bounds it, so what counts is
// workgroups per CU: the cells' derived values are formed in each slice's turn
// (kept for all cells across the slices they took 163 registers: two workgroups
// of 384 threads; 112 now).  16 slices of 3072 x 3072 cells: 1.76 -> 1.23 ms.
// 768 threads are held to 80 registers (some spill): two workgroups on a CU
// instead of one, 8 slices of 6144 x 6144 cells, the call 3.26 -> 3.16 ms (3.40 with
// one).  Below 256 threads few workgroups run at all and keeping the values is
// faster (16 slices of 600 x 600: 34 us against 37).
constexpr int BST_SPB = 8;
struct BstRowsK {
    const float2* polar; // [S][A2][n/2]
    float2* out;         // [S][s][N]
    int n, A2, s, S, N, L;
};

template <int THREADS, int E, int EC>
__global__ __launch_bounds__(THREADS, THREADS == 768 ? 6 : (THREADS >= 256 ? 4 : 1)) void k_bst_rows(BstRowsK a, const float2* twg, FftK p)
{
    constexpr bool BY_SLICE = THREADS >= 256;
    extern __shared__ float2 z[];
    const int n = a.n, s = a.s;
    float2* tws = z + lds_elems(n);
    const int ntw = 128 + n / 128 + 1;
    for (int k = threadIdx.x; k < ntw; k += THREADS) tws[k] = twg[k];
    const Tw tw{tws, tws + 128};
    // runs of 8 neighbouring rows on one XCD (workgroups go to the 8 XCDs round
    // robin): their cells share lines of the polar rows
    const int tyd = (int)(blockIdx.x / 64u * 64u + (blockIdx.x & 7u) * 8u + (blockIdx.x >> 3) % 8u);
    if (tyd >= s) return;
    const int sl0 = blockIdx.y * BST_SPB, sl1 = min(a.S, sl0 + BST_SPB);
    const int ty = (tyd + s - s / 2) % s; // (ty + s/2) % s == tyd
    // the cells txd = threadIdx.x + j THREADS of this row (THREADS EC >= s), in
    // three registers each: oc = polar offset of (iarc, irho), with bit 30 set
    // when uarc wraps to 0 (-1: zero cell or past s); ps = the radial fraction
    // with the cell's checkerboard sign in its sign bit; tf = the angular one
    int oc[EC];
    float ps[EC], tf[EC];
    const int h = n / 2;               // polar rows hold radii [0, n/2)
    const int wrapb = (a.A2 - 1) * h; // (iarc, irho) -> (0, irho)
#pragma unroll
    for (int j = 0; j < EC; ++j) {
        const int txd = threadIdx.x + j * THREADS;
        oc[j] = -1;
        ps[j] = tf[j] = 0.0f;
        if (txd < s) {
            const int tx = (txd + s - s / 2) % s;
            const int posx = tx - s / 2, posy = ty - s / 2;
            const double rho = (double)n * hypot((double)posx, (double)posy) / (double)s;
            const double angle = (double)a.A2 * (0.5 * atan2((double)posy, (double)posx) / M_PI + 0.5);
            const long long irho = (long long)rho;
            int iarc = (int)angle;
            float pf = 0.0f;
            if (irho < n / 2 - 1) {
                pf = (float)(rho - (double)irho);
                tf[j] = (float)((double)iarc - angle);
                iarc = iarc % a.A2;
                oc[j] = (iarc * h + (int)irho) | (iarc + 1 == a.A2 ? (1 << 30) : 0);
            }
            ps[j] = ((tx & 1) == (ty & 1)) ? pf : -pf;
        }
    }
    for (int sl = sl0; sl < sl1; ++sl) {
        const float2* P = a.polar + (size_t)sl * a.A2 * h;
        // opaque: what depends on the cells is formed in each slice's turn, not
        // kept in registers for all cells
        int tid = threadIdx.x;
        if (BY_SLICE) asm volatile("" : "+v"(tid));
        __syncthreads(); // the previous slice's row is read (and the twiddles are in)
#pragma unroll
        for (int j = 0; j < EC; ++j) {
            const int txd = tid + j * THREADS;
            int o = oc[j];
            float pj = ps[j], tfrac = tf[j];
            if (BY_SLICE) asm volatile("" : "+v"(o), "+v"(pj), "+v"(tfrac));
            if (txd < s) {
                float2 val = make_float2(0.0f, 0.0f);
                const float pfrac = fabsf(pj);
                if (o >= 0) {
                    const int o0 = o & ((1 << 30) - 1);
                    const int o1 = (o >> 30) ? o0 - wrapb : o0 + h;
                    const float2 a0 = P[o0], a1 = P[o0 + 1];
                    const float2 b0 = P[o1], b1 = P[o1 + 1];
                    const float2 i0 = make_float2(a0.x * (1.0f - pfrac) + a1.x * pfrac,
                                                  a0.y * (1.0f - pfrac) + a1.y * pfrac);
                    const float2 i1 = make_float2(b0.x * (1.0f - pfrac) + b1.x * pfrac,
                                                  b0.y * (1.0f - pfrac) + b1.y * pfrac);
                    val = make_float2(i0.x * tfrac + i1.x * (1.0f - tfrac), i0.y * tfrac + i1.y * (1.0f - tfrac));
                }
                const float sg = __builtin_signbit(pj) ? -1.0f : 1.0f;
                const float2 v = make_float2(val.x * sg, val.y * sg);
                z[pix(txd)] = make_float2(v.x, -v.y);
            }
        }
        __syncthreads();
        fft_run<THREADS, E>(z, tw, p, tid);
        for (int c = tid; c < a.N; c += THREADS) {
            const float2 v = z[pix(a.L + c)];
            a.out[((size_t)sl * s + tyd) * a.N + c] = make_float2(v.x, -v.y);
        }
    }
}

// out[sl][c][y] = in[sl][y][c0 + c] for the nc columns [c0, c0 + nc) of an
// s-row slice of row pitch ip: the columns the crop keeps, as rows for the
// second 1-D pass (32 x 32 LDS tiles)
__global__ __launch_bounds__(256) void k_transpose_c(const float2* in, float2* out, int s, int c0, int nc, int ip)
{
    __shared__ float2 t[32][33];
    const int sl = blockIdx.z;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    const float2* src = in + (size_t)sl * s * ip;
    float2* dst = out + (size_t)sl * nc * s;
    for (int k = threadIdx.x; k < 32 * 32; k += 256) {
        const int dy = k / 32, dx = k % 32;
        if (y0 + dy < s && x0 + dx < nc) t[dy][dx] = src[(size_t)(y0 + dy) * ip + c0 + x0 + dx];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 32 * 32; k += 256) {
        const int dx = k / 32, dy = k % 32;
        if (y0 + dy < s && x0 + dx < nc) dst[(size_t)(x0 + dx) * s + y0 + dy] = t[dy][dx];
    }
}

// obj[sl][j][i] = Re(R[sl][i][j + L]) / scale, R the inverse FFT along the
// rows of the kept columns ([sl][N][s])
__global__ void k_bst_extract(const float2* R, float* obj, int s, int N, int L, float scale, int S)
{
    const long long total = (long long)S * N * N;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(e % N), j = (int)((e / N) % N);
        const long long sl = e / ((long long)N * N);
        obj[e] = R[(sl * N + i) * (long long)s + j + L].x / scale;
    }
}

template <int THREADS, int E>
void launch_bst_polar_t(const BstPolarK& k, const FftK& p, size_t lds, hipStream_t st)
{
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_bst_polar<THREADS, E>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_bst_polar<THREADS, E>), dim3((unsigned)((long long)k.S * k.A)), dim3(THREADS), lds, st, k,
                       p);
}

template <int THREADS, int E>
void launch_bst_filter_polar_t(const FilterK& f, const BstPolarK& k, const FftK& p, size_t lds, hipStream_t st)
{
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_bst_filter_polar<THREADS, E>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const long long blocks = (long long)((f.S + f.SB - 1) / f.SB) * f.A * (f.SB / 2);
    hipLaunchKernelGGL((k_bst_filter_polar<THREADS, E>), dim3((unsigned)blocks), dim3(THREADS), lds, st, f, k, p);
}

template <int THREADS, int E, int EC = E>
void launch_bst_rows_t(const BstRowsK& k, const float2* tw, const FftK& p, size_t lds, hipStream_t st)
{
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_bst_rows<THREADS, E, EC>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_bst_rows<THREADS, E, EC>), dim3((unsigned)(k.s + 63) / 64u * 64u, (unsigned)((k.S + BST_SPB - 1) / BST_SPB)),
                       dim3(THREADS), lds, st, k, tw, p);
}

template <int THREADS, int E>
void launch_ifft_t(float2* data, const float2* tw, const FftK& p, long long rows, size_t lds, hipStream_t st)
{
    RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_ifft_rows<THREADS, E>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_ifft_rows<THREADS, E>), dim3((unsigned)rows), dim3(THREADS), lds, st, data, tw, p);
}

FftK fftk_of(const FftPlan& plan)
{
    FftK p;
    p.n = plan.n;
    p.nstages = plan.nstages;
    for (int i = 0; i < 24; ++i) {
        p.radix[i] = plan.radix[i];
        p.twstep[i] = 0;
        p.nsm[i] = 0;
        p.nss[i] = 0;
    }
    // stage st works on Ns = radix[0] * .. * radix[st-1] and j < nb = n / radix[st]:
    // nsm = ceil(2^nss / Ns) with 2^nss >= nb * Ns makes (j * nsm) >> nss == j / Ns
    // for every j < nb (the error j * (nsm Ns - 2^nss) / (Ns 2^nss) stays below the
    // gap 1/Ns); nsm <= 2 nb + 1 < 2^24 and j * nsm < 2^32, as the 24-bit multiplies need
    long long Ns = 1;
    for (int st = 0; st < p.nstages; ++st) {
        const int R = p.radix[st];
        const long long nb = p.n / R;
        p.twstep[st] = (int)(p.n / (Ns * R));
        int k = 0;
        while ((1LL << k) < nb * Ns) ++k;
        const long long m = ((1LL << k) + Ns - 1) / Ns;
        if (m >= (1LL << 24) || (nb - 1) * m >= (1LL << 32) || nb >= (1LL << 24))
            fail(RAFT_EUNSUPPORTED, "internal: FFT stage index out of the 24-bit range");
        if ((Ns & (Ns - 1)) != 0)
            for (long long j = 0; j < nb; ++j)
                if ((long long)(((unsigned long long)j * (unsigned long long)m) >> k) != j / Ns)
                    fail(RAFT_EUNSUPPORTED, "internal: FFT stage division check failed");
        p.nsm[st] = (unsigned)m;
        p.nss[st] = k;
        Ns *= R;
    }
    return p;
}

} // namespace

FftPlan fft_plan(int n)
{
    FftPlan p;
    p.n = n;
    if (n < 2 || n > 16384) return p;
    int m = n;
    static const int order[] = {8, 4, 2, 3, 5};
    for (int r : order) {
        while (m % r == 0 && m > 1) {
            if (p.nstages >= 24) return p;
            p.radix[p.nstages++] = r;
            m /= r;
        }
    }
    if (m != 1) return p;
    // threads = n / 8 when that is an allowed block size, so every radix-8
    // butterfly of a pass has its own thread (6144 -> 768, 3072 -> 384)
    static const int tsz[] = {64, 128, 192, 256, 384, 512, 768, 1024};
    int t = 1024;
    for (int c : tsz)
        if (c * 8 >= n) {
            t = c;
            break;
        }
    p.threads = t;
    p.ok = true;
    return p;
}

// first radix of the FP32 form (k_filter_dif), 0: none
static int dif_radix(int n)
{
    for (int m : {8, 10, 12, 16})
        if (n == 64 * m) return m;
    for (int m : {3, 4, 5, 6, 8, 10, 12, 16})
        if (n == 512 * m) return m;
    return 0;
}

// frequency held at each position after forward passes of these radices:
// position q (block / radix) + r holds radix f(r) + q
static std::vector<int> dif_order(const int* radix, int passes)
{
    std::vector<int> freq(1, 0);
    for (int i = passes - 1; i >= 0; --i) {
        std::vector<int> up;
        for (int q = 0; q < radix[i]; ++q)
            for (int f : freq) up.push_back(radix[i] * f + q);
        freq.swap(up);
    }
    return freq;
}

bool dif_tables(int n, const std::vector<float2>& H, std::vector<float2>& Hp, std::vector<float2>& tw)
{
    const int m = dif_radix(n);
    if (!m) return false;
    const int radix[4] = {m, 8, 8, 8};
    const std::vector<int> freq = dif_order(radix, n == 64 * m ? 3 : 4);
    Hp.resize(n);
    for (int e = 0; e < n; ++e) Hp[e] = H[freq[e]];
    // exp(-2 pi i q j / (R M)), [q < R][j < M], of the first pass and of the
    // radix-8 passes over blocks of 512 and 64
    tw.clear();
    for (int R : {m, 8, 8}) {
        const int M = tw.empty() ? n / m : (tw.size() == (size_t)n ? 64 : 8);
        for (int q = 0; q < R; ++q)
            for (int j = 0; j < M; ++j) {
                const double ang = -2.0 * M_PI * (double)q * (double)j / ((double)R * M);
                tw.push_back(make_float2((float)std::cos(ang), (float)std::sin(ang)));
            }
    }
    return true;
}

ConvPlan conv_plan(int n, int N)
{
    ConvPlan best;
    if (n < CV_LEAST_N || (n < CV_MIN_N && N < CV_LEAST_RAYS)) return best;
    long long cost = 0;
    for (int m : {1, 3, 5})
        for (int len = m * 64, k = 6; len <= CV_MAX_LEN; len *= 2, ++k) {
            const int chunk = std::min(len - N + 1, n);
            if (chunk < 1) continue;
            const int chunks = (n + chunk - 1) / chunk;
            // of equal cost one long transform instead of two (51 rays padded to 153, 4800
            // pairs: 85 -> 50 us), but for 8192, of which one workgroup fits a CU (1601 padded
            // to 4803: 150 us by two of 4096, 228 by one)
            const long long c = (long long)chunks * len;
            if (best.len && (c > cost || (c == cost && (chunks >= best.chunks || len > CV_MAX_LEN / 2)))) continue;
            cost = c;
            best = ConvPlan();
            best.len = len; best.chunk = chunk; best.chunks = chunks;
            if (m > 1) best.radix[best.passes++] = m;
            const int fours = k % 3 == 0 ? 0 : (k % 3 == 2 ? 1 : 2);
            for (int i = 0; i < fours; ++i) best.radix[best.passes++] = 4;
            for (int i = 0; i < (k - 2 * fours) / 3; ++i) best.radix[best.passes++] = 8;
        }
    if (best.chunks > CV_MAX_CHUNKS) best = ConvPlan();
    return best;
}

bool conv_pays_lowpass(int n, int N) { return (N + 63) / 64 * n >= CV_LEAST_LOWPASS; }

void conv_tables(const ConvPlan& p, const double* g, int n, int N, int L, std::vector<double>& spec,
                 std::vector<double>& tw, std::vector<double>& edge)
{
    const int len = p.len;
    std::vector<double> w(2 * (size_t)len);
    for (int k = 0; k < len; ++k) {
        const double ang = -2.0 * M_PI * (double)k / (double)len;
        w[2 * k] = std::cos(ang);
        w[2 * k + 1] = std::sin(ang);
    }
    const std::vector<int> freq = dif_order(p.radix, p.passes);
    spec.assign(2 * (size_t)len * p.chunks, 0.0);
    std::vector<double> x(2 * (size_t)len), y(2 * (size_t)len);
    for (int c = 0; c < p.chunks; ++c) {
        std::fill(x.begin(), x.end(), 0.0);
        const long long T0 = (long long)c * p.chunk;
        for (int t = -(N - 1); t < p.chunk; ++t)
            x[2 * (size_t)((t + len) % len)] = g[(((T0 + t - L) % n) + n) % n] / (double)len;
        // forward transform, radix-2 steps down to the odd factor (decimation in time)
        int m = len;
        while (m % 2 == 0) m /= 2;
        const int q = len / m; // q interleaved transforms of length m
        for (int r = 0; r < q; ++r)
            for (int k = 0; k < m; ++k) {
                double re = 0.0, im = 0.0;
                for (int i = 0; i < m; ++i) {
                    const size_t e = 2 * ((size_t)r + (size_t)q * i), f = 2 * (size_t)((long long)i * k % m * q);
                    re += x[e] * w[f] - x[e + 1] * w[f + 1];
                    im += x[e] * w[f + 1] + x[e + 1] * w[f];
                }
                y[2 * ((size_t)r * m + k)] = re;
                y[2 * ((size_t)r * m + k) + 1] = im;
            }
        // y: [r][k], transforms of x[r + q i]; pairs r, r + h combine to length 2 s
        for (int h = q / 2, s = m; h >= 1; h /= 2, s *= 2) {
            for (int r = 0; r < h; ++r)
                for (int k = 0; k < s; ++k) {
                    const double* e = &y[2 * ((size_t)r * s + k)];
                    const double* o = &y[2 * ((size_t)(r + h) * s + k)];
                    const double* f = &w[2 * (size_t)k * h];
                    const double re = o[0] * f[0] - o[1] * f[1], im = o[0] * f[1] + o[1] * f[0];
                    double* d0 = &x[2 * ((size_t)r * 2 * s + k)];
                    double* d1 = &x[2 * ((size_t)r * 2 * s + k + s)];
                    d0[0] = e[0] + re; d0[1] = e[1] + im;
                    d1[0] = e[0] - re; d1[1] = e[1] - im;
                }
            x.swap(y);
        }
        for (int e = 0; e < len; ++e) {
            spec[2 * ((size_t)c * len + e)] = y[2 * (size_t)freq[e]];
            spec[2 * ((size_t)c * len + e) + 1] = y[2 * (size_t)freq[e] + 1];
        }
    }
    tw = w;
    edge.assign(2 * (size_t)n, 0.0);
    for (int T = 0; T < n; ++T) {
        double e0 = 0.0, e1 = 0.0;
        for (int j = 0; j < L; ++j) e0 += g[(T - j + n) % n];
        for (int j = L + N; j < n; ++j) e1 += g[(T - j + n) % n];
        edge[T] = e0;
        edge[(size_t)n + T] = e1;
    }
}

bool launch_fbp_filter(const FilterArgs& a, const FftPlan& plan, int store, hipStream_t st)
{
    if (a.S <= 0 || a.A <= 0) return a.rows != nullptr && store == RAFT_STORE_F32;
    FilterK k;
    k.tomo = a.tomo; k.q = a.q; k.H = a.H; k.tw = a.tw; k.g = a.g; k.wa = a.wa;
    k.N = a.N; k.A = a.A; k.S = a.S; k.npad = a.npad; k.L = a.L; k.tlo = a.tlo; k.W = a.W; k.none = a.none;
    k.SB = (store == RAFT_STORE_F16) ? 8 : 4;
    k.split = store == RAFT_STORE_F32 ? a.mx : 0;
    k.rg = a.mx ? 1 : a.A;
    k.ra = a.mx ? (a.S + k.SB - 1) / k.SB : 1;
    k.rows = store == RAFT_STORE_F32 ? a.rows : nullptr;
    bool direct = false;
    const long long groups = (a.S + k.SB - 1) / k.SB;
    const long long blocks = groups * a.A * (k.SB / 2);
    if (blocks > 0x7fffffffLL) fail(RAFT_EUNSUPPORTED, "too many sinogram rows for one filter launch");
    const size_t lds = sizeof(float2) * lds_elems(a.npad);
    const size_t lds_fft = lds + sizeof(float2) * (size_t)(128 + a.npad / 128 + 1);
    bool done = false;
    if (a.dif_H && !a.none) {
        if (store == RAFT_STORE_F16) done = launch_dif<__half>(k, a, st);
        else done = launch_dif<float>(k, a, st);
        direct = done && k.rows != nullptr;
    }
    if (done) {
    } else if (plan.ok || a.none) {
        const FftK p = fftk_of(plan);
        const int threads = plan.ok ? plan.threads : 256;
        if (store == RAFT_STORE_F16) launch_fft<__half>(k, p, threads, (int)blocks, lds_fft, st);
        else direct = launch_fft<float>(k, p, threads, (int)blocks, lds_fft, st);
    } else {
        if (lds > 160 * 1024) fail(RAFT_EUNSUPPORTED, "padded row too long for the direct filter path");
        if (a.conv.len > 0) {
            if (store == RAFT_STORE_F16) launch_conv<__half>(k, a, st);
            else launch_conv<float>(k, a, st);
        } else if (store == RAFT_STORE_F16) {
            RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_filter_direct<__half>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            hipLaunchKernelGGL((k_filter_direct<__half>), dim3((int)blocks), dim3(256), lds, st, k);
        } else {
            RAFT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_filter_direct<float>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            hipLaunchKernelGGL((k_filter_direct<float>), dim3((int)blocks), dim3(256), lds, st, k);
        }
    }
    RAFT_HIP(hipGetLastError());
    return direct;
}

bool bst_filter_polar_fits(int n)
{
    return sizeof(float2) * (lds_elems(n) + (size_t)(128 + n / 128 + 1) + (size_t)(n / 2)) <= 160 * 1024;
}

void launch_bst(const BstArgs& a, const FftPlan& plan, hipStream_t st, const FilterArgs* filt)
{
    if (a.S <= 0) return;
    if (!plan.ok) fail(RAFT_EUNSUPPORTED, "BST needs a padded size n = N(1+pad) <= 16384 with factors 2, 3, 5");
    const int n = plan.n, s = n;
    const FftK p = fftk_of(plan);
    const size_t lds = sizeof(float2) * (lds_elems(n) + (size_t)(128 + n / 128 + 1));
    if ((long long)a.S * 2 * a.A > 0x7fffffffLL || (long long)a.S * s > 0x7fffffffLL)
        fail(RAFT_EUNSUPPORTED, "BST block too large for one launch");
    BstPolarK k{a.q, a.polar, a.tw, n, a.A, a.S};
    if (filt) {
        // filter + polar FFTs in one pass from the sinogram (k_bst_filter_polar)
        if (filt->npad != n || filt->S != a.S || filt->A != a.A)
            fail(RAFT_EINVAL, "BST filter arguments do not match the transform");
        FilterK f;
        f.tomo = filt->tomo; f.q = nullptr; f.H = filt->H; f.tw = filt->tw; f.g = nullptr; f.wa = filt->wa;
        f.N = filt->N; f.A = filt->A; f.S = filt->S; f.npad = n; f.L = filt->L; f.tlo = 0; f.W = n;
        f.none = filt->none;
        f.SB = 4;
        f.split = 0;
        f.rg = f.A;
        f.ra = 1;
        f.rows = nullptr;
        if ((long long)((f.S + f.SB - 1) / f.SB) * f.A * (f.SB / 2) > 0x7fffffffLL)
            fail(RAFT_EUNSUPPORTED, "too many sinogram rows for one BST launch");
        const size_t lds_fp = lds + sizeof(float2) * (size_t)(n / 2);
        if (lds_fp > 160 * 1024) fail(RAFT_EUNSUPPORTED, "padded row too long for the BST filter pass");
        if (n > 8192) launch_bst_filter_polar_t<1024, 16>(f, k, p, lds_fp, st);
        else {
            switch (plan.threads) {
            case 64: launch_bst_filter_polar_t<64, 8>(f, k, p, lds_fp, st); break;
            case 128: launch_bst_filter_polar_t<128, 8>(f, k, p, lds_fp, st); break;
            case 192: launch_bst_filter_polar_t<192, 8>(f, k, p, lds_fp, st); break;
            case 256: launch_bst_filter_polar_t<256, 8>(f, k, p, lds_fp, st); break;
            case 384: launch_bst_filter_polar_t<384, 8>(f, k, p, lds_fp, st); break;
            case 512: launch_bst_filter_polar_t<512, 8>(f, k, p, lds_fp, st); break;
            case 768: launch_bst_filter_polar_t<768, 8>(f, k, p, lds_fp, st); break;
            default: launch_bst_filter_polar_t<1024, 8>(f, k, p, lds_fp, st); break;
            }
        }
    } else if (n > 8192) launch_bst_polar_t<1024, 16>(k, p, lds, st);
    else {
        switch (plan.threads) {
        case 64: launch_bst_polar_t<64, 8>(k, p, lds, st); break;
        case 128: launch_bst_polar_t<128, 8>(k, p, lds, st); break;
        case 192: launch_bst_polar_t<192, 8>(k, p, lds, st); break;
        case 256: launch_bst_polar_t<256, 8>(k, p, lds, st); break;
        case 384: launch_bst_polar_t<384, 8>(k, p, lds, st); break;
        case 512: launch_bst_polar_t<512, 8>(k, p, lds, st); break;
        case 768: launch_bst_polar_t<768, 8>(k, p, lds, st); break;
        default: launch_bst_polar_t<1024, 8>(k, p, lds, st); break;
        }
    }
    RAFT_HIP(hipGetLastError());
    if (a.fused) {
        // polar -> Cartesian rows, inverse-transformed in LDS, N kept columns
        // per row -> cart [S][s][N]; then transposed to cartT [S][N][s]
        const BstRowsK rk{a.polar, a.cart, n, 2 * a.A, s, a.S, a.N, a.L};
        if (n > 8192) launch_bst_rows_t<1024, 16>(rk, a.tw, p, lds, st);
        else {
            switch (plan.threads) {
            case 64: launch_bst_rows_t<64, 8>(rk, a.tw, p, lds, st); break;
            case 128: launch_bst_rows_t<128, 8>(rk, a.tw, p, lds, st); break;
            case 192: launch_bst_rows_t<192, 8>(rk, a.tw, p, lds, st); break;
            case 256: launch_bst_rows_t<256, 8>(rk, a.tw, p, lds, st); break;
            case 384: launch_bst_rows_t<384, 8>(rk, a.tw, p, lds, st); break;
            case 512: launch_bst_rows_t<512, 8>(rk, a.tw, p, lds, st); break;
            case 768: launch_bst_rows_t<768, 8>(rk, a.tw, p, lds, st); break;
            default: launch_bst_rows_t<1024, 8>(rk, a.tw, p, lds, st); break;
            }
        }
        RAFT_HIP(hipGetLastError());
        dim3 g((a.N + 31) / 32, (s + 31) / 32, a.S);
        hipLaunchKernelGGL(k_transpose_c, g, dim3(256), 0, st, a.cart, a.cartT, s, 0, a.N, a.N);
        RAFT_HIP(hipGetLastError());
    } else {
        const long long cells = (long long)a.S * s * s;
        hipLaunchKernelGGL(k_bst_p2c, dim3((unsigned)std::min<long long>((cells + 255) / 256, 65536)), dim3(256), 0,
                           st, a.polar, a.cart, n, 2 * a.A, s, a.S);
        RAFT_HIP(hipGetLastError());
    }
    // 2-D inverse FFT: all rows (unfused form), then only the N columns
    // [L, L + N) the crop keeps (transposed to rows); the other columns are
    // never needed
    for (int pass = a.fused ? 1 : 0; pass < 2; ++pass) {
        float2* d = pass == 0 ? a.cart : a.cartT;
        const long long rows = (long long)a.S * (pass == 0 ? s : a.N);
        if (n > 8192) launch_ifft_t<1024, 16>(d, a.tw, p, rows, lds, st);
        else {
            switch (plan.threads) {
            case 64: launch_ifft_t<64, 8>(d, a.tw, p, rows, lds, st); break;
            case 128: launch_ifft_t<128, 8>(d, a.tw, p, rows, lds, st); break;
            case 192: launch_ifft_t<192, 8>(d, a.tw, p, rows, lds, st); break;
            case 256: launch_ifft_t<256, 8>(d, a.tw, p, rows, lds, st); break;
            case 384: launch_ifft_t<384, 8>(d, a.tw, p, rows, lds, st); break;
            case 512: launch_ifft_t<512, 8>(d, a.tw, p, rows, lds, st); break;
            case 768: launch_ifft_t<768, 8>(d, a.tw, p, rows, lds, st); break;
            default: launch_ifft_t<1024, 8>(d, a.tw, p, rows, lds, st); break;
            }
        }
        RAFT_HIP(hipGetLastError());
        if (pass == 0) {
            dim3 g((a.N + 31) / 32, (s + 31) / 32, a.S);
            hipLaunchKernelGGL(k_transpose_c, g, dim3(256), 0, st, a.cart, a.cartT, s, a.L, a.N, s);
            RAFT_HIP(hipGetLastError());
        }
    }
    const long long outn = (long long)a.S * a.N * a.N;
    hipLaunchKernelGGL(k_bst_extract, dim3((unsigned)std::min<long long>((outn + 255) / 256, 65536)), dim3(256), 0,
                       st, a.cartT, a.obj, s, a.N, a.L, a.scale, a.S);
    RAFT_HIP(hipGetLastError());
}

} // namespace raft
