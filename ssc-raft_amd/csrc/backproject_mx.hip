// backproject_mx.hip -- backprojection of many slices on the matrix cores
// (gfx950, wave64): the same sums as backproject.hip's kernels, for calls with
// enough slices to fill a matrix tile.
//
// For one angle a, the pixels of a small patch read bins of a short window:
// out[pixel][slice] += sum_b sel[pixel][b] rows[b][slice], with one 1 per row
// of sel.  sel is built from the same IEEE-double bin index as the gather
// kernels, T = (int)fma(X, cA, fma(Y, cB, c0)); the contraction runs as
// v_smfmac_f32_32x32x32 (sparse A: at most two of every four k): 32 pixels x
// (4 angles x 8 bins) x 32 columns per instruction.  A patch is 6 x 5 pixels
// (30 of 32 rows used): every pixel lies within |(2.5, 2)| = 3.2016 pixels of its
// centre, so with base = (int)(u_centre - 3.45) every T of the patch lies in
// [base, base + 7] (truncation is monotone and maps an interval shorter than 7
// onto at most 8 integers), for every angle at FBP's one bin per pixel.
//
// FP32 rows: each value is split exactly into three bf16 pieces h + m + l
// (8 + 8 + 8 significant bits, truncated, so nothing overflows); products
// with the selection are exact.  h sums and m + l sums have accumulators of
// their own.  An h carries 8 bits, so its running sum is exact while it stays
// below 2^16 times the smallest term, and the m + l sum sits 2^-8 below: there the
// total rounds less than a sum of FP32 values does, and past it the h sum rounds as
// that would (64 slices of 2048^2: 7.6e-7 from 64 bits, the gather form 9.8e-7).
// Subnormal pieces count: the instruction does not flush them.  FP16 rows are used
// as they are, one accumulator, FP32 sums.
//
// Workgroup: 8 waves, a tile of 4 x 8 patches (24 x 40 pixels), 4 patches in x
// per wave (they share the Y part of the coordinate), up to 32 (FP32) or 64
// (FP16) slices.  Per round of 4 angles the windows of BM_SLOT bins are staged
// in LDS, the loads of the next two or three rounds in flight.  The B operand
// (bins x slices) comes from LDS through ds_read_b64_tr_b16: the LDS holds
// [segment of 4 (FP16: 8) slices][bin], a segment pitch of 32 (64) bytes mod
// 256, so a read of 4 bins x 32 columns touches every bank once.
//
// What bounds it: 64 slices of 2048^2 pixels and 2048 angles move 187 GB from L2
// into LDS, about 9 TB/s, and the operand reads keep the LDS pipe at 0.175 wave
// instructions per clock per CU, as many as it does of 16-byte reads in a loop of
// nothing else; VALU issue is at 0.36 and the waves wait a third of their cycles
// (two per SIMD hold the FP32 accumulators: 128 registers each).  The gather kernels take
// 29.5 ms there (one LDS read per pixel, angle and 4 slices), FP16 rows 23.8 ms
// against 9.3 here.
//
// Staging: by default the filter writes the rows in the layout the LDS wants
// (FP32: [angle][group of 4 slices][piece][bin], 8 bytes each; FP16:
// [angle][group of 8][bin], 16 bytes) and they move with loads straight into
// LDS.  The checked form takes the gather kernels' rows and splits them on the
// way, for callers whose scratch is fixed; the sums are the same bit for bit.
//
// A window that holds a non-finite value makes every pixel that shares it
// non-finite (0 * inf); such pixels are summed again one by one in the gather
// kernels' order, so they get what those give.
#include "raft_internal.hpp"

#include <algorithm>
#include <cmath>

namespace raft {

namespace {

constexpr int BM_PX = 6, BM_PY = 5;          // patch
constexpr int BM_PIX = BM_PX * BM_PY;        // 30 of the 32 matrix rows
constexpr int BM_NX = 4, BM_NY = 8;          // patches per tile (NX per wave, one wave per row of patches)
constexpr int BM_TX = BM_PX * BM_NX, BM_TY = BM_PY * BM_NY;
constexpr int BM_CH = 4;                     // angles per round
constexpr int BM_SLOT = 52;                  // staged bins per angle
constexpr double BM_REACH = 3.45;            // base = (int)(u_centre - BM_REACH)
constexpr double BM_SPREAD = 19.6787;        // |(9, 17.5)|: farthest patch centre from the tile centre
// a round's windows hold base .. base + 7 of every patch: first bin
// (int)(u_tile - BM_TILE_REACH), one less where that makes the source 16-byte
// aligned
constexpr double BM_TILE_REACH = BM_SPREAD + BM_REACH + 0.01;
static_assert(2 * BM_SPREAD + 0.02 + 1 + 8 + 1 <= BM_SLOT, "staged window too short");

typedef short s4v __attribute__((ext_vector_type(4)));
typedef short s8v __attribute__((ext_vector_type(8)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h16x16 __attribute__((ext_vector_type(16)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef double d2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) s4v lds_s4;

// wait for every vector-memory load of this wave, loads into LDS included
// (s_waitcnt vmcnt(0))
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0xF70); }

// N loads of 16 bytes per lane straight into LDS: load j takes lane l's bytes at
// base + off[j] + 1024 j to LDS byte dst + 1024 j + 16 l (the instruction's
// offset counts on both sides; base and dst uniform).  In assembly because the
// compiler, which cannot see that the loads fill another buffer than the one
// being read, would wait for them before the next LDS read; no register is
// written, and the caller waits for them itself (wait_loads_but, then a
// barrier).
template <int N, int M> __device__ __forceinline__ void load_lds(const char* base, const unsigned (&off)[M], unsigned dst)
{
    static_assert(N >= 1 && N <= 5 && N <= M, "loads per round");
    const unsigned d = __builtin_amdgcn_readfirstlane(dst + 1024u);
    if constexpr (N == 1)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:-1024"
                     : : "s"(d), "v"(off[0]), "s"(base) : "memory", "m0");
    if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3 offset:-1024\n\t"
                     "global_load_lds_dwordx4 %2, %3"
                     : : "s"(d), "v"(off[0]), "v"(off[1]), "s"(base) : "memory", "m0");
    if constexpr (N == 3)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %4 offset:-1024\n\t"
                     "global_load_lds_dwordx4 %2, %4\n\tglobal_load_lds_dwordx4 %3, %4 offset:1024"
                     : : "s"(d), "v"(off[0]), "v"(off[1]), "v"(off[2]), "s"(base) : "memory", "m0");
    if constexpr (N == 4)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %5 offset:-1024\n\t"
                     "global_load_lds_dwordx4 %2, %5\n\tglobal_load_lds_dwordx4 %3, %5 offset:1024\n\t"
                     "global_load_lds_dwordx4 %4, %5 offset:2048"
                     : : "s"(d), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base) : "memory", "m0");
    if constexpr (N == 5)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %6 offset:-1024\n\t"
                     "global_load_lds_dwordx4 %2, %6\n\tglobal_load_lds_dwordx4 %3, %6 offset:1024\n\t"
                     "global_load_lds_dwordx4 %4, %6 offset:2048\n\tglobal_load_lds_dwordx4 %5, %6 offset:3072"
                     : : "s"(d), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "s"(base)
                     : "memory", "m0");
}

// 4 bytes per lane from base + off to LDS byte dst + 4 l
__device__ __forceinline__ void load_lds4(const char* base, unsigned off, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 : : "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(off), "s"(base) : "memory", "m0");
}

// wait until at most N of this wave's vector-memory loads are outstanding
template <int N> __device__ __forceinline__ void wait_loads_but()
{
    __builtin_amdgcn_s_waitcnt(0xF70 & ~0xF | (N & 15)); // vmcnt bits 3:0, N < 16
}

// lane L of this lane's row of 16
__device__ __forceinline__ int row_lane(int v, int l)
{
    switch (l) { // the control is an immediate; l is known once the loop is unrolled
#define BM_LANE(L) case L: return __builtin_amdgcn_update_dpp(0, v, 0x150 + L, 0xf, 0xf, true);
        BM_LANE(0) BM_LANE(1) BM_LANE(2) BM_LANE(3) BM_LANE(4) BM_LANE(5) BM_LANE(6) BM_LANE(7)
        BM_LANE(8) BM_LANE(9) BM_LANE(10) BM_LANE(11) BM_LANE(12) BM_LANE(13) BM_LANE(14) BM_LANE(15)
#undef BM_LANE
    }
    return v;
}

struct BmArgs {
    const char* q;      // FP32: [A][G][3][W] 8-byte entries (4 slices of one piece); FP16: [A][G][W] 16-byte
                        // entries (8 slices); the checked form: [G][A][W] 16-byte entries (4 FP32 or 8 FP16)
    float* out;         // [S][n][n]
    const d2v* cs;  // per angle {cA, cB}
    double xc, c0;
    int n, A, tlo, W, S, G; // S: slices of the call, G: its 16-byte row groups
    int s_first;            // first slice of this launch's first pack
    int tiles_x, tiles_y, total;
};

// FORM: 0 = FP32 rows, 32 slices; 1 = FP32 rows, 16 slices (h and m side by
// side in one operand, l under m in the second); 2 = FP16 rows, 64 slices;
// 3 = FP16 rows, 32 slices
template <int FORM> struct Form {
    static constexpr bool F16 = FORM >= 2;
    static constexpr int SLICES = FORM == 0 ? 32 : (FORM == 1 ? 16 : (FORM == 2 ? 64 : 32));
    static constexpr int NG = F16 ? SLICES / 8 : SLICES / 4;  // row groups of 16-byte entries
    static constexpr int ES = F16 ? 16 : 8;                   // bytes per (segment, bin)
    static constexpr int NSEG = F16 ? NG : 3 * NG;            // staged segments per angle
    static constexpr int GS = BM_SLOT * ES;                   // segment pitch
    static constexpr int UPS = GS / 16;                       // 16-byte units per segment
    static constexpr int UNITS = NSEG * UPS;
    static constexpr int NI = (UNITS + 63) / 64;              // wave loads per angle (64 units each, the last fewer)
    static constexpr int NACC = (FORM == 0 || FORM == 2) ? 2 : 1;
    static constexpr int NB = FORM == 0 ? 3 : (FORM == 3 ? 1 : 2); // B operands per step
    // Two accumulators per patch (128 registers a wave): two waves per SIMD, the
    // operands read one step ahead.  One accumulator: four waves per SIMD (two
    // workgroups per CU) that read them in place.
    static constexpr bool PIPE = NACC == 2;
    static constexpr int WAVES = 8, THREADS = 64 * WAVES;
    static constexpr int PPW = BM_NX * BM_NY / WAVES;         // patches per wave, side by side in x
    static constexpr int WPA = WAVES / BM_CH;                 // waves that stage one angle
    static constexpr int NJ = (NI + WPA - 1) / WPA;           // loads per wave and round; the last of the WPA: NL
    static constexpr int NL = NI - (WPA - 1) * NJ;
    static_assert(NL >= 1 && NL <= NJ, "staging split");
    static constexpr int ZERO = NSEG * GS;                    // FORM 1: a segment of zeros behind the others
    static constexpr int AS = (NSEG + (FORM == 1)) * GS;      // angle pitch
    static constexpr int BUF = BM_CH * AS + 256 + 16;         // a round's windows, 16 coefficient pairs, 4 offsets
    static constexpr int DEPTH = FORM == 1 ? 3 : 4;                           // LDS buffers; loads run DEPTH - 1 rounds ahead
    static constexpr int STAGE = DEPTH * BUF;
    static constexpr int COLS = PIPE ? 32 : 16;              // slices of one round of the output exchange
    static constexpr int OP = COLS + 4;                       // its floats per pixel
    static constexpr int OUT = BM_TX * BM_TY * OP * 4;
};
template <int FORM> constexpr int bm_lds() { return std::max(Form<FORM>::STAGE, Form<FORM>::OUT); }

// the FP32 value behind three bf16 pieces (a non-finite one sits in h alone)
__device__ __forceinline__ float bm_join(const unsigned short* h, size_t piece)
{
    const float fh = __uint_as_float((unsigned)h[0] << 16);
    if (!(fh - fh == 0.0f)) return fh;
    return (fh + __uint_as_float((unsigned)h[piece] << 16)) + __uint_as_float((unsigned)h[2 * piece] << 16);
}

// one slice's sum at pixel (X, Y), in the gather kernels' order (FP32: partial
// sums over BP_GROUP angles; FP16: one running sum)
// (arguments by value: a reference to the kernel's own would move them to memory)
template <bool F16, bool CHECKED>
__device__ __noinline__ float bm_one(const char* q, const d2v* cs, double c0, int A, int G, int W_, int tlo, int sl, double X,
                                     double Y)
{
    constexpr int SB = F16 ? 8 : 4;
    constexpr bool SPLIT = !F16 && !CHECKED;
    const size_t W = (size_t)W_, arow = W * (SPLIT ? 24 : 16); // bytes of one angle of one group
    const char* row = q + (size_t)(sl / SB) * (CHECKED ? A : 1) * arow;
    const size_t step = arow * (CHECKED ? 1 : G); // to the next angle
    const int s = sl % SB;
    float tot = 0.0f;
    for (int a0 = 0; a0 < A; a0 += BP_GROUP) {
        float part = 0.0f;
        const int a1 = min(A, a0 + BP_GROUP);
        for (int ang = a0; ang < a1; ++ang) {
            const size_t b = (size_t)((int)fma(X, cs[ang].x, fma(Y, cs[ang].y, c0)) - tlo);
            if (F16) tot += __half2float(reinterpret_cast<const __half*>(row + (size_t)ang * step + b * 16)[s]);
            else if (SPLIT)
                part += bm_join(reinterpret_cast<const unsigned short*>(row + (size_t)ang * step + b * 8) + s, W * 4);
            else part += reinterpret_cast<const float*>(row + (size_t)ang * step + b * 16)[s];
        }
        if (!F16) tot += part;
        if (tot != tot) break; // NaN stays NaN
    }
    return tot;
}

template <int FORM, bool CHECKED>
__global__ __launch_bounds__(Form<FORM>::THREADS, Form<FORM>::PIPE ? 2 : 4) void k_backproject_mx(BmArgs a)
{
    using F = Form<FORM>;
    extern __shared__ __align__(16) char bm_smem[];
    lds_char* lds = (lds_char*)bm_smem;

    // XCD-contiguous order: the hardware deals workgroups to the 8 XCDs round
    // robin; XCD x takes the tiles [x per, (x + 1) per), walked in strips of 4
    // tile rows, so the tiles it runs together share bins in its L2
    const unsigned per = ((unsigned)a.total + 7u) >> 3;
    const unsigned id = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (id >= (unsigned)a.total) return;
    const unsigned ntile = (unsigned)(a.tiles_x * a.tiles_y);
    const unsigned pack = id / ntile;
    unsigned t = id - pack * ntile;
    const unsigned strip = t / (4u * a.tiles_x);
    t -= strip * 4u * a.tiles_x;
    const unsigned srows = min(4u, (unsigned)a.tiles_y - strip * 4u);
    const int i0 = (int)(t / srows) * BM_TX;
    const int j0 = (int)(strip * 4u + t % srows) * BM_TY;
    const int s0 = a.s_first + (int)pack * F::SLICES;  // first slice of the pack
    const int g0 = s0 / (F::F16 ? 8 : 4);              // its first row group

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    // pixel of this lane's matrix row (rows 30 and 31 repeat pixel 0)
    const int m = (lane & 31) < BM_PIX ? (lane & 31) : 0;
    const int px0 = i0 + BM_PX * F::PPW * (wave % (BM_NX / F::PPW)); // this wave's patches
    const int py0 = j0 + BM_PY * (wave / (BM_NX / F::PPW));
    double X[F::PPW];
#pragma unroll
    for (int k = 0; k < F::PPW; ++k) X[k] = (double)(px0 + BM_PX * k + m % BM_PX) - a.xc;
    const double Y = (double)(py0 + m / BM_PX) - a.xc;
    const double Yc = (double)(py0 + 2) - a.xc;
    double Xt = ((double)i0 + 0.5 * (BM_TX - 1)) - a.xc;
    double Yt = ((double)j0 + 0.5 * (BM_TY - 1)) - a.xc;
    const double c0c = a.c0 - BM_REACH;
    double c0t = a.c0 - BM_TILE_REACH;
    // in vector registers: an FP64 operation reads one scalar operand only
    asm volatile("" : "+v"(Xt), "+v"(Yt), "+v"(c0t));

    // B operand addresses: lane i of a 16-lane group reads bin row i / 4, column
    // chunk i % 4 (4 columns of 2 bytes); lanes 16..31 the next 16 columns
    const int cc = 4 * ((lane >> 4) & 1) + (lane & 3);
    const int rb = ((lane & 15) >> 2) * F::ES;
    const int lofs0 = F::F16 ? (cc >> 1) * F::GS + (cc & 1) * 8 + rb : cc * F::GS + rb;
    // FORM 1, second operand: zeros under the h columns, l under the m columns
    const int lofs1 = FORM == 1 ? (cc < 4 ? F::ZERO : (2 * F::NG + cc - 4) * F::GS) + rb : 0;

    f16x acc[F::PPW][F::NACC];
#pragma unroll
    for (int k = 0; k < F::PPW; ++k)
#pragma unroll
        for (int c = 0; c < F::NACC; ++c)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[k][c][i] = 0.0f;

    if (FORM == 1) {
        // the segment of zeros of every angle slot
        for (int e = tid; e < F::DEPTH * BM_CH * BM_SLOT; e += F::THREADS)
            *reinterpret_cast<u2v*>(bm_smem + e / (BM_CH * BM_SLOT) * F::BUF + e / BM_SLOT % BM_CH * F::AS + F::ZERO +
                                    e % BM_SLOT * 8) = u2v{0u, 0u};
    }

    // ---- staging.  Waves WPA al .. WPA al + WPA - 1 move angle slot al.
    // Unchecked: NJ loads of 64 16-byte units each straight into LDS; unit u is
    // 16 bytes of segment u / UPS.  Checked: rows (angle, group) through
    // registers, half of the groups each of the angle's two waves.
    const int al = wave / F::WPA, ws = wave % F::WPA;
    constexpr int SG = CHECKED ? F::NG / F::WPA : 1; // checked: groups per wave
    const unsigned arow = (unsigned)a.W * (!F::F16 && !CHECKED ? 24u : 16u); // bytes of one angle of one group
    const char* src[SG];
    unsigned off[F::NJ];
    if (CHECKED) {
#pragma unroll
        for (int u = 0; u < SG; ++u) src[u] = a.q + (size_t)min(g0 + SG * ws + u, a.G - 1) * a.A * arow;
    } else {
#pragma unroll
        for (int j = 0; j < F::NJ; ++j) {
            const int u = min((ws * F::NJ + j) * 64 + lane, F::UNITS - 1);
            const int seg = u / F::UPS, pos = u % F::UPS;
            const int g = min(g0 + seg % F::NG, a.G - 1);
            // less the instruction's offset, 4096 more to stay positive
            off[j] = (unsigned)g * arow + (unsigned)(seg / F::NG) * (unsigned)a.W * 8u + (unsigned)pos * 16u +
                     (4096u - 1024u * (unsigned)(j - 1));
        }
    }
    // the loads of a round's last 64 units are fewer; this lane takes part in them
    const bool tail_lane = lane < F::UNITS - 64 * (F::NI - 1);
    u4v st[SG];
    unsigned stc = 0; // checked, wave 0: a dword of the round's coefficient pairs
    // Coefficients of the round at a0: this lane's two angles as matrix row
    // (a0 + half, a0 + 2 + half) and its angle as role lane (below).
    // From the round's LDS buffer (vector loads would have to be waited for
    // together with the younger window loads).
    const int rk = lane & 3, rj = (lane >> 2) & 3; // role: patch and job
    const int ra = rj == 0 ? half : (rj == 1 ? 2 + half : 2 * half + (rj & 1));
    auto coefs = [&](int bufo, d2v (&c)[3], int& bias) __attribute__((always_inline)) {
        const d2v* t = reinterpret_cast<const d2v*>(bm_smem + bufo + BM_CH * F::AS);
        c[0] = t[half];
        c[1] = t[2 + half];
        c[2] = t[ra];
        bias = reinterpret_cast<const int*>(bm_smem + bufo + BM_CH * F::AS + 256)[ra];
    };
    // Role lanes: in every row of 16 lanes, lane rk + 4 rj holds for patch rk
    // minus the window base of the row's first (rj = 0) and second (1)
    // matrix-row angle (minus: row broadcasts fold into additions; folded into
    // a subtraction the compiler's form gave wrong values), and the LDS offset of that base in the windows of the two angles
    // (2 half, 2 half + 1) this half reads as operand (2, 3); the step of
    // patch k takes them with row broadcasts.
    const double Xr = ((double)(px0 + BM_PX * (rk % F::PPW)) + 2.5) - a.xc;
    auto roles = [&](const d2v c, int bias) __attribute__((always_inline)) {
        const int base = (int)fma(Xr, c.x, fma(Yc, c.y, c0c));
        return rj < 2 ? -base : base * F::ES + bias;
    };
    // the LDS offset of bin 0 of angle slot u of a buffer (from the window's first
    // bin), left in the buffer by the wave that stages that window
    int* const bias_at = reinterpret_cast<int*>(bm_smem + BM_CH * F::AS + 256);
    // this wave's angle slot of the round at a0 (uniform: scalar loads)
    typedef const __attribute__((address_space(4))) d2v* cptr;
    auto slot = [&](int a0) __attribute__((always_inline)) { return ((cptr)a.cs)[CHECKED ? min(a0 + al, a.A - 1) : a0 + al]; };
    auto issue = [&](int a0, int bufo, const d2v c) __attribute__((always_inline)) {
        const int ang = min(a0 + al, a.A - 1);
        int w = __builtin_amdgcn_readfirstlane((int)fma(Xt, c.x, fma(Yt, c.y, c0t))) - a.tlo;
        if (!F::F16 && !CHECKED) w &= ~1;
        if (tid == wave * 64) bias_at[bufo / 4 + al] = bufo + al * F::AS - (a.tlo + w) * F::ES;
        if (CHECKED) {
            if (wave == 0 && lane < 4 * BM_CH)
                stc = reinterpret_cast<const unsigned*>(a.cs)[4 * min(a0 + (lane >> 2), a.A - 1) + (lane & 3)];
            // bins outside the rows are zeros no pixel of the image reads
            const int b = w + lane;
#pragma unroll
            for (int u = 0; u < SG; ++u) {
                st[u] = u4v{0u, 0u, 0u, 0u};
                if (lane < BM_SLOT && (unsigned)b < (unsigned)a.W)
                    st[u] = *reinterpret_cast<const u4v*>(src[u] + (size_t)ang * arow + (size_t)b * 16);
            }
        } else {
            const unsigned dst = (unsigned)(size_t)lds + (unsigned)bufo;
            if (wave == 0) load_lds4(reinterpret_cast<const char*>(a.cs + a0), 4u * lane, dst + BM_CH * F::AS);
            const char* base = a.q + (size_t)ang * ((size_t)arow * a.G) + (w * F::ES - 4096);
            const unsigned d = dst + (unsigned)(al * F::AS + ws * F::NJ * 1024);
            if (ws < F::WPA - 1) {
                load_lds<F::NJ>(base, off, d);
            } else {
                if constexpr (F::NL > 1) load_lds<F::NL - 1>(base, off, d);
                const unsigned last[1] = {off[F::NL - 1] - 1024u};
                if (tail_lane) load_lds<1>(base + 1024 * F::NL, last, d + 1024u * (F::NL - 1));
            }
        }
    };
    auto commit = [&](int bufo) __attribute__((always_inline)) {
        if (!CHECKED || lane >= BM_SLOT) return;
        if (wave == 0 && lane < 4 * BM_CH) *reinterpret_cast<unsigned*>(bm_smem + bufo + BM_CH * F::AS + 4 * lane) = stc;
#pragma unroll
        for (int u = 0; u < SG; ++u) {
            char* d = bm_smem + bufo + al * F::AS + (SG * ws + u) * F::GS + lane * F::ES;
            if (F::F16) {
                *reinterpret_cast<u4v*>(d) = st[u];
            } else {
                uint2 h, md, l;
                split4(make_float4(__uint_as_float(st[u][0]), __uint_as_float(st[u][1]), __uint_as_float(st[u][2]),
                                   __uint_as_float(st[u][3])), h, md, l);
                *reinterpret_cast<uint2*>(d) = h;
                *reinterpret_cast<uint2*>(d + F::NG * F::GS) = md;
                *reinterpret_cast<uint2*>(d + 2 * F::NG * F::GS) = l;
            }
        }
    };
    constexpr unsigned ONE = F::F16 ? 0x3c00u : 0x3f80u;
    // Round r uses buffer r % DEPTH.  In the middle of round r (before the last
    // but one of its steps) the workgroup meets: from there on the windows of
    // round r + 1 are in LDS and nobody reads those of round r - 1, so the loads
    // of round r + DEPTH - 1 start.  A step's operands are read one step ahead,
    // across rounds too, so neither the products nor the reads drain at the
    // meeting point.  Rounds past the last angle load the last one again.
    constexpr int AHEAD = CHECKED ? 2 : F::DEPTH - 1;
    if (CHECKED) {
        issue(0, 0, slot(0));
        commit(0);
        issue(BM_CH, F::BUF, slot(BM_CH));
    } else {
#pragma unroll
        for (int r = 0; r < AHEAD; ++r) issue(r * BM_CH, r * F::BUF, slot(r * BM_CH));
    }
    d2v sl_c = slot(AHEAD * BM_CH);
    if (!CHECKED) wait_loads();
    __syncthreads();

    // selection of a step: the patch's matrix rows and its operand offsets
    constexpr int SLOTS = F::PIPE ? 2 : 1;
    u4v av[SLOTS];
    int idx[SLOTS], e0, e1, d0, d1;
    double cA0, cA1, rt0, rt1;
    unsigned one0, one1;
    int rv;
    auto enter = [&](int a0, const d2v (&c)[3], int bias) __attribute__((always_inline)) {
        cA0 = c[0].x;
        cA1 = c[1].x;
        rt0 = fma(Y, c[0].y, a.c0);
        rt1 = fma(Y, c[1].y, a.c0);
        // angles past A select nothing
        one0 = a0 + half < a.A ? ONE : 0u;
        one1 = a0 + 2 + half < a.A ? ONE : 0u;
        rv = roles(c[2], bias);
    };
    auto address = [&](int k) __attribute__((always_inline)) {
        e0 = row_lane(rv, 8 + k);
        e1 = row_lane(rv, 12 + k);
    };
    auto bins = [&](int k) __attribute__((always_inline)) {
        d0 = (int)fma(X[k], cA0, rt0) + row_lane(rv, k);
        d1 = (int)fma(X[k], cA1, rt1) + row_lane(rv, 4 + k);
    };
    // matrix row: slots 0, 1 = bins 0..3 and 2, 3 = bins 4..7 of the first angle,
    // slots 4..7 of the second; one 1 per angle, the selected bin of a slot pair
    // in its index (bits 2 of d fall into the indices of the zero slots)
    auto select = [&](int k) __attribute__((always_inline)) {
        const int q = k % SLOTS;
        av[q] = u4v{d0 < 4 ? one0 : 0u, d0 < 4 ? 0u : one0, d1 < 4 ? one1 : 0u, d1 < 4 ? 0u : one1};
        const int ix = d0 | (d1 << 8);
        idx[q] = ix | (ix << 4);
    };
    union Operand {
        s4v h[4];
        bf16x16 v;
        h16x16 f;
    } O[F::NB];
    auto read = [&](int b) __attribute__((always_inline)) {
        const int lo = FORM == 1 && b == 1 ? lofs1 : lofs0;
        const int bo = FORM == 1 ? 0 : b * (F::F16 ? 4 : 8) * F::GS;
        lds_char* p0 = lds + (e0 + lo);
        lds_char* p1 = lds + (e1 + lo);
        O[b].h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p0 + bo));
        O[b].h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p0 + bo + 4 * F::ES));
        O[b].h[2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p1 + bo));
        O[b].h[3] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p1 + bo + 4 * F::ES));
    };
    auto product = [&](int k, int b) __attribute__((always_inline)) {
        f16x& A = acc[k][b == 0 ? 0 : F::NACC - 1];
        if constexpr (F::F16)
            A = __builtin_amdgcn_smfmac_f32_32x32x32_f16(__builtin_bit_cast(h8v, av[k % SLOTS]), O[b].f, A, idx[k % SLOTS], 0, 0);
        else
            A = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(__builtin_bit_cast(bf8v, av[k % SLOTS]), O[b].v, A, idx[k % SLOTS], 0, 0);
    };

    d2v cn[3];
    int bias;
    coefs(0, cn, bias);
    enter(0, cn, bias);
    if (F::PIPE) {
        address(0);
#pragma unroll
        for (int b = 0; b < F::NB; ++b) read(b);
        bins(0);
        select(0);
    }
    int b1 = F::BUF, bf = (AHEAD % F::DEPTH) * F::BUF; // buffers of round r + 1 and of round r + AHEAD
    auto next_buf = [](int b) __attribute__((always_inline)) { return b == (F::DEPTH - 1) * F::BUF ? 0 : b + F::BUF; };
    // the windows of round r + 1 are in LDS and nobody reads those of round r - 1
    // any more; the last round's look-ahead finds the last angle again
    auto meet = [&](int a0) __attribute__((always_inline)) {
        if (CHECKED) commit(b1);
        else if (ws == F::WPA - 1) wait_loads_but<(AHEAD - 2) * F::NL>();
        else wait_loads_but<(AHEAD - 2) * F::NJ>();
        __syncthreads();
        issue(a0 + AHEAD * BM_CH, bf, sl_c);
        sl_c = slot(a0 + (AHEAD + 1) * BM_CH);
        asm volatile("" ::: "memory"); // keeps that load here, not at its use in the next round
        coefs(b1, cn, bias);
        b1 = next_buf(b1);
        bf = next_buf(bf);
    };
#pragma unroll 1
    for (int a0 = 0; a0 < a.A; a0 += BM_CH) {
#pragma unroll
        for (int k = 0; k < F::PPW; ++k) {
            if constexpr (F::PIPE) {
                if (k == F::PPW - 2) meet(a0);
                const int kn = (k + 1) % F::PPW;
                if (kn == 0) enter(a0 + BM_CH, cn, bias);
                address(kn);
                // a product, the next step's operand in its place, the next
                // step's selection in between
#pragma unroll
                for (int b = 0; b < F::NB; ++b) {
                    product(k, b);
                    read(b);
                    if (b == 0) bins(kn);
                    if (b == 1) select(kn);
                }
            } else {
                address(k);
#pragma unroll
                for (int b = 0; b < F::NB; ++b) read(b);
                bins(k);
                select(k);
#pragma unroll
                for (int b = 0; b < F::NB; ++b) product(k, b);
            }
        }
        if (!F::PIPE) {
            meet(a0);
            enter(a0 + BM_CH, cn, bias);
        }
    }
    wait_loads();
    __syncthreads(); // LDS is free for the exchange

    // ---- output: accumulators through LDS ([pixel][column]), then one pixel
    // per thread.  Lane l holds column l % 32 of rows 8 (i / 4) + 4 (l / 32) + i % 4.
    constexpr int ROUNDS = F::SLICES / F::COLS;
    float* ex = reinterpret_cast<float*>(bm_smem);
    const size_t nn = (size_t)a.n * a.n;
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
        if (rd > 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < F::PPW; ++k)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 8 * (i >> 2) + 4 * half + (i & 3);
                const int px = (py0 - j0 + r / BM_PX) * BM_TX + px0 - i0 + BM_PX * k + r % BM_PX;
                float v = acc[k][FORM == 2 ? rd : 0][i];
                if (FORM == 0) v += acc[k][1][i];
                if (FORM == 1) v += __shfl_xor(v, 16); // h + (m + l), the columns 16 apart
                const bool mine = F::COLS == 32 || ((lane >> 4) & 1) == rd;
                if (r < BM_PIX && mine) ex[px * F::OP + (lane & (F::COLS - 1))] = v;
            }
        __syncthreads();
        for (int px = tid; px < BM_TX * BM_TY; px += F::THREADS) {
            const int i = i0 + px % BM_TX, j = j0 + px / BM_TX;
            if (i >= a.n || j >= a.n) continue;
            const float4* e4 = reinterpret_cast<const float4*>(ex + px * F::OP);
#pragma unroll 1
            for (int qd = 0; qd < F::COLS / 4; ++qd) {
                const int sl = s0 + F::COLS * rd + 4 * qd;
                if (sl >= a.S) break;
                float4 tv = e4[qd];
                // x - x is 0 for finite values only
                const float chk = (tv.x - tv.x) + (tv.y - tv.y) + (tv.z - tv.z) + (tv.w - tv.w);
                if (!(chk == 0.0f)) {
                    const double Xp = (double)i - a.xc, Yp = (double)j - a.xc;
                    if (!(tv.x - tv.x == 0.0f)) tv.x = bm_one<F::F16, CHECKED>(a.q, a.cs, a.c0, a.A, a.G, a.W, a.tlo, sl, Xp, Yp);
                    if (!(tv.y - tv.y == 0.0f) && sl + 1 < a.S) tv.y = bm_one<F::F16, CHECKED>(a.q, a.cs, a.c0, a.A, a.G, a.W, a.tlo, sl + 1, Xp, Yp);
                    if (!(tv.z - tv.z == 0.0f) && sl + 2 < a.S) tv.z = bm_one<F::F16, CHECKED>(a.q, a.cs, a.c0, a.A, a.G, a.W, a.tlo, sl + 2, Xp, Yp);
                    if (!(tv.w - tv.w == 0.0f) && sl + 3 < a.S) tv.w = bm_one<F::F16, CHECKED>(a.q, a.cs, a.c0, a.A, a.G, a.W, a.tlo, sl + 3, Xp, Yp);
                }
                float* o = a.out + (size_t)sl * nn + (size_t)j * a.n + i;
                o[0] = tv.x;
                if (sl + 1 < a.S) o[nn] = tv.y;
                if (sl + 2 < a.S) o[2 * nn] = tv.z;
                if (sl + 3 < a.S) o[3 * nn] = tv.w;
            }
        }
    }
}

constexpr long long BM_CUS = 256;
long long bm_tiles(int n) { return (long long)((n + BM_TX - 1) / BM_TX) * ((n + BM_TY - 1) / BM_TY); }

template <int FORM, bool CHECKED> void bm_launch(BmArgs a, int first, int packs, hipStream_t st)
{
    if (packs <= 0) return;
    a.s_first = first;
    a.tiles_x = (a.n + BM_TX - 1) / BM_TX;
    a.tiles_y = (a.n + BM_TY - 1) / BM_TY;
    const long long total = (long long)a.tiles_x * a.tiles_y * packs;
    if (total > 0x7ffffff0LL) fail(RAFT_EUNSUPPORTED, "too many tiles for one backprojection launch");
    a.total = (int)total;
    const void* fn = reinterpret_cast<const void*>(&k_backproject_mx<FORM, CHECKED>);
    constexpr int lds = bm_lds<FORM>();
    RAFT_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    void* args[] = {&a};
    RAFT_HIP(hipLaunchKernel(fn, dim3(8u * (((unsigned)total + 7u) / 8u)), dim3(Form<FORM>::THREADS), args, lds, st));
}

} // namespace

// Packs of a launch: wide ones, and a narrow one (half as many slices) for a
// rest that fits it, unless one more wide pack starts at once on idle CUs.
struct BmPlan {
    int wide, narrow;
};
static BmPlan bm_plan(int S, int n, bool f16)
{
    const int w = f16 ? Form<2>::SLICES : Form<0>::SLICES;
    const long long tiles = bm_tiles(n);
    BmPlan p = {S / w, 0};
    const int rest = S % w;
    if (rest > w / 2 || (rest > 0 && tiles * (p.wide + 1) <= BM_CUS)) ++p.wide;
    else if (rest > 0) p.narrow = 1;
    return p;
}

// Whether an FBP call of S slices of n x n from A angles runs here.
// Backprojection time, gather form -> this file, n angles and rays (ms):
//   FP32 rows   S = 16            32             64
//     n =  512  0.188 -> 0.206  0.277 -> 0.298  0.531 -> 0.465
//     n = 1024  0.985 -> 1.040  1.97  -> 1.54   3.96  -> 2.91
//     n = 2048  7.95  -> 7.25   15.1  -> 11.1   29.5  -> 21.1
//   FP16 rows   S = 8             16             64
//     n =  512  0.203 -> 0.154  0.210 -> 0.155  0.478 -> 0.265
//     n = 1024  0.514 -> 0.727  0.902 -> 0.732  3.08  -> 1.32
//     n = 2048  3.18  -> 4.55   6.15  -> 4.70   23.8  -> 9.31
// FP16 rows gain from half a narrow pack on, at every n.  FP32 rows need full
// packs and enough tiles: per angle a round of wide packs over the chip (one
// workgroup on each of 256 CUs) takes 0.30 us and a round of narrow ones (two on
// each) 0.39 us, the gather form 0.057 us per 10^6 pixels and slices (a little
// more where it cannot fill the chip).
// The image leaves through LDS here, 0.8 to 0.9 us per 10^6 pixels and slices more
// than in the gather form, which the angles have to earn back.  Few angles (us):
//   FP32 2048, S = 64   A = 2  190 -> 447   32  559 -> 670   64  1010 -> 930
//         512, S = 200       35 -> 77          113 -> 138        201 -> 205
//         200, S = 150       12 -> 14           31 -> 22          52 -> 30
//   FP16 2048, S = 32       120 -> 220        215 -> 219        394 -> 277
//        1024, S = 16        16 -> 34          37 -> 50          65 -> 70
//          64, S = 70         7 -> 16          18 -> 22          31 -> 29
// There the gather form takes 0.44 ns a workgroup and angle and 0.14 us an angle
// (FP16 0.6 ns and 0.2 us, 0.37 us at least), a round here 0.27 us (narrow 0.36, FP16
// 0.22; FP16's small images 2.6 us and 0.09 us a slice of a pack besides).
bool bp_matrix_form(int S, int n, int A, int store)
{
    if (S < 16 || n < 1) return false;
    const bool f16 = store == RAFT_STORE_F16;
    const BmPlan p = bm_plan(S, n, f16);
    const long long tiles = bm_tiles(n);
    const double wide = (double)((tiles * p.wide + BM_CUS - 1) / BM_CUS);
    const double narrow = (double)((tiles * p.narrow + 2 * BM_CUS - 1) / (2 * BM_CUS));
    const double image = 1.0e-6 * (double)n * n * S;
    const int sb = f16 ? BP_SLICES_F16 : BP_SLICES_F32;
    const double groups = (double)bp_tiles(n) * ((S + sb - 1) / sb); // workgroups of the gather form
    if (f16) {
        const double once = 2.6 + 0.09 * std::min(S, Form<2>::SLICES) + 0.8 * image;
        return A * 0.22 * (wide + narrow) + once < A * std::max(0.37, 0.6e-3 * groups + 0.2);
    }
    return 0.30 * wide + 0.39 * narrow < 0.057 * image &&
           A * (0.27 * wide + 0.36 * narrow) + 0.9 * image < A * (0.437e-3 * groups + 0.14);
}

// One launch addresses an angle's rows with 32-bit byte offsets, and takes no
// more slice groups than the gather form does (a larger call is left to that
// form, which refuses it).  A row holds less than 1.5 n + 128 bins.
constexpr long long BM_GROUPS = 65535, BM_BYTES = (1LL << 32) - 8192;
bool bp_matrix_fits(int slices, int n, int store)
{
    const int pack = bp_matrix_pack(store), sb = store == RAFT_STORE_F16 ? BP_SLICES_F16 : BP_SLICES_F32;
    const long long groups = ((long long)slices + pack - 1) / pack * (pack / sb);
    return groups <= BM_GROUPS && groups * (3LL * n / 2 + 128) * (long long)bp_matrix_entry(store) <= BM_BYTES;
}

int bp_matrix_pack(int store) { return store == RAFT_STORE_F16 ? 32 : 16; }

size_t bp_matrix_entry(int store) { return store == RAFT_STORE_F16 ? 16 : 24; }

void bp_window_matrix(BpGeom& g)
{
    const int tx = (g.n + BM_TX - 1) / BM_TX, ty = (g.n + BM_TY - 1) / BM_TY;
    const double h = 0.5 * (BM_TX - 1), v = 0.5 * (BM_TY - 1);
    const double xlo = h - g.xc, xhi = (double)((tx - 1) * BM_TX) + h - g.xc;
    const double ylo = v - g.xc, yhi = (double)((ty - 1) * BM_TY) + v - g.xc;
    long long tmin = 0x7fffffffLL, tmax = -0x7fffffffLL;
    for (int a = 0; a < g.nangles; ++a) {
        // first bins of the corner tiles' windows; every other tile's lies between
        for (double X : {xlo, xhi})
            for (double Y : {ylo, yhi}) {
                const long long t = (long long)std::floor(X * g.cA[a] + Y * g.cB[a] + g.c0 - BM_TILE_REACH);
                tmin = std::min(tmin, t);
                tmax = std::max(tmax, t);
            }
    }
    // one bin for truncation toward zero, one for the 16-byte alignment, one
    // for rounding on each side; an even width keeps every row aligned
    tmin -= 3;
    tmax += 2 + BM_SLOT;
    g.tlo = (int)tmin;
    g.width = (int)((tmax - tmin + 2) & ~1LL);
}

template <bool CHECKED> static void bm_launch_plan(const BmArgs& a, const BmPlan& p, bool f16, hipStream_t st)
{
    if (f16) {
        bm_launch<2, CHECKED>(a, 0, p.wide, st);
        bm_launch<3, CHECKED>(a, p.wide * Form<2>::SLICES, p.narrow, st);
    } else {
        bm_launch<0, CHECKED>(a, 0, p.wide, st);
        bm_launch<1, CHECKED>(a, p.wide * Form<0>::SLICES, p.narrow, st);
    }
}

void launch_backproject_mx(const BpArgs& b, int store, hipStream_t st)
{
    const bool f16 = store == RAFT_STORE_F16;
    BmArgs a;
    a.q = static_cast<const char*>(b.q);
    a.out = b.out;
    a.cs = reinterpret_cast<const d2v*>(b.cs); a.xc = b.xc; a.c0 = b.c0;
    a.n = b.n; a.A = b.A; a.tlo = b.tlo; a.W = b.W; a.S = b.S;
    a.G = (b.S + (f16 ? 8 : 4) - 1) / (f16 ? 8 : 4);
    const bool checked = b.chunk == BP_MX_CHECKED;
    if (!b.cs || b.mode != 0) fail(RAFT_EINVAL, "internal: the matrix form runs FBP sums with the paired coefficient table");
    const size_t need = (size_t)a.G * a.A * a.W * (checked ? 16 : bp_matrix_entry(store));
    if (b.q_bytes && need > b.q_bytes)
        fail(RAFT_EINVAL, "internal: backprojection would read past its staged rows");
    if (a.G > BM_GROUPS || (!checked && (long long)a.G * a.W * (long long)bp_matrix_entry(store) > BM_BYTES))
        fail(RAFT_EUNSUPPORTED, "too many slice groups for one backprojection launch");
    const BmPlan p = bm_plan(b.S, b.n, f16);
    if (checked) bm_launch_plan<true>(a, p, f16, st);
    else bm_launch_plan<false>(a, p, f16, st);
}

} // namespace raft
