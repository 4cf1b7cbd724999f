// Fused sector kernel with wave-private FFTs, N = 256..8192: the plain form,
// and the chosen form off the producer/consumer kernels (N = 4096 / 8192, or
// stations on different band starts; phased sums from N = 2048 on); ACF / XCF
// products or the phased sum.
//
// M = N / 2 complex points per station-frame, split M = 32 x M2:
//   m = M2 m1 + m2,  k = k1 + 32 k2
//   stage 1:  Y[m2][k1]    = W_M^{m2 k1} sum_m1 z[M2 m1 + m2] W32^{m1 k1}
//   stage 2:  Z[k1 + 32 k2] = sum_m2 Y[m2][k1] W_M2^{m2 k2}
// Every wave holds 2048 points, 32 per lane, whatever M is: 2048 / M
// station-frames for M <= 2048, a half (quarter) of one above.  Stage 1 is a
// DFT-32 per lane on the VALU (lane = row m2), or, for the chosen form, the
// FP16 hi/lo MFMA GEMM on 16-row tiles of the same rows.  Stage 2 is one
// DFT-M2 per column in a lane's registers for M2 <= 32 (M <= 1024), two
// passes (8 x 8, 16 x 8) for M2 = 64 / 128.  The passes exchange through LDS
// within the wave, with no barrier for M <= 2048.  Between stages the data
// stay in place (slot k1 M2 + position), under an XOR swizzle that gives every
// pass's reads and writes all 64 banks once per half-wave (wk_slot).
//
// A workgroup is four waves, two per station: F = 4096 / M frames a round.
// After one barrier all 256 threads form the round's products, each thread the
// same bin pairs (p, M - p) of every frame: both stations' untangles share the
// pair's reads, and the masks of bins outside the overlap are applied once, to
// the sums.  64 KB of Z and 15 KB of tables: two workgroups per CU, whose
// rounds overlap (one's products with the other's FFTs).
//
// Samples reach the FFT as FP16 (exact: the plan checks the levels) from a
// zero-padded row that byte tables decode into, as in the MFMA kernels; the
// integer shift is an offset into it.  The row shares the Z slot's memory.
//
// Bound by VALU issue: at N = 1024 1,264 VALU instructions per frame pair (the
// Stockham kernel: 2,973; half of the 1,264 are the DFTs' additions), 75 % of
// its SIMD cycles; HBM and the LDS are far from their rates.  Two waves per
// SIMD, because 32 points, the FP64 sums and the twiddles of a lane take
// 180..256 VGPRs; from N = 4096 on they leave a third to a half of the cycles
// to LDS latency and, at 8192, the transform's barriers.  2^27 samples per
// station, 2-bit, whole calls, Stockham kernel -> this one (microseconds; plain
// from N = 2048 with the phase chains): plain 256: 1052 -> 399, 512: 975 ->
// 378, 1024: 778 -> 390, 2048: 1456 -> 629, 4096: 1604 -> 750, 8192: 1340 ->
// 899; chosen 4096: 710 -> 491, 8192: 912 -> 736; phased power, plain 256: 1677
// -> 663, 1024: 1266 -> 637, 4096: 1560 -> 818; chosen 2048: 697 -> 472, 4096:
// 791 -> 552, 8192: 1068 -> 584.
#include <type_traits>

#include "fxc_dev.h"

namespace fxc {

namespace wk {
template <int LOGM>
struct Shape {
    static constexpr int M = 1 << LOGM, N = 2 * M, M2 = M / 32;
    static constexpr int WAVES = 4, NT = 64 * WAVES;
    static constexpr int F = WAVES * 2048 / (2 * M);          // frames per round
    static constexpr int SPW = M <= 2048 ? 2048 / M : 1;      // station-frames per wave
    static constexpr int WPS = M <= 2048 ? 1 : M / 2048;      // waves per station-frame
    static constexpr int PAD = N >= 512 ? 64 : 32;            // zero samples each side of a staged frame
    static constexpr int A = M2 <= 32 ? 1 : (M2 == 64 ? 8 : 16), B = M2 / A;   // stage 2 = A x B
    static constexpr int RB = 32 / B;                         // runs of B slots per 64 banks
    static constexpr int PPT = M / 2 >= NT ? M / 2 / NT : 1;  // bin pairs per thread
    static constexpr int G = M / 2 >= NT ? 1 : NT / (M / 2);  // thread groups sharing the pairs
    // staged rows: SK dwords of skew after every M2 dwords (the MFMA operand
    // reads of lane groups g lie M2 dwords apart), and station-frame q of a
    // wave QO q dwords into its slot (their rows' reads run side by side)
    static constexpr int SK = M2 >= 32 ? 16 : 0, QO = M2 < 64 ? M2 : 0;
    static_assert(F >= 1, "frames per round");
};

}  // namespace wk

template <int LOGM, typename P>
struct WkShared {
    using S = wk::Shape<LOGM>;
    alignas(16) float2 z[2][S::F][S::M];
    uint32_t slut[2][4 * 256];
    alignas(16) uint16_t dlut[2][kWkDlutHalves];
    float2 w2[S::A > 1 ? S::M2 : 1];
    P pp[S::F];   // the iteration's frames
};

// Slot of element (row k1, position a B + b) of the wave's station-frame q.
// Runs of B slots rotate over the bank groups with k1 (two-pass stage 2) or
// with q (single pass), and the slots of a run are permuted by the remaining
// index bits; each pass's 32 concurrent lanes then differ in (run, slot).
template <int LOGM>
__device__ __forceinline__ int wk_slot(int q, int k1, int a, int b) {
    using S = wk::Shape<LOGM>;
    if constexpr (S::A == 1) {
        const int row = k1 ^ (q & (S::RB - 1));
        return row * S::M2 + (b ^ ((k1 / S::RB) & (S::B - 1)));
    } else {
        return k1 * S::M2 + S::B * (a ^ (k1 & (S::RB - 1))) + (b ^ ((a ^ (k1 / S::RB)) & (S::B - 1)));
    }
}

// Slot of Z[k] (k < M).
template <int LOGM>
__device__ __forceinline__ int wk_zslot(int q, int k) {
    using S = wk::Shape<LOGM>;
    const int k1 = k & 31, k2 = k >> 5;
    if constexpr (S::A == 1) return wk_slot<LOGM>(q, k1, 0, k2);
    else return wk_slot<LOGM>(q, k1, k2 % S::A, k2 / S::A);
}

// cos(2 pi n / 32), n = 0..8.
constexpr double kCos32[9] = {1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
                              0.70710678118654752440, 0.55557023301960222474, 0.38268343236508977173,
                              0.19509032201612826785, 0.0};
constexpr double cos32(int n) {
    n &= 31;
    if (n > 16) n = 32 - n;
    return n <= 8 ? kCos32[n] : -kCos32[16 - n];
}

// x W32^n, W32 = exp(-2 pi i / 32).  The f32 roundings of these constants all
// shorten them (by up to 2.9e-8), which would show as a common loss of power
// in the summed spectra (8e-8 at M = 1024, in place of the 5.5e-8 that radix-8
// passes have); the larger part of each constant is therefore applied as a
// high and a low part, two more multiply-adds a product (3e-8).
template <int n>
__device__ __forceinline__ float2 mul_w32(float2 x) {
    constexpr int q = n & 31;
    if constexpr (q == 0) return x;
    else if constexpr (q == 8) return make_float2(x.y, -x.x);
    else if constexpr (q == 16) return make_float2(-x.x, -x.y);
    else {
        constexpr double c = cos32(q), s = cos32(q - 8);
        constexpr float ch = (float)c, sh = (float)s;
        // re = x c + y s, im = y c - x s
        if constexpr ((c < 0 ? -c : c) >= (s < 0 ? -s : s)) {
            constexpr float cl = (float)(c - (double)ch);
            return make_float2(fmaf(x.x, ch, fmaf(x.y, sh, x.x * cl)), fmaf(x.y, ch, fmaf(-x.x, sh, x.y * cl)));
        } else {
            constexpr float sl = (float)(s - (double)sh);
            return make_float2(fmaf(x.y, sh, fmaf(x.x, ch, x.y * sl)), fmaf(-x.x, sh, fmaf(x.y, ch, -x.x * sl)));
        }
    }
}

// DFT-8 in place: dft8 with the 1/sqrt2 products folded into the last sums.
__device__ __forceinline__ void wk_dft8(float2 *a) {
    float2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6];
    float2 o0 = a[1], o1 = a[3], o2 = a[5], o3 = a[7];
    dft4(e0, e1, e2, e3);
    dft4(o0, o1, o2, o3);
    constexpr float r = (float)kCos32[4];
    const float2 v1 = make_float2(o1.x + o1.y, o1.y - o1.x);     // W8^1 o1 / r
    const float2 v3 = make_float2(o3.y - o3.x, -o3.x - o3.y);    // W8^3 o3 / r
    a[0] = c_add(e0, o0);
    a[4] = c_sub(e0, o0);
    a[1] = make_float2(fmaf(v1.x, r, e1.x), fmaf(v1.y, r, e1.y));
    a[5] = make_float2(fmaf(-v1.x, r, e1.x), fmaf(-v1.y, r, e1.y));
    a[2] = make_float2(e2.x + o2.y, e2.y - o2.x);
    a[6] = make_float2(e2.x - o2.y, e2.y + o2.x);
    a[3] = make_float2(fmaf(v3.x, r, e3.x), fmaf(v3.y, r, e3.y));
    a[7] = make_float2(fmaf(-v3.x, r, e3.x), fmaf(-v3.y, r, e3.y));
}

// DFT-(4 Q) of a[0 .. 4Q) in place (natural order), Q = 4 or 8, as 4 x Q:
// n = Q p + b, k = c + 4 d.
template <int Q, int B>
__device__ __forceinline__ void dft4q_row(float2 (&u)[4][Q], const float2 *a) {
    float2 y0 = a[B], y1 = a[Q + B], y2 = a[2 * Q + B], y3 = a[3 * Q + B];
    dft4(y0, y1, y2, y3);
    u[0][B] = y0;
    u[1][B] = mul_w32<(8 / Q) * B>(y1);
    u[2][B] = mul_w32<2 * (8 / Q) * B>(y2);
    u[3][B] = mul_w32<3 * (8 / Q) * B>(y3);
}
template <int Q>
__device__ __forceinline__ void dft4q(float2 *a) {
    float2 u[4][Q];
    dft4q_row<Q, 0>(u, a);
    dft4q_row<Q, 1>(u, a);
    dft4q_row<Q, 2>(u, a);
    dft4q_row<Q, 3>(u, a);
    if constexpr (Q == 8) {
        dft4q_row<Q, 4>(u, a);
        dft4q_row<Q, 5>(u, a);
        dft4q_row<Q, 6>(u, a);
        dft4q_row<Q, 7>(u, a);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if constexpr (Q == 8) wk_dft8(u[c]);
        else dft4(u[c][0], u[c][1], u[c][2], u[c][3]);
#pragma unroll
        for (int d = 0; d < Q; ++d) a[c + 4 * d] = u[c][d];
    }
}
template <int R>
__device__ __forceinline__ void wk_dft(float2 *a) {
    if constexpr (R == 4) dft4(a[0], a[1], a[2], a[3]);
    else if constexpr (R == 8) wk_dft8(a);
    else dft4q<R / 4>(a);
}

// ---------------------------------------------------------------- decode
// This wave's packed words of its station's next round: word l + 64 u of the
// SPW station-frames' contiguous run (M <= 2048), or of the whole
// station-frame by the WPS waves that share it; 2 BITS words per lane.
template <int LOGM, int BITS>
__device__ __forceinline__ void wk_load_t(const uint32_t *p, int nvalid, int t, uint32_t (&w)[16]) {
    using S = wk::Shape<LOGM>;
    constexpr int T = 64 * S::WPS;
    const int nw = nvalid * (S::N * BITS / 32);
#pragma unroll
    for (int u = 0; u < 2 * BITS; ++u)
        if (t + T * u < nw) w[u] = __builtin_nontemporal_load(p + t + T * u);
}
template <int LOGM>
__device__ __forceinline__ void wk_load(const uint8_t *src, int nvalid, int bits, int t, uint32_t (&w)[16]) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(src);
    if (bits == 2) wk_load_t<LOGM, 2>(p, nvalid, t, w);
    else if (bits == 1) wk_load_t<LOGM, 1>(p, nvalid, t, w);
    else if (bits == 4) wk_load_t<LOGM, 4>(p, nvalid, t, w);
    else wk_load_t<LOGM, 8>(p, nvalid, t, w);
}

__device__ __forceinline__ uint32_t wk_shuffle(uint32_t v, int kind, const uint32_t *slut) {
    if (kind == SHUF_PAIRSWAP) return ((v & 0xAAAAAAAAu) >> 1) | ((v & 0x55555555u) << 1);
    if (kind == SHUF_GENERIC)
        return slut[v & 255u] | slut[256 + ((v >> 8) & 255u)] | slut[512 + ((v >> 16) & 255u)] |
               slut[768 + (v >> 24)];
    return v;
}

// One word decoded into its 32 / BITS FP16 samples at dst (utils.rs:215-376:
// codes LSB first, levels, odd samples negated for LSB stations: the sign is
// in the table).  Tables: 8 bits, one sample per byte, odd bytes at +256; 4
// bits, two samples per byte; 2 bits, four; 1 bit, four samples per nibble.
template <int BITS>
__device__ __forceinline__ void wk_stage_word(uint32_t v, const uint16_t *dlut, uint32_t *dst) {
    if constexpr (BITS == 2) {
        const uint2 *t = reinterpret_cast<const uint2 *>(dlut);
        const uint2 e0 = t[v & 255u], e1 = t[(v >> 8) & 255u], e2 = t[(v >> 16) & 255u], e3 = t[v >> 24];
        uint4 *d = reinterpret_cast<uint4 *>(dst);
        d[0] = make_uint4(e0.x, e0.y, e1.x, e1.y);
        d[1] = make_uint4(e2.x, e2.y, e3.x, e3.y);
    } else if constexpr (BITS == 1) {
        const uint2 *t = reinterpret_cast<const uint2 *>(dlut);
        uint4 *d = reinterpret_cast<uint4 *>(dst);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint2 e0 = t[(v >> (8 * i)) & 15u], e1 = t[(v >> (8 * i + 4)) & 15u];
            d[i] = make_uint4(e0.x, e0.y, e1.x, e1.y);
        }
    } else if constexpr (BITS == 4) {
        const uint32_t *t = reinterpret_cast<const uint32_t *>(dlut);
        *reinterpret_cast<uint4 *>(dst) =
            make_uint4(t[v & 255u], t[(v >> 8) & 255u], t[(v >> 16) & 255u], t[v >> 24]);
    } else {
        const uint32_t h0 = dlut[v & 255u], h1 = dlut[256 + ((v >> 8) & 255u)],
                       h2 = dlut[(v >> 16) & 255u], h3 = dlut[256 + (v >> 24)];
        *reinterpret_cast<uint2 *>(dst) = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
    }
}

// The staged row of station-frame q of a wave: PAD zeros, N samples, PAD
// zeros as FP16 pairs, at the start of its Z slot, offset and skewed (Shape).
template <int LOGM>
__device__ __forceinline__ uint32_t *wk_row(float2 *z, int q) {
    using S = wk::Shape<LOGM>;
    return reinterpret_cast<uint32_t *>(z + q * S::M) + (S::QO * q) % 64;
}
// Position of dword d of a row (d < M + PAD).
template <int LOGM>
__device__ __forceinline__ int wk_pos(int d) {
    using S = wk::Shape<LOGM>;
    return d + S::SK * (d / S::M2);
}

template <int LOGM, int BITS>
__device__ __forceinline__ void wk_stage_t(const uint32_t (&w)[16], int kind, const uint32_t *slut,
                                           const uint16_t *dlut, float2 *z, int t) {
    using S = wk::Shape<LOGM>;
    constexpr int T = 64 * S::WPS, NWF = S::N * BITS / 32;   // words per station-frame
    static_assert(S::SK == 0 || (S::M2 % (16 / BITS) == 0 && S::PAD / 2 % S::M2 % (16 / BITS) == 0),
                  "a word's samples stay within a skew block");
#pragma unroll
    for (int u = 0; u < 2 * BITS; ++u) {
        const int wi = t + T * u, q = wi / NWF, wf = wi % NWF;
        wk_stage_word<BITS>(wk_shuffle(w[u], kind, slut), dlut,
                            wk_row<LOGM>(z, q) + wk_pos<LOGM>(S::PAD / 2 + (16 / BITS) * wf));
    }
}
template <int LOGM>
__device__ __forceinline__ void wk_stage(const uint32_t (&w)[16], int bits, int kind, const uint32_t *slut,
                                         const uint16_t *dlut, float2 *z, int t) {
    using S = wk::Shape<LOGM>;
    if (bits == 2) wk_stage_t<LOGM, 2>(w, kind, slut, dlut, z, t);
    else if (bits == 1) wk_stage_t<LOGM, 1>(w, kind, slut, dlut, z, t);
    else if (bits == 4) wk_stage_t<LOGM, 4>(w, kind, slut, dlut, z, t);
    else wk_stage_t<LOGM, 8>(w, kind, slut, dlut, z, t);
    // the zero padding: PAD / 2 dwords each side
    constexpr int T = 64 * S::WPS;
    for (int i = t; i < S::SPW * S::PAD; i += T) {
        const int q = i / S::PAD, j = i % S::PAD;
        wk_row<LOGM>(z, q)[wk_pos<LOGM>(j < S::PAD / 2 ? j : S::M + j)] = 0u;
    }
}

// The FP16 pairs (samples 2m - sh and 2m + 1 - sh) of a shifted frame's
// complex elements m = M2 (g + m1(k)) + m2, k = 0..K-1.  Shifts
// within the padding: two dwords and a funnel shift; beyond it: each sample
// checked against the frame.
template <int LOGM, int K, typename M1>
__device__ __forceinline__ void wk_pairs(const uint32_t *row, int m2, int g, int sh, M1 m1, uint32_t (&d)[K]) {
    using S = wk::Shape<LOGM>;
    constexpr int STEP = S::M2 + S::SK;
    if (sh >= -S::PAD && sh <= S::PAD) {
        const int i = S::PAD + 2 * m2 - sh;   // >= 0
        const uint32_t odd = (uint32_t)(i & 1) * 2u;
        const uint32_t *p0 = row + STEP * g + wk_pos<LOGM>(i >> 1);
        const uint32_t *p1 = row + STEP * g + wk_pos<LOGM>((i >> 1) + 1);
#pragma unroll
        for (int k = 0; k < K; ++k) d[k] = __builtin_amdgcn_alignbyte(p1[STEP * m1(k)], p0[STEP * m1(k)], odd);
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = 2 * (S::M2 * (g + m1(k)) + m2) - sh;
            auto sample = [&](int j) -> uint32_t {
                if ((unsigned)j >= (unsigned)S::N) return 0u;
                const int h = S::PAD + j;
                return reinterpret_cast<const uint16_t *>(row + wk_pos<LOGM>(h >> 1))[h & 1];
            };
            d[k] = sample(i) | (sample(i + 1) << 16);
        }
    }
}

__device__ __forceinline__ float2 wk_f32(uint32_t p) {
    typedef _Float16 half2v __attribute__((ext_vector_type(2)));
    const half2v h = __builtin_bit_cast(half2v, p);
    return make_float2((float)h.x, (float)h.y);
}

// tab[i] of a uniform table, addressed by a 32-bit byte offset.
__device__ __forceinline__ float2 wk_at(const float2 *tab, int i) {
    return *reinterpret_cast<const float2 *>(reinterpret_cast<const uint8_t *>(tab) + (uint32_t)i * 8u);
}

// Orders the LDS accesses of the waves that share a station-frame.
template <int LOGM>
__device__ __forceinline__ void wk_sync() {
    if constexpr (wk::Shape<LOGM>::WPS == 1) wave_lds_sync();
    else __syncthreads();
}

// Both FFT stages of this wave's points: staged rows in, Z in place out.
// t: index among the station-frame's 64 WPS lanes; sh: this lane's row's shift
// (MF: of tile row l % 16 per tile, sht).
template <int LOGM, bool MF>
__device__ __forceinline__ void wk_fft(float2 *z, const int *sht, const float2 *tw, const float2 *w2,
                                       const uint4 *b1, int l, int t) {
    using S = wk::Shape<LOGM>;
    constexpr int M = S::M, M2 = S::M2;
    if constexpr (MF) {
        // four 16-row tiles; tile row r of tile tp is row 16 tp + r of the
        // wave's 64: station-frame q, m2
        const int c = l & 15, g = l >> 4;
        const int r0 = t - l;   // first row of this wave (M2 > 64)
        half8 A[4][2];
#pragma unroll
        for (int tp = 0; tp < 4; ++tp) {
            const int row = r0 + 16 * tp + c, q = row / M2, m2 = row % M2;
            uint32_t d[8];
            wk_pairs<LOGM>(wk_row<LOGM>(z, q), m2, g, sht[tp], [](int k) { return 16 * (k >> 2) + 4 * (k & 3); },
                           d);
            A[tp][0] = __builtin_bit_cast(half8, make_uint4(d[0], d[1], d[2], d[3]));
            A[tp][1] = __builtin_bit_cast(half8, make_uint4(d[4], d[5], d[6], d[7]));
        }
        wk_sync<LOGM>();   // every row is read before Y overwrites it
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            half8 b[2][4];   // re / im column tile: hi / lo of both K-steps
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    b[p][e] = __builtin_bit_cast(half8, b1[((4 * (e >> 1) + h + 2 * p) * 2 + (e & 1)) * 64 + l]);
            const int k1 = c + 16 * h;
#pragma unroll
            for (int tp = 0; tp < 4; ++tp) {
                const f4 re = mf_stage1(A[tp][0], A[tp][1], b[0][0], b[0][1], b[0][2], b[0][3]);
                const f4 im = mf_stage1(A[tp][0], A[tp][1], b[1][0], b[1][1], b[1][2], b[1][3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = r0 + 16 * tp + 4 * g + i, q = row / M2, m2 = row % M2;
                    z[q * M + wk_slot<LOGM>(q, k1, m2 / S::B, m2 % S::B)] =
                        c_mul(make_float2(re[i], im[i]), wk_at(tw, m2 * 32 + k1));
                }
            }
        }
    } else {
        const int q = t / M2, m2 = t % M2;   // this lane's row
        uint32_t d[32];
        wk_pairs<LOGM>(wk_row<LOGM>(z, q), m2, 0, sht[0], [](int k) { return k; }, d);
        float2 x[32];
#pragma unroll
        for (int r = 0; r < 32; ++r) x[r] = wk_f32(d[r]);
        wk_sync<LOGM>();
        wk_dft<32>(x);
        float2 *zq = z + q * M;
#pragma unroll
        for (int k1 = 0; k1 < 32; ++k1) {
            if (k1 > 0) x[k1] = c_mul(x[k1], wk_at(tw, k1 * M2 + m2));
            zq[wk_slot<LOGM>(q, k1, m2 / S::B, m2 % S::B)] = x[k1];
        }
    }
    wk_sync<LOGM>();
    if constexpr (S::A == 1) {
        constexpr int CPL = 32 / M2;   // columns per lane
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            const int col = l + 64 * u, k1 = col & 31, q = col >> 5;
            float2 *zq = z + q * M;
            float2 x[M2];
#pragma unroll
            for (int b = 0; b < M2; ++b) x[b] = zq[wk_slot<LOGM>(q, k1, 0, b)];
            wk_dft<M2>(x);
#pragma unroll
            for (int b = 0; b < M2; ++b) zq[wk_slot<LOGM>(q, k1, 0, b)] = x[b];
        }
    } else {
        constexpr int T = 64 * S::WPS, A = S::A, B = S::B;
#pragma unroll
        for (int u = 0; u < 32 / A; ++u) {
            const int id = t + T * u, b = id % B, k1 = id / B;
            float2 x[A];
#pragma unroll
            for (int a = 0; a < A; ++a) x[a] = z[wk_slot<LOGM>(0, k1, a, b)];
            wk_dft<A>(x);
#pragma unroll
            for (int c = 0; c < A; ++c) {
                if (c > 0) x[c] = c_mul(x[c], w2[b * c]);
                z[wk_slot<LOGM>(0, k1, c, b)] = x[c];
            }
        }
        wk_sync<LOGM>();
        constexpr int CL = A < B ? A : B;
#pragma unroll
        for (int u = 0; u < 32 / B; ++u) {
            const int id = t + T * u;
            const int c = (id % CL) + (id / (CL * 32)) * CL, k1 = (id / CL) & 31;
            float2 x[B];
#pragma unroll
            for (int b = 0; b < B; ++b) x[b] = z[wk_slot<LOGM>(0, k1, c, b)];
            wk_dft<B>(x);
#pragma unroll
            for (int d = 0; d < B; ++d) z[wk_slot<LOGM>(0, k1, c, d)] = x[d];
        }
    }
}

// The chosen form's DFT-32 on MFMA: the operand table (scale 1), N >= 1024.
__host__ __device__ inline bool wave_mfma(const SectorArgs &a, int precision) {
    return precision != 0 && a.mf_tab != nullptr && a.N >= 1024;
}

// The frames' parameters, one thread each, ahead of the sector kernel: in it
// the FP64 phases (eight sines and cosines and two arctangents in the plain
// form) would be a serial stretch of a few lanes per workgroup.  k_sector's
// values (make_frame_param), the plain form's f32 start and step as FP64
// angles and log magnitudes, so that a bin's phasor needs one FP64
// multiply-add instead of a product of powers.
__global__ __launch_bounds__(64) void k_wave_params(SectorArgs a, int precision, WkParam *out) {
    const int64_t f = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (f >= a.nf) return;
    const int64_t idx = a.first_frame + f;
    WkParam p;
    const int gs = a.grid == 0 ? a.a1s : a.a2s;
    p.l0 = 1.0;
    p.lam = 0.0;
    FrameDelayDev d;
    compute_frame_delay(idx, a.dly, d, nullptr, nullptr);
    p.s1 = (int16_t)clamp_shift(d.int1, a.N);
    p.s2 = (int16_t)clamp_shift(d.int2, a.N);
    p.frmix = make_float2(1.0f, 0.0f);
    if (precision != 0) {
        double tau1, tau2, tf1, tf2;
        frame_taus(idx, a.dly, tau1, tau2, tf1, tf2);
        const double w1 = a.dly.lo1 == 0.0 ? 0.0 : wrap_turns(-a.dly.lo1 * tf1);
        const double w2 = a.dly.lo2 == 0.0 ? 0.0 : wrap_turns(-a.dly.lo2 * tf2);
        p.dth = -a.df * (d.frac1 - d.frac2);
        p.phw = wrap_turns(w1 - w2 - a.df * (d.frac1 * (double)a.a1s - d.frac2 * (double)a.a2s));
    } else {
        double ang0, angs;
        {
#pragma clang fp contract(off)
            const double two_pi_df = -2.0 * FXC_PI * a.df;   // main.rs:133-149
            const double step1 = two_pi_df * d.frac1, step2 = two_pi_df * d.frac2;
            ang0 = step1 * (double)a.a1s - step2 * (double)a.a2s;
            angs = step1 - step2;
            p.frmix = c_mul(make_float2(d.fr1[0], d.fr1[1]), make_float2(d.fr2[0], -d.fr2[1]));
        }
        const float2 st = polar1_f32((float)ang0), sp = polar1_f32((float)angs);
        const cd s = d_mul(cd{(double)st.x, (double)st.y}, cd{(double)p.frmix.x, (double)p.frmix.y});
        const double inv = 0.5 / FXC_PI;
        p.phw = atan2(s.y, s.x) * inv;
        p.dth = atan2((double)sp.y, (double)sp.x) * inv;
        // |start| |step|^k to first order in ln |.|, for values within 1e-7 of 1
        p.l0 = 0.5 * (s.x * s.x + s.y * s.y + 1.0);
        p.lam = 0.5 * ((double)sp.x * sp.x + (double)sp.y * sp.y - 1.0);
    }
    const double mirror = 2.0 * p.phw + (double)(a.M - 2 * gs) * p.dth;
    if (wave_mfma(a, precision)) {   // taken as f32 (k_sector_wave)
        const float2 C = sincos_turns((float)wrap_turns(mirror));
        p.C = make_double2(C.x, C.y);
    } else {
        const cd C = phasor_turns_f64(mirror);
        p.C = make_double2(C.x, C.y);
    }
    p.F1 = sincos_turns((float)wrap_turns(256.0 * p.dth));
    out[f] = p;
}

// The phased sum's parameters (make_phased_param), and for the chosen form the
// rotations of bin M and of a step of 256 bins.
template <int PREC>
__global__ __launch_bounds__(64) void k_wave_phased_params(SectorArgs a, WkPhased *out) {
    const int64_t f = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (f >= a.nf) return;
    PhasedParam p;
    make_phased_param<PREC>(a.first_frame + f, a, p);
    WkPhased o;
    o.th[0] = p.th1;
    o.th[1] = p.th2;
    o.fr[0] = p.fr1;
    o.fr[1] = p.fr2;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        o.RM[s] = sincos_turns((float)wrap_turns((double)a.M * o.th[s]));
        o.F1[s] = sincos_turns((float)wrap_turns(256.0 * o.th[s]));
    }
    o.s1 = (int16_t)p.s1;
    o.s2 = (int16_t)p.s2;
    o.pad = 0;
    out[f] = o;
}

// X[p] and X[M - p] (times 2) from Z[p], Z[M - p]; w = W_N^p.
__device__ __forceinline__ void wk_untangle(float2 a, float2 b, float2 w, float2 &xp, float2 &xm) {
    const float ex = a.x + b.x, ey = a.y - b.y;
    const float ox = a.x - b.x, oy = a.y + b.y;
    const float tx = w.x * ox - w.y * oy, ty = w.x * oy + w.y * ox;
    xp = make_float2(ex + ty, ey - tx);
    xm = make_float2(ex - ty, -(ey + tx));
}
// X[j] alone (times 2), from Z[j], Z[M - j] and w = W_N^j.
__device__ __forceinline__ float2 wk_untangle1(float2 a, float2 b, float2 w) {
    const float ex = a.x + b.x, ey = a.y - b.y;
    const float ox = a.x - b.x, oy = a.y + b.y;
    return make_float2(ex + (w.x * oy + w.y * ox), ey - (w.x * ox - w.y * oy));
}

// SHIFT: the stations' band starts differ, so the other station's bins of a
// pair are p + sb and M - p + sb, untangled one by one.  PH: the phased sum
// in place of the ACF / XCF products: per bin the stations' rotations (the
// reference's f32 chains, or phasors of the FP64 phases), fringe phasors, the
// weighted sum cb, |cb|^2 and, for the .raw output, cb.  CHAIN: the XCF takes
// its phases from the reference's chains (overlaps above 512 bins, plain form).
template <int LOGM, bool MF, bool SHIFT, bool PH, bool CHAIN>
__global__ __launch_bounds__(wk::Shape<LOGM>::NT)
__attribute__((amdgpu_waves_per_eu(2, 2))) void k_sector_wave(SectorArgs a) {
    using Par = std::conditional_t<PH, WkPhased, WkParam>;
    using S = wk::Shape<LOGM>;
    constexpr int M = S::M, H = M + 1, NT = S::NT, F = S::F, PPT = S::PPT, G = S::G;
    extern __shared__ __align__(16) uint8_t smem[];
    WkShared<LOGM, Par> &sh = *reinterpret_cast<WkShared<LOGM, Par> *>(smem);
    const int tid = threadIdx.x, l = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s = wv / (S::WAVES / 2), ws = wv % (S::WAVES / 2);   // station, wave of the station
    const WkTables tab = wk_tables(a.wk_tab, M);
    for (int i = tid; i < 2 * 4 * 256; i += NT) (&sh.slut[0][0])[i] = tab.slut[i];
    for (int i = tid; i < 2 * kWkDlutHalves / 2; i += NT)
        reinterpret_cast<uint32_t *>(&sh.dlut[0][0])[i] = reinterpret_cast<const uint32_t *>(tab.dlut)[i];
    if constexpr (S::A > 1)
        for (int i = tid; i < S::M2; i += NT) sh.w2[i] = tab.w2[i];

    const bool do_acf = (a.flags & FLAG_ACF) != 0, do_xcf = (a.flags & FLAG_XCF) != 0;
    const int gs = a.grid == 0 ? a.a1s : a.a2s, ge = gs + a.ov;
    const int sb = a.grid == 0 ? a.a2s - a.a1s : a.a1s - a.a2s;   // other station's bin - grid bin
    const int gst = a.grid;                                       // station on the grid

    const int grp = G > 1 ? tid / (M / 2) : 0;
    auto wn = [&](int k) {   // W_N^k, 0 <= k <= M
        const float2 v = a.tw_post[k];
        return make_float2(v.x, -v.y);
    };
    constexpr int NP = PH ? 1 : 4;   // sums per bin
    double acc[PPT][2][NP], mid[NP];
#pragma unroll
    for (int c = 0; c < NP; ++c) mid[c] = 0.0;
#pragma unroll
    for (int j = 0; j < PPT; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int c = 0; c < NP; ++c) acc[j][e][c] = 0.0;

    const int64_t f_begin = (int64_t)blockIdx.x * a.frames_per_wg;
    int64_t f_end = f_begin + a.frames_per_wg;
    if (f_end > a.nf) f_end = a.nf;
    const int bits = a.st[s].bits, kind = a.st[s].shuffle_kind;
    const int64_t bpf = a.st[s].bpf;
    const uint8_t *raw = s ? a.raw2 : a.raw1;
    const int t = S::WPS > 1 ? ws * 64 + l : l;
    const int fw = S::WPS > 1 ? 0 : ws * S::SPW;   // this wave's first frame of a round
    auto nvalid = [&](int64_t fr) {                // valid station-frames of this wave in round fr
        const int64_t n = f_end - fr - fw;
        return (int)(n < 0 ? 0 : (n > S::SPW ? S::SPW : n));
    };
    uint32_t w[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) w[u] = 0u;
    wk_load<LOGM>(raw + (f_begin + fw) * bpf, nvalid(f_begin), bits, t, w);
    __syncthreads();   // the tables are filled by all waves, and read by each on its own from here on
    float2 *zw = &sh.z[s][fw][0];

    const Par *params = reinterpret_cast<const Par *>(a.wk_params);
    for (int64_t fr = f_begin; fr < f_end; fr += F) {
        {
            const int nf = (int)((f_end - fr) < F ? (f_end - fr) : F);   // frames of this iteration
            const int lr = loop_local(l), tr = loop_local(t);   // see loop_local
            int sht[MF ? 4 : 1];
#pragma unroll
            for (int tp = 0; tp < (MF ? 4 : 1); ++tp) {
                int q = fw;
                if constexpr (S::WPS == 1) q += (MF ? 16 * tp + (lr & 15) : lr) / S::M2;
                const Par &P = params[fr + (q < nf ? q : nf - 1)];
                sht[tp] = s ? P.s2 : P.s1;
            }
            // the round's parameters (read after the barrier below)
            {
                constexpr int PW = sizeof(Par) / 4;
                const uint32_t *src = reinterpret_cast<const uint32_t *>(params + fr);
                uint32_t *dst = reinterpret_cast<uint32_t *>(sh.pp);
                for (int i = tid; i < nf * PW; i += NT) dst[i] = src[i];
            }
            wk_stage<LOGM>(w, bits, kind, sh.slut[s], sh.dlut[s], zw, tr);
            if (fr + F < f_end)
                wk_load<LOGM>(raw + (fr + F + fw) * bpf, nvalid(fr + F), bits, tr, w);
            wk_sync<LOGM>();
            wk_fft<LOGM, MF>(zw, sht, tab.tw, sh.w2, reinterpret_cast<const uint4 *>(a.mf_tab), lr, tr);
            // this thread's bin pairs (p, M - p): Z slots of the grid station
            // (both stations without SHIFT) in a wave's first frame, untangle
            // twiddles W_N^p; SHIFT: the other station's slots and twiddles of
            // bins p + sb and M - p + sb (clamped into the band; sums of bins
            // outside the overlap are dropped)
            const int pt = loop_local(G > 1 ? tid % (M / 2) : tid);
            int zp[PPT], zm[PPT];
            float2 wp[PPT];
            int op[SHIFT ? PPT : 1][4];
            float2 ow[SHIFT ? PPT : 1][2];
#pragma unroll
            for (int j = 0; j < PPT; ++j) {
                const int p = pt + NT * j;
                zp[j] = wk_zslot<LOGM>(0, p);
                zm[j] = wk_zslot<LOGM>(0, (M - p) & (M - 1));
                wp[j] = wn(p);
                if constexpr (SHIFT) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        int o = (e ? M - p : p) + sb;
                        o = o < 0 ? 0 : (o > M ? M : o);
                        op[j][2 * e] = wk_zslot<LOGM>(0, o & (M - 1));
                        op[j][2 * e + 1] = wk_zslot<LOGM>(0, (M - o) & (M - 1));
                        ow[j][e] = wn(o);
                    }
                }
            }
            __syncthreads();
            if constexpr (PH) {
                // ---- phased sum of the round's frames (main.rs:2238-2302)
                const float wg = 0.5f * (float)(gst == 0 ? a.w1 : a.w2);   // 1/2: the untangle's factor
                const float wo = 0.5f * (float)(gst == 0 ? a.w2 : a.w1);
                const bool chain = a.chain != nullptr;
                const bool write_cb = (a.flags & FLAG_RAW_OUT) != 0 && a.cb_out != nullptr;
                // cb of grid bin g from both stations' bins X (times 2) and
                // rotations R; the Nyquist bins lose their imaginary part
                // after the rotation (utils.rs:118-123)
                auto combine = [&](int g, float2 Xg, float2 Rg, float2 frg, float2 Xo, float2 Ro, float2 fro) {
                    float2 sg = c_mul(Xg, Rg);
                    if (g == M) sg.y = 0.0f;
                    const float2 cg = c_mul(sg, frg);
                    float2 co = make_float2(0.f, 0.f);
                    if (g >= gs && g < ge) {
                        float2 so = c_mul(Xo, Ro);
                        if (g + sb == M) so.y = 0.0f;
                        co = c_mul(so, fro);
                    }
                    const float2 c1 = gst == 0 ? cg : co, c2 = gst == 0 ? co : cg;
                    const float u1 = gst == 0 ? wg : wo, u2 = gst == 0 ? wo : wg;
                    float2 cb;
                    {
#pragma clang fp contract(off)
                        const float2 a1 = c_scale(c1, u1), a2 = c_scale(c2, u2);
                        cb = make_float2(a1.x + a2.x, a1.y + a2.y);
                    }
                    return cb;
                };
                auto put_cb = [&](int64_t f, int g, float2 cb) {
                    if (g == 0 || g == M) cb.y = 0.0f;   // main.rs:2283-2284
                    a.cb_out[f * (M + 1) + g] = cb;
                };
                auto clampo = [&](int g) { const int o = g + sb; return o < 0 ? 0 : (o > M ? M : o); };
                auto link = [&](int64_t f, int st, int b) {   // station st's chain, all ones without a delay
                    if (st == 1 && a.chains == 1) return make_float2(1.f, 0.f);
                    return chain_at(a, f * a.chains + st, b);
                };
#pragma unroll 1
                for (int f = grp; f < nf; f += G) {
                    const Par &P = sh.pp[f];
                    const float2 *zg = &sh.z[gst][f][0], *zo = &sh.z[gst ^ 1][f][0];
                    const int qx = S::A == 1 ? ((f % S::SPW) & (S::RB - 1)) * S::M2 : 0;
                    const float2 frg = P.fr[gst], fro = P.fr[gst ^ 1];
                    float2 Ug = make_float2(1.f, 0.f), Uo = Ug, Uom = Ug;   // rotations of p, p + sb, M - p + sb
                    if (!chain) {
                        Ug = sincos_turns((float)wrap_turns((double)pt * P.th[gst]));
                        Uo = sincos_turns((float)wrap_turns((double)(pt + sb) * P.th[gst ^ 1]));
                        if constexpr (SHIFT)
                            Uom = sincos_turns((float)wrap_turns((double)(M - pt + sb) * P.th[gst ^ 1]));
                    }
#pragma unroll
                    for (int j = 0; j < PPT; ++j) {
                        const int p = pt + NT * j;
                        float2 gp, gm, xp, xm;   // grid station, other station
                        wk_untangle(zg[zp[j] ^ qx], zg[zm[j] ^ qx], wp[j], gp, gm);
                        if constexpr (SHIFT) {
                            xp = wk_untangle1(zo[op[j][0] ^ qx], zo[op[j][1] ^ qx], ow[j][0]);
                            xm = wk_untangle1(zo[op[j][2] ^ qx], zo[op[j][3] ^ qx], ow[j][1]);
                        } else {
                            wk_untangle(zo[zp[j] ^ qx], zo[zm[j] ^ qx], wp[j], xp, xm);
                        }
                        float2 Rgp, Rgm, Rop, Rom;
                        if (chain) {
                            Rgp = link(fr + f, gst, p);
                            Rgm = link(fr + f, gst, M - p);
                            Rop = link(fr + f, gst ^ 1, clampo(p));
                            Rom = link(fr + f, gst ^ 1, clampo(M - p));
                        } else {
                            Rgp = Ug;
                            Rgm = c_mul(P.RM[gst], c_conj(Ug));
                            Rop = Uo;
                            Rom = SHIFT ? Uom : c_mul(P.RM[gst ^ 1], c_conj(Uo));
                            if (j + 1 < PPT) {
                                Ug = c_mul(Ug, P.F1[gst]);
                                Uo = c_mul(Uo, P.F1[gst ^ 1]);
                                if constexpr (SHIFT) Uom = c_mul(Uom, c_conj(P.F1[gst ^ 1]));
                            }
                        }
                        const float2 cp = combine(p, gp, Rgp, frg, xp, Rop, fro);
                        const float2 cm = combine(M - p, gm, Rgm, frg, xm, Rom, fro);
                        acc[j][0][0] += (double)norm_sqr(cp);
                        acc[j][1][0] += (double)norm_sqr(cm);
                        if (write_cb) {
                            put_cb(fr + f, p, cp);
                            put_cb(fr + f, M - p, cm);
                        }
                    }
                }
                // bin M / 2 pairs with itself; thread f takes frame f's
                if (tid < nf) {
                    const int f = tid, g = M / 2;
                    const Par &P = sh.pp[f];
                    const int qf = S::WPS == 1 ? f % S::SPW : 0;
                    const float2 zg = sh.z[gst][f][wk_zslot<LOGM>(qf, g)];
                    const float2 g2 = make_float2(2.0f * zg.x, -2.0f * zg.y);
                    const int o = clampo(g);
                    const float2 x2 = wk_untangle1(sh.z[gst ^ 1][f][wk_zslot<LOGM>(qf, o & (M - 1))],
                                                   sh.z[gst ^ 1][f][wk_zslot<LOGM>(qf, (M - o) & (M - 1))], wn(o));
                    const float2 Rg = chain ? link(fr + f, gst, g)
                                            : sincos_turns((float)wrap_turns((double)g * P.th[gst]));
                    const float2 Ro = chain ? link(fr + f, gst ^ 1, o)
                                            : sincos_turns((float)wrap_turns((double)o * P.th[gst ^ 1]));
                    const float2 cb = combine(g, g2, Rg, P.fr[gst], x2, Ro, P.fr[gst ^ 1]);
                    mid[0] += (double)norm_sqr(cb);
                    if (write_cb) put_cb(fr + f, g, cb);
                }
            } else {
                // ---- products of the round's frames (main.rs:2491-2568)
                // FP64 phasor u of overlap index k with the f32 step's magnitude, rounded to f32
                auto scaled = [](cd u, const Par &P, int k) {
                    const double l = fma((double)k, P.lam, P.l0);
                    return make_float2((float)(u.x * l), (float)(u.y * l));
                };
                auto phasor = [&](const Par &P, int k) {   // zero outside the overlap, whose sums are dropped
                    if ((unsigned)k >= (unsigned)a.ov) return make_float2(0.f, 0.f);
                    return scaled(phasor_turns_f64(fma((double)k, P.dth, P.phw)), P, k);
                };
    #pragma unroll 1
                for (int f = grp; f < nf; f += G) {
                    const Par &P = sh.pp[f];
                    const float2 *zg = &sh.z[gst][f][0], *zo = &sh.z[gst ^ 1][f][0];
                    // rows of the wave's station-frame q are XORed by q in the
                    // single-pass swizzle
                    const int qx = S::A == 1 ? ((f % S::SPW) & (S::RB - 1)) * S::M2 : 0;
                    // XCF phasors.  MFMA instances (chosen form): f32 from the
                    // reduced FP64 phase on.  The others hold them in FP64 to
                    // the bin, as the plain form's powers of the f32 step are
                    // rounded there: parts within 2^-25, where an f32
                    // polynomial, step and mirror product gave up to 1.8e-7.
                    // 2^27 samples of both stations, plain N = 1024: 386 us
                    // against 377 (FP64 literals in vector registers and the
                    // phasor ahead of the untangle: 404)
                    float2 U = make_float2(1.f, 0.f);
                    if constexpr (MF)
                        if (do_xcf) U = sincos_turns((float)wrap_turns(fma((double)(pt - gs), P.dth, P.phw)));
    #pragma unroll
                    for (int j = 0; j < PPT; ++j) {
                        const int p = pt + NT * j;
                        float2 gp, gm, xp, xm;   // grid station, other station
                        wk_untangle(zg[zp[j] ^ qx], zg[zm[j] ^ qx], wp[j], gp, gm);
                        if constexpr (SHIFT) {
                            xp = wk_untangle1(zo[op[j][0] ^ qx], zo[op[j][1] ^ qx], ow[j][0]);
                            xm = wk_untangle1(zo[op[j][2] ^ qx], zo[op[j][3] ^ qx], ow[j][1]);
                        } else {
                            wk_untangle(zo[zp[j] ^ qx], zo[zm[j] ^ qx], wp[j], xp, xm);
                        }
                        if (do_acf) {
                            acc[j][0][0] += (double)norm_sqr(gp);
                            acc[j][0][1] += (double)norm_sqr(xp);
                            acc[j][1][0] += (double)norm_sqr(gm);
                            acc[j][1][1] += (double)norm_sqr(xm);
                        }
                        if (do_xcf) {
                            float2 Pp, Pm;
                            if constexpr (CHAIN) {
                                const int kp = p - gs, km = M - p - gs;
                                Pp = c_mul(P.frmix, chain_at(a, fr + f, kp < 0 ? 0 : (kp >= a.ov ? a.ov - 1 : kp)));
                                Pm = c_mul(P.frmix, chain_at(a, fr + f, km < 0 ? 0 : (km >= a.ov ? a.ov - 1 : km)));
                            } else if constexpr (MF) {
                                Pp = U;
                                Pm = c_mul(make_float2((float)P.C.x, (float)P.C.y), c_conj(U));
                                if (j + 1 < PPT) U = c_mul(U, P.F1);
                            } else if constexpr (PPT == 1) {
                                const cd Ud = phasor_turns_f64(fma((double)(pt - gs), P.dth, P.phw));
                                const cd Um = d_mul(cd{P.C.x, P.C.y}, cd{Ud.x, -Ud.y});
                                Pp = scaled(Ud, P, p - gs);
                                Pm = scaled(Um, P, M - p - gs);
                            } else {   // overlaps of at most 512 bins: each bin's own
                                Pp = phasor(P, p - gs);
                                Pm = phasor(P, M - p - gs);
                            }
                            // station 1 times conj(station 2)
                            const float2 vp = c_mul(gst == 0 ? c_mul(gp, c_conj(xp)) : c_mul(xp, c_conj(gp)), Pp);
                            const float2 vm = c_mul(gst == 0 ? c_mul(gm, c_conj(xm)) : c_mul(xm, c_conj(gm)), Pm);
                            acc[j][0][2] += (double)vp.x;
                            acc[j][0][3] += (double)vp.y;
                            acc[j][1][2] += (double)vm.x;
                            acc[j][1][3] += (double)vm.y;
                        }
                    }
                }
                // bin M / 2 pairs with itself; thread f takes frame f's
                if (tid < nf) {
                    const int f = tid;
                    const Par &P = sh.pp[f];
                    const int qf = S::WPS == 1 ? f % S::SPW : 0;
                    const float2 zg = sh.z[gst][f][wk_zslot<LOGM>(qf, M / 2)];
                    const float2 g2 = make_float2(2.0f * zg.x, -2.0f * zg.y);
                    int o = M / 2 + (SHIFT ? sb : 0);
                    o = o < 0 ? 0 : (o > M ? M : o);
                    const float2 x2 = wk_untangle1(sh.z[gst ^ 1][f][wk_zslot<LOGM>(qf, o & (M - 1))],
                                                   sh.z[gst ^ 1][f][wk_zslot<LOGM>(qf, (M - o) & (M - 1))], wn(o));
                    if (do_acf) {
                        mid[0] += (double)norm_sqr(g2);
                        mid[1] += (double)norm_sqr(x2);
                    }
                    const int k = M / 2 - gs;
                    if (do_xcf && k >= 0 && k < a.ov) {
                        float2 ph;
                        if constexpr (CHAIN) ph = c_mul(P.frmix, chain_at(a, fr + f, k));
                        else if constexpr (MF) ph = sincos_turns((float)wrap_turns(fma((double)k, P.dth, P.phw)));
                        else ph = phasor(P, k);
                        const float2 v = c_mul(gst == 0 ? c_mul(g2, c_conj(x2)) : c_mul(x2, c_conj(g2)), ph);
                        mid[2] += (double)v.x;
                        mid[3] += (double)v.y;
                    }
                }
            }
            __syncthreads();
        }
    }

    // ---- workgroup partial: thread groups added in order, bins outside the
    // overlap dropped, the untangle's factor 2 (4 in the products) taken out
    const bool ov_only = (a.flags & FLAG_ACF_OVERLAP) != 0;
    double *out = a.part + (size_t)blockIdx.x * kNumProducts * H;
    auto put = [&](int c, int g, double v) {   // c 0 / 1: grid / other station's ACF; 2 / 3: XCF
        int prod = P_PH;
        if constexpr (!PH) {
            const bool in_ov = g >= gs && g < ge;
            v = in_ov || (c == 0 && !ov_only) ? 0.25 * v : 0.0;
            prod = c >= 2 ? P_12R + (c - 2) : ((c == 0) == (gst == 0) ? P_11 : P_22);
        }
        double *o = out + prod * H + g;
        *o = a.accumulate ? *o + v : v;
    };
    double *red = reinterpret_cast<double *>(&sh.z[0][0][0]);   // [F][NP] mids, then G > 1: [G - 1][NP][M + 2]
    if (tid < F)
#pragma unroll
        for (int c = 0; c < NP; ++c) red[tid * NP + c] = mid[c];
    if constexpr (G > 1) {
        static_assert(PPT == 1 && (NP * F + (G - 1) * NP * (M + 2)) * 8 <= (int)sizeof(sh.z), "group sums");
        double *gr = red + NP * F;
        const int p = tid % (M / 2);
        if (grp > 0)
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                gr[((grp - 1) * NP + c) * (M + 2) + p] = acc[0][0][c];
                gr[((grp - 1) * NP + c) * (M + 2) + M - p] = acc[0][1][c];
            }
        __syncthreads();
        if (grp == 0)
#pragma unroll
            for (int c = 0; c < NP; ++c)
                for (int k = 0; k < G - 1; ++k) {
                    acc[0][0][c] += gr[(k * NP + c) * (M + 2) + p];
                    acc[0][1][c] += gr[(k * NP + c) * (M + 2) + M - p];
                }
    } else {
        __syncthreads();
    }
    if (grp == 0) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            const int p = (G > 1 ? tid % (M / 2) : tid) + NT * j;
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                put(c, p, acc[j][0][c]);
                put(c, M - p, acc[j][1][c]);
            }
        }
    }
    if (tid < NP) {
        double v = 0.0;
        for (int f = 0; f < F; ++f) v += red[f * NP + tid];
        put(tid, M / 2, v);
    }
}

template <int LOGM, bool MF, bool PH, bool CHAIN = false>
static hipError_t launch_wave_t(const SectorArgs &a, int n_wg, hipStream_t s) {
    constexpr size_t lds = sizeof(WkShared<LOGM, std::conditional_t<PH, WkPhased, WkParam>>);
    static_assert(2 * lds <= 160 * 1024 && wk::Shape<LOGM>::NT == 256, "two workgroups per CU");
    const dim3 grid(n_wg), block(wk::Shape<LOGM>::NT);
    if (a.a1s == a.a2s) hipLaunchKernelGGL((k_sector_wave<LOGM, MF, false, PH, CHAIN>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((k_sector_wave<LOGM, MF, true, PH, CHAIN>), grid, block, lds, s, a);
    return hipGetLastError();
}

hipError_t launch_wave_params(const SectorArgs &a, int precision, WkParam *out, hipStream_t s) {
    if (a.nf <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_wave_params, dim3((unsigned)((a.nf + 63) / 64)), dim3(64), 0, s, a, precision, out);
    return hipGetLastError();
}

hipError_t launch_wave_phased_params(const SectorArgs &a, int precision, WkPhased *out, hipStream_t s) {
    if (a.nf <= 0) return hipSuccess;
    const dim3 grid((unsigned)((a.nf + 63) / 64));
    if (precision == 0) hipLaunchKernelGGL(k_wave_phased_params<0>, grid, dim3(64), 0, s, a, out);
    else hipLaunchKernelGGL(k_wave_phased_params<1>, grid, dim3(64), 0, s, a, out);
    return hipGetLastError();
}

template <bool PH>
static hipError_t launch_wave_n(const SectorArgs &a, int precision, int n_wg, hipStream_t s) {
    if (a.wk_tab == nullptr || a.wk_params == nullptr || a.frames_per_wg % wave_frames(a.N) != 0)
        return hipErrorInvalidValue;
    const bool mf = wave_mfma(a, precision);
    const bool chain = !PH && a.chain != nullptr;            // the phased sum's instances hold both
    if (chain && (mf || a.N < 2048)) return hipErrorInvalidValue;   // at most 512 bins
    switch (a.N) {
    case 256: return launch_wave_t<7, false, PH>(a, n_wg, s);
    case 512: return launch_wave_t<8, false, PH>(a, n_wg, s);
    case 1024: return mf ? launch_wave_t<9, true, PH>(a, n_wg, s) : launch_wave_t<9, false, PH>(a, n_wg, s);
    case 2048: return mf ? launch_wave_t<10, true, PH>(a, n_wg, s)
                    : chain ? launch_wave_t<10, false, PH, !PH>(a, n_wg, s) : launch_wave_t<10, false, PH>(a, n_wg, s);
    case 4096: return mf ? launch_wave_t<11, true, PH>(a, n_wg, s)
                    : chain ? launch_wave_t<11, false, PH, !PH>(a, n_wg, s) : launch_wave_t<11, false, PH>(a, n_wg, s);
    case 8192: return mf ? launch_wave_t<12, true, PH>(a, n_wg, s)
                    : chain ? launch_wave_t<12, false, PH, !PH>(a, n_wg, s) : launch_wave_t<12, false, PH>(a, n_wg, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_sector_wave(const SectorArgs &a, int precision, int n_wg, hipStream_t s) {
    return launch_wave_n<false>(a, precision, n_wg, s);
}
hipError_t launch_phased_wave(const SectorArgs &a, int precision, int n_wg, hipStream_t s) {
    return launch_wave_n<true>(a, precision, n_wg, s);
}

}  // namespace fxc
