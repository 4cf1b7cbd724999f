// FX path for FFT lengths beyond one workgroup's LDS (N = 32768, 65536:
// M = N/2 complex points = 128/256 KB of FP32 per station-frame).  Frames
// are processed in chunks through HBM scratch:
//
//   1. k_frame_params   per-frame delay entries (main.rs:184-241) and the
//                       XCF phase start/step (main.rs:133-149)
//   2. k_decode_frames  decode + integer shift to FP32 (the bit-exact decode)
//   3. k_fft_pass       four-step FFT, m = M2 m1 + m2, k = k1 + M1 k2:
//                       column DFTs over m1 (length M1) times W_M^{m2 k1},
//                       then row DFTs over m2 (length M2) into Z in natural
//                       order; each pass is a batch of LDS Stockham FFTs
//   4. k_mac_large      realfft untangle and ACF/XCF products, one output
//                       bin per thread looping over a group of frames, FP64
//                       accumulators (any band shift)
//
// Where both stations' bins share the four-step's rows, the fused four-step
// (also N = 16384): the plain form's first pass with the decode in it
// (k_large_pass1_f32; the chosen form's is in fxc_mfma.hip) and the second
// passes with the untangle and the products or the phased bin in them.
#include "fxc_dev.h"

namespace fxc {

// ---------------------------------------------------------------- params
template <int PREC>
__global__ void k_frame_params(SectorArgs a, int logm, FrameParam *params, int64_t *shifts) {
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= a.nf) return;
    FrameParam p;
    make_frame_param<PREC>(a.first_frame + f, a, logm, p);
    params[f] = p;
    shifts[2 * f] = p.s1;
    shifts[2 * f + 1] = p.s2;
}

hipError_t launch_frame_params(const SectorArgs &a, int precision, FrameParam *params,
                               int64_t *shifts, hipStream_t s) {
    if (a.nf <= 0) return hipSuccess;
    const int logm = __builtin_ctz((unsigned)a.M) + 1;
    const dim3 grid((unsigned)((a.nf + 127) / 128));
    if (precision == 0)
        hipLaunchKernelGGL(k_frame_params<0>, grid, dim3(128), 0, s, a, logm, params, shifts);
    else
        hipLaunchKernelGGL(k_frame_params<1>, grid, dim3(128), 0, s, a, logm, params, shifts);
    return hipGetLastError();
}

// ------------------------------------------------------- four-step passes
// A batch of CB independent L-point FFTs (L = E*T), column c of the batch
// at in[c*ics + m*ims] (m < L), result k written to out[c*ocs + k*oks],
// multiplied by W_M^{(c0 + c) k} when `twiddle` (tw_m = W_M^j, j < M).
// Loads and stores walk the unit-stride index across the threads.
// ROWS (the inverse of spectra kept as four-step rows): in holds per frame
// the M1 = cols rows X[k1][k2] of bin k1 + M1 k2 and then bin M; element
// (column k1, k2) is conj(Z'[k1 + M1 k2]) of the half-length inverse,
// irfft_pre_elem's arithmetic formed on the way in (bins k and M - k are in
// rows k1 and M1 - k1, row 0 its own mirror).
template <bool ROWS>
__device__ __forceinline__ float2 pass_input(const float2 *src, int64_t c, int64_t m, int64_t ics, int64_t ims,
                                             int64_t cols, int L, const float2 *tw_post) {
    if constexpr (!ROWS) return src[c * ics + m * ims];
    const int M1 = (int)cols, M = M1 * L, k1 = (int)c, k2 = (int)m;
    float2 z;
    if (k1 == 0 && k2 == 0) {
        z = make_float2(src[0].x + src[M].x, src[0].x - src[M].x);
    } else {
        const int km = k1 == 0 ? L - k2 : L - 1 - k2, rm = k1 == 0 ? 0 : M1 - k1;
        z = irfft_pre_pair(src[k1 * L + k2], src[rm * L + km], tw_post[k1 + M1 * k2]);
    }
    return c_conj(z);
}

template <int E, int T, int CB, bool ROWS>
__global__ __launch_bounds__(CB *T) void k_fft_pass(const float2 *in, float2 *out, int64_t nbatch,
                                                    int64_t cols, int64_t ics, int64_t ims,
                                                    int64_t ocs, int64_t oks, int64_t frame_in,
                                                    int64_t frame_out, const float2 *tw_l,
                                                    const float2 *tw_m, int M, int twiddle,
                                                    const float2 *tw_post) {
    constexpr int L = E * T;
    constexpr int LP = L + L / 16 + 2;
    __shared__ float2 buf[CB][LP];
    const int tid = threadIdx.x;
    const int64_t blocks_per_frame = cols / CB;
    const int64_t f = blockIdx.x / blocks_per_frame;
    const int64_t c0 = (blockIdx.x % blocks_per_frame) * CB;
    if (f >= nbatch) return;
    const float2 *src = in + f * frame_in;
    float2 *dst = out + f * frame_out;
    // load: unit stride along c (ics == 1) or along m (ims == 1)
    for (int i = tid; i < CB * L; i += CB * T) {
        int c, m;
        // (rows of a spectrum: along c, where the W_N^{-k} table is contiguous)
        if (ics == 1 || ROWS) { c = i % CB; m = i / CB; }
        else { m = i % L; c = i / L; }
        buf[c][pad(m)] = pass_input<ROWS>(src, c0 + c, m, ics, ims, cols, L, tw_post);
    }
    __syncthreads();
    const int c = tid / T, t = tid % T;
    float2 v[E];
#pragma unroll
    for (int r = 0; r < E; ++r) v[r] = buf[c][pad(t + T * r)];
    __syncthreads();
    fft_forward<E, T>(buf[c], v, tw_l, t);
    for (int i = tid; i < CB * L; i += CB * T) {
        int cc, k;
        if (ocs == 1) { cc = i % CB; k = i / CB; }
        else { k = i % L; cc = i / L; }
        float2 y = buf[cc][pad(k)];
        if (twiddle) y = c_mul(y, tw_m[((c0 + cc) * (int64_t)k) % M]);
        dst[(c0 + cc) * ocs + (int64_t)k * oks] = y;
    }
}

template <int E, int T>
static hipError_t launch_pass_t(const float2 *in, float2 *out, int64_t nbatch, int64_t cols,
                                int64_t ics, int64_t ims, int64_t ocs, int64_t oks,
                                int64_t frame_in, int64_t frame_out, const float2 *tw_l,
                                const float2 *tw_m, int M, int twiddle, hipStream_t s,
                                const float2 *rows_tw_post) {
    constexpr int CB = 16;
    if (cols % CB != 0) return hipErrorInvalidValue;
    const int64_t grid = nbatch * (cols / CB);
    auto kern = rows_tw_post ? k_fft_pass<E, T, CB, true> : k_fft_pass<E, T, CB, false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(CB * T), 0, s, in, out, nbatch, cols, ics, ims,
                       ocs, oks, frame_in, frame_out, tw_l, tw_m, M, twiddle, rows_tw_post);
    return hipGetLastError();
}

static hipError_t launch_pass(int L, const float2 *in, float2 *out, int64_t nbatch, int64_t cols,
                              int64_t ics, int64_t ims, int64_t ocs, int64_t oks,
                              int64_t frame_in, int64_t frame_out, const float2 *tw_l,
                              const float2 *tw_m, int M, int twiddle, hipStream_t s,
                              const float2 *rows_tw_post = nullptr) {
    switch (L) {
    case 128: return launch_pass_t<4, 32>(in, out, nbatch, cols, ics, ims, ocs, oks, frame_in,
                                          frame_out, tw_l, tw_m, M, twiddle, s, rows_tw_post);
    case 256: return launch_pass_t<8, 32>(in, out, nbatch, cols, ics, ims, ocs, oks, frame_in,
                                          frame_out, tw_l, tw_m, M, twiddle, s, rows_tw_post);
    default: return hipErrorInvalidValue;
    }
}

// Z (natural order, M complex per station-frame) of nframes frames from the
// decoded samples x (N floats per frame): x read as z[m] = x[2m] + i x[2m+1].
// With mf_b1 the first pass's DFT-32 runs on FP16 MFMA (fxc_mfma.hip).
hipError_t launch_fft_large(const void *x, bool x_fp16, float2 *ybuf, float2 *z, int64_t nframes,
                            int M1, int M2, const float2 *tw1, const float2 *tw2,
                            const float2 *twm, const void *mf_b1, hipStream_t s) {
    const int M = M1 * M2;
    if (x_fp16 && !mf_b1) return hipErrorInvalidValue;   // FP16 input feeds the MFMA pass only
    const float2 *zin = reinterpret_cast<const float2 *>(x);
    // columns c = m2 (M2 of them): input z[m2 + M2 m1], output Y[k1][m2] * W_M^{m2 k1}
    hipError_t e = mf_b1 ? launch_fft_pass1_mfma(x, x_fp16, ybuf, nframes, M1, M2, mf_b1, twm, s)
                         : launch_pass(M1, zin, ybuf, nframes, M2, 1, M2, 1, M2, M, M, tw1, twm, M, 1, s);
    if (e != hipSuccess) return e;
    // rows c = k1 (M1 of them): input Y[k1][m2], output Z[k1 + M1 k2]
    return launch_pass(M2, ybuf, z, nframes, M1, M2, 1, 1, M1, M, M, tw2, twm, M, 0, s);
}

size_t frame_param_bytes() { return sizeof(FrameParam); }

__global__ void k_untangle_large(const float2 *z, int64_t nframes, int M, const float2 *tw_post,
                                 float2 *out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t f = i / (M + 1);
    const int k = (int)(i % (M + 1));
    if (f >= nframes) return;
    out[i] = untangle_np(z + f * M, k, M, tw_post);
}

hipError_t launch_untangle_large(const float2 *z, int64_t nframes, int M, const float2 *tw_post,
                                 float2 *out, hipStream_t s) {
    const int64_t n = nframes * (M + 1);
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_untangle_large, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, z,
                       nframes, M, tw_post, out);
    return hipGetLastError();
}

// ------------------------------------------------ inverse real FFT, N >= 32768
// inverse_c2r_process (utils.rs:60-66) through the HBM four-step: conj(Z')
// of each frame's half spectrum, a forward FFT, then the real samples
// interleaved and scaled 1/N (odd samples negated once more for an LSB
// output stream, main.rs:2290-2292), as k_irfft_frames does in LDS.
__global__ void k_irfft_prepare_large(const float2 *X, int64_t nframes, int M, const float2 *tw_post,
                                      float2 *zc) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t f = i / M;
    const int k = (int)(i - f * M);
    if (f >= nframes) return;
    zc[i] = irfft_pre_elem(X + f * (M + 1), k, M, tw_post);
}

__global__ void k_irfft_finish_large(const float2 *z, int64_t nframes, int M, int negate_odd,
                                     float *out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nframes * M) return;
    const float scale = 1.0f / (float)(2 * M);
    const float odd_sign = negate_odd ? 1.0f : -1.0f;
    const float2 v = z[i];
    out[2 * i] = v.x * scale;
    out[2 * i + 1] = odd_sign * (v.y * scale);
}

hipError_t launch_irfft_large(const float2 *X, int64_t nframes, int M1, int M2, const float2 *tw1,
                              const float2 *tw2, const float2 *twm, const float2 *tw_post,
                              float2 *zc, float2 *ybuf, float2 *z, bool negate_odd, float *out,
                              const SectorArgs *q, uint8_t *q_out, hipStream_t s) {
    const int M = M1 * M2;
    const int64_t n = nframes * M;
    if (n <= 0) return hipSuccess;
    const dim3 grid((unsigned)((n + 255) / 256));
    hipLaunchKernelGGL(k_irfft_prepare_large, grid, dim3(256), 0, s, X, nframes, M, tw_post, zc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (q != nullptr) {   // rows c = k1: result n1 = k2 of row k1 is element k1 + M1 k2 of the series
        e = launch_pass(M1, zc, ybuf, nframes, M2, 1, M2, 1, M2, M, M, tw1, twm, M, 1, s);
        return e != hipSuccess ? e : launch_fft_cols_quantise(*q, ybuf, nframes, M1, M2, M2, 1, tw2, q_out, negate_odd, s);
    }
    e = launch_fft_large(zc, false, ybuf, z, nframes, M1, M2, tw1, tw2, twm, nullptr, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_irfft_finish_large, grid, dim3(256), 0, s, z, nframes, M, negate_odd ? 1 : 0,
                       out);
    return hipGetLastError();
}

// The same transform of spectra kept as the four-step's rows (M1 rows of M2
// bins, then bin M, per frame), quantised: y[k1 + M1 k2] = conj(Z'[k1 + M1
// k2]) is row k1's entry k2, so the first pass is the rows' DFT-M2 over k2
// (formed on the way in, no pass of its own) times W_M^{n2 k1}, the second
// the columns' DFT-M1 over k1 into n2 + M2 n1.
hipError_t launch_irfft_rows_quantise(const SectorArgs &a, const float2 *X, int64_t nframes, int M1, int M2,
                                      const float2 *tw1, const float2 *tw2, const float2 *twm, float2 *ybuf,
                                      uint8_t *out, bool negate_odd, hipStream_t s) {
    const int M = M1 * M2;
    if (nframes <= 0) return hipSuccess;
    hipError_t e = launch_pass(M2, X, ybuf, nframes, M1, M2, 1, M2, 1, M + 1, M, tw2, twm, M, 1, s, a.tw_post);
    if (e != hipSuccess) return e;
    return launch_fft_cols_quantise(a, ybuf, nframes, M2, M1, 1, M2, tw1, out, negate_odd, s);
}

// ---------------------------------------------------------- untangle + MAC
// Bin g of the output grid per thread; frames [g0, g1) of the chunk; the
// per-frame phase terms come from k_frame_params.
template <int PREC>
__global__ __launch_bounds__(256) void k_mac_large(SectorArgs a, const float2 *z1, const float2 *z2,
                                                   const FrameParam *params, int64_t fpg,
                                                   int accumulate) {
    const int M = a.M;
    const int half = M + 1;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t f0 = (int64_t)blockIdx.y * fpg;
    int64_t f1 = f0 + fpg;
    if (f1 > a.nf) f1 = a.nf;
    if (g >= half) return;
    const bool do_acf = (a.flags & FLAG_ACF) != 0;
    const bool do_xcf = (a.flags & FLAG_XCF) != 0;
    const bool ov_only = (a.flags & FLAG_ACF_OVERLAP) != 0;
    const int gs = (a.grid == 0) ? a.a1s : a.a2s;
    const bool in_ov = g >= gs && g < gs + a.ov;
    const int sb_other = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    const float2 *zg = a.grid == 0 ? z1 : z2;
    const float2 *zo = a.grid == 0 ? z2 : z1;
    const int kk = g - gs;   // overlap index (XCF phase exponent)
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t f = f0; f < f1; ++f) {
        const float2 Xg = untangle_np(zg + f * M, g, M, a.tw_post);
        float2 Xo = make_float2(0.0f, 0.0f);
        if (in_ov) Xo = untangle_np(zo + f * M, g + sb_other, M, a.tw_post);
        if (do_acf) {
            const float pgrid = (!ov_only || in_ov) ? norm_sqr(Xg) : 0.0f;
            const float poth = in_ov ? norm_sqr(Xo) : 0.0f;
            acc[0] += (double)(a.grid == 0 ? pgrid : poth);
            acc[1] += (double)(a.grid == 0 ? poth : pgrid);
        }
        if (in_ov && do_xcf) {
            const FrameParam &P = params[f];
            float2 phf;
            if (PREC == 0 && a.chain != nullptr) {
                phf = chain_at(a, f, kk);   // the reference's own chain
            } else if (PREC != 0) {
                // chosen form: the FP64 phase in turns, reduced mod 1, then the f32 sincos
                const float r = (float)wrap_turns(fma((double)kk, P.dth, P.phw));
                phf = make_float2(__builtin_amdgcn_cosf(r), __builtin_amdgcn_sinf(r));
            } else {
                cd ph = P.start;
                for (int b = 0; b < kMaxPow; ++b)
                    if ((kk >> b) & 1) ph = d_mul(ph, P.pw[b]);
                phf = make_float2((float)ph.x, (float)ph.y);
            }
            const float2 X1 = (a.grid == 0) ? Xg : Xo;
            const float2 X2 = (a.grid == 0) ? Xo : Xg;
            float2 v2 = c_mul(X1, c_conj(X2));
            if (PREC == 0) v2 = c_mul(v2, P.frmix);
            v2 = c_mul(v2, phf);
            acc[2] += (double)v2.x;
            acc[3] += (double)v2.y;
        }
    }
    double *out = a.part + (size_t)blockIdx.y * kNumProducts * half;
    const double prev[4] = {accumulate ? out[P_11 * half + g] : 0.0,
                            accumulate ? out[P_22 * half + g] : 0.0,
                            accumulate ? out[P_12R * half + g] : 0.0,
                            accumulate ? out[P_12I * half + g] : 0.0};
    out[P_11 * half + g] = prev[0] + acc[0];
    out[P_22 * half + g] = prev[1] + acc[1];
    out[P_12R * half + g] = prev[2] + acc[2];
    out[P_12I * half + g] = prev[3] + acc[3];
}

// ------------------------------------ FP32 first pass fused with the decode
// The plain form's first pass of the fused four-step (M1 = 128): workgroup
// (frame, part p) takes the columns m2 in [64 p, 64 p + 64) of all 128 rows
// m1 (element m = m2 + M2 m1).  The rows' packed words are staged in LDS as
// k_large_pass1_fused does; thread (column n, j) decodes inputs m1 = j + 8 r,
// takes the DFT-16 over r (index e) times W_128^{j e}, and after an LDS
// transpose (over the words) the DFT-8 over j for e = 2 j and 2 j + 1, giving
// k1 = e + 16 b; the output twiddle W_M^{m2 k1} comes from a table in store
// order.  Against the decode kernel and the LDS Stockham pass it replaces
// (FP32 samples to memory and back, then the columns), 2^27 samples of both
// stations at N = 32768: 311 + 690 us to 424.
template <int BITS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_large_pass1_f32(
    SectorArgs a, int station, const int64_t *shifts, float2 *out, int M2, int parts,
    const float2 *tw_m, const float2 *tw_y) {
    __shared__ float2 zb[128 * 64];
    __shared__ float2 w128[128];
    __shared__ float lev[256];
    uint32_t *words = reinterpret_cast<uint32_t *>(zb);   // 128 rows x K words, one zero word after them
    const StationDev &st = a.st[station];
    const int bits = BITS ? BITS : st.bits;
    const int K = 4 * bits + 1, rw = M2 * bits / 16;      // 128 K + 1 <= 8321 words (16 bits)
    const int M = a.M;
    const int tid = threadIdx.x;
    const int n = tid & 63;
    const int jw = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a contiguous run of (frame, part) per XCD, as k_large_pass1_fused
    const int nb = (int)gridDim.x, xcd = (int)blockIdx.x & 7, kb = (int)blockIdx.x >> 3;
    const int lb = xcd * (nb >> 3) + min(xcd, nb & 7) + kb;
    const int64_t f = lb / parts;
    const int part = lb % parts;
    if (f >= a.nf) return;   // uniform per workgroup
    if (tid < 128) w128[tid] = tw_m[tid * M2];
    if (st.bits >= 2 && st.bits <= 8 && tid >= 256)
        lev[tid - 256] = (tid - 256 <= (int)st.code_mask) ? st.levels[tid - 256] : 0.0f;
    const int sh = clamp_shift(shifts[f * 2 + station], a.N);
    const int base0 = ((128 * part - sh) * bits) >> 5;   // arithmetic shift: floor
    {
        const uint8_t *frame = (station == 0 ? a.raw1 : a.raw2) + f * st.bpf;
        const int nst = 128 * K;
        for (int i0 = 0; i0 < nst; i0 += 512 * 4) {   // four loads in flight per thread
            uint32_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int idx = i0 + tid + 512 * u;
                const int m1 = idx / K;
                v[u] = idx < nst ? frame_word(frame, st, m1 * rw + base0 + (idx - m1 * K)) : 0u;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int idx = i0 + tid + 512 * u;
                if (idx < nst) words[idx] = v[u];
            }
        }
        if (tid == 0) words[nst] = 0u;
    }
    __syncthreads();
    // LSB flip (odd samples of the unshifted frame): sample 2m - sh is odd iff sh is
    const uint32_t fm0 = (st.lsb && (sh & 1)) ? 0x80000000u : 0u;
    const uint32_t fm1 = (st.lsb && !(sh & 1)) ? 0x80000000u : 0u;
    const int m2 = 64 * part + n;
    float2 v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m1 = jw + 8 * r;
        const int src0 = 2 * (m2 + M2 * m1) - sh;
        const int bp = src0 * bits;
        v[r] = decode_pair_local<BITS>(words, st, lev, src0, (bp >> 5) - base0 + m1 * (K - rw),
                                       (uint32_t)bp & 31u, a.N, fm0, fm1);
    }
    dft16(v);
#pragma unroll
    for (int e = 1; e < 16; ++e) v[e] = c_mul(v[e], w128[jw * e]);
    float2 ty[2][8];   // output twiddles, loaded across the barriers
    const float2 *ty0 = tw_y + m2;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int b = 0; b < 8; ++b) ty[h][b] = ty0[(2 * jw + h + 16 * b) * M2];
    __syncthreads();   // every thread is done with the words
#pragma unroll
    for (int e = 0; e < 16; ++e) zb[(e * 8 + jw) * 64 + n] = v[e];
    __syncthreads();
    float2 *dst = out + f * (int64_t)M + m2;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = 2 * jw + h;
        float2 u[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) u[q] = zb[(e * 8 + q) * 64 + n];
        dftR<8>(u);
#pragma unroll
        for (int b = 0; b < 8; ++b) dst[(e + 16 * b) * M2] = c_mul(u[b], ty[h][b]);
    }
}

hipError_t launch_large_pass1_f32(const SectorArgs &a, const int64_t *shifts, float2 *out0, float2 *out1,
                                  int M1, int M2, const float2 *tw_m, const float2 *tw_y, hipStream_t s) {
    if (tw_y == nullptr || M1 != 128 || (M2 != 64 && M2 != 128 && M2 != 256) || M1 * M2 != a.M)
        return hipErrorInvalidValue;
    if (a.nf <= 0) return hipSuccess;
    const int parts = M2 / 64;
    for (int st = 0; st < 2; ++st) {
        const int bits = a.st[st].bits;
        if (bits < 1 || bits > 16) return hipErrorInvalidValue;
        auto kern = bits == 1   ? k_large_pass1_f32<1>
                    : bits == 2 ? k_large_pass1_f32<2>
                    : bits == 4 ? k_large_pass1_f32<4>
                    : bits == 8 ? k_large_pass1_f32<8>
                                : k_large_pass1_f32<0>;
        hipLaunchKernelGGL(kern, dim3((unsigned)(a.nf * parts)), dim3(512), 0, s, a, st, shifts,
                           st == 0 ? out0 : out1, M2, parts, tw_m, tw_y);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ------------------------------------ second pass fused with the products
// Both stations' bins on the same rows of the four-step (the band shift a
// multiple of M1).  Z[k1 + M1 k2] is row k1's DFT over m2 of
// Y[k1][m2], and bin M - k lies in row M1 - k1 (row 0 and row M1/2 are their
// own mirrors), so the untangle of a bin needs only its row pair.
// Workgroup (pair p, frame group): rows ra = p, rb = M1 - p (p = 0: rows 0
// and M1/2) of both stations; the pair's post twiddles W_N^{-g} are staged
// in LDS once.  The four rows of a frame are transformed by one wave (its
// next frames' rows are loaded into registers meanwhile); after a barrier
// each thread takes bins g = row + M1 k2 of the pair (and bin M in pair 0):
// the split-method untangle of both stations, then the ACF/XCF products with
// the XCF phasor from the frame's FP64 phase (k_mac_large's arithmetic) or
// the phased bin, and FP64 sums.  The frame group's partial slot holds the
// pair's bins contiguously (coalesced stores); the reduce over the slots
// puts them back in bin order.
__device__ __forceinline__ float2 untangle_ab(float2 A, float2 B, int k, int M, float2 w) {
    if (k == 0 || k == M) return make_float2(k == 0 ? A.x + A.y : A.x - A.y, 0.0f);
    const float ex = 0.5f * (A.x + B.x), ey = 0.5f * (A.y - B.y);
    const float dx = 0.5f * (A.x - B.x), dy = 0.5f * (A.y + B.y);
    return make_float2(ex + (w.x * dy - w.y * dx), ey - (w.x * dx + w.y * dy));
}

// What a second pass forms of its bins: the products; the phased power; the
// power and the phased spectra, rows of M2 as they come (a.cb_out, per frame
// M1 rows, then bin M).
enum { P2_PRODUCTS = 0, P2_PHASED = 1, P2_PHASED_CB = 2 };

// A thread's sums into its entry of the partial slot (phased: the power
// alone, the other products are not read)
template <int NA>
__device__ __forceinline__ void store_pair_sums(double *out, int half, int g, const double (&acc)[NA],
                                                int accumulate) {
    if constexpr (NA == 1) {
        out[P_PH * half + g] = accumulate ? out[P_PH * half + g] + acc[0] : acc[0];
    } else {
        const int prod[4] = {P_11, P_22, P_12R, P_12I};
#pragma unroll
        for (int c = 0; c < 4; ++c)
            out[prod[c] * half + g] = (accumulate ? out[prod[c] * half + g] : 0.0) + acc[c];
    }
}

// The plain form's phase chains for the second pass: link kk of the frames
// of the span side by side (a.chain_ld per link), so that a thread, which
// owns a bin and walks the frames, reads its frames' links as one run.  (Rows
// of one frame's links, k_phase_chain's, would have each lane read 4 bytes of
// its own line, M1 links apart, twice a frame.)  M2 = 64 / 128 take them two
// frames at a time, the next two on their way; all eight in registers spill.
__device__ __forceinline__ const float2 *chain_link(const SectorArgs &a, int kk, int64_t f) {
    return reinterpret_cast<const float2 *>(a.chain) + (int64_t)kk * a.chain_ld + f;
}
template <int F>
struct ChainLinks {
    float2 v[F];
    __device__ __forceinline__ void load(const float2 *p) {   // F frames (the row's padding included)
#pragma unroll
        for (int i = 0; i < F; ++i) v[i] = p[i];
    }
    // phased: rotations of station st's bin; a station without a chain
    // (a.chains = 1, the second) is not rotated
    __device__ __forceinline__ void load_rot(const SectorArgs &a, int bin, int st, int64_t f) {
        if (st < a.chains) load(chain_link(a, bin * a.chains + st, f));
        else
#pragma unroll
            for (int i = 0; i < F; ++i) v[i] = make_float2(1.f, 0.f);
    }
};

// One bin of a row pair for the second pass: bin g = row + M1 k2
// of row ra (rb_sel false) or rb, or bin M (nyq: row 0, k2 = M2); the
// untangle of both stations and the ACF/XCF products (k_mac_large's arithmetic).
// PLAIN: the reference's own f32 phase, chv (a link of the frame's chain),
// after the fringe phasor frmix.
template <int M2, int LP, bool PLAIN>
__device__ __forceinline__ void row_bin(const float2 (*zb)[LP], const float2 (*twp)[M2], bool rb_sel,
                                        int k2, bool nyq, int M, int M1, int ra, int rb, int gs, int ov,
                                        int sbo, int jo, int grid, bool do_acf, bool do_xcf,
                                        bool ov_only, double dth, double phw, float2 frmix, float2 chv,
                                        double (&acc)[4]) {
    const int row = nyq ? 0 : (rb_sel ? rb : ra);
    if (nyq) k2 = M2;
    const int g = nyq ? M : row + M1 * k2;
    const int bg = row == ra ? 0 : 1;
    const int bm = (row == 0 ? row : M1 - row) == ra ? 0 : 1;
    const int km = row == 0 ? (M2 - k2) & (M2 - 1) : M2 - 1 - k2;
    const float2 Zg = zb[bg][pad(k2 & (M2 - 1))], Zm = zb[bm][pad(km)];
    const float2 Xg = untangle_ab(Zg, Zm, g, M, twp[bg][k2 & (M2 - 1)]);
    const bool in_ov = g >= gs && g < gs + ov;
    float2 Xo = make_float2(0.0f, 0.0f);
    if (in_ov) {
        const int h = g + sbo, kh = k2 + jo;
        const int khm = row == 0 ? (M2 - kh) & (M2 - 1) : M2 - 1 - kh;
        const float2 Oh = zb[2 + bg][pad(kh & (M2 - 1))];
        const float2 Om = zb[2 + bm][pad(khm & (M2 - 1))];
        Xo = untangle_ab(Oh, Om, h, M, twp[bg][kh & (M2 - 1)]);
    }
    if (do_acf) {
        const float pgrid = (!ov_only || in_ov) ? norm_sqr(Xg) : 0.0f;
        const float poth = in_ov ? norm_sqr(Xo) : 0.0f;
        acc[0] += (double)(grid == 0 ? pgrid : poth);
        acc[1] += (double)(grid == 0 ? poth : pgrid);
    }
    if (in_ov && do_xcf) {
        float2 phf = chv;
        if constexpr (!PLAIN) {
            const float r = (float)wrap_turns(fma((double)(g - gs), dth, phw));
            phf = make_float2(__builtin_amdgcn_cosf(r), __builtin_amdgcn_sinf(r));
        }
        const float2 X1 = (grid == 0) ? Xg : Xo;
        const float2 X2 = (grid == 0) ? Xo : Xg;
        float2 v2 = c_mul(X1, c_conj(X2));
        if constexpr (PLAIN) v2 = c_mul(v2, frmix);
        v2 = c_mul(v2, phf);
        acc[2] += (double)v2.x;
        acc[3] += (double)v2.y;
    }
}

// One bin of a row pair for the phased sum (k_phased_large's per-bin
// arithmetic, main.rs:2264-2302): both stations' untangled bins, each
// rotated by exp(2 pi i b th) from the FP64 phase and by its fringe phasor,
// cb = w1 c1 + w2 c2, |cb|^2 into the FP64 sum.  Returns cb as the inverse
// FFT takes it (DC and Nyquist imaginary parts zeroed).  PLAIN: rotated by
// the reference's own f32 values rg (this bin) and ro (the other station's).
template <int M2, int LP, bool PLAIN>
__device__ __forceinline__ float2 row_bin_ph(const float2 (*zb)[LP], const float2 (*twp)[M2], bool rb_sel,
                                             int k2, bool nyq, int M, int M1, int ra, int rb, int gs,
                                             int ov, int sbo, int jo, int grid, const PhasedParam &P,
                                             float w1, float w2, float2 rg, float2 ro, double &acc) {
    const int row = nyq ? 0 : (rb_sel ? rb : ra);
    if (nyq) k2 = M2;
    const int g = nyq ? M : row + M1 * k2;
    const int bg = row == ra ? 0 : 1;
    const int bm = (row == 0 ? row : M1 - row) == ra ? 0 : 1;
    const int km = row == 0 ? (M2 - k2) & (M2 - 1) : M2 - 1 - k2;
    const float2 Zg = zb[bg][pad(k2 & (M2 - 1))], Zm = zb[bm][pad(km)];
    const float2 Xg = untangle_ab(Zg, Zm, g, M, twp[bg][k2 & (M2 - 1)]);
    const bool in_ov = g >= gs && g < gs + ov;
    const double thg = grid == 0 ? P.th1 : P.th2, tho = grid == 0 ? P.th2 : P.th1;
    const float2 frg = grid == 0 ? P.fr1 : P.fr2, fro = grid == 0 ? P.fr2 : P.fr1;
    float2 sg = c_mul(Xg, PLAIN ? rg : phasor_turns((double)g * thg));
    if (g == M) sg.y = 0.0f;                              // Nyquist (utils.rs:118-123)
    const float2 cg = c_mul(sg, frg);
    float2 co = make_float2(0.0f, 0.0f);
    if (in_ov) {
        const int h = g + sbo, kh = k2 + jo;
        const int khm = row == 0 ? (M2 - kh) & (M2 - 1) : M2 - 1 - kh;
        const float2 Oh = zb[2 + bg][pad(kh & (M2 - 1))];
        const float2 Om = zb[2 + bm][pad(khm & (M2 - 1))];
        float2 so = c_mul(untangle_ab(Oh, Om, h, M, twp[bg][kh & (M2 - 1)]),
                          PLAIN ? ro : phasor_turns((double)h * tho));
        if (h == M) so.y = 0.0f;
        co = c_mul(so, fro);
    }
    const float2 c1 = grid == 0 ? cg : co, c2 = grid == 0 ? co : cg;
    float2 cb;
    {
#pragma clang fp contract(off)
        const float2 a1 = c_scale(c1, w1), a2 = c_scale(c2, w2);
        cb = make_float2(a1.x + a2.x, a1.y + a2.y);
    }
    acc += (double)norm_sqr(cb);
    if (g == 0 || g == M) cb.y = 0.0f;                    // main.rs:2283-2284
    return cb;
}

// Bin M's phased bin (pair 0's first threads), its rotations read here
template <int M2, int LP, bool PLAIN>
__device__ __forceinline__ float2 nyq_bin_ph(const SectorArgs &a, const float2 (*zb)[LP], const float2 (*twp)[M2],
                                             int M1, int ra, int rb, int gs, int sbo, int jo,
                                             const PhasedParam &P, float w1, float w2, int64_t f, double &acc) {
    ChainLinks<1> rg = {}, ro = {};
    if constexpr (PLAIN) {
        rg.load_rot(a, a.M, a.grid, f);
        if (a.M >= gs && a.M < gs + a.ov) ro.load_rot(a, a.M + sbo, 1 - a.grid, f);
    }
    return row_bin_ph<M2, LP, PLAIN>(zb, twp, false, 0, true, a.M, M1, ra, rb, gs, a.ov, sbo, jo, a.grid, P, w1, w2,
                                     rg.v[0], ro.v[0], acc);
}

// The same second pass at M2 = 256 with two radix-16 passes per row: each
// wave transforms one frame's four rows (lane = 16 q + j: row q, butterfly
// j) -- the first pass from registers, its outputs multiplied by the second
// pass's twiddles W_256^{j r} and transposed through LDS, the second pass
// writing X[j + 16 r].  The four waves transform four frames, then after a
// barrier every thread forms two bins of all four, and a second barrier
// frees the rows.  The twiddles are read from LDS, which leaves registers
// (and, with rows of 271 entries, LDS) for four workgroups per CU instead of
// three: 2^27 samples 703 -> 683 us.
template <int MODE, bool PLAIN>
__global__ __launch_bounds__(256, PLAIN ? 3 : 4) void k_large_pass2_r16(SectorArgs a, const float2 *y1,
                                                         const float2 *y2, const void *params, int M1, const float2 *tw_m2, int64_t fpg,
                                                         int accumulate) {
    constexpr int M2 = 256, LP = 271;   // pad(255) + 1
    constexpr int NA = MODE == P2_PRODUCTS ? 4 : 1;
    __shared__ float2 zr[4][4][LP];   // [frame of the iteration = wave][grid ra, grid rb, other ra, other rb]
    __shared__ float2 twp[2][M2];     // tw_post[row + M1 k2], rows ra / rb
    __shared__ float2 twj[16][16];    // W_256^{j r}
    const int M = a.M;
    const int half = M + 1;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int q = lane >> 4, j = lane & 15;
    const int p = blockIdx.x;
    const int ra = p, rb = p == 0 ? M1 / 2 : M1 - p;
    for (int i = tid; i < 2 * M2; i += 256)
        twp[i / M2][i % M2] = a.tw_post[(i < M2 ? ra : rb) + M1 * (i % M2)];
    twj[tid >> 4][tid & 15] = tw_m2[(tid >> 4) * (tid & 15)];
    const int64_t g0 = (int64_t)blockIdx.y * fpg;
    int64_t g1 = g0 + fpg;
    if (g1 > a.nf) g1 = a.nf;
    const bool do_acf = (a.flags & FLAG_ACF) != 0;
    const bool do_xcf = (a.flags & FLAG_XCF) != 0;
    const bool ov_only = (a.flags & FLAG_ACF_OVERLAP) != 0;
    const int gs = (a.grid == 0) ? a.a1s : a.a2s;
    const int sbo = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    const int jo = sbo / M1;
    const float2 *src_row = ((q & 2) ? (a.grid == 0 ? y2 : y1) : (a.grid == 0 ? y1 : y2)) +
                            (int64_t)((q & 1) ? rb : ra) * M2 + j;
    const bool nyq = p == 0 && tid == 0;
    const float w1 = (float)a.w1, w2 = (float)a.w2;   // phased sum
    double acc[3][NA];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int c = 0; c < NA; ++c) acc[i][c] = 0.0;
    float2 cur[16];
    {
        const int64_t f = g0 + w;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            cur[r] = f < g1 ? src_row[f * (int64_t)M + 16 * r] : make_float2(0.f, 0.f);
    }
    bool in_ov[2];   // the thread's bins (rows ra / rb) lie in the overlap
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int kk = (i ? rb : ra) + M1 * tid - gs;
        in_ov[i] = kk >= 0 && kk < a.ov;
    }
    __syncthreads();   // twiddles staged
    float2 *z = zr[w][q];
    for (int64_t it = g0; it < g1; it += 4) {
        const int64_t f = it + w, fn = f + 4;
        float2 nxt[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            nxt[r] = fn < g1 ? src_row[fn * (int64_t)M + 16 * r] : make_float2(0.f, 0.f);
        ChainLinks<PLAIN ? 4 : 1> cg[2] = {}, co[2] = {};
#pragma unroll
        for (int i = 0; PLAIN && i < 2; ++i) {
            const int g = (i ? rb : ra) + M1 * tid;
            if constexpr (MODE == P2_PRODUCTS) {
                if (do_xcf && in_ov[i]) cg[i].load(chain_link(a, g - gs, it));
            } else {
                cg[i].load_rot(a, g, a.grid, it);
                if (in_ov[i]) co[i].load_rot(a, g + sbo, 1 - a.grid, it);
            }
        }
        if (f < g1) {
            dft16(cur);                                  // pass 1: inputs j + 16 r
#pragma unroll
            for (int r = 1; r < 16; ++r) cur[r] = c_mul(cur[r], twj[r][loop_local(j)]);
#pragma unroll
            for (int r = 0; r < 16; ++r) z[pad(16 * j + r)] = cur[r];
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) cur[r] = z[pad(j + 16 * r)];
            dft16(cur);                                  // pass 2
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) z[pad(j + 16 * r)] = cur[r];   // X[j + 16 r]
        }
        __syncthreads();   // the iteration's rows are ready
        const int nfr = (int)((g1 - it) < 4 ? (g1 - it) : 4);
        auto bins = [&](int s2) {
            if constexpr (MODE != P2_PRODUCTS) {
                const PhasedParam P = static_cast<const PhasedParam *>(params)[it + s2];
                float2 *cbo = MODE == P2_PHASED_CB ? a.cb_out + (it + s2) * half : nullptr;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float2 cb = row_bin_ph<M2, LP, PLAIN>(
                        zr[s2], twp, i == 1, tid, false, M, M1, ra, rb, gs, a.ov, sbo, jo, a.grid, P, w1, w2,
                        cg[i].v[PLAIN ? s2 : 0], co[i].v[PLAIN ? s2 : 0], acc[i][0]);
                    if constexpr (MODE == P2_PHASED_CB) cbo[(i ? rb : ra) * M2 + tid] = cb;
                }
                if (nyq) {
                    const float2 cn = nyq_bin_ph<M2, LP, PLAIN>(a, zr[s2], twp, M1, ra, rb, gs, sbo, jo, P, w1, w2,
                                                                it + s2, acc[2][0]);
                    if constexpr (MODE == P2_PHASED_CB) cbo[M] = cn;
                }
            } else {
                const FrameParam &F = static_cast<const FrameParam *>(params)[it + s2];
                const double dth = PLAIN ? 0.0 : F.dth, phw = PLAIN ? 0.0 : F.phw;
                const float2 frmix = PLAIN ? F.frmix : make_float2(0.f, 0.f);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    row_bin<M2, LP, PLAIN>(zr[s2], twp, i == 1, tid, false, M, M1, ra, rb, gs, a.ov, sbo, jo,
                                           a.grid, do_acf, do_xcf, ov_only, dth, phw, frmix, cg[i].v[PLAIN ? s2 : 0], acc[i]);
                if (nyq) {
                    const bool cn = PLAIN && do_xcf && M >= gs && M - gs < a.ov;
                    row_bin<M2, LP, PLAIN>(zr[s2], twp, false, 0, true, M, M1, ra, rb, gs, a.ov, sbo, jo,
                                           a.grid, do_acf, do_xcf, ov_only, dth, phw, frmix,
                                           cn ? *chain_link(a, M - gs, it + s2) : make_float2(0.f, 0.f), acc[2]);
                }
            }
        };
        if constexpr (PLAIN) {   // the frames' links in registers
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2)
                if (s2 < nfr) bins(s2);
        } else {
            for (int s2 = 0; s2 < nfr; ++s2) bins(s2);
        }
        __syncthreads();   // every thread is done with the rows
#pragma unroll
        for (int r = 0; r < 16; ++r) cur[r] = nxt[r];
    }
    // partial slot in pair-major order (as k_large_pass2_r8)
    double *out = a.part + (size_t)blockIdx.y * kNumProducts * half;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        int g;
        if (i < 2) {
            g = p * 2 * M2 + tid + 256 * i;
        } else {
            if (!nyq) continue;
            g = M;
        }
        store_pair_sums<NA>(out, half, g, acc[i], accumulate);
    }
}

// The second pass at M2 = 64 (N = 16384) and 128 (N = 32768) with two radix
// passes per row, E = M2 / 8 points each lane: lane 8 q + j of wave w takes
// row slot q (frame 2 w + q / 4 of the iteration, row q % 4 of [grid ra, grid
// rb, other ra, other rb]) -- first the DFT-E of inputs j + 8 r from
// registers, its outputs e multiplied by W_M2^{j e} and transposed through
// LDS, then lane j the DFT-8 for e = j (and j + 8), writing X[e + E b] -- so
// the four waves transform eight frames per iteration.  After a barrier each
// thread forms one bin of the pair (bin t % (2 M2): row ra for the first M2,
// else rb) of every frame (M2 = 64: of every second, threads t and t + 128
// hold the same bin and their sums are added in that order at the end; bin M,
// pair 0: the threads of bin 0), and a second barrier frees the rows.
// The E-point registers cost a row two LDS round trips.  M2 = 128 had seven
// radix-2 passes (two points per lane, one row per wave), fourteen LDS
// accesses per point: 512 frames 65 us (products) and 75 us (phased power),
// here 48 and 53.  M2 = 128 keeps the twiddles in LDS: in registers they
// spill at four waves per SIMD (746 us for 2^27 samples against 699; 735
// with three waves and no spill).
template <int M2, int MODE, bool PLAIN>
__global__ __launch_bounds__(256, PLAIN ? (MODE == P2_PRODUCTS ? 4 : 3) : M2 == 64 ? 5 : 4) void k_large_pass2_r8(
    SectorArgs a, const float2 *y1, const float2 *y2, const void *params, int M1, const float2 *tw_m2,
    int64_t fpg, int accumulate) {
    constexpr int E = M2 / 8, LP = M2 + M2 / 16 + 2;
    constexpr int FS = 128 / M2;                        // threads per bin
    constexpr int FT = 8 / FS;                          // frames per thread and iteration
    constexpr int NA = MODE == P2_PRODUCTS ? 4 : 1;
    __shared__ float2 zr[8][4][LP];   // [frame of the iteration][grid ra, grid rb, other ra, other rb]
    __shared__ float2 twp[2][M2];     // tw_post[row + M1 k2], rows ra / rb
    __shared__ double hsum[FS > 1 ? 128 : 1][NA];   // FS = 2: threads 128..255's sums
    __shared__ double msum[NA];                     // and thread 128's bin-M sums (pair 0)
    const int M = a.M;
    const int half = M + 1;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int q = lane >> 3, j = lane & 7;
    const int fw = q >> 2, rk = q & 3;
    const int p = blockIdx.x;
    const int ra = p, rb = p == 0 ? M1 / 2 : M1 - p;
    for (int i = tid; i < 2 * M2; i += 256)
        twp[i / M2][i % M2] = a.tw_post[(i < M2 ? ra : rb) + M1 * (i % M2)];
    __shared__ float2 twj[M2 == 128 ? E : 1][8];   // W_M2^{j e}, M2 = 128 (M2 = 64: registers)
    float2 tw[E];
#pragma unroll
    for (int r = 1; r < E; ++r) tw[r] = M2 == 64 ? tw_m2[(j * r) & (M2 - 1)] : make_float2(0.f, 0.f);
    if (M2 == 128 && tid < 8 * E) twj[tid >> 3][tid & 7] = tw_m2[((tid & 7) * (tid >> 3)) & (M2 - 1)];
    const int64_t g0 = (int64_t)blockIdx.y * fpg;
    int64_t g1 = g0 + fpg;
    if (g1 > a.nf) g1 = a.nf;
    const bool do_acf = (a.flags & FLAG_ACF) != 0;
    const bool do_xcf = (a.flags & FLAG_XCF) != 0;
    const bool ov_only = (a.flags & FLAG_ACF_OVERLAP) != 0;
    const float w1 = (float)a.w1, w2 = (float)a.w2;   // phased sum
    const int gs = (a.grid == 0) ? a.a1s : a.a2s;
    const int sbo = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    const int jo = sbo / M1;   // the other station's k2 offset (sbo is a multiple of M1)
    const float2 *src_row = ((rk & 2) ? (a.grid == 0 ? y2 : y1) : (a.grid == 0 ? y1 : y2)) +
                            (int64_t)((rk & 1) ? rb : ra) * M2 + j;
    const int bsel = tid % (2 * M2), fsel = tid / (2 * M2);
    const bool rb_sel = bsel >= M2;
    const int k2 = bsel & (M2 - 1);
    const bool nyq = p == 0 && bsel == 0;   // these threads also take bin M
    double acc[NA], nacc[NA];
#pragma unroll
    for (int c = 0; c < NA; ++c) acc[c] = nacc[c] = 0.0;
    const int kk = (rb_sel ? rb : ra) + M1 * k2 - gs;   // overlap index of this thread's bin
    const bool in_ov = kk >= 0 && kk < a.ov;
    auto links = [&](ChainLinks<2> &cg, ChainLinks<2> &co, int64_t f) {   // plain: this bin's, frames f, f + 1
        if constexpr (MODE == P2_PRODUCTS) {
            if (do_xcf && in_ov) cg.load(chain_link(a, kk, f));
        } else {
            cg.load_rot(a, kk + gs, a.grid, f);
            if (in_ov) co.load_rot(a, kk + gs + sbo, 1 - a.grid, f);
        }
    };
    const int slot = 2 * w + fw;   // this lane's frame of the iteration
    float2 cur[E];
    {
        const int64_t f = g0 + slot;
#pragma unroll
        for (int r = 0; r < E; ++r)
            cur[r] = f < g1 ? src_row[f * (int64_t)M + 8 * r] : make_float2(0.f, 0.f);
    }
    __syncthreads();   // twiddles staged
    float2 *z = zr[slot][rk];
    for (int64_t it = g0; it < g1; it += 8) {
        const int64_t f = it + slot, fn = f + 8;
        float2 nxt[E];
#pragma unroll
        for (int r = 0; r < E; ++r)
            nxt[r] = fn < g1 ? src_row[fn * (int64_t)M + 8 * r] : make_float2(0.f, 0.f);
        ChainLinks<2> cg = {}, co = {};   // plain: the first pair's links, loaded behind the rows' transforms
        if constexpr (PLAIN) links(cg, co, it + fsel * FT);
        if (f < g1) {
            dftR<E>(cur);                                // pass 1: inputs j + 8 r
#pragma unroll
            for (int r = 1; r < E; ++r) cur[r] = c_mul(cur[r], M2 == 64 ? tw[r] : twj[r][loop_local(j)]);
#pragma unroll
            for (int r = 0; r < E; ++r) z[pad(8 * r + j)] = cur[r];
            wave_lds_sync();
            float2 u[E / 8][8];
#pragma unroll
            for (int h = 0; h < E / 8; ++h)
#pragma unroll
                for (int r = 0; r < 8; ++r) u[h][r] = z[pad(8 * (j + 8 * h) + r)];
            wave_lds_sync();
#pragma unroll
            for (int h = 0; h < E / 8; ++h) {
                dftR<8>(u[h]);                           // pass 2
#pragma unroll
                for (int r = 0; r < 8; ++r) z[pad(j + 8 * h + E * r)] = u[h][r];   // X[e + E b]
            }
        }
        __syncthreads();   // the iteration's rows are ready
        const int nfr = (int)((g1 - it) < 8 ? (g1 - it) : 8);
        auto bins = [&](int s2, float2 chv, float2 cho) {
            if constexpr (MODE == P2_PRODUCTS) {
                const FrameParam &F = static_cast<const FrameParam *>(params)[it + s2];
                const double dth = PLAIN ? 0.0 : F.dth, phw = PLAIN ? 0.0 : F.phw;
                const float2 frmix = PLAIN ? F.frmix : make_float2(0.f, 0.f);
                row_bin<M2, LP, PLAIN>(zr[s2], twp, rb_sel, k2, false, M, M1, ra, rb, gs, a.ov, sbo, jo,
                                       a.grid, do_acf, do_xcf, ov_only, dth, phw, frmix, chv, acc);
                if (nyq) {
                    const bool cn = PLAIN && do_xcf && M >= gs && M - gs < a.ov;
                    row_bin<M2, LP, PLAIN>(zr[s2], twp, false, 0, true, M, M1, ra, rb, gs, a.ov, sbo, jo,
                                           a.grid, do_acf, do_xcf, ov_only, dth, phw, frmix,
                                           cn ? *chain_link(a, M - gs, it + s2) : make_float2(0.f, 0.f), nacc);
                }
            } else {
                const PhasedParam P = static_cast<const PhasedParam *>(params)[it + s2];
                float2 *cbo = MODE == P2_PHASED_CB ? a.cb_out + (it + s2) * half : nullptr;
                const float2 cb = row_bin_ph<M2, LP, PLAIN>(zr[s2], twp, rb_sel, k2, false, M, M1, ra, rb, gs,
                                                            a.ov, sbo, jo, a.grid, P, w1, w2, chv, cho, acc[0]);
                if constexpr (MODE == P2_PHASED_CB) cbo[(rb_sel ? rb : ra) * M2 + k2] = cb;
                if (nyq) {
                    const float2 cn = nyq_bin_ph<M2, LP, PLAIN>(a, zr[s2], twp, M1, ra, rb, gs, sbo, jo, P, w1, w2,
                                                                it + s2, nacc[0]);
                    if constexpr (MODE == P2_PHASED_CB) cbo[M] = cn;
                }
            }
        };
        if constexpr (PLAIN) {   // consecutive frames, their links in pairs, the next pair on its way
            for (int i = 0; i < FT && fsel * FT + i < nfr; i += 2) {
                const ChainLinks<2> ng = cg, no = co;
                if (i + 2 < FT) links(cg, co, it + fsel * FT + i + 2);
                bins(fsel * FT + i, ng.v[0], no.v[0]);
                if (fsel * FT + i + 1 < nfr) bins(fsel * FT + i + 1, ng.v[1], no.v[1]);
            }
        } else {
            for (int s2 = fsel; s2 < nfr; s2 += FS) bins(s2, make_float2(0.f, 0.f), make_float2(0.f, 0.f));
        }
        __syncthreads();   // every thread is done with the rows
#pragma unroll
        for (int r = 0; r < E; ++r) cur[r] = nxt[r];
    }
    if constexpr (FS > 1) {
        if (tid >= 128) {
#pragma unroll
            for (int c = 0; c < NA; ++c) hsum[bsel][c] = acc[c];
            if (nyq)
#pragma unroll
                for (int c = 0; c < NA; ++c) msum[c] = nacc[c];
        }
        __syncthreads();
        if (tid >= 128) return;
#pragma unroll
        for (int c = 0; c < NA; ++c) {
            acc[c] += hsum[bsel][c];
            if (nyq) nacc[c] += msum[c];
        }
    }
    // partial slot in pair-major order: index p 2 M2 + i (i < M2: row ra,
    // k2 = i; else row rb, k2 = i - M2), bin M last (phased: the power alone,
    // the other products are not read); launch_reduce_pairs restores bin order
    double *out = a.part + (size_t)blockIdx.y * kNumProducts * half;
    store_pair_sums<NA>(out, half, p * 2 * M2 + bsel, acc, accumulate);
    if (nyq) store_pair_sums<NA>(out, half, M, nacc, accumulate);
}

// The phased sum with the .raw output on the second pass at M2 = 64 (N =
// 16384): k_large_pass2_r8 with the phased bin and the first half of the
// inverse real FFT as well.  The pair's cb
// rows of the iteration's frames are kept in LDS; after the barrier that
// ends the bins, lanes 0..31 of wave w take (frame, row) tasks 4 w ..
// 4 w + 3 (frame task / 2, row ra or rb), 8 lanes each: y[k] = conj(Z'[k])
// of the half-length complex inverse (irfft_pre_elem's arithmetic: bins k
// and M - k lie in the pair), the row's DFT-64 over k2 (two radix-8 passes,
// the wave's own row buffers as scratch), times W_M^{n2 k1}, stored as row
// k1 of the frame's 128 x 64 block in a.cb_out (M entries per frame).
// k_irfft_cols_quantise finishes the transform over k1 and quantises.
template <bool PLAIN>
__global__ __launch_bounds__(256, PLAIN ? 3 : 4) void k_large_pass2_r8_ph(SectorArgs a, const float2 *y1,
                                                           const float2 *y2, const PhasedParam *pp,
                                                           int M1, const float2 *tw_m2,
                                                           const float2 *tw_m, int64_t fpg,
                                                           int accumulate) {
    constexpr int M2 = 64, LP = M2 + M2 / 16 + 2;
    __shared__ float2 zr[8][4][LP];   // [frame of the iteration][grid ra, grid rb, other ra, other rb]
    __shared__ float2 twp[2][M2];     // tw_post[row + M1 k2], rows ra / rb
    __shared__ double hsum[128];      // threads 128..255's sums
    __shared__ double msum;           // thread 128's bin-M sum (pair 0)
    __shared__ float2 cbl[8][2][M2];   // cb of the pair's rows, per frame
    __shared__ float2 cbn[8];                    // cb of bin M (pair 0)
    __shared__ float2 twr[2][M2];      // W_M^{n2 row}, rows ra / rb
    const int M = a.M;
    const int half = M + 1;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int q = lane >> 3, j = lane & 7;
    const int fw = q >> 2, rk = q & 3;
    const int p = blockIdx.x;
    const int ra = p, rb = p == 0 ? M1 / 2 : M1 - p;
    for (int i = tid; i < 2 * M2; i += 256) {
        twp[i / M2][i % M2] = a.tw_post[(i < M2 ? ra : rb) + M1 * (i % M2)];
        twr[i / M2][i % M2] = tw_m[((i % M2) * (i < M2 ? ra : rb)) & (M - 1)];
    }
    float2 tw[8];
#pragma unroll
    for (int r = 1; r < 8; ++r) tw[r] = tw_m2[(j * r) & (M2 - 1)];
    const int64_t g0 = (int64_t)blockIdx.y * fpg;
    int64_t g1 = g0 + fpg;
    if (g1 > a.nf) g1 = a.nf;
    const float w1 = (float)a.w1, w2 = (float)a.w2;
    const int gs = (a.grid == 0) ? a.a1s : a.a2s;
    const int sbo = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    const int jo = sbo / M1;
    const float2 *src_row = ((rk & 2) ? (a.grid == 0 ? y2 : y1) : (a.grid == 0 ? y1 : y2)) +
                            (int64_t)((rk & 1) ? rb : ra) * M2 + j;
    const int bsel = tid & 127, fsel = tid >> 7;
    const bool rb_sel = bsel >= M2;
    const int k2 = bsel & (M2 - 1);
    const bool nyq = p == 0 && bsel == 0;   // threads 0 and 128 also take bin M
    double acc = 0.0, nacc = 0.0;
    const int slot = 2 * w + fw;   // this lane's frame of the iteration
    float2 cur[8];
    {
        const int64_t f = g0 + slot;
#pragma unroll
        for (int r = 0; r < 8; ++r)
            cur[r] = f < g1 ? src_row[f * (int64_t)M + 8 * r] : make_float2(0.f, 0.f);
    }
    __syncthreads();   // twiddles staged
    float2 *z = zr[slot][rk];
    for (int64_t it = g0; it < g1; it += 8) {
        const int64_t f = it + slot, fn = f + 8;
        float2 nxt[8];
#pragma unroll
        for (int r = 0; r < 8; ++r)
            nxt[r] = fn < g1 ? src_row[fn * (int64_t)M + 8 * r] : make_float2(0.f, 0.f);
        ChainLinks<PLAIN ? 4 : 1> cg = {}, co = {};   // this thread's frames it + 4 fsel ..
        if constexpr (PLAIN) {
            const int g = (rb_sel ? rb : ra) + M1 * k2;
            cg.load_rot(a, g, a.grid, it + 4 * fsel);
            if (g >= gs && g < gs + a.ov) co.load_rot(a, g + sbo, 1 - a.grid, it + 4 * fsel);
        }
        if (f < g1) {
            dftR<8>(cur);                                // pass 1: inputs j + 8 r
#pragma unroll
            for (int r = 1; r < 8; ++r) cur[r] = c_mul(cur[r], tw[r]);
#pragma unroll
            for (int r = 0; r < 8; ++r) z[pad(8 * j + r)] = cur[r];
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 8; ++r) cur[r] = z[pad(j + 8 * r)];
            dftR<8>(cur);                                // pass 2
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 8; ++r) z[pad(j + 8 * r)] = cur[r];   // X[j + 8 r]
        }
        __syncthreads();   // the iteration's rows are ready
        const int nfr = (int)((g1 - it) < 8 ? (g1 - it) : 8);
        auto bins = [&](int s2, float2 rg, float2 ro) {
            const PhasedParam P = pp[it + s2];
            cbl[s2][rb_sel][k2] = row_bin_ph<M2, LP, PLAIN>(zr[s2], twp, rb_sel, k2, false, M, M1, ra, rb, gs, a.ov,
                                                            sbo, jo, a.grid, P, w1, w2, rg, ro, acc);
            if (nyq)
                cbn[s2] = nyq_bin_ph<M2, LP, PLAIN>(a, zr[s2], twp, M1, ra, rb, gs, sbo, jo, P, w1, w2, it + s2, nacc);
        };
        if constexpr (PLAIN) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * fsel + i < nfr) bins(4 * fsel + i, cg.v[i], co.v[i]);
        } else {
            for (int s2 = fsel; s2 < nfr; s2 += 2) bins(s2, make_float2(0.f, 0.f), make_float2(0.f, 0.f));
        }
        __syncthreads();   // every thread is done with the rows; cb complete
        {
            // the wave's row buffers zr[2 w][*] are scratch here: the next
            // frames' rows are written to them by this wave only
            const int task = 4 * w + (lane >> 3);
            const int s3 = task >> 1, b = task & 1;
            if (lane < 32 && s3 < nfr) {
                const int row = b ? rb : ra;
                const int bm = (row == 0 ? row : M1 - row) == ra ? 0 : 1;
                float2 v[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int kk = j + 8 * r;                  // k2 of bin k = row + M1 kk
                    float2 zq;
                    if (row == 0 && kk == 0) {
                        const float2 x0 = cbl[s3][0][0], xm = cbn[s3];
                        zq = make_float2(x0.x + xm.x, x0.x - xm.x);
                    } else {
                        const int km = row == 0 ? (M2 - kk) & (M2 - 1) : M2 - 1 - kk;
                        const float2 A = cbl[s3][b][kk], Bc = cbl[s3][bm][km];
                        const float er = A.x + Bc.x, ei = A.y - Bc.y;
                        const float dr = A.x - Bc.x, di = A.y + Bc.y;
                        const float2 wp = twp[b][kk];
                        const float orr = dr * wp.x - di * wp.y;
                        const float oi = dr * wp.y + di * wp.x;
                        zq = make_float2(er - oi, ei + orr);
                    }
                    v[r] = c_conj(zq);
                }
                float2 *zs = zr[2 * w][lane >> 3];
                dftR<8>(v);                                  // pass 1: inputs j + 8 r
#pragma unroll
                for (int r = 1; r < 8; ++r) v[r] = c_mul(v[r], tw[r]);
#pragma unroll
                for (int r = 0; r < 8; ++r) zs[pad(8 * j + r)] = v[r];
                wave_lds_sync();
#pragma unroll
                for (int r = 0; r < 8; ++r) v[r] = zs[pad(j + 8 * r)];
                dftR<8>(v);                                  // pass 2: outputs n2 = j + 8 r
                float2 *bo = a.cb_out + (it + s3) * (int64_t)M + row * M2;
#pragma unroll
                for (int r = 0; r < 8; ++r) bo[j + 8 * r] = c_mul(v[r], twr[b][j + 8 * r]);
                wave_lds_sync();
            }
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) cur[r] = nxt[r];
    }
    if (tid >= 128) {
        hsum[bsel] = acc;
        if (nyq) msum = nacc;
    }
    __syncthreads();
    if (tid >= 128) return;
    // partial slot in pair-major order (as k_large_pass2_r8); the other
    // products stay zero
    double *out = a.part + (size_t)blockIdx.y * kNumProducts * half;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int g;
        double v;
        if (i == 0) {
            g = p * 2 * M2 + bsel;
            v = acc + hsum[bsel];
        } else {
            if (!nyq) continue;
            g = M;
            v = nacc + msum;
        }
        out[P_PH * half + g] = accumulate ? out[P_PH * half + g] + v : v;
    }
}

hipError_t launch_large_pass2_phased(const SectorArgs &a, const float2 *y1, const float2 *y2,
                                     const void *pp, int M1, int M2, const float2 *tw_m2,
                                     const float2 *tw_m, bool raw, int n_groups, int accumulate,
                                     bool plain, hipStream_t s) {
    const int sbo = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    if (M1 * M2 != a.M || sbo % M1 != 0 || (M2 != 64 && M2 != 128 && M2 != 256) || M1 != 128 ||
        (raw && !a.cb_out))
        return hipErrorInvalidValue;
    int64_t fpg = (a.nf + n_groups - 1) / n_groups;
    if (plain) {   // whole iterations, so that the chain runs start on their 64-byte lines
        if (a.chain == nullptr || a.chain_ld < a.nf + 8) return hipErrorInvalidValue;
        fpg = (fpg + 7) & ~(int64_t)7;
    }
    const dim3 grid((unsigned)(M1 / 2), (unsigned)n_groups);
    if (raw && M2 == 64) {
        auto kern = plain ? k_large_pass2_r8_ph<true> : k_large_pass2_r8_ph<false>;
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a, y1, y2, (const PhasedParam *)pp, M1, tw_m2, tw_m,
                           fpg, accumulate);
        return hipGetLastError();
    }
    auto pick = [raw](auto cb, auto power) { return raw ? cb : power; };
    auto kern = M2 == 64    ? (plain ? k_large_pass2_r8<64, P2_PHASED, true> : k_large_pass2_r8<64, P2_PHASED, false>)
                : M2 == 128 ? (plain ? pick(k_large_pass2_r8<128, P2_PHASED_CB, true>, k_large_pass2_r8<128, P2_PHASED, true>)
                                     : pick(k_large_pass2_r8<128, P2_PHASED_CB, false>, k_large_pass2_r8<128, P2_PHASED, false>))
                            : (plain ? pick(k_large_pass2_r16<P2_PHASED_CB, true>, k_large_pass2_r16<P2_PHASED, true>)
                                     : pick(k_large_pass2_r16<P2_PHASED_CB, false>, k_large_pass2_r16<P2_PHASED, false>));
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a, y1, y2, pp, M1, tw_m2, fpg, accumulate);
    return hipGetLastError();
}

hipError_t launch_large_pass2_mac(const SectorArgs &a, const float2 *y1, const float2 *y2,
                                  const FrameParam *params, int M1, int M2, const float2 *tw_m2,
                                  int n_groups, int accumulate, bool plain, hipStream_t s) {
    const int sbo = (a.grid == 0) ? (a.a2s - a.a1s) : (a.a1s - a.a2s);
    if (M1 * M2 != a.M || sbo % M1 != 0 || (M2 != 64 && M2 != 128 && M2 != 256)) return hipErrorInvalidValue;
    int64_t fpg = (a.nf + n_groups - 1) / n_groups;
    if (plain) {   // whole iterations, so that the chain runs start on their 64-byte lines
        if ((a.flags & FLAG_XCF) && (a.chain == nullptr || a.chain_ld < a.nf + 8)) return hipErrorInvalidValue;
        fpg = (fpg + 7) & ~(int64_t)7;
    }
    const dim3 grid((unsigned)(M1 / 2), (unsigned)n_groups);
    auto kern = M2 == 64    ? (plain ? k_large_pass2_r8<64, P2_PRODUCTS, true> : k_large_pass2_r8<64, P2_PRODUCTS, false>)
                : M2 == 128 ? (plain ? k_large_pass2_r8<128, P2_PRODUCTS, true> : k_large_pass2_r8<128, P2_PRODUCTS, false>)
                            : (plain ? k_large_pass2_r16<P2_PRODUCTS, true> : k_large_pass2_r16<P2_PRODUCTS, false>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a, y1, y2, (const void *)params, M1, tw_m2, fpg,
                       accumulate);
    return hipGetLastError();
}

hipError_t launch_mac_large(const SectorArgs &a, int precision, const float2 *z1, const float2 *z2,
                            const FrameParam *params, int n_groups, int accumulate,
                            hipStream_t s) {
    const int64_t fpg = (a.nf + n_groups - 1) / n_groups;
    const dim3 grid((unsigned)((a.M + 1 + 255) / 256), (unsigned)n_groups);
    if (precision == 0)
        hipLaunchKernelGGL(k_mac_large<0>, grid, dim3(256), 0, s, a, z1, z2, params, fpg, accumulate);
    else
        hipLaunchKernelGGL(k_mac_large<1>, grid, dim3(256), 0, s, a, z1, z2, params, fpg, accumulate);
    return hipGetLastError();
}

}  // namespace fxc
