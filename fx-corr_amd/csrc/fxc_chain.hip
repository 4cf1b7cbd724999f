// The reference's f32 phase chains, replayed per frame for the plain form.
//
// XCF phase (main.rs:2513-2527, start/step from xcf_phase_start_and_step,
// main.rs:133-149):
//     p_0 = from_polar(1, ang0 as f32),  p_{k+1} = p_k * from_polar(1, angs as f32)
// Phased per-station rotation (utils.rs:93-117 with start_bin = 0, rate =
// accel = t = 0, USB sign; main.rs:2238-2262):
//     r_0 = from_polar(1, (step * 0) as f32),  r_{b+1} = r_b * from_polar(1, step as f32)
//
// Each link is Rust's Complex<f32> product: four f32 products and two f32
// sums, no fused multiply-add, so a chain carries the reference's rounding
// bit for bit.  from_polar's cos/sin are the correctly rounded f32 values;
// for the step angles of N >= 2048 (|angle| < 3.1e-3) glibc's cosf/sinf
// return exactly those, and a start one ulp away (larger band-shifted start
// angles) moves a chain by at most ~5e-7 over 30720 links.
//
// Two adjacent lanes walk one chain, one holding its real part and the other
// its imaginary part: a link is then own * re(step) + other * (-/+ im(step)),
// the same products and sums, with the other lane's part read through the
// multiply's DPP operand -- three VALU instructions and one wait state on the
// walk's critical path.  Each chain is one sequential walk (a launch holds a
// few hundred to a few thousand of them, far fewer than the chip's lanes), so
// the launch time is the latency of a link.  One thread per chain with both
// parts took 22.6 ns a link (six VALU instructions, an address and a store per
// pair); this form takes 11..13 ns (a 128-frame FFT-2048 sector 46 -> 34 us,
// four frames at FFT 65536 870 -> 434).  Rows are planar (chain_at): each lane
// stores four links of its part as one 16-byte store.  Blocks of one wave, so
// that the few long chains of a launch spread over the compute units.
#include "fxc_dev.h"

namespace fxc {

// The next link's part held by this lane: v * qx + other * c, other = the
// partner lane's part (quad_perm [1, 0, 3, 2]).  Real part (c = -im step):
// re*qx - im*qy; imaginary part (c = im step): im*qx + re*qy.
__device__ __forceinline__ float chain_next(float v, float qx, float c) {
#pragma clang fp contract(off)
    const float other = __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
    const float own = v * qx;
    const float cross = other * c;
    return own + cross;
}

// Link 0 and the step of a frame's chain (phased: station s's)
__device__ __forceinline__ void chain_start(const SectorArgs &a, int kind, int64_t frame, int s, float2 &p,
                                            float2 &step) {
    FrameDelayDev d;
    compute_frame_delay(frame, a.dly, d, nullptr, nullptr);
    {
#pragma clang fp contract(off)
        if (kind == CHAIN_XCF) {
            const double two_pi_df = -2.0 * FXC_PI * a.df;
            const double step1 = two_pi_df * d.frac1;
            const double step2 = two_pi_df * d.frac2;
            p = polar1_f32((float)(step1 * (double)a.a1s - step2 * (double)a.a2s));
            step = polar1_f32((float)(step1 - step2));
        } else {
            const double total = s ? d.frac2 : d.frac1;
            const double phase_step = -1.0 * 2.0 * FXC_PI * a.df * total;
            p = polar1_f32((float)(phase_step * 0.0));
            step = polar1_f32((float)phase_step);
        }
    }
}

__global__ __launch_bounds__(64) void k_phase_chain(SectorArgs a, int kind, float *out) {
    const int nch = kind == CHAIN_XCF ? 1 : a.chains;
    const int len = kind == CHAIN_XCF ? a.ov : a.M + 1;
    const int64_t i = (int64_t)blockIdx.x * (blockDim.x / 2) + (threadIdx.x >> 1);   // chain
    const bool im = threadIdx.x & 1;
    if (i >= a.nf * nch) return;   // both lanes of a pair together
    const int64_t f = i / nch;
    const int s = (int)(i - f * nch);
    float2 p, step;
    chain_start(a, kind, a.first_frame + f, s, p, step);
    // this part's row: a.chain_ld floats (a multiple of 16, >= len)
    float4 *o = reinterpret_cast<float4 *>(out + (2 * i + (im ? 1 : 0)) * (int64_t)a.chain_ld);
    const float qx = step.x, c = im ? step.y : -step.y;
    float v = im ? p.y : p.x;
    for (int k = 0; k < len; k += 16, o += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float4 r;
            r.x = v;
            r.y = chain_next(r.x, qx, c);
            r.z = chain_next(r.y, qx, c);
            r.w = chain_next(r.z, qx, c);
            o[u] = r;
            v = chain_next(r.w, qx, c);
        }
    }
}

typedef __attribute__((address_space(1))) float global_float;
typedef __attribute__((address_space(1))) char global_char;

// The chains link-major (link k of frame f's chain c at (((k chains + c) ld +
// f) 2 + im), ld = a.chain_ld >= the frames, links up to a multiple of 8): for
// the second pass of the four-step, whose threads own a bin and walk the
// frames.  A block's 32 frames store 256 contiguous bytes per link; 16 ns a
// link against the rows' 12.7 (the store and its scalar address).  grid.y: the chain.
__global__ __launch_bounds__(64) void k_phase_chain_links(SectorArgs a, int kind, float *out) {
    const int64_t f = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 1);
    const bool im = threadIdx.x & 1;
    if (f >= a.nf) return;   // both lanes of a pair together
    const int len = kind == CHAIN_XCF ? a.ov : a.M + 1;
    const int ch = (int)blockIdx.y;
    float2 p, step;
    chain_start(a, kind, a.first_frame + f, ch, p, step);
    const float qx = step.x, c = im ? step.y : -step.y;
    float v = im ? p.y : p.x;
    // a uniform row pointer and the lane's offset: the walk's only vector work is the link
    global_float *o = (global_float *)(out + 2 * (ch * (int64_t)a.chain_ld + (int64_t)blockIdx.x * 32));
    const int64_t ld = 2 * (int64_t)gridDim.y * a.chain_ld;
    unsigned off = threadIdx.x * 4u;
    for (int k = 0; k < len; k += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u, o += ld) {
            asm volatile("" : "+s"(o), "+v"(off));   // stay a scalar pair and a 32-bit offset
            *(global_float *)((global_char *)o + off) = v;
            v = chain_next(v, qx, c);
        }
    }
}

hipError_t launch_phase_chain_links(const SectorArgs &a, int kind, float *out, hipStream_t s) {
    if (kind == CHAIN_PHASED && a.chains != 1 && a.chains != 2) return hipErrorInvalidValue;
    if (a.nf <= 0) return hipSuccess;
    if (a.chain_ld < a.nf) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((a.nf + 31) / 32), kind == CHAIN_XCF ? 1u : (unsigned)a.chains);
    hipLaunchKernelGGL(k_phase_chain_links, grid, dim3(64), 0, s, a, kind, out);
    return hipGetLastError();
}

hipError_t launch_phase_chain(const SectorArgs &a, int kind, float *out, hipStream_t s) {
    if (kind == CHAIN_PHASED && a.chains != 1 && a.chains != 2) return hipErrorInvalidValue;
    const int64_t n = a.nf * (kind == CHAIN_XCF ? 1 : a.chains);
    if (n <= 0) return hipSuccess;
    const int len = kind == CHAIN_XCF ? a.ov : a.M + 1;
    if (a.chain_ld < chain_ld_for(len) || (a.chain_ld & 15)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_phase_chain, dim3((unsigned)((n + 31) / 32)), dim3(64), 0, s, a, kind,
                       out);
    return hipGetLastError();
}

}  // namespace fxc
