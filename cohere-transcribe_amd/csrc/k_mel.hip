// k_mel.hip — log-mel front-end on the GPU (transcribe.c:177-214).
//
// Per frame t of a clip: samples [t*160, t*160+400) of the zero-padded
// (200 each side), pre-emphasised (x[i] - 0.97 x[i-1]) signal, Hann window,
// 512-point FFT, power spectrum (257 bins), 128 Slaney mel filters,
// log(x + 2^-24).  Then each mel bin is normalised over the clip's frames
// with mean and var/(T-1).  One wavefront, or with few frames four, transform
// one frame in LDS (radix-2, twiddles from a host table); a second kernel
// normalises rows.
#include "ct_dev.h"
#include "ct_launch.h"
#include "../../include/model_types.h"

namespace {

constexpr int NF = N_FFT;   // 512

// Orders one wavefront's LDS accesses: the hardware keeps them in issue order,
// so only the compiler has to be held.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// A workgroup of four wavefronts takes WPF of them per frame.  With many frames
// each wavefront transforms one alone (WPF 1): four butterflies a lane and
// stage, no barriers.  With few, nothing hides that chain, and the frame is
// split over the workgroup (WPF 4): one butterfly a lane and a barrier per
// stage.  Both do the same arithmetic per element.  us, WPF 1 and 4: 51 frames
// 11.3 and 6.3, 301 11.9 and 6.7, 1019 12.5 and 9.7, 2001 14.2 and 14.4, 3001
// 18.3 and 18.4, 4096 20.9 and 22.9, 6251 29 and 32; 16503 with WPF 1 58 (89
// with twiddles from memory and two barriers a stage).
constexpr int MEL_FEW_FRAMES = 2048;
template <int WPF>
__global__ __launch_bounds__(256) void mel_frames_kernel(float *mel,
                                                         const CtMelClip *clips, const int *frame_clip,
                                                         const float *hann, const float *twr,
                                                         const float *twi, const float *fb,
                                                         const int *fb_lo, const int *fb_hi, int n_frames) {
    constexpr int FPW = 4 / WPF, LANES = 64 * WPF;
    __shared__ float s_re[FPW][NF], s_im[FPW][NF], s_wr[NF / 2], s_wi[NF / 2];
    const int w = threadIdx.x / LANES, lane = threadIdx.x % LANES;
    const int f = blockIdx.x * FPW + w;
    s_wr[threadIdx.x] = twr[threadIdx.x];
    s_wi[threadIdx.x] = twi[threadIdx.x];
    auto frame_sync = [] {
        if (WPF == 1) wave_lds_fence();
        else __syncthreads();
    };
    if (WPF == 1) __syncthreads();
    if (f >= n_frames) return;
    float *re = s_re[w], *im = s_im[w];
    const CtMelClip c = clips[frame_clip[f]];
    const int t = f - c.frame0;
    const int off = t * HOP_LEN;
    const int pad = WIN_LEN / 2;
    // load windowed, pre-emphasised samples in bit-reversed order
#pragma unroll
    for (int j0 = 0; j0 < NF; j0 += LANES) {
        const int j = j0 + lane;
        float v = 0.0f;
        if (j < WIN_LEN) {
            const int a = off + j - pad;              // index into the clip
            const float x1 = (a >= 0 && a < c.n) ? c.pcm[a] : 0.0f;
            const float x0 = (a - 1 >= 0 && a - 1 < c.n && off + j > 0) ? c.pcm[a - 1] : 0.0f;
            v = (x1 - 0.97f * x0) * hann[j];
        }
        const int r = __brev((unsigned)j) >> (32 - 9);
        re[r] = v;
        im[r] = 0.0f;
    }
    frame_sync();
    for (int half = 1; half < NF; half <<= 1) {
#pragma unroll
        for (int u = 0; u < NF / 2 / LANES; u++) {     // 256 butterflies per stage
            const int k = lane + LANES * u, pos = k & (half - 1);
            const int i0 = 2 * k - pos, i1 = i0 + half;
            const int tw = pos * (NF / (2 * half));
            const float wr = s_wr[tw], wi = s_wi[tw];
            const float vr = re[i1] * wr - im[i1] * wi;
            const float vi = re[i1] * wi + im[i1] * wr;
            const float ur = re[i0], ui = im[i0];
            re[i0] = ur + vr; im[i0] = ui + vi;
            re[i1] = ur - vr; im[i1] = ui - vi;
        }
        frame_sync();
    }
    // the power spectrum over the real parts (each lane reads only what it writes)
    for (int i = lane; i < N_BINS; i += LANES) re[i] = re[i] * re[i] + im[i] * im[i];
    frame_sync();
    for (int m = lane; m < N_MELS; m += LANES) {
        float acc = 0.0f;
        const int lo = fb_lo[m], hi = fb_hi[m];
        const float *wm = fb + m * N_BINS;
        for (int i = lo; i < hi; i += 8) {             // eight weights in flight
            float wt[8];
#pragma unroll
            for (int u = 0; u < 8; u++) wt[u] = i + u < hi ? wm[i + u] : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (i + u < hi) acc += wt[u] * re[i + u];
        }
        mel[c.mel0 + (long)m * c.T + t] = logf(acc + 5.9604644775390625e-8f);
    }
}

// One row of a clip's spectrogram per wavefront.  A lane sums frames lane,
// lane + 64, .. in turn and the lanes' sums are added by wave_sum, in fp32, the
// same chain whatever the clip's length; what is spread wide is the loads: a
// row of up to 64 * PER frames is fetched whole, every load in flight, and
// stays in registers between the passes.  A frame past the clip adds zero,
// which changes no sum.  2001 frames 16.2 us with a load at a time, 4.2 here;
// 6251 frames 44 and 12.4.
template <int PER>
__device__ __forceinline__ void norm_row(float *row, int T, int lane) {
    float v[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) v[i] = row[min(lane + 64 * i, T - 1)];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) s += lane + 64 * i < T ? v[i] : 0.0f;
    const float mu = wave_sum(s) / (float)T;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const float d = lane + 64 * i < T ? v[i] - mu : 0.0f;
        q = __builtin_fmaf(d, d, q);
    }
    const float var = wave_sum(q) / (float)(T - 1);
    const float r = 1.0f / sqrtf(var + 1e-5f);
#pragma unroll
    for (int i = 0; i < PER; i++)
        if (lane + 64 * i < T) row[lane + 64 * i] = (v[i] - mu) * r;
}
__global__ __launch_bounds__(64) void mel_norm_kernel(float *mel, const CtMelClip *clips) {
    const CtMelClip c = clips[blockIdx.y];
    const int lane = threadIdx.x, T = c.T;
    float *row = mel + c.mel0 + (long)blockIdx.x * T;
    if (T <= 64 * 4) return norm_row<4>(row, T, lane);
    if (T <= 64 * 16) return norm_row<16>(row, T, lane);
    if (T <= 64 * 32) return norm_row<32>(row, T, lane);
    if (T <= 64 * 64) return norm_row<64>(row, T, lane);
    // longer than 40 s: read again for each pass, 16 loads in flight
    constexpr int U = 16;
    float s = 0.0f, q = 0.0f;
    for (int t0 = lane; t0 < T; t0 += 64 * U) {
        float v[U];
#pragma unroll
        for (int i = 0; i < U; i++) v[i] = row[min(t0 + 64 * i, T - 1)];
#pragma unroll
        for (int i = 0; i < U; i++) s += t0 + 64 * i < T ? v[i] : 0.0f;
    }
    const float mu = wave_sum(s) / (float)T;
    for (int t0 = lane; t0 < T; t0 += 64 * U) {
        float v[U];
#pragma unroll
        for (int i = 0; i < U; i++) v[i] = row[min(t0 + 64 * i, T - 1)];
#pragma unroll
        for (int i = 0; i < U; i++) {
            const float d = t0 + 64 * i < T ? v[i] - mu : 0.0f;
            q = __builtin_fmaf(d, d, q);
        }
    }
    const float var = wave_sum(q) / (float)(T - 1);
    const float r = 1.0f / sqrtf(var + 1e-5f);
    for (int t0 = lane; t0 < T; t0 += 64 * U) {
        float v[U];
#pragma unroll
        for (int i = 0; i < U; i++) v[i] = row[min(t0 + 64 * i, T - 1)];
#pragma unroll
        for (int i = 0; i < U; i++)
            if (t0 + 64 * i < T) row[t0 + 64 * i] = (v[i] - mu) * r;
    }
}

}  // namespace

extern "C" void ctk_mel(float *mel, const CtMelClip *clips, int n_clips,
                        const int *frame_clip, int n_frames, const CtMelTables *tab, hipStream_t s) {
    if (n_frames <= 0) return;
    if (n_frames <= MEL_FEW_FRAMES)
        hipLaunchKernelGGL(mel_frames_kernel<4>, dim3(n_frames), dim3(256), 0, s, mel, clips, frame_clip, tab->hann,
                           tab->twr, tab->twi, tab->fb, tab->fb_lo, tab->fb_hi, n_frames);
    else
        hipLaunchKernelGGL(mel_frames_kernel<1>, dim3((n_frames + 3) / 4), dim3(256), 0, s, mel, clips, frame_clip,
                           tab->hann, tab->twr, tab->twi, tab->fb, tab->fb_lo, tab->fb_hi, n_frames);
    hipLaunchKernelGGL(mel_norm_kernel, dim3(N_MELS, n_clips), dim3(64), 0, s, mel, clips);
}
