// k_mel.hip — log-mel front-end on the GPU (transcribe.c:177-214).
//
// Per frame t of a clip: samples [t*160, t*160+400) of the zero-padded
// (200 each side), pre-emphasised (x[i] - 0.97 x[i-1]) signal, Hann window,
// 512-point FFT, power spectrum (257 bins), 128 Slaney mel filters,
// log(x + 2^-24).  Then each mel bin is normalised over the clip's frames
// with mean and var/(T-1).  One wavefront transforms one frame in LDS
// (radix-2, twiddles from a host table); a second kernel normalises rows.
#include "ct_dev.h"
#include "ct_launch.h"
#include "../../include/model_types.h"

namespace {

constexpr int NF = N_FFT;   // 512
constexpr int FPW = 4;      // frames of a workgroup, one per wavefront

// Orders one wavefront's LDS accesses: the hardware keeps them in issue order,
// so only the compiler has to be held.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// A wavefront transforms one frame alone, four butterflies a lane and stage,
// so no stage waits for other wavefronts (one frame on four wavefronts spent
// its time at 18 barriers): 2001 frames 16.5 -> 15.1 us, 16503 89 -> 63.
__global__ __launch_bounds__(64 * FPW) void mel_frames_kernel(float *mel,
                                                         const CtMelClip *clips, const int *frame_clip,
                                                         const float *hann, const float *twr,
                                                         const float *twi, const float *fb,
                                                         const int *fb_lo, const int *fb_hi, int n_frames) {
    __shared__ float s_re[FPW][NF], s_im[FPW][NF], s_wr[NF / 2], s_wi[NF / 2];
    for (int i = threadIdx.x; i < NF / 2; i += 64 * FPW) { s_wr[i] = twr[i]; s_wi[i] = twi[i]; }
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int f = blockIdx.x * FPW + w;
    if (f >= n_frames) return;
    float *re = s_re[w], *im = s_im[w];
    const CtMelClip c = clips[frame_clip[f]];
    const int t = f - c.frame0;
    const int off = t * HOP_LEN;
    const int pad = WIN_LEN / 2;
    // load windowed, pre-emphasised samples in bit-reversed order
#pragma unroll
    for (int j0 = 0; j0 < NF; j0 += 64) {
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
    wave_lds_fence();
    for (int half = 1; half < NF; half <<= 1) {
#pragma unroll
        for (int u = 0; u < NF / 128; u++) {           // 256 butterflies per stage
            const int k = lane + 64 * u, pos = k & (half - 1);
            const int i0 = 2 * k - pos, i1 = i0 + half;
            const int tw = pos * (NF / (2 * half));
            const float wr = s_wr[tw], wi = s_wi[tw];
            const float vr = re[i1] * wr - im[i1] * wi;
            const float vi = re[i1] * wi + im[i1] * wr;
            const float ur = re[i0], ui = im[i0];
            re[i0] = ur + vr; im[i0] = ui + vi;
            re[i1] = ur - vr; im[i1] = ui - vi;
        }
        wave_lds_fence();
    }
    // the power spectrum over the real parts (each lane reads only what it writes)
    for (int i = lane; i < N_BINS; i += 64) re[i] = re[i] * re[i] + im[i] * im[i];
    wave_lds_fence();
    for (int m = lane; m < N_MELS; m += 64) {
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
    hipLaunchKernelGGL(mel_frames_kernel, dim3((n_frames + FPW - 1) / FPW), dim3(64 * FPW), 0, s, mel, clips, frame_clip,
                       tab->hann, tab->twr, tab->twi, tab->fb, tab->fb_lo, tab->fb_hi, n_frames);
    hipLaunchKernelGGL(mel_norm_kernel, dim3(N_MELS, n_clips), dim3(64), 0, s, mel, clips);
}
