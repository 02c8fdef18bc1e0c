// Log-mel front end (i_whisper/audio.py:216-267) in float32: centred STFT
// frames of a periodic Hann window with reflect padding, |X|^2, the mel
// filterbank, log10 of max(., 1e-10); then per audio the floor
// max(log, max_all - 8) and log / 4 + 1.
#include "../../include/iwhisper_amd.h"
#include "iw_common.hpp"
#include "iw_kernels.hpp"

#include <mutex>

// Block maxima of iw_log_mel_noalloc: a fixed device array instead of a
// caller workspace, for callers that cannot allocate. Each GPU holds its own
// copy (at its own address, looked up once per device below) until the process
// ends; every call on one GPU shares it, so calls that overlap on one GPU race.
static __device__ __align__(256) float scratch[IW_LOG_MEL_SCRATCH_FLOATS];

namespace iw {

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
float *g_scratch_ptr[kMaxScratchDevices] = {};
}  // namespace

int log_mel_scratch(hipStream_t stream, float **ptr) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices)
    return fail("iw_log_mel_noalloc: no usable current device");
  if (stream != nullptr) {
    hipDevice_t sdev = -1;
    if (hipStreamGetDevice(stream, &sdev) != hipSuccess || sdev != dev)
      return fail("iw_log_mel_noalloc: the stream does not belong to the current device");
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    // device address of this device's copy (the host-side name `scratch` is
    // not a device address and is never passed to a kernel)
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(std::string("iw_log_mel_noalloc: hipGetSymbolAddress failed: ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<float *>(p);
  }
  *ptr = g_scratch_ptr[dev];
  return IW_OK;
}

namespace {

constexpr int kFft = 512;         // N_FFT
constexpr int kBins = kFft / 2 + 1;
constexpr int kFramesPerBlock = 64;
constexpr int kMaxMels = 128;
constexpr int kMaxFilterTaps = 2048;  // nonzero filterbank weights

constexpr int kWaves = 16;
constexpr int kFramesPerWave = kFramesPerBlock / kWaves;

struct Cplx {
  float re, im;
};
__device__ __forceinline__ Cplx operator+(Cplx a, Cplx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ Cplx operator-(Cplx a, Cplx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ Cplx operator*(Cplx a, Cplx b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ Cplx minus_i(Cplx a) { return {a.im, -a.re}; }  // -i a

constexpr float kR = 0.70710678118654752f;

// 8-point DFT (exp(-2 pi i jk / 8)) of eight real values
__device__ __forceinline__ void dft8_real(const float (&a)[8], Cplx (&y)[8]) {
  const float b0 = a[0] + a[4], b1 = a[0] - a[4], b2 = a[2] + a[6], b3 = a[2] - a[6];
  const float c0 = a[1] + a[5], c1 = a[1] - a[5], c2 = a[3] + a[7], c3 = a[3] - a[7];
  const float p = kR * (c1 - c3), q = kR * (c1 + c3);
  y[0] = {(b0 + b2) + (c0 + c2), 0.f};
  y[4] = {(b0 + b2) - (c0 + c2), 0.f};
  y[2] = {b0 - b2, c2 - c0};
  y[6] = {b0 - b2, c0 - c2};
  y[1] = {b1 + p, -b3 - q};
  y[7] = {b1 + p, b3 + q};
  y[3] = {b1 - p, b3 - q};
  y[5] = {b1 - p, q - b3};
}

// the same of eight complex values, in place
__device__ __forceinline__ void dft8(Cplx (&a)[8]) {
  Cplx e[4], o[4];
  auto dft4 = [](Cplx x0, Cplx x1, Cplx x2, Cplx x3, Cplx (&y)[4]) {
    const Cplx t0 = x0 + x2, t1 = x0 - x2, t2 = x1 + x3, t3 = minus_i(x1 - x3);
    y[0] = t0 + t2, y[2] = t0 - t2, y[1] = t1 + t3, y[3] = t1 - t3;
  };
  dft4(a[0], a[2], a[4], a[6], e);
  dft4(a[1], a[3], a[5], a[7], o);
  o[1] = Cplx{kR * (o[1].re + o[1].im), kR * (o[1].im - o[1].re)};
  o[2] = minus_i(o[2]);
  o[3] = Cplx{kR * (o[3].im - o[3].re), -kR * (o[3].re + o[3].im)};
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = e[k] + o[k], a[k + 4] = e[k] - o[k];
}

// this wave's LDS accesses so far are done before the later ones
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One block = 16 waves = 64 consecutive frames of one audio (four per wave, one
// at a time; one audio of 30 s is only 47 blocks, so what counts is the chain
// of a wave). A frame's 512-point transform is three radix-8 steps in
// registers, eight values per lane, with two exchanges through the wave's own
// LDS rows:
//   A_q[l]    = W512^(l q) sum_k x[l + 64 k] W8^(k q)          lane l
//   B[q][m][s] = W64^(m s) sum_j A_q[m + 8 j] W8^(j s)          lane 8 q + m
//   X[q + 8 s + 64 t] = sum_m B[q][m][s] W8^(m t)               lane 8 s + q
// (W_n = exp(-2 pi i / n), from a table computed in float64 on the host). The
// LDS rows are laid out so that an exchange's lanes spread over the banks (the writes
// of B alone meet seven of the 64 banks twice: 72 s + 9 m + q). Each mel bin then sums its
// filter's nonzero taps (sparse rows: first
// bin, tap count, offset into the weights), and the block writes [n_mels][64]
// rows of log10 values plus its maximum. With 4 waves of 16 frames and nine
// radix-2 steps in LDS this took 85.8 us for 30 s of audio at 80 mels; now 21.8.
__global__ __launch_bounds__(64 * kWaves) void logmel_kernel(
    const float *__restrict__ audio, int64_t n_samples, int64_t audio_ld, const float2 *__restrict__ twiddle,
    const float *__restrict__ window, const int *__restrict__ fstart, const int *__restrict__ flen,
    const int *__restrict__ foff, const float *__restrict__ fw, int n_taps, int n_mels, int n_frames,
    float *__restrict__ out, int64_t out_ld_b, float *__restrict__ blockmax) {
  constexpr int NT = 64 * kWaves, XLD = 8 * 72;
  __shared__ float sRe[kWaves][XLD], sIm[kWaves][XLD];
  __shared__ int sStart[kMaxMels], sLen[kMaxMels], sOff[kMaxMels];
  __shared__ float sW[kMaxFilterTaps];
  __shared__ float sOut[kMaxMels][kFramesPerBlock + 1];
  __shared__ float sMax[kWaves];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t b = blockIdx.y;
  const int t0 = blockIdx.x * kFramesPerBlock;
  const float *x = audio + b * audio_ld;
  // this lane's window values and twiddles (the table holds half a turn)
  const int hi = lane >> 3, lo = lane & 7;
  auto w512 = [&](int j) {
    const float2 w = twiddle[j & 255];
    return j & 256 ? Cplx{-w.x, -w.y} : Cplx{w.x, w.y};
  };
  float win[8];
  Cplx tw1[8], tw2[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    win[k] = window[lane + 64 * k];
    tw1[k] = w512(lane * k);
    tw2[k] = w512(8 * lo * k);
  }
  for (int i = tid; i < n_mels; i += NT) sStart[i] = fstart[i], sLen[i] = flen[i], sOff[i] = foff[i];
  for (int i = tid; i < n_taps; i += NT) sW[i] = fw[i];
  __syncthreads();

  float vmax = -__builtin_inff();
  float *re = sRe[wave], *im = sIm[wave];
  for (int f = 0; f < kFramesPerWave; ++f) {
    const int fl = wave * kFramesPerWave + f;  // frame within the block
    const int t = t0 + fl;
    if (t >= n_frames) break;  // uniform per wave
    // windowed frame t: padded samples [t*160, t*160 + 512) of the signal
    // reflect-padded by 256 on each side (torch.stft center=True)
    float a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      int64_t u = (int64_t)t * 160 - kFft / 2 + lane + 64 * k;
      u = u < 0 ? -u : (u >= n_samples ? 2 * (n_samples - 1) - u : u);
      a[k] = x[u] * win[k];
    }
    Cplx y[8];
    dft8_real(a, y);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      y[q] = q == 0 ? y[q] : y[q] * tw1[q];
      re[q * 72 + lane] = y[q].re, im[q * 72 + lane] = y[q].im;
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = {re[hi * 72 + lo + 8 * j], im[hi * 72 + lo + 8 * j]};
    wave_lds_sync();
    dft8(y);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      y[s] = s == 0 ? y[s] : y[s] * tw2[s];
      re[(s * 8 + lo) * 9 + hi] = y[s].re, im[(s * 8 + lo) * 9 + hi] = y[s].im;
    }
    wave_lds_sync();
#pragma unroll
    for (int m = 0; m < 8; ++m) y[m] = {re[(hi * 8 + m) * 9 + lo], im[(hi * 8 + m) * 9 + lo]};
    wave_lds_sync();
    dft8(y);
    // power spectrum of bins 0 .. 256, into re[]
#pragma unroll
    for (int u = 0; u < 4; ++u) re[lane + 64 * u] = y[u].re * y[u].re + y[u].im * y[u].im;
    if (lane == 0) re[256] = y[4].re * y[4].re + y[4].im * y[4].im;
    wave_lds_sync();
    for (int m = lane; m < n_mels; m += 64) {
      float acc = 0.f;
      const int st = sStart[m], len = sLen[m], off = sOff[m];
      for (int e = 0; e < len; ++e) acc = __fmaf_rn(sW[off + e], re[st + e], acc);
      const float lv = log10f(fmaxf(acc, 1e-10f));
      sOut[m][fl] = lv;
      vmax = fmaxf(vmax, lv);
    }
    wave_lds_sync();
  }
  // block maximum and the [n_mels][64] rows
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o));
  if (lane == 0) sMax[wave] = vmax;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < kWaves; ++w) vmax = fmaxf(vmax, sMax[w]);
    blockmax[b * gridDim.x + blockIdx.x] = vmax;
  }
  const int nf = min(kFramesPerBlock, n_frames - t0);
  for (int i = tid; i < n_mels * kFramesPerBlock; i += NT) {
    const int m = i / kFramesPerBlock, f = i % kFramesPerBlock;
    if (f < nf) out[b * out_ld_b + (int64_t)m * n_frames + t0 + f] = sOut[m][f];
  }
}

// log_spec = max(log_spec, max(log_spec) - 8) / 4 + 1 over one audio
__global__ __launch_bounds__(256) void logmel_finish_kernel(float *__restrict__ out, int64_t out_ld_b, int64_t count,
                                                            const float *__restrict__ blockmax, int nblk) {
  __shared__ float sM[4];
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x;
  float m = -__builtin_inff();
  for (int i = tid; i < nblk; i += 256) m = fmaxf(m, blockmax[b * nblk + i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((tid & 63) == 0) sM[tid >> 6] = m;
  __syncthreads();
  const float floor8 = __fsub_rn(fmaxf(fmaxf(sM[0], sM[1]), fmaxf(sM[2], sM[3])), 8.0f);
  float *o = out + b * out_ld_b;
  for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < count; i += (int64_t)gridDim.x * 256)
    o[i] = __fadd_rn(__fmul_rn(fmaxf(o[i], floor8), 0.25f), 1.0f);
}

}  // namespace

int launch_log_mel(const float *audio, int64_t batch, int64_t n_samples, int64_t audio_ld, const float *twiddle,
                   const float *window, const int *fstart, const int *flen, const int *foff, const float *fw,
                   int n_taps, int n_mels, float *out, int64_t out_ld_b, float *blockmax, hipStream_t s) {
  const int n_frames = (int)(n_samples / 160);
  const int nblk = (n_frames + kFramesPerBlock - 1) / kFramesPerBlock;
  hipLaunchKernelGGL(logmel_kernel, dim3((unsigned)nblk, (unsigned)batch), dim3(64 * kWaves), 0, s, audio, n_samples,
                     audio_ld, reinterpret_cast<const float2 *>(twiddle), window, fstart, flen, foff, fw, n_taps,
                     n_mels, n_frames, out, out_ld_b, blockmax);
  int rc = check_launch("logmel_kernel");
  if (rc) return rc;
  const int64_t count = (int64_t)n_mels * n_frames;
  hipLaunchKernelGGL(logmel_finish_kernel, dim3(64, (unsigned)batch), dim3(256), 0, s, out, out_ld_b, count,
                     blockmax, nblk);
  return check_launch("logmel_finish_kernel");
}

int log_mel_limits(int *max_mels, int *max_taps) {
  *max_mels = kMaxMels;
  *max_taps = kMaxFilterTaps;
  return 0;
}

}  // namespace iw
