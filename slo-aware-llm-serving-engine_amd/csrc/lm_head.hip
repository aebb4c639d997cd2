// LM head on the sampled rows with the greedy argmax fused in (gfx950).
//
// Replaces compute_logits on hidden.index_select(0, sample_indices) and the
// argmax of run_mixed (nanovllm/engine/mixed_model_runner.py:115-126;
// ParallelLMHead.forward, nanovllm/layers/embed_head.py:56-66, at TP=1):
//   logits[r, v] = bf16(sum_k hidden[r, k] * weight[v, k])   (fp32 sums)
//   token[r]     = the first v with the largest logits[r, v]
// The weight (vocab x hidden, 778 MB for Qwen3-4B) is streamed from HBM once;
// the logits need not be written at all.
//
// Two kernels: lm_head_stream_kernel (see there; up to 64 sampled rows) and
// lm_head_argmax_kernel:
// Workgroup b owns vocab rows [128 b, 128 b + 128): wavefront w the 32 rows
// from 128 b + 32 w, as two 16-row MFMA tiles (v_mfma_f32_16x16x32_bf16, A =
// weight rows, B = hidden^T, so C[vocab][row] leaves every sampled row's
// logits in one lane column).  The hidden rows are staged in LDS 256 or 128
// columns at a time (double-buffered, shared by the 4 wavefronts); each
// wavefront loads the next chunk's weight fragments into registers as soon as
// this chunk's MFMAs have consumed them.  Loads past the last sampled row or
// vocab row repeat the last one, so every lane issues the same loads.  The argmax
// is reduced in registers, across lanes, across wavefronts in LDS, and across
// workgroups with one 64-bit atomicMax per sampled row on the key
// (orderable bf16 bits << 32) | (0xffffffff - v), so the largest value and
// then the smallest index win.  A one-wavefront launch turns the keys into
// token ids and clears them for the next call.
#include <algorithm>
#include <atomic>
#include "common.h"
#include "capi_internal.h"
#include "tile_io.h"

namespace slo {

constexpr int LM_RT = 2;            // 16-row weight tiles per wavefront
constexpr int LM_VT = 64 * LM_RT;   // vocab rows per workgroup
// Hidden columns per chunk for NCT row tiles: 256 (each weight row is then
// read 512 contiguous bytes at a time, measured 3% faster than 256 bytes at 26
// sampled rows), halved until the two LDS buffers of the hidden chunk fit in
// 64 KiB (128 from NCT = 3 on).
constexpr int lm_kc(int nct) {
  int kc = 256;
  while (kc > 128 && 2 * nct * 16 * (kc * 2 + 16) > 65536) kc /= 2;
  return kc;
}

__device__ __forceinline__ uint32_t bf16_order(uint32_t b) { return (b & 0x8000u) ? (b ^ 0xffffu) : (b | 0x8000u); }

// Logits and best keys of a wavefront's 32 vocab rows from vbase on.
template <int NCT>
__device__ __forceinline__ void lm_rank(const f32x4 (&acc)[LM_RT][NCT], int vbase, int M, int V, uint16_t* logits,
                                        int64_t lstride, unsigned long long* best, int n, int g) {
  // Lane (n, g) holds logits of vocab vbase + 16 rt + 4 g + i for sampled row 16 ct + n.
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int row = 16 * ct + n;
    unsigned long long key = 0;
#pragma unroll
    for (int rt = 0; rt < LM_RT; ++rt) {
      const int v0 = vbase + 16 * rt + 4 * g;
      const uint32_t p01 = pack_bf16x2(acc[rt][ct][0], acc[rt][ct][1]);
      const uint32_t p23 = pack_bf16x2(acc[rt][ct][2], acc[rt][ct][3]);
      const uint32_t bits[4] = {p01 & 0xffffu, p01 >> 16, p23 & 0xffffu, p23 >> 16};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (v0 + i >= V) continue;
        const unsigned long long k =
            ((unsigned long long)bf16_order(bits[i]) << 32) | (0xffffffffu - (uint32_t)(v0 + i));
        key = k > key ? k : key;
      }
      if (logits != nullptr && row < M && v0 < V) {
        const int64_t off = (int64_t)row * lstride + v0;
        uint16_t* dst = logits + off;
        if (v0 + 3 < V && (off & 3) == 0) {
          *reinterpret_cast<u32x2*>(dst) = u32x2{p01, p23};
        } else {
          for (int i = 0; i < 4 && v0 + i < V; ++i) dst[i] = (uint16_t)bits[i];
        }
      }
    }
#pragma unroll
    for (int m = 16; m < 64; m <<= 1) {
      const unsigned long long o = __shfl_xor(key, m, 64);
      key = o > key ? o : key;
    }
    if (g == 0) best[row] = key;
  }
}

template <int NCT, int LM_KC = lm_kc(NCT)>  // 16-row tiles of sampled rows, hidden columns per chunk
__global__ void __launch_bounds__(256)
lm_head_argmax_kernel(const uint16_t* __restrict__ hidden, int64_t hstride, int M, const uint16_t* __restrict__ w,
                      int64_t wstride, int V, int H, uint16_t* __restrict__ logits, int64_t lstride,
                      unsigned long long* __restrict__ keys) {
  constexpr int RT = LM_RT;
  constexpr int LM_KS = LM_KC / 32;        // MFMA k-steps per chunk
  constexpr int LM_ROWB = LM_KC * 2 + 16;  // padded LDS row of one hidden chunk (bytes)
  constexpr int HL = NCT * LM_KC / 128;  // 16-byte hidden pieces per thread and chunk
  __shared__ __attribute__((aligned(16))) uint8_t hs[2][NCT * 16 * LM_ROWB];
  __shared__ unsigned long long best[4][NCT * 16];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int vbase = blockIdx.x * LM_VT + wave * 16 * RT;

  // Hidden chunk kc: NCT*16 rows x LM_KC/8 pieces of 16 bytes, spread over the
  // threads, loaded into registers, later written to hs[buf].  Rows past M
  // repeat row M - 1 (their logits are never used), so every lane issues the
  // same loads and the waits stay exact counts.
  auto load_h = [&](int kc, u32x4 (&x)[HL]) {
#pragma unroll
    for (int i = 0; i < HL; ++i) {
      const int c = tid + 256 * i, row = min(c / (LM_KC / 8), M - 1), col = c % (LM_KC / 8);
      x[i] = *reinterpret_cast<const u32x4*>(hidden + row * hstride + kc + 8 * col);
    }
  };
  auto store_h = [&](const u32x4 (&x)[HL], int buf) {
#pragma unroll
    for (int i = 0; i < HL; ++i) {
      const int c = tid + 256 * i;
      *reinterpret_cast<u32x4*>(hs[buf] + (c / (LM_KC / 8)) * LM_ROWB + 16 * (c % (LM_KC / 8))) = x[i];
    }
  };
  // Weight fragments of one chunk: row tile rt, k-step s (32 columns each); a
  // row's LM_KC columns are read by consecutive instructions.
  auto load_a = [&](int kc, u32x4 (&a)[RT][LM_KS]) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int v = vbase + 16 * rt + n;
      const uint16_t* src = w + (int64_t)min(v, V - 1) * wstride + kc + 8 * g;  // rows past V: never ranked
#pragma unroll
      for (int s = 0; s < LM_KS; ++s) a[rt][s] = *reinterpret_cast<const u32x4*>(src + 32 * s);
    }
  };

  f32x4 acc[RT][NCT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = f32x4{0, 0, 0, 0};

  auto mma = [&](const u32x4 (&cur)[RT][LM_KS], int buf) {
#pragma unroll
    for (int s = 0; s < LM_KS; ++s) {
      u32x4 b[NCT];
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
        b[ct] = *reinterpret_cast<const u32x4*>(hs[buf] + (16 * ct + n) * LM_ROWB + 2 * (32 * s + 8 * g));
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = mfma16(as_bf16x8(cur[rt][s]), as_bf16x8(b[ct]), acc[rt][ct]);
    }
  };

  const int nchunks = H / LM_KC;
  u32x4 hx[HL];
  // The next chunk's hidden piece is loaded before this chunk's MFMAs and its
  // weight fragments after them, into the same registers (two register sets
  // measured slower: fewer workgroups per CU).
  u32x4 a0[RT][LM_KS];
  load_a(0, a0);
  load_h(0, hx);
  store_h(hx, 0);
  __syncthreads();
  for (int c = 0; c < nchunks; ++c) {
    const int buf = c & 1;
    const bool more = c + 1 < nchunks;
    if (more) load_h((c + 1) * LM_KC, hx);
    mma(a0, buf);
    if (more) {
      load_a((c + 1) * LM_KC, a0);
      store_h(hx, buf ^ 1);
    }
    __syncthreads();
  }

  lm_rank<NCT>(acc, vbase, M, V, logits, lstride, best[wave], n, g);
  __syncthreads();
  for (int row = tid; row < min(M, NCT * 16); row += 256) {
    unsigned long long key = best[0][row];
#pragma unroll
    for (int q = 1; q < 4; ++q) key = best[q][row] > key ? best[q][row] : key;
    if (key) atomicMax(keys + row, key);
  }
}

// The same product with the weight streamed HBM -> LDS (up to 64 sampled rows).
// The stream is the bound, and a non-temporal LDS-DMA stream that reads every
// 128-byte line in one instruction is the fastest read this GPU has (6.4-6.7
// against 5.6 TB/s); the register fragments above read a line in two
// instructions and lose with that policy (153 -> 180 us at 26 rows of 151,936
// x 2,560).  One persistent workgroup per CU takes the blocks of 128 vocab rows
// blockIdx, blockIdx + grid, ... as one stream of 128-column chunks: 32 weight
// rows (8 KiB) a wavefront and NCT * 4 KiB of hidden rows a workgroup, three
// LDS stages, two chunks in flight also across blocks, one barrier a chunk.
// Rows of both operands are 256 bytes with chunk c of row r in slot
// c ^ (r & 15), so the fragment reads of 16 lanes fall on distinct banks.
constexpr int LS_KC = 128, LS_STAGES = 3;
template <int NCT>
__global__ void __launch_bounds__(256, 1)
lm_head_stream_kernel(const uint16_t* __restrict__ hidden, int64_t hstride, int M, const uint16_t* __restrict__ w,
                      int64_t wstride, int V, int H, uint16_t* __restrict__ logits, int64_t lstride,
                      unsigned long long* __restrict__ keys) {
  constexpr int OPS = 8 + NCT;                   // LDS-DMA loads per wavefront and chunk
  constexpr int WBYTES = LM_VT * 256;            // weight stage: 128 rows of 256 bytes
  constexpr int SBYTES = WBYTES + NCT * 16 * 256;
  __shared__ __attribute__((aligned(16))) uint8_t lds[LS_STAGES * SBYTES];
  __shared__ unsigned long long best[4][NCT * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int blocks = (V + LM_VT - 1) / LM_VT, nchunks = H / LS_KC;
  const uint32_t base = lds_addr(lds);

  // Byte offsets of this lane's rows (weight rows 32 wave + 4 i + g of the
  // block, hidden rows 4 (NCT wave + i) + g), 16-byte chunk n ^ (row & 15).
  uint32_t wo[8], ho[NCT];
#pragma unroll
  for (int i = 0; i < NCT; ++i) {
    const int r = 4 * (NCT * wave + i) + g;
    ho[i] = (uint32_t)min(r, M - 1) * (uint32_t)(2 * hstride) + 16u * (uint32_t)(n ^ (r & 15));
  }
  int pb = blockIdx.x, pc = 0;  // next chunk to request
  const uint8_t* wp = nullptr;
  auto produce = [&](uint32_t dst) -> bool {
    if (pb >= blocks) return false;
    if (pc == 0) {
      // Rows past the vocabulary repeat the last one: never ranked.
      wp = reinterpret_cast<const uint8_t*>(w + (int64_t)pb * LM_VT * wstride);
      const int last = V - 1 - pb * LM_VT;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 32 * wave + 4 * i + g;
        wo[i] = (uint32_t)min(r, last) * (uint32_t)(2 * wstride) + 16u * (uint32_t)(n ^ (r & 15));
      }
    }
    const void* ws = uniform_ptr(wp + 2 * LS_KC * pc);
    const void* hp = uniform_ptr(reinterpret_cast<const uint8_t*>(hidden) + 2 * LS_KC * pc);
#pragma unroll
    for (int i = 0; i < 8; ++i) dma16_nt_at(ws, wo[i], dst + 8192 * wave + 1024 * i);
#pragma unroll
    for (int i = 0; i < NCT; ++i) dma16_at(hp, ho[i], dst + WBYTES + 1024 * (NCT * wave + i));
    if (++pc == nchunks) {
      pc = 0;
      pb += gridDim.x;
    }
    return true;
  };

  produce(base);
  bool ahead = produce(base + SBYTES);  // whether the chunk after the current one is requested
  int st = 0;
  for (int b = blockIdx.x; b < blocks; b += gridDim.x) {
    f32x4 acc[LM_RT][NCT];
#pragma unroll
    for (int rt = 0; rt < LM_RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = f32x4{0, 0, 0, 0};
    for (int c = 0; c < nchunks; ++c) {
      if (ahead) __builtin_amdgcn_s_waitcnt(vmcnt_imm(OPS));
      else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      lds_sync();  // every wavefront's loads of this chunk landed, the stage before it is free
      ahead = produce(base + SBYTES * (st == 0 ? 2 : st - 1));
      const uint8_t* wt = lds + SBYTES * st + 8192 * wave;
      const uint8_t* ht = lds + SBYTES * st + WBYTES;
#pragma unroll
      for (int s = 0; s < LS_KC / 32; ++s) {
        u32x4 a[LM_RT], x[NCT];
#pragma unroll
        for (int rt = 0; rt < LM_RT; ++rt) a[rt] = ld16(wt + rt * 4096 + k_off(n, 4 * s + g));
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) x[ct] = ld16(ht + ct * 4096 + k_off(n, 4 * s + g));
#pragma unroll
        for (int rt = 0; rt < LM_RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = mfma16(as_bf16x8(a[rt]), as_bf16x8(x[ct]), acc[rt][ct]);
      }
      st = st == 2 ? 0 : st + 1;
    }
    lm_rank<NCT>(acc, b * LM_VT + wave * 16 * LM_RT, M, V, logits, lstride, best[wave], n, g);
    lds_sync();
    // (best is written again only after the next block's barriers.)
    for (int row = tid; row < min(M, NCT * 16); row += 256) {
      unsigned long long key = best[0][row];
#pragma unroll
      for (int q = 1; q < 4; ++q) key = best[q][row] > key ? best[q][row] : key;
      if (key) atomicMax(keys + row, key);
    }
  }
}

__global__ void lm_head_tokens_kernel(unsigned long long* __restrict__ keys, int64_t* __restrict__ tokens, int M) {
  for (int r = threadIdx.x; r < M; r += blockDim.x) {
    const unsigned long long k = keys[r];
    tokens[r] = (int64_t)(0xffffffffu - (uint32_t)(k & 0xffffffffu));
    keys[r] = 0;
  }
}

template <int NCT>
void launch_lm(dim3 grid, hipStream_t s, const uint16_t* hidden, int64_t hstride, int M, const uint16_t* w,
               int64_t wstride, int V, int H, uint16_t* logits, int64_t lstride, unsigned long long* keys, int cus) {
  // The stream kernel up to 64 sampled rows (three stages of weight and hidden
  // chunks fit the LDS; row offsets within a block are 32 bits): 151,936 x
  // 2,560 at 1, 26 and 64 rows 139 -> 122, 148 -> 131, 165 -> 145 us; 33,333 x
  // 1,024 at 26 rows 26.6 -> 24.1 us.  Weight rows a multiple of 8 KiB apart
  // put a chunk of every row on the same memory channels, where the register
  // kernel's 512-byte chunks are faster up to 32 sampled rows (151,936 x 4,096
  // at 26 rows 242 against 251 us, 32,000 x 4,096 at one row 61 against 63).
  // Above that it stays faster with rows of exactly 16 KiB, and up to 48 sampled
  // rows of 8 KiB (us, register / stream: 33-48 rows, 32,000 x 4,096 55 / 62,
  // 151,936 x 4,096 255 / 262, 60,000 x 8,192 200 / 237; 49-64 rows, 60,000 x
  // 8,192 228 / 235), and loses beyond (33-48 rows, 60,000 x 12,288 307 / 270,
  // 40,000 x 16,384 328 / 264, 40,000 x 20,480 450 / 351; 49-64 rows, 151,936 x
  // 4,096 279 / 271, 60,000 x 12,288 325 / 281).
  if constexpr (NCT <= 4) {
    const bool same_channels =
        wstride % 4096 == 0 && (NCT <= 2 || wstride == 8192 || (NCT == 3 && wstride == 4096));
    if (wstride < (1 << 23) && hstride < (1 << 23) && !same_channels) {
      const dim3 sgrid(std::min<unsigned>(grid.x, (unsigned)cus));
      hipLaunchKernelGGL((lm_head_stream_kernel<NCT>), sgrid, dim3(256), 0, s, hidden, hstride, M, w, wstride, V, H,
                         logits, lstride, keys);
      return;
    }
  }
  if (H % lm_kc(NCT) == 0)
    hipLaunchKernelGGL((lm_head_argmax_kernel<NCT, lm_kc(NCT)>), grid, dim3(256), 0, s, hidden, hstride, M, w, wstride, V,
                       H, logits, lstride, keys);
  else
    hipLaunchKernelGGL((lm_head_argmax_kernel<NCT, 128>), grid, dim3(256), 0, s, hidden, hstride, M, w, wstride, V, H,
                       logits, lstride, keys);
}

}  // namespace slo

using namespace slo;

extern "C" int slo_lm_head_argmax(const void* hidden, int64_t hidden_row_stride, int32_t num_rows, const void* weight,
                                  int64_t weight_row_stride, int32_t vocab_size, int32_t hidden_size, void* logits,
                                  int64_t logits_row_stride, uint64_t* keys, int64_t* tokens, slo_stream_t stream) {
  if (num_rows < 0 || vocab_size <= 0 || hidden_size <= 0) return fail(SLO_ERR_INVALID, "lm_head_argmax: bad sizes");
  if (num_rows > 128) return fail(SLO_ERR_UNSUPPORTED, "lm_head_argmax: at most 128 sampled rows per call");
  if (hidden_size % 128) return fail(SLO_ERR_UNSUPPORTED, "lm_head_argmax: hidden_size must be a multiple of 128");
  if (num_rows == 0) return SLO_OK;
  if (!hidden || !weight || !keys || !tokens) return fail(SLO_ERR_INVALID, "lm_head_argmax: null pointer");
  if ((hidden_row_stride % 8) || (weight_row_stride % 8) || hidden_row_stride < hidden_size ||
      weight_row_stride < hidden_size || (reinterpret_cast<uintptr_t>(hidden) % 16) ||
      (reinterpret_cast<uintptr_t>(weight) % 16) || (reinterpret_cast<uintptr_t>(keys) % 8))
    return fail(SLO_ERR_INVALID, "lm_head_argmax: rows must be 16-byte aligned");
  if (logits && (logits_row_stride < vocab_size || (reinterpret_cast<uintptr_t>(logits) % 8)))
    return fail(SLO_ERR_INVALID, "lm_head_argmax: logits must be 8-byte aligned with rows of at least vocab_size");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((vocab_size + LM_VT - 1) / LM_VT);
  const auto* h16 = static_cast<const uint16_t*>(hidden);
  const auto* w16 = static_cast<const uint16_t*>(weight);
  auto* l16 = static_cast<uint16_t*>(logits);
  auto* k64 = reinterpret_cast<unsigned long long*>(keys);
  static std::atomic<int> cu_count[64];  // per device, 0 until asked
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return fail(SLO_ERR_HIP, "lm_head_argmax: hipGetDevice failed");
  int cus = cu_count[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return fail(SLO_ERR_HIP, "lm_head_argmax: hipDeviceGetAttribute failed");
    cu_count[dev].store(cus, std::memory_order_relaxed);
  }
  switch ((num_rows + 15) / 16) {
    case 1: launch_lm<1>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 2: launch_lm<2>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 3: launch_lm<3>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 4: launch_lm<4>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 5: launch_lm<5>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 6: launch_lm<6>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    case 7: launch_lm<7>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
    default: launch_lm<8>(grid, s, h16, hidden_row_stride, num_rows, w16, weight_row_stride, vocab_size, hidden_size, l16, logits_row_stride, k64, cus); break;
  }
  int rc = check_launch("lm_head_argmax");
  if (rc) return rc;
  hipLaunchKernelGGL(lm_head_tokens_kernel, dim3(1), dim3(128), 0, s, k64, tokens, num_rows);
  return check_launch("lm_head_tokens");
}
