// Dense causal per-block attention mass for gfx950 (CDNA4): the teacher that
// SelectOracle selects from.
//
//   mass[b, h, i, j] = mean over the query rows t of block i of
//                      sum over the keys s of block j, s <= t, of softmax_s(S[t, :])
//   S[t, s]          = rnd(rnd(q_t . k_s) * scale)  (rounded to the operand dtype,
//                      as torch rounds a 16-bit matmul and the scale multiply)
//
// with the softmax in fp32 (src/eval_qwen_ppl.py:65-108, capture_mass; the
// group mean over each KV head's query heads is left to the caller, as there).
//
// The scores are formed once. One workgroup per (b, query head, query block),
// one wave per 32 query rows (two 16-row operand fragments, so each K fragment
// read from LDS feeds two products), K tiles through a direct-to-LDS ring. Each
// row keeps a reference score (a running maximum moved only when it is exceeded
// by 8 log2 units) and its sum of exp(S - reference); at the end of every key
// block the block's sums and the references they were formed under (scores, so
// exact in 16 bits) go to the workspace. Once a row's total is known, the
// workgroup reads them back and forms
//   mass[i, j] = 1/BS sum_t sum[t, j] * exp(reference[t, j] - reference[t]) / total[t].
// That traffic is 6 bytes per (row, key block) each way against BS x D products
// per pair. The second pass over all scores that it replaces (row log-sum-exp
// first, then the normalised sums) took as long as the first.
// Measured (bf16, 16384 tokens, 16 query heads over 2 KV heads, d 256, blocks of
// 128): 3.98 ms for two passes of 16-row waves, 1.11 ms now (0.99 PFLOP/s of the
// causal products against 1.26 that a 8192^3 library product reaches on the card).
#include "fbsa_common.h"
#include "fbsa_internal.h"

namespace fbsa {

struct MassArgs {
  const void *q, *k;
  float *mass;  // (B, Hq, nblk, nblk)
  char *ws;     // one slot of slot_bytes per workgroup of this launch
  int64_t B, Hq, Hkv, L, nblk;
  int64_t sq[3], sk[3];
  int64_t first;       // launch-order index of the launch's first workgroup
  int64_t slot_rows;   // (row, key block) entries of a slot
  float scale;
  int grp;
};

template <typename T, int BS, int D> struct MassCfg {
  static constexpr int QT = 2;  // 16-row query fragments per wave
  static constexpr int NW = BS / (16 * QT);
  static constexpr int NT = NW * 64;
  static constexpr int KC = D >= 256 ? 32 : 64;  // keys per chunk
  static constexpr int NCH = BS / KC;
  static constexpr int CPR = D * 2 / 16;
  static constexpr int TILE_BYTES = KC * D * 2;
  static constexpr int LPT = TILE_BYTES / (NT * 16);
  static constexpr int NSTAGE = 3;
  static constexpr int LDS_BYTES = NSTAGE * TILE_BYTES + 2 * BS * 4;
  static_assert(LPT * NT * 16 == TILE_BYTES, "tile must split evenly over threads");
  static_assert(KC <= BS, "chunk larger than a block");
};

constexpr float kMassSlack = 8.f;  // log2 units by which a score may pass its row's reference

template <typename T> __device__ __forceinline__ float round_to_t(float x) { return (float)(T)x; }

// Launch order: query blocks with the longest walks first; the query heads of a
// KV group back to back on one XCD (they read the same K tiles).
__host__ __device__ inline int64_t mass_block_of_unit(int64_t unit, int64_t bh, int64_t nblk) {
  return nblk - 1 - unit / bh;
}

// FOLD: bf16 with a power-of-two scale. Multiplying by it is exact, so the
// second rounding returns its argument and the scale joins the exponent's
// factor (a product too small for a normal bf16 leaves exp(S) at 1 either way).
template <typename T, int BS, int D, bool FOLD>
__global__ __launch_bounds__(BS * 2) void mass_kernel(MassArgs a) {
  using C = MassCfg<T, BS, D>;
  constexpr int QT = C::QT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char *stages = smem;
  float *s_ref = (float *)(smem + C::NSTAGE * C::TILE_BYTES);  // [BS] final reference (times the exponent factor)
  float *s_inv = s_ref + BS;                                   // [BS] 1 / (BS * total)

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4,
            p = lane & 15;
  int hin;
  const int64_t bh = a.B * a.Hkv;
  const int64_t unit = gqa_unit(a.first + blockIdx.x, bh * a.nblk, a.grp, &hin);
  const int i = (int)mass_block_of_unit(unit, bh, a.nblk);
  const int hk = (int)(unit % bh % a.Hkv), hq = hk * a.grp + hin;
  const int64_t b = unit % bh / a.Hkv;
  float *sums = (float *)(a.ws + (int64_t)blockIdx.x * a.slot_rows * 6);
  T *refs = (T *)(sums + a.slot_rows);

  // Q fragments (B operands of S^T = K Q^T): lane (p, g) holds q[row][32 ks + 8 g .. + 7]
  // of rows 32 w + 16 n + p, n < QT
  s16x8 qf[QT][D / 32];
#pragma unroll
  for (int n = 0; n < QT; ++n) {
    const T *qr = (const T *)a.q + b * a.sq[0] + hq * a.sq[1] + ((int64_t)i * BS + 16 * (QT * w + n) + p) * a.sq[2];
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) qf[n][ks] = *(const s16x8 *)(qr + 32 * ks + 8 * g);
  }

  // direct-to-LDS plan: per-lane byte offsets of this thread's LPT loads of a K chunk
  int32_t koff[C::LPT];
#pragma unroll
  for (int n = 0; n < C::LPT; ++n) {
    const int u = (n * C::NW + w) * 64 + lane;
    const int row = u / C::CPR, pos = u % C::CPR;
    koff[n] = (int32_t)(((int64_t)row * a.sk[2] + (pos ^ swz(row, C::CPR)) * 8) * 2);
  }
  const char *knext = (const char *)((const T *)a.k + b * a.sk[0] + hk * a.sk[1]);  // next chunk to issue
  const int64_t kstep = (int64_t)C::KC * a.sk[2] * 2;
  const int nchunks = (i + 1) * C::NCH;
  int ist = 0;  // its stage
  auto issue = [&]() {
    char *st = stages + ist * C::TILE_BYTES;
#pragma unroll
    for (int n = 0; n < C::LPT; ++n) g2lds16(knext + koff[n], st + (n * C::NW + w) * 1024);
    knext += kstep;
    ist = ist + 1 == C::NSTAGE ? 0 : ist + 1;
  };
#pragma unroll
  for (int c = 0; c < C::NSTAGE - 1; ++c)
    if (c < nchunks) issue();
  // the register-operand loads above and the first stages have landed (issued
  // together, so their latencies overlap): the compiler then waits for nothing
  // inside the ring loop, where its own waits would also drain the prefetch
  wait_vmcnt<0>();

  // exponent of a score: exp2(S * cexp + nref), nref = -reference * cexp (0 while the
  // row has seen nothing above -inf, so that those keys add exp2(-inf) = 0)
  const float cexp = FOLD ? a.scale * kLog2e : kLog2e;
  const float slack = kMassSlack / cexp;
  float ref[QT], lim[QT], nref[QT], tot[QT], bsum[QT];
#pragma unroll
  for (int n = 0; n < QT; ++n) {
    ref[n] = lim[n] = -INFINITY;
    nref[n] = tot[n] = bsum[n] = 0.f;
  }
  int c = 0, cst = 0;  // chunk and its stage
  auto chunk = [&](auto MASKED, int ch) {
    constexpr bool masked = decltype(MASKED)::value;
    const int ahead = nchunks - 1 - c;
    wait_ring<C::LPT>(ahead < C::NSTAGE - 2 ? ahead : C::NSTAGE - 2);
    lds_barrier();  // chunk c landed for every wave; chunk c-1's stage is free
    if (c + C::NSTAGE - 1 < nchunks) issue();
    const char *Ks = stages + cst * C::TILE_BYTES;
    ++c;
    cst = cst + 1 == C::NSTAGE ? 0 : cst + 1;
    constexpr int NM = C::KC / 16, KL = D / 32 < 4 ? D / 32 : 4;
    float x[QT][NM][4];
    const char *kb[KL];
#pragma unroll
    for (int l = 0; l < KL; ++l) kb[l] = Ks + tile_kbase(l, g, p, C::CPR);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      f32x4 acc[QT];
#pragma unroll
      for (int n = 0; n < QT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks) {
        const s16x8 kf = *(const s16x8 *)(kb[ks % 4] + (ks / 4) * 256 + m * 256 * C::CPR);
#pragma unroll
        for (int n = 0; n < QT; ++n) acc[n] = Mfma16<T>::run(kf, qf[n][ks], acc[n]);
      }
      // lane (p, g) holds keys 16 m + 4 g + r of the chunk for the rows 16 n + p
#pragma unroll
      for (int n = 0; n < QT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = round_to_t<T>(acc[n][r]);
          if constexpr (!FOLD) v = round_to_t<T>(v * a.scale);
          if constexpr (masked)
            if (ch * C::KC + 16 * m + 4 * g + r > 16 * (QT * w + n) + p) v = -INFINITY;  // key after the query
          x[n][m][r] = v;
        }
    }
    bool over = false;
    float cm[QT];
#pragma unroll
    for (int n = 0; n < QT; ++n) {
      cm[n] = x[n][0][0];
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) cm[n] = fmaxf(cm[n], x[n][m][r]);
      over |= cm[n] > lim[n];
    }
    if (__any(over)) {
#pragma unroll
      for (int n = 0; n < QT; ++n) {
        // a row's keys are spread over the lanes p, p + 16, p + 32, p + 48
        float rm = fmaxf(cm[n], __shfl_xor(cm[n], 16, 64));
        rm = fmaxf(rm, __shfl_xor(rm, 32, 64));
        if (rm > lim[n]) {
          const float f = __builtin_amdgcn_exp2f((ref[n] - rm) * cexp);  // 0 from -inf
          tot[n] *= f;
          bsum[n] *= f;
          ref[n] = rm;
          lim[n] = rm + slack;
          nref[n] = -rm * cexp;
        }
      }
    }
#pragma unroll
    for (int n = 0; n < QT; ++n)
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          bsum[n] += __builtin_amdgcn_exp2f(__builtin_fmaf(x[n][m][r], cexp, nref[n]));
  };
  // the sums of key block j, and the references they were formed under
  auto flush = [&](int j) {
    float v[QT];
#pragma unroll
    for (int n = 0; n < QT; ++n) {
      tot[n] += bsum[n];
      v[n] = bsum[n] + __shfl_xor(bsum[n], 16, 64);
      v[n] += __shfl_xor(v[n], 32, 64);
      bsum[n] = 0.f;
    }
    if (g < QT) {
      const int64_t at = (int64_t)j * BS + 16 * (QT * w + g) + p;
      sums[at] = g ? v[1] : v[0];
      refs[at] = (T)(g ? ref[1] : ref[0]);
    }
  };
  for (int j = 0; j < i; ++j) {
#pragma unroll 1
    for (int ch = 0; ch < C::NCH; ++ch) chunk(std::false_type{}, ch);
    flush(j);
  }
#pragma unroll 1
  for (int ch = 0; ch < C::NCH; ++ch) chunk(std::true_type{}, ch);
  flush(i);

#pragma unroll
  for (int n = 0; n < QT; ++n) {
    float t = tot[n] + __shfl_xor(tot[n], 16, 64);
    t += __shfl_xor(t, 32, 64);
    if (g == n) {
      s_ref[16 * (QT * w + n) + p] = ref[n];
      s_inv[16 * (QT * w + n) + p] = (1.f / BS) / t;
    }
  }
  __syncthreads();  // every wave's totals are in LDS and its sums in memory
  constexpr int RPL = BS / 64;  // rows per lane
  float fref[RPL], finv[RPL];
#pragma unroll
  for (int e = 0; e < RPL; ++e) {
    fref[e] = s_ref[RPL * lane + e];
    finv[e] = s_inv[RPL * lane + e];
  }
  const int64_t rowoff = ((b * a.Hq + hq) * a.nblk + i) * a.nblk;
  for (int j = w; j <= i; j += C::NW) {
    float v = 0.f;
#pragma unroll
    for (int e = 0; e < RPL; ++e) {
      const int64_t at = (int64_t)j * BS + RPL * lane + e;
      v += sums[at] * finv[e] * __builtin_amdgcn_exp2f(((float)refs[at] - fref[e]) * cexp);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) a.mass[rowoff + j] = v;
  }
  for (int64_t jj = i + 1 + tid; jj < a.nblk; jj += C::NT) a.mass[rowoff + jj] = 0.f;  // above the diagonal
}

// Workspace: every workgroup's sums and references, up to kMassSlots bytes (and
// at least kMassMin workgroups); a longer sequence runs in several launches,
// each over the workgroups whose slots fit.
constexpr int64_t kMassSlots = (int64_t)1 << 30;
constexpr int64_t kMassMin = 256;
static int64_t mass_slot_rows(const fbsa_attn_desc *d, int64_t first) {
  // the longest walk from launch index `first` on (a round of 8 units runs together)
  const int64_t grp = d->Hq / d->Hkv;
  return (mass_block_of_unit(first / (8 * grp) * 8, d->B * d->Hkv, d->nblk) + 1) * d->bs;
}
size_t mass_workspace_bytes(const fbsa_attn_desc *d) {
  const int64_t n = d->B * d->Hq * d->nblk, slot = mass_slot_rows(d, 0) * 6;
  const int64_t most = kMassSlots / slot > kMassMin ? kMassSlots / slot : kMassMin;
  return (size_t)((n < most ? n : most) * slot);
}

template <typename T, int BS, int D, bool FOLD> static int launch_mass(MassArgs a, const fbsa_attn_desc *d, hipStream_t s) {
  using C = MassCfg<T, BS, D>;
  int e = lds_optin((const void *)mass_kernel<T, BS, D, FOLD>, C::LDS_BYTES, "hipFuncSetAttribute(mass)");
  if (e) return e;
  const int64_t n = a.B * a.Hq * a.nblk, ws = (int64_t)mass_workspace_bytes(d);
  for (a.first = 0; a.first < n;) {
    a.slot_rows = mass_slot_rows(d, a.first);
    int64_t nwg = ws / (a.slot_rows * 6);
    if (nwg > n - a.first) nwg = n - a.first;
    hipLaunchKernelGGL((mass_kernel<T, BS, D, FOLD>), dim3((unsigned)nwg), dim3(C::NT), C::LDS_BYTES, s, a);
    e = hip_check(hipGetLastError(), "mass_kernel launch");
    if (e) return e;
    a.first += nwg;
  }
  return FBSA_OK;
}

template <typename T, int BS, int D> static int mass_fold(const MassArgs &a, const fbsa_attn_desc *d, hipStream_t s) {
  if constexpr (__is_same(T, bf16)) {
    int ex;
    if (a.scale >= 0x1p-60f && a.scale <= 1.f && frexpf(a.scale, &ex) == 0.5f)
      return launch_mass<T, BS, D, true>(a, d, s);
  }
  return launch_mass<T, BS, D, false>(a, d, s);
}

template <typename T, int BS> static int mass_d(const MassArgs &a, const fbsa_attn_desc *d, hipStream_t s) {
  switch (d->D) {
    case 64: return mass_fold<T, BS, 64>(a, d, s);
    case 128: return mass_fold<T, BS, 128>(a, d, s);
    case 256: return mass_fold<T, BS, 256>(a, d, s);
  }
  return fail(FBSA_EUNSUPPORTED, "fbsa_block_mass: head dim %lld not in {64,128,256}", (long long)d->D);
}

template <typename T> static int mass_bs(const MassArgs &a, const fbsa_attn_desc *d, hipStream_t s) {
  switch (d->bs) {
    case 64: return mass_d<T, 64>(a, d, s);
    case 128: return mass_d<T, 128>(a, d, s);
  }
  return fail(FBSA_EUNSUPPORTED, "fbsa_block_mass: block size %lld not in {64,128}", (long long)d->bs);
}

int run_block_mass(const fbsa_attn_desc *d, const void *q, const void *k, float *mass, void *ws, hipStream_t s) {
  MassArgs a;
  a.q = q; a.k = k; a.mass = mass; a.ws = (char *)ws;
  a.B = d->B; a.Hq = d->Hq; a.Hkv = d->Hkv; a.L = d->L; a.nblk = d->nblk;
  for (int x = 0; x < 3; ++x) { a.sq[x] = d->sq[x]; a.sk[x] = d->sk[x]; }
  a.scale = d->scale;
  a.grp = (int)(d->Hq / d->Hkv);
  if (d->dtype == FBSA_BF16) return mass_bs<bf16>(a, d, s);
  if (d->dtype == FBSA_F16) return mass_bs<f16>(a, d, s);
  return fail(FBSA_EUNSUPPORTED, "fbsa_block_mass: 16-bit operands only (bf16, f16)");
}

}  // namespace fbsa
