// Forward for a few query rows per sequence against many keys (decoding a token, or a handful of drafted ones): every key
// and value is read once and used for at most 32 query rows, so the kernel is a stream of K and V through the chip and what
// bounds it is HBM.  fa_fwd_kernel is the wrong shape for that: its workgroup owns 128 query rows, of which one wave's 32
// hold all there is, the other three waves only help with the staging, and every tile is a workgroup barrier.
//
// Here the waves of a workgroup own keys, not rows: wave w takes the 32-key tiles w, w + NW, ... of the workgroup's share
// of the keys, stages them into a double buffer of its own with direct-to-LDS loads (one tile is always in flight while
// the one before it is used) and never meets another wave before the end, when the NW partial (maximum, sum, output)
// triples are merged through LDS.  All products are MFMAs in the forward kernel's orientation (S^T = K Q^T, O^T = V^T P^T):
// the up to 32 query rows are the 32 columns, so one row costs what 32 do and the matrix work stays far below the stream.
// Two waves (four at d <= 32): two stages of a (K, V) tile pair per wave are then 64 KB a workgroup at d = 128, and two
// workgroups a compute unit keep up to 128 KB in flight; at d = 64 (32 KB) four waves took 8.3 us where two take 6.1 (1024
// pairs with 70 keys) and 73.5 against 76.5 where every stream is long (2000 keys).  Measured with the merge, inputs that change from
// call to call, bf16, one new token, us of fa_fwd_kernel with its own split / here: 8 sequences of 1024 to 4096 keys, 16 heads, d = 128 (168 MB) 96.6 /
// 42.8 (the kernel alone 38.8: FETCH_SIZE gives K and V once, 4.3 TB/s); all of 5000 keys 122.8 / 66.2 (5.0 TB/s, what a large copy reaches), of 12000
// 288 / 144 (5.5 TB/s).
#include "fa_params.h"
#include "fa_stage.h"

namespace fa {

namespace {

template <int D>
struct DecodeCfg {
  static constexpr int NW = kDecodeWaves(D);
  static constexpr int BN = 32;
  static constexpr int DV = D < 32 ? 32 : D;
  static constexpr int CH = D / 8;
  static constexpr int RPI = 64 / CH;             // tile rows per direct-to-LDS instruction
  static constexpr int NI = BN / RPI;             // instructions per tile and tensor
  static constexpr int NOFF = 16 / RPI > 0 ? 16 / RPI : 1;  // distinct source offsets (swizzle period 16 rows)
  static constexpr int kTile = BN * D * 2;
  static constexpr int kWave = 2 * 2 * kTile;     // two stages of (K tile, V tile)
  static constexpr int kSlack = D < 32 ? 64 : 0;  // the 32-wide transposed reads run past a 16-wide V row
  static constexpr int XS = DV + 4;               // merge: floats per (wave, query row)
  static constexpr int kMerge = NW * 32 * XS * 4 + 2 * NW * 32 * 4;
  static constexpr int kTiles = NW * kWave + kSlack;
  static constexpr int kLds = kTiles > kMerge ? kTiles : kMerge;
};

template <int N>
FA_DEVICE void wait_vmcnt() {  // at most N of this wave's global loads (direct-to-LDS ones included) are still outstanding
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

}  // namespace

template <typename T, int D>
__global__ void __launch_bounds__(64 * DecodeCfg<D>::NW) fa_decode_kernel(const FwdParams p) {
  using Cfg = DecodeCfg<D>;
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  constexpr int NW = Cfg::NW, BN = Cfg::BN, DV = Cfg::DV, NI = Cfg::NI;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[Cfg::kLds];

  // heads innermost: the workgroups that run at one time read neighbouring rows of a (token, head, d) cache; the first
  // splits of all sequences come first, the ones that may lie past a sequence's end last
  const int h = blockIdx.x % p.H;
  const int b = (blockIdx.x / p.H) % p.B;
  const int split = blockIdx.x / (p.H * p.B);
  int q_begin, Lq, k_begin = 0, Lk = 0;
  if (!seq_extent(p.cu_q, b, p.total_q, p.max_sq, &q_begin, &Lq)) return;
  if (!seq_extent(p.cu_k, b, p.total_k, p.max_sk, &k_begin, &Lk)) Lk = 0;  // no keys: o = 0, lse = -inf
  const int k_lo = split * p.split_keys;
  if (split > 0 && k_lo >= Lk) return;  // (the combine kernel knows how many splits a sequence has)
  const int k_hi = Lk - k_lo < p.split_keys ? Lk : k_lo + p.split_keys;
  const int ntiles = (k_hi - k_lo + BN - 1) / BN;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hf = lane >> 5;

  vec8 qreg[D / 16];
  {
    const int qr = c < Lq ? c : Lq - 1;  // (columns past the last row repeat it and are dropped at the end)
    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)(q_begin + qr) * p.q_rs + (int64_t)h * p.q_hs + hf * 8;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++) qreg[ks] = bitcast<vec8>(ld_global16(qp + ks * 16));
  }

  // ---- staging (see fa_stage.h): this wave's tiles only
  const char* const kb = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.k) + (int64_t)(k_begin + k_lo) * p.k_rs + (int64_t)h * p.k_hs);
  const char* const vb = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.v) + (int64_t)(k_begin + k_lo) * p.v_rs + (int64_t)h * p.v_hs);
  const int64_t krsb = p.k_rs * 2, vrsb = p.v_rs * 2;
  const int rl = lane / Cfg::CH, pch = lane % Cfg::CH;
  uint32_t koff_g[Cfg::NOFF], voff_g[Cfg::NOFF];
#pragma unroll
  for (int j = 0; j < Cfg::NOFF; j++) {
    koff_g[j] = (uint32_t)(rl * krsb) + 16u * (uint32_t)(pch ^ tile_swz<D, kSwzRow>(j * Cfg::RPI + rl));
    voff_g[j] = (uint32_t)(rl * vrsb) + 16u * (uint32_t)(pch ^ tile_swz<D, kSwzTr>(j * Cfg::RPI + rl));
  }
  unsigned char* const lds_wave = lds_raw + wave * Cfg::kWave;
  auto issue_one = [&](const char* base, int64_t rsb, const uint32_t (&off)[Cfg::NOFF], bool is_v, int r0, unsigned char* dst) {
    const int valid = k_hi - k_lo - r0;  // rows of the tile that exist
    const char* const tb = base + (int64_t)r0 * rsb;
    if (__builtin_expect(valid >= BN, 1)) {
#pragma unroll
      for (int i = 0; i < NI; i++) dma16(tb + i * Cfg::RPI * rsb, off[i % Cfg::NOFF], dst + i * 1024);
    } else {  // rows past the end repeat the last one: LDS holds tensor data only, their scores are masked
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const int r = i * Cfg::RPI + rl;
        const int rc = r < valid ? r : valid - 1;
        const int swz = is_v ? tile_swz<D, kSwzTr>(r) : tile_swz<D, kSwzRow>(r);
        dma16(tb, (uint32_t)(rc * rsb) + 16u * (uint32_t)(pch ^ swz), dst + i * 1024);
      }
    }
  };
  auto issue = [&](int t, int stage) {
    unsigned char* const dst = lds_wave + stage * 2 * Cfg::kTile;
    issue_one(kb, krsb, koff_g, false, t * BN, dst);
    issue_one(vb, vrsb, voff_g, true, t * BN, dst + Cfg::kTile);
  };

  int koff[D / 16], voff[DV / 32];
#pragma unroll
  for (int ks = 0; ks < D / 16; ks++) koff[ks] = frag_off<D, kSwzRow>(c, ks * 2 + hf);
#pragma unroll
  for (int db = 0; db < DV / 32; db++) voff[db] = tr_off<D, kSwzTr>(0, db * 4, lane);

  f32x16 o_acc[DV / 32];
#pragma unroll
  for (int i = 0; i < DV / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) o_acc[i][r] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;  // l_i: this lane's share, the other half's in lane ^ 32
  const float cs = p.scale_log2;

  int t = wave, stage = 0;
  if (t < ntiles) issue(t, 0);
  if (t + NW < ntiles) issue(t + NW, 1);
  if (p.rot_cos != nullptr) {  // rotary embedding of the queries, as in fa_fwd_kernel: turned here, left in q_rot once
    const int row = c < Lq ? c : Lq - 1, tr = row < p.rot_rows ? row : p.rot_rows - 1;
    const T* const ct = reinterpret_cast<const T*>(p.rot_cos) + (int64_t)tr * (D / 2) + hf * 4;
    const T* const st = reinterpret_cast<const T*>(p.rot_sin) + (int64_t)tr * (D / 2) + hf * 4;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++)
      qreg[ks] = rotate8<T>(qreg[ks], *reinterpret_cast<const typename E::vec4*>(ct + ks * 8),
                            *reinterpret_cast<const typename E::vec4*>(st + ks * 8), false);
    if (p.q_rot != nullptr && wave == 0 && split == 0 && c < Lq) {
      T* const qo = reinterpret_cast<T*>(p.q_rot) + (int64_t)(q_begin + c) * p.qr_rs + (int64_t)h * p.qr_hs + hf * 8;
#pragma unroll
      for (int ks = 0; ks < D / 16; ks++) st_global16(qo + ks * 16, bitcast<u32x4>(qreg[ks]));
    }
    wait_vmcnt<0>();  // (the main loop counts this wave's outstanding accesses: these are not to be among them)
  }
  for (; t < ntiles; t += NW) {
    const bool next = t + NW < ntiles;  // its 2 * NI loads were issued after this tile's
    if (next) wait_vmcnt<3 * NI>();
    else wait_vmcnt<NI>();
    const T* const Ks = reinterpret_cast<const T*>(lds_wave + stage * 2 * Cfg::kTile);
    const T* const Vs = Ks + BN * D;
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++) s = E::mfma32(*reinterpret_cast<const vec8*>(Ks + koff[ks]), qreg[ks], s);
    const int n0 = k_lo + t * BN;
    if (n0 + BN > k_hi) {
#pragma unroll
      for (int r = 0; r < 16; r++)
        if (n0 + 8 * (r >> 2) + 4 * hf + (r & 3) >= k_hi) s[r] = -INFINITY;
    }
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mt = fmaxf(mt, s[r]);
    mt = half_max(mt);
    if (__any(mt > m_i)) {
      const float m_new = fmaxf(m_i, mt);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2((m_i - m_new) * cs);
      m_i = m_new;
      l_i *= alpha;
#pragma unroll
      for (int i = 0; i < DV / 32; i++) o_acc[i] = o_acc[i] * alpha;
    }
    const float mc = (m_i == -INFINITY ? 0.f : m_i) * cs;
    vec8 pb[2];
#pragma unroll
    for (int tt = 0; tt < 2; tt++) {
      f32x8 pf;
#pragma unroll
      for (int i = 0; i < 8; i++) pf[i] = fast_exp2(__builtin_fmaf(s[8 * tt + i], cs, -mc));
      pb[tt] = cvt8<T>(pf);
      l_i = sum8_acc(pb[tt], l_i);
    }
    if (next) wait_vmcnt<2 * NI>();
    else wait_vmcnt<0>();
#pragma unroll
    for (int tt = 0; tt < 2; tt++)
#pragma unroll
      for (int db = 0; db < DV / 32; db++) {
        const T* vp = Vs + 16 * tt * D + voff[db];
        const u32x2 lo = lds_read_tr16(vp), hi = lds_read_tr16(vp + 8 * D);
        o_acc[db] = E::mfma32(bitcast<vec8>(u32x4{lo[0], lo[1], hi[0], hi[1]}), pb[tt], o_acc[db]);
      }
    if (t + 2 * NW < ntiles) {
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stage has been read before it is refilled
      issue(t + 2 * NW, stage);
    }
    stage ^= 1;
  }

  // ---- merge the waves' partial results: row q of wave w at X[(w * 32 + q) * XS], its maximum and sum behind all rows
  __syncthreads();
  float* const X = reinterpret_cast<float*>(lds_raw);
  float* const Xm = X + NW * 32 * Cfg::XS;
  float* const Xl = Xm + NW * 32;
  l_i = half_sum(l_i);
  if (c < Lq) {
    if (hf == 0) {
      Xm[wave * 32 + c] = m_i;
      Xl[wave * 32 + c] = l_i;
    }
#pragma unroll
    for (int db = 0; db < DV / 32; db++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = o_acc[db][g4 * 4 + i];
        *reinterpret_cast<f32x4*>(X + (wave * 32 + c) * Cfg::XS + db * 32 + g4 * 8 + hf * 4) = x;
      }
  }
  __syncthreads();
  for (int idx = tid; idx < Lq * (D / 4); idx += 64 * NW) {
    const int q = idx / (D / 4), d0 = idx % (D / 4) * 4;
    float m = Xm[q];
#pragma unroll
    for (int w = 1; w < NW; w++) m = fmaxf(m, Xm[w * 32 + q]);
    const float mu = m == -INFINITY ? 0.f : m;
    float l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = fast_exp2((Xm[w * 32 + q] - mu) * cs);  // 0 for a wave without keys
      l = __builtin_fmaf(Xl[w * 32 + q], f, l);
      o = o + *reinterpret_cast<const f32x4*>(X + (w * 32 + q) * Cfg::XS + d0) * f;
    }
    const bool empty = !(l > 0.f);
    o = o * (empty ? 1.f : fast_rcp(l));
    const float lse = empty ? -INFINITY : (m * cs + fast_log2(l)) * kLn2;
    if (p.n_splits > 1) {
      if (d0 == 0) p.lse_part[(((int64_t)split * p.B + b) * p.H + h) * p.sq_r + q] = lse;
      *reinterpret_cast<f32x4*>(p.o_part + (((int64_t)split * p.total_q + q_begin + q) * p.H + h) * D + d0) = o;
    } else {
      if (d0 == 0) p.lse[((int64_t)b * p.H + h) * p.sq_r + q] = lse;
      T* const op = reinterpret_cast<T*>(p.o) + (int64_t)(q_begin + q) * p.o_rs + (int64_t)h * p.o_hs + d0;
      *reinterpret_cast<typename E::vec4*>(op) = cvt4<T>(o);
    }
  }
}

namespace {
template <typename T>
hipError_t launch_decode_t(const FwdParams& p, int head_dim, hipStream_t stream) {
  const int grid = p.B * p.H * (p.n_splits > 1 ? p.n_splits : 1);
  switch (head_dim) {
    case 16: hipLaunchKernelGGL((fa_decode_kernel<T, 16>), dim3(grid), dim3(64 * DecodeCfg<16>::NW), 0, stream, p); break;
    case 32: hipLaunchKernelGGL((fa_decode_kernel<T, 32>), dim3(grid), dim3(64 * DecodeCfg<32>::NW), 0, stream, p); break;
    case 64: hipLaunchKernelGGL((fa_decode_kernel<T, 64>), dim3(grid), dim3(64 * DecodeCfg<64>::NW), 0, stream, p); break;
    case 128: hipLaunchKernelGGL((fa_decode_kernel<T, 128>), dim3(grid), dim3(64 * DecodeCfg<128>::NW), 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_decode(const FwdParams& p, int dtype, int head_dim, hipStream_t stream) {
  return dtype == 0 ? launch_decode_t<_Float16>(p, head_dim, stream) : launch_decode_t<__bf16>(p, head_dim, stream);
}

}  // namespace fa
