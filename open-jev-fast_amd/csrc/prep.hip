// The two consumers of the in-projection output that forward_gtree calls by default: the full-attention prep and
// the linear-attention prep on the tree layout. Both give every wave a piece of a token row that it reads, finishes
// and writes out by itself, with whole 8- or 16-byte vector stores.
#include "ojx_internal.h"

#include <algorithm>

namespace ojx {

namespace {

__device__ __forceinline__ void unpack8(uint4 a, float (&v)[8]) {
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[2 * j] = bf2f(w[j] & 0xffffu);
    v[2 * j + 1] = bf2f(w[j] >> 16);
  }
}

// Store of a lane's 16 bytes; NT: non-temporal, past the caches.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ void store16(uint16_t* dst, uint4 v) {
  if constexpr (NT) __builtin_nontemporal_store(__builtin_bit_cast(u32x4, v), reinterpret_cast<u32x4*>(dst));
  else *reinterpret_cast<uint4*>(dst) = v;
}

}  // namespace

// ------------------------------------------------------------------------------------------------ full attention
// Reference behaviour: fullattn_prep2 (src/kernels.cu:302-355), called from forward_gtree as
// K.fullattn_prep2(proj, qw1, kw1, cos, sin, 1, N, HQ, HKV, D, eps) (src/fastmodel.py:462). proj [N, P] bf16 with
// P = HQ 2D + 2 HKV D; for token n:
//   q head h: x = proj[n][2hD .. 2hD+D), gate head h = proj[n][2hD+D .. 2hD+2D);
//   k head h: x = proj[n][2 HQ D + hD ..); v head h = proj[n][2 HQ D + HKV D + hD ..).
//   q and k: xn = bf16((x * rsqrt(sum x^2 / D + eps)) * w1[d]) with w1 = qw1 / kw1 [D] fp32, then on the first RD
//   dims the rotate-half RoPE: out = bf16(bf16(xn * cos[n][d]) + bf16(rh * sin[n][d])), rh = -xn[d + RD/2] for
//   d < RD/2 and xn[d - RD/2] for RD/2 <= d < RD; dims >= RD keep xn.
//   Outputs: qt [HQ, N, D], kt [HKV, N, D], vt [HKV, N, D] (head-major for attention) and gate [N, HQ D].
//
// Work layout: half a wave per (token, head task), eight tasks per workgroup. Task t of a token: t < HQ the q head t
// (the half wave also copies gate head t), HQ <= t < HQ + HKV the k head t - HQ, then the v heads (copies). Lane l of
// the 32 owns dims 8l .. 8l+7: one 16-byte load and store each, 512 contiguous bytes per head. A q/k head's sum of
// squares is five shuffles; the rotary partner dims d -+ RD/2 are all held by lane l ^ (RD / 16) (RD is 16 times a
// power of two), so the exchange is a shuffle of the eight values: no LDS, no barrier.
// What bounds it: the launch up to a few hundred tokens, then its bytes. Graph replays over rotating inputs, an
// earlier kernel (a wave of 8-byte lanes per task, the partner through LDS) -> this one: M = 288 6.5 -> 6.1 us, M =
// 539 11.4 -> 9.6, M = 1024 17.7 -> 14.9 (4.0 TB/s), M = 2048 31.6 -> 24.2 (4.8 TB/s).
// Its stores are ordinary ones. Non-temporal stores make the prep itself up to 1.3 us shorter, but the attention's
// reads then miss the caches: with a kernel that reads the four outputs behind it, M = 7 10.8 -> 11.6 us, M = 539 26.0
// -> 27.1, M = 1024 31.9 -> 33.9, M = 2048 48.3 -> 54.0; with the projection in front as well M = 288 73.4 -> 73.4, M
// = 1024 156.0 -> 158.0, M = 2048 301.2 -> 304.3.
__global__ void __launch_bounds__(256) fullattn_prep_k(const uint16_t* __restrict__ proj, int64_t N, int HQ, int HKV,
                                                       int RD, float eps, const float* __restrict__ qw1,
                                                       const float* __restrict__ kw1, const uint16_t* __restrict__ cosb,
                                                       const uint16_t* __restrict__ sinb, uint16_t* __restrict__ qt,
                                                       uint16_t* __restrict__ kt, uint16_t* __restrict__ vt,
                                                       uint16_t* __restrict__ gate) {
  constexpr int D = 256;
  const int l = threadIdx.x & 31;
  const int T = HQ + 2 * HKV, G = (T + 7) >> 3;  // tasks per token, workgroups per token
  const int64_t n = blockIdx.x / G;
  const int t = (int)(blockIdx.x - n * G) * 8 + (threadIdx.x >> 5);
  if (t >= T) return;  // whole half wave; the shuffles below stay within one
  const int64_t P = (int64_t)(2 * HQ + 2 * HKV) * D;
  const uint16_t* row = proj + n * P;
  const int d0 = l * 8;
  if (t >= HQ + HKV) {  // v head: a copy into [HKV, N, D]
    const int hv = t - HQ - HKV;
    *reinterpret_cast<uint4*>(vt + ((int64_t)hv * N + n) * D + d0) =
        *reinterpret_cast<const uint4*>(row + (int64_t)(2 * HQ + HKV) * D + hv * D + d0);
    return;
  }
  const bool isq = t < HQ;
  const uint4 xa = *reinterpret_cast<const uint4*>(
      row + (isq ? (int64_t)t * 2 * D : (int64_t)2 * HQ * D + (int64_t)(t - HQ) * D) + d0);
  if (isq)  // gate head: a copy into [N, HQ D]
    *reinterpret_cast<uint4*>(gate + n * (int64_t)(HQ * D) + t * D + d0) =
        *reinterpret_cast<const uint4*>(row + (int64_t)t * 2 * D + D + d0);
  const float* w1 = (isq ? qw1 : kw1) + d0;
  const float4 wa = *reinterpret_cast<const float4*>(w1), wb = *reinterpret_cast<const float4*>(w1 + 4);
  const bool rot = d0 < RD;
  uint4 ca = make_uint4(0u, 0u, 0u, 0u), sa = ca;
  if (rot) {
    ca = *reinterpret_cast<const uint4*>(cosb + n * RD + d0);
    sa = *reinterpret_cast<const uint4*>(sinb + n * RD + d0);
  }
  float x[8];
  unpack8(xa, x);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) ss += __shfl_xor(ss, o);
  const float r = rsqrtf(ss / (float)D + eps);
  const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = rbf((x[j] * r) * wv[j]);
  float cs[8], sn[8];
  unpack8(ca, cs);
  unpack8(sa, sn);
  const bool lo = d0 < RD / 2;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float pv = __shfl_xor(x[j], RD / 16);  // every lane of the half wave takes part
    o[j] = rot ? rbf(rbf(x[j] * cs[j]) + rbf((lo ? -pv : pv) * sn[j])) : x[j];
  }
  uint16_t* dst = isq ? qt + ((int64_t)t * N + n) * D : kt + ((int64_t)(t - HQ) * N + n) * D;
  *reinterpret_cast<uint4*>(dst + d0) =
      make_uint4(pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7]));
}

hipError_t launch_fullattn_prep(const uint16_t* proj, int64_t N, int HQ, int HKV, int RD, float eps,
                                const float* qw1, const float* kw1, const uint16_t* cosb, const uint16_t* sinb,
                                uint16_t* qt, uint16_t* kt, uint16_t* vt, uint16_t* gate, hipStream_t st) {
  const int64_t G = (HQ + 2 * HKV + 7) / 8;
  hipLaunchKernelGGL(fullattn_prep_k, dim3((unsigned)(N * G)), dim3(256), 0, st, proj, N, HQ, HKV, RD, eps, qw1, kw1,
                     cosb, sinb, qt, kt, vt, gate);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------ linear attention
// Reference behaviour: linattn_prep_dedup2 (src/kernels.cu:1176-1265), called from forward_gtree as
// K.linattn_prep_dedup2(proj, lay.hist, lay.rep_ptr, lay.rep_pos, lay.L2, convw, A_log, dt_bias, KD, VD, HV, HK, HD,
// rep_qk) (src/fastmodel.py:420,438). proj [N, P] bf16, P = C + VD + 2 HV with C = 2 KD + VD conv channels
// (q | k | v), then the z gate (VD, read later by the gated norm), then b [HV] and a [HV]. Each packed row n is
// computed once and written to every slot s = rep_pos[p], p in [rep_ptr[n], rep_ptr[n+1]) (the candidate paths that
// contain it); the slots of group N (rep_ptr[N] .. rep_ptr[N+1]) are the paths' end padding and receive zeros.
//   channel c: conv = sum_{i=0..3} convw[c][i] * proj[hist[n][i]][c], added in that order (hist[n] = the rows
//   t-3 .. t on the row's path, -1 = none); o = bf16(silu(conv)). q and k channels (c < 2 KD) are then
//   L2-normalised over their head of HD = 128 channels: bf16(o * (1 / sqrt(sum o^2 + 1e-6))).
//   head h < HV: beta = bf16(sigmoid(b_h)), g = -exp(A_log[h]) * softplus(a_h + dt_bias[h]) (fp32, softplus(x) = x
//   above 20), b and a read from row hist[n][3].
//   Outputs: q, k [R, HK RQ HD] (RQ = 1, or 3 = HV / HK copies of each head side by side), v [R, VD], g [R, HV] fp32,
//   beta [R, HV] bf16; R = rep_pos's length.
// Products of two bf16 values are exact in fp32, so the conv's sum order is the only one that fixes its bits; it is
// kept. The head sums of squares are added in another order than the reference's (one rounding step at most).
//
// Work layout: one wave per (row, 512 channels), eight consecutive channels per lane; four consecutive rows of one
// channel block per workgroup, so that the block's weights and the rows' shared history come from L1 after the first
// wave. A lane keeps its finished channels as one 16-byte value in registers and stores it to every slot of the row:
// 1 KB contiguous per wave and slot, slot ids fetched 64 at a time beside the row's loads and read lane by lane (a
// uniform address per store). A head of 128 channels is 16 lanes, so its sum of squares is four shuffles. No LDS and
// no barrier: the waves are independent, where an earlier kernel of one workgroup per row (about one workgroup per CU
// on a 288-row tree) exposed every latency of its conv -> barrier -> norm -> barrier -> write chain. One more channel
// block, the last, computes the gates. The row groups after the rows write zeros to the padding slots, kPadGroups
// slots at a time.
// What bounds it: the slot rows written, once a tree has a few hundred slots (below that, the launch and one chain of
// loads). The channel blocks of a row are neighbouring workgroups, so that its 20 KB of each slot go out at about the
// same time. Graph replays on MI355X over rotating inputs, earlier kernel -> this one, and the algorithmic rate: 200
// shared rows x 8 paths 15.8 -> 10.3 us (4.2 TB/s), 480 x 8 26.3 -> 20.6 (4.6 TB/s), 1500 x 16 125.3 -> 99.6 (5.4
// TB/s).
// NT, non-temporal slot stores, from 256 MB of outputs on (what the Infinity Cache holds). Below, the next kernel
// finds much of the slots there after ordinary stores and none of them after non-temporal ones; above, it misses
// either way and the stores are faster. Prep and a kernel that reads its outputs, ordinary -> non-temporal: 200 x 8
// (37 MB) 32.8 -> 36.8 us, 480 x 8 (82 MB) 54.8 -> 64.8, 900 x 8 (154 MB) 93.6 -> 107.6, 900 x 12 (231 MB) 150.4 ->
// 149.7, 900 x 16 (308 MB) 189.7 -> 188.0 (with the projection in front 369.5 -> 359.7), 1500 x 16 (505 MB) 299.2 ->
// 294.3.
constexpr int kLinRows = 4;      // rows (waves) per workgroup
constexpr int kPadGroups = 256;  // padding slots written at a time
constexpr int64_t kNtBytes = 256LL << 20;  // outputs of this size and more go past the caches

// Calls put(s) for each of the slots rep_pos[p0], rep_pos[p0 + step], ... below p1; sid holds the first 64 of them,
// one per lane. Every lane of the wave takes part.
template <typename F>
__device__ __forceinline__ void each_slot(const int* __restrict__ rep_pos, int p0, int p1, int step, int sid, F put) {
  const int lane = threadIdx.x & 63;
  for (int base = p0; base < p1; base += 64 * step) {
    const int cnt = min(64, (p1 - base + step - 1) / step);
    if (base != p0) sid = lane < cnt ? rep_pos[base + lane * step] : 0;
    for (int j = 0; j < cnt; ++j) put((int64_t)__builtin_amdgcn_readlane(sid, j));
  }
}

template <int RQ, bool NT>
__global__ void __launch_bounds__(64 * kLinRows) linattn_prep_k(
    const uint16_t* __restrict__ proj, const int4* __restrict__ hist, const int* __restrict__ rep_ptr,
    const int* __restrict__ rep_pos, const uint16_t* __restrict__ convw, const uint16_t* __restrict__ A_log,
    const uint16_t* __restrict__ dt_bias, uint16_t* __restrict__ q, uint16_t* __restrict__ k,
    uint16_t* __restrict__ v, float* __restrict__ g, uint16_t* __restrict__ beta, int N, int KD, int VD, int HV,
    int rg0) {
  constexpr int HD = 128;
  const int C = 2 * KD + VD;
  const int64_t P = (int64_t)C + VD + 2 * HV;
  const int lane = threadIdx.x & 63;
  const int rb = (N + kLinRows - 1) / kLinRows;  // row groups; padding groups follow
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = (C / 8 + 63) / 64 + 1;           // channel blocks of a row, the gates last
  const int rgl = blockIdx.x / T, cb = blockIdx.x - rgl * T, rg = rg0 + rgl;  // this launch starts at row group rg0
  const bool pad = rg >= rb;
  const int n = pad ? N : rg * kLinRows + wave;
  if (n >= N && !pad) return;
  int p0 = rep_ptr[n], step = 1;
  const int p1 = rep_ptr[n + 1];
  if (pad) {
    p0 += (rg - rb) * kLinRows + wave;
    step = kPadGroups;
  }
  if (p0 >= p1) return;  // whole wave
  const int sid = p0 + lane * step < p1 ? rep_pos[p0 + lane * step] : 0;
  const int4 hr = hist[n];  // row N holds no history

  if (cb == T - 1) {  // the gates
    for (int h0 = 0; h0 < HV; h0 += 64) {
      const int h = h0 + lane;
      const bool on = h < HV;
      float gv = 0.f;
      uint16_t bv = 0;
      if (on && !pad) {
        const uint16_t* br = proj + (int64_t)hr.w * P + C + VD;
        bv = (uint16_t)f2bf(sigmoid_f(bf2f(br[h])));
        const float xs = bf2f(br[HV + h]) + bf2f(dt_bias[h]);
        gv = -expf(bf2f(A_log[h])) * (xs > 20.f ? xs : log1pf(expf(xs)));
      }
      each_slot(rep_pos, p0, p1, step, sid, [&](int64_t s) {
        if (on) {
          g[s * HV + h] = gv;
          beta[s * HV + h] = bv;
        }
      });
    }
    return;
  }

  const int c0 = (cb * 64 + lane) * 8;
  const bool live = c0 < C;
  const bool isqk = c0 < 2 * KD;  // the same for all 16 lanes of a head (KD is a multiple of HD)
  uint4 val = make_uint4(0u, 0u, 0u, 0u);
  if (live && !pad) {
    const int rows[4] = {hr.x, hr.y, hr.z, hr.w};
    uint4 xr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      xr[i] = rows[i] >= 0 ? *reinterpret_cast<const uint4*>(proj + (int64_t)rows[i] * P + c0)
                           : make_uint4(0u, 0u, 0u, 0u);
    const uint4* wp = reinterpret_cast<const uint4*>(convw + (int64_t)c0 * 4);  // [8 channels][4 taps]
    const uint4 wq[4] = {wp[0], wp[1], wp[2], wp[3]};
    const uint32_t* wv = &wq[0].x;
    float o[8];
    float ss = 0.f;
#pragma unroll
    for (int ch = 0; ch < 8; ++ch) {
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t* xw = &xr[i].x;
        const float xv = bf2f((xw[ch >> 1] >> ((ch & 1) * 16)) & 0xffffu);
        const int wi = ch * 4 + i;
        const float wf = bf2f((wv[wi >> 1] >> ((wi & 1) * 16)) & 0xffffu);
        acc += wf * xv;
      }
      o[ch] = rbf(silu_f(acc));
      ss += o[ch] * o[ch];
    }
    if (isqk) {
#pragma unroll
      for (int off = 1; off < HD / 8; off <<= 1) ss += __shfl_xor(ss, off);
      const float rs = 1.0f / sqrtf(ss + 1e-6f);
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) o[ch] *= rs;
    }
    val = make_uint4(pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7]));
  }
  // the lane's place in a slot's row: q / k rows hold each head RQ times side by side
  const int64_t ld = isqk ? (int64_t)RQ * KD : VD;
  const int cq = c0 < KD ? c0 : c0 - KD;
  uint16_t* const dst = isqk ? (c0 < KD ? q : k) + (cq / HD) * (RQ * HD) + cq % HD : v + (c0 - 2 * KD);
  each_slot(rep_pos, p0, p1, step, sid, [&](int64_t s) {
    if (!live) return;
    uint16_t* const d = dst + s * ld;
    store16<NT>(d, val);
    if (RQ > 1 && isqk) {
#pragma unroll
      for (int r = 1; r < RQ; ++r) store16<NT>(d + r * HD, val);
    }
  });
}

hipError_t launch_linattn_prep(const uint16_t* proj, const int32_t* hist, const int32_t* rep_ptr,
                               const int32_t* rep_pos, int64_t N, int64_t R, const uint16_t* convw,
                               const uint16_t* A_log, const uint16_t* dt_bias, int KD, int VD, int HV, int RQ,
                               uint16_t* q, uint16_t* k, uint16_t* v, float* g, uint16_t* beta, hipStream_t st) {
  const int C = 2 * KD + VD;
  const int64_t T = (C / 8 + 63) / 64 + 1, groups = (N + kLinRows - 1) / kLinRows + kPadGroups / kLinRows;
  const bool nt = R * (2LL * (2 * RQ * (int64_t)KD + VD) + 6LL * HV) >= kNtBytes;
  const auto kernel = RQ == 3 ? (nt ? linattn_prep_k<3, true> : linattn_prep_k<3, false>)
                              : (nt ? linattn_prep_k<1, true> : linattn_prep_k<1, false>);
  // A launch has fewer than 2^32 threads: row groups beyond that (rows in the millions) go in further launches.
  const int64_t per = ((1LL << 32) - 1) / (64 * kLinRows * T);
  for (int64_t g0 = 0; g0 < groups; g0 += per) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(std::min(per, groups - g0) * T)), dim3(64 * kLinRows), 0, st, proj,
                       reinterpret_cast<const int4*>(hist), rep_ptr, rep_pos, convw, A_log, dt_bias, q, k, v, g, beta,
                       (int)N, KD, VD, HV, (int)g0);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace ojx
