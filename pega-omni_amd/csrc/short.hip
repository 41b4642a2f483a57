// Head-64 attentions over short rings (gfx950, wave64): the Mimi codec
// transformer's ring attention and the rotary + ring write before it, the
// Qwen3-TTS codec decoder's fused rotary + ring write + attention, and the
// PersonaPlex depformer's fused K/V write + causal attention.
//
//   mimi_rope_kv64      crates/omni-personaplex/kernels/mimi.cu:226-246
//   mimi_attend64       crates/omni-personaplex/kernels/mimi.cu:248-263
//   codec_attention64   crates/omni-qwen3-tts/kernels/codec.cu:168-277
//   dep_kv_attend64     crates/omni-personaplex/kernels/lm.cu:314-366
//
// One wave per (row, head), eight per (rows of a session, head) for Mimi's
// rings. Lane l holds dims 8c .. 8c + 7 (c = l % 8, one
// 16-byte load of a 128-byte K or V row) of key row r = l / 8, so one load
// instruction covers 8 keys; scores are 8-lane DPP sums and the softmax runs
// online in base 2 with the scale folded into q. The key a fused kernel has
// just produced (the current frame or step) stays in each lane's registers
// and replaces the loaded value by a select, so no lane reads memory another
// lane of the same kernel has just written.
#include "common.h"
#include "kernels.h"

namespace omni {

namespace {

constexpr int kD = 64;
constexpr int kCodecWindow = 72;
constexpr int kDepSteps = 8;

__device__ __forceinline__ float row8_sum64(float v) {
  v += dpp<kQuadSwap1>(v);
  v += dpp<kQuadSwap2>(v);
  v += dpp<kRowHalfMirror>(v);
  return v;
}

// Combine the 8 key rows of the wave (lanes 8 apart), per lane.
template <bool MAX>
__device__ __forceinline__ float across_rows8(float v) {
  v = MAX ? fmaxf(v, dpp<kRowRor8>(v)) : v + dpp<kRowRor8>(v);
  v = MAX ? fmaxf(v, xor_lane(v, 16)) : v + xor_lane(v, 16);
  v = MAX ? fmaxf(v, xor_lane(v, 32)) : v + xor_lane(v, 32);
  return v;
}

__device__ __forceinline__ uint4 pack8(const float* v) {
  return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                    pack_bf16x2(v[6], v[7]));
}

// Online-softmax state of one (row, head) spread over the wave.
struct Row64 {
  float q[8];  // q dims 8c .. 8c + 7, times scale * log2(e)
  float m, l, acc[8];

  __device__ void init(const float* qv, float scale) {
    const float s = scale * kLog2e;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[e] = qv[e] * s;
      acc[e] = 0.f;
    }
    m = -INFINITY;
    l = 0.f;
  }

  // The K and V rows of keys tb .. tb + 8 NI - 1 (clamped to len - 1): key
  // row r = lane / 8 of load i is key tb + 8 i + r.
  template <int NI>
  struct Tile {
    uint4 kr[NI], vr[NI];
  };
  template <int NI, class KV>
  __device__ static void load(Tile<NI>& x, int tb, int len, const KV& kv) {
    const int lane = threadIdx.x & 63, r = lane >> 3, c = lane & 7;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int t = min(tb + 8 * i + r, len - 1);
      x.kr[i] = ldg16(kv.k(t) + 8 * c);
      x.vr[i] = ldg16(kv.v(t) + 8 * c);
    }
  }

  // Online softmax over one loaded tile; key `cur` (if in it) comes from
  // (cur_k, cur_v) instead of memory.
  template <int NI>
  __device__ void step(Tile<NI>& x, int tb, int len, int cur, const uint4& cur_k, const uint4& cur_v) {
    const int lane = threadIdx.x & 63, r = lane >> 3;
    float sc[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int t = tb + 8 * i + r;
      if (t == cur) {
        x.kr[i] = cur_k;
        x.vr[i] = cur_v;
      }
      float kf[8];
      widen8(x.kr[i], kf);
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) d = fmaf(q[e], kf[e], d);
      d = row8_sum64(d);
      sc[i] = t < len ? d : -INFINITY;
    }
    float mx = sc[0];
#pragma unroll
    for (int i = 1; i < NI; ++i) mx = fmaxf(mx, sc[i]);
    mx = across_rows8<true>(mx);
    const float mn = fmaxf(m, mx);
    const float corr = fast_exp2(m - mn);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= corr;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float p = fast_exp2(sc[i] - mn);
      ps += p;
      float vf[8];
      widen8(x.vr[i], vf);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(p, vf[e], acc[e]);
    }
    l = fmaf(l, corr, ps);
  }

  // Sum the 8 key rows and write dims 8c .. 8c + 7 (lanes of key row 0).
  __device__ void finish(bf16_t* out) {
    const int lane = threadIdx.x & 63, c = lane & 7;
    const float lt = across_rows8<false>(l);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = across_rows8<false>(acc[e]) / lt;
    if (lane < 8) *reinterpret_cast<uint4*>(out + 8 * c) = pack8(o);
  }
};

// ----------------------------------------------------------------- Mimi ring
// Slots of one session's ring. A row at position p sees slots
// (p - len + 1 + t) % context, t < len = min(p + 1, context): slots 0 .. len - 1
// whether the ring has wrapped (all of them) or not, so the keys are walked in
// slot order and the rows of one session see nested sets of slots.
//
// TR consecutive rows of one session (TR divides T) and one head per workgroup:
// each K and V row is read once for the TR rows, and eight waves of two loads
// of 8 slots each cover 128 slots per memory round trip (two for a full
// 250-slot ring) where one wave per (row, head) walked it in sixteen. Bound by
// those round trips in small batches and by memory in large ones. One frame of
// eight layers at T = 2 with its codec and depformer calls, as a replayed
// graph: 32 sessions 166 -> 79 us, 128 sessions 211 -> 152 us. Waves x loads
// per trip, 4 / 32 / 128 sessions: 8 x 2 63 / 79 / 152, 4 x 4 66 / 83 / 150,
// 8 x 4 61 / 80 / 180, 4 x 8 64 / 83 / 196 us (more loads per trip cost
// registers, and so occupancy); one row per workgroup 58-60 / 91-95 / 199-209;
// two heads per workgroup (256-byte runs) 71 / 85 / 153 us.
//
// Few workgroups take one row each (kMimiAlone): a pair's code is twice as long
// and its call 0.6 us longer at the least, and CUs that would idle read the K and
// V rows again. us per layer, pairs / single rows, 8 heads, T = 2, positions
// 3-400 (0-7): 1 session 3.25 / 2.67 (3.23 / 2.63), 8 5.6 / 4.8 (3.35 / 2.82), 16
// (256 workgroups) 5.8 / 5.3 (3.56 / 2.83), 24 6.1 / 6.7 (3.7 / 3.0), 32 6.3 / 7.7
// (3.7 / 3.0), 128 14.2 / 20.0 (7.1 / 4.9).
// A context of at most one wave's slots takes one wave: context 8, 32 sessions
// 3.65 -> 2.68, 128 6.97 -> 3.79. One wave per (row, head) throughout would take
// 3.0 and 3.8 us for 32 and 128 sessions that are all at positions 0-7, where
// pairs take 3.7 and 7.1, but 13.4 and 20.8 at positions 3-400, and a call lasts
// as long as its longest ring. (Ending the waves that have no slots at once: 128
// sessions at 0-7 5.2, all other calls 3-5% longer.)
constexpr int kMimiWaves = 8;
constexpr int kMimiLoads = 2;
constexpr int kMimiAlone = 256;  // workgroups of one row: one per CU

template <int TR, int W = kMimiWaves>
__global__ __launch_bounds__(64 * W) void mimi_attend64(ShortArgs a) {
  constexpr int NI = kMimiLoads, R = 8;  // R slots per load instruction
  const int n0 = blockIdx.x * TR, h = blockIdx.y;
  const int lane = threadIdx.x & 63, c = lane & 7, r = lane >> 3;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = n0 / a.T;
  const int p0 = a.pos[s] * a.T + n0 % a.T;
  float q[TR][8], m[TR], l[TR], acc[TR][8];
  int len[TR];
#pragma unroll
  for (int j = 0; j < TR; ++j) {
    widen8(ldg16(a.qkv + ((int64_t)min(n0 + j, a.rows - 1) * 3 * a.heads + h) * kD + 8 * c), q[j]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[j][e] *= a.scale * kLog2e;
      acc[j][e] = 0.f;
    }
    m[j] = -INFINITY;
    l[j] = 0.f;
    len[j] = min(p0 + j + 1, a.context);
  }
  const int64_t width = (int64_t)a.heads * kD;  // elements of a slot's K (and V) heads
  const bf16_t* kb = reinterpret_cast<const bf16_t*>(static_cast<const uint8_t*>(a.state) +
                                                     (int64_t)a.lines[s] * a.stride) + h * kD + 8 * c;
  const int slots = len[TR - 1];
  for (int tb = wave * R * NI; tb < slots; tb += W * R * NI) {
    uint4 kr[NI], vr[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const bf16_t* at = kb + (int64_t)min(tb + R * i + r, slots - 1) * 2 * width;
      kr[i] = ldg16_stream(at);
      vr[i] = ldg16_stream(at + width);
    }
#pragma unroll
    for (int j = TR - 1; j >= 0; --j) {
      if (tb >= len[j]) continue;
      // A lane past the row's slots (one that only a later row of the session
      // sees, or past the last): its p is 0 here, and the V row it holds must not
      // reach the sum (0 times an infinity would).
      if (tb + R * NI > len[j]) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
          if (tb + R * i + r >= len[j]) vr[i] = uint4{};
      }
      float sc[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        float kf[8];
        widen8(kr[i], kf);
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d = fmaf(q[j][e], kf[e], d);
        d = row8_sum64(d);
        sc[i] = tb + R * i + r < len[j] ? d : -INFINITY;
      }
      float mx = sc[0];
#pragma unroll
      for (int i = 1; i < NI; ++i) mx = fmaxf(mx, sc[i]);
      mx = across_rows8<true>(mx);
      const float mo = m[j];
      m[j] = fmaxf(mo, mx);
      // Slots whose scores are all -inf (infinite keys) weigh 0: -inf less -inf
      // would make this wave's share NaN beside another wave's finite one.
      const float mn = m[j] == -INFINITY ? 0.f : m[j];
      const float corr = fast_exp2(mo - mn);
      float ps = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[j][e] *= corr;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const float p = fast_exp2(sc[i] - mn);
        ps += p;
        float vf[8];
        widen8(vr[i], vf);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[j][e] = fmaf(p, vf[e], acc[j][e]);
      }
      l[j] = fmaf(l[j], corr, ps);
    }
  }
  // Merge the waves (a wave whose slots lie past the row's has m = -inf, l = 0).
  __shared__ float sm_m[TR][W], sm_l[TR][W], sm_o[TR][W][kD];
#pragma unroll
  for (int j = 0; j < TR; ++j) {
    l[j] = across_rows8<false>(l[j]);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[j][e] = across_rows8<false>(acc[j][e]);
    if (r == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sm_o[j][wave][8 * c + e] = acc[j][e];
      if (c == 0) {
        sm_m[j][wave] = m[j];
        sm_l[j][wave] = l[j];
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TR * kD; i += 64 * W) {
    const int d = i % kD, j = i / kD;
    if (n0 + j >= a.rows) break;
    float top = sm_m[j][0];
#pragma unroll
    for (int w = 1; w < W; ++w) top = fmaxf(top, sm_m[j][w]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float e = sm_m[j][w] == -INFINITY ? 0.f : fast_exp2(sm_m[j][w] - top);
      num = fmaf(sm_o[j][w][d], e, num);
      den = fmaf(sm_l[j][w], e, den);
    }
    a.out[((int64_t)(n0 + j) * a.heads + h) * kD + d] = (bf16_t)f2bf(num / den);
  }
}

// Mimi's rotary + ring write: row n of session s = n / T at p = pos[s] T +
// n % T. One 256-thread workgroup per row; the row's 32 angles (pair i turns
// by p exp(i coef), computed with expf and sincosf as the reference does) go
// to LDS once. Thread u takes the 16-byte chunk u % 8 (dims 8c .. 8c + 7,
// interleaved pairs 4c .. 4c + 3) of head u / 8 of [q | k | v]: q heads are
// turned in place, k heads turned into ring slot p % context (its K heads),
// v heads copied there (its V heads), each rotated value rounded to bf16.
__global__ __launch_bounds__(256) void mimi_rope_kv64(ShortArgs a) {
  const int n = blockIdx.x, s = n / a.T;
  const int p = a.pos[s] * a.T + n % a.T;
  __shared__ float s_cos[kD / 2], s_sin[kD / 2];
  if (threadIdx.x < kD / 2) {
    const float freq = expf((float)threadIdx.x * a.coef);
    sincosf(freq * (float)p, &s_sin[threadIdx.x], &s_cos[threadIdx.x]);
  }
  __syncthreads();
  bf16_t* row = a.qkv_rw + (int64_t)n * 3 * a.heads * kD;
  bf16_t* slot = reinterpret_cast<bf16_t*>(static_cast<uint8_t*>(a.state) + (int64_t)a.lines[s] * a.stride) +
                 (int64_t)(p % a.context) * 2 * a.heads * kD;
  for (int u = threadIdx.x; u < 3 * a.heads * 8; u += blockDim.x) {
    const int hh = u >> 3, c = u & 7;
    const uint4 w = ldg16(row + hh * kD + 8 * c);
    if (hh >= 2 * a.heads) {  // v: copied into the slot's V heads
      *reinterpret_cast<uint4*>(slot + (int64_t)(hh - a.heads) * kD + 8 * c) = w;
      continue;
    }
    float x[8], y[8];
    widen8(w, x);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float cs = s_cos[4 * c + j], sn = s_sin[4 * c + j];
      y[2 * j] = x[2 * j] * cs - x[2 * j + 1] * sn;
      y[2 * j + 1] = x[2 * j] * sn + x[2 * j + 1] * cs;
    }
    bf16_t* dst = hh < a.heads ? row + hh * kD : slot + (int64_t)(hh - a.heads) * kD;
    *reinterpret_cast<uint4*>(dst + 8 * c) = pack8(y);
  }
}

// ------------------------------------------------------ Qwen3-TTS codec ring
struct CodecRing {
  const bf16_t* ring;  // K[72][width] then V[72][width]
  int first, width, h;
  __device__ const bf16_t* k(int t) const { return ring + (int64_t)((first + t) % kCodecWindow) * width + h * kD; }
  __device__ const bf16_t* v(int t) const {
    return ring + ((int64_t)kCodecWindow + (first + t) % kCodecWindow) * width + h * kD;
  }
};

__global__ __launch_bounds__(64) void codec_attention64(ShortArgs a) {
  const int r = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63, c = lane & 7;
  const int width = a.heads * kD;
  const bf16_t* row = a.qkv + (int64_t)r * 3 * width + h * kD;
  bf16_t* ring = reinterpret_cast<bf16_t*>(static_cast<uint8_t*>(a.state) + (int64_t)a.lines[r] * a.stride);
  const int p = a.pos[r];
  const int n = min(p + 1, kCodecWindow);
  // The whole window (at most 72 keys, 9 rows of 8) is loaded first, in one
  // round trip that overlaps the rotary below. The slot of frame p, written
  // below, reads stale here and is replaced by the registers' values.
  const CodecRing kv{ring, p - n + 1, width, h};
  Row64::Tile<kCodecWindow / 8> win;
  Row64::load(win, 0, n, kv);

  // Half-split rotary of q and k at p: pair i = dims i, i + 32; lane c holds
  // dims 8c .. 8c + 7, whose partners are in lane c ^ 4.
  float qk[2][8];
  widen8(ldg16(row + 8 * c), qk[0]);
  widen8(ldg16(row + width + 8 * c), qk[1]);
  const uint4 cur_v = ldg16(row + 2 * width + 8 * c);
  // The 32 angles once, one pair per lane, through LDS.
  __shared__ float s_cos[kD / 2], s_sin[kD / 2];
  if (lane < kD / 2) {
    const float inv_freq = 1.f / powf(a.theta, (float)(2 * lane) / kD);
    sincosf((float)p * inv_freq, &s_sin[lane], &s_cos[lane]);
  }
  __syncthreads();
  const bool lo = c < 4;
  float rot[2][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int i = 8 * (c & 3) + e;
    const float cs = s_cos[i], sn = s_sin[i];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const float partner = xor_lane(qk[w][e], 4);
      rot[w][e] = lo ? qk[w][e] * cs - partner * sn : qk[w][e] * cs + partner * sn;
    }
  }
  const uint4 qb = pack8(rot[0]), cur_k = pack8(rot[1]);  // both rounded to bf16
  float qv[8];
  widen8(qb, qv);
  if (lane < 8) {  // frame p % 72 of the ring: the rotated k and the v row
    const int64_t at = (int64_t)(p % kCodecWindow) * width + h * kD + 8 * c;
    *reinterpret_cast<uint4*>(ring + at) = cur_k;
    *reinterpret_cast<uint4*>(ring + (int64_t)kCodecWindow * width + at) = cur_v;
  }
  Row64 st;
  st.init(qv, 0.125f);  // 1 / sqrt(64)
  st.step(win, 0, n, n - 1, cur_k, cur_v);
  st.finish(a.out + (int64_t)r * width + h * kD);
}

// ------------------------------------------------------- depformer steps
struct DepSteps {
  const bf16_t* ws;  // the session's [8][K | V][width]
  int width, h;
  __device__ const bf16_t* k(int t) const { return ws + (int64_t)t * 2 * width + h * kD; }
  __device__ const bf16_t* v(int t) const { return ws + (int64_t)t * 2 * width + width + h * kD; }
};

__global__ __launch_bounds__(64) void dep_kv_attend64(ShortArgs a) {
  const int s = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63, c = lane & 7;
  const int width = a.heads * kD;
  const bf16_t* row = a.qkv + (int64_t)s * 3 * width;
  bf16_t* ws = a.ws + (int64_t)s * kDepSteps * 2 * width;
  // Steps 0 .. step (at most 8, one row of 8 keys) load together with the
  // row; step `step`, written below, is replaced by the registers' values.
  Row64::Tile<kDepSteps / 8> win;
  Row64::load(win, 0, a.step + 1, DepSteps{ws, width, h});
  const uint4 cur_k = ldg16(row + width + h * kD + 8 * c);
  const uint4 cur_v = ldg16(row + 2 * width + h * kD + 8 * c);
  if (lane < 8) {
    *reinterpret_cast<uint4*>(ws + (int64_t)a.step * 2 * width + h * kD + 8 * c) = cur_k;
    *reinterpret_cast<uint4*>(ws + (int64_t)a.step * 2 * width + width + h * kD + 8 * c) = cur_v;
  }
  float qv[8];
  widen8(ldg16(row + h * kD + 8 * c), qv);
  Row64 st;
  st.init(qv, a.scale);
  st.step(win, 0, a.step + 1, a.step, cur_k, cur_v);
  st.finish(a.out + (int64_t)s * width + h * kD);
}

}  // namespace

int launch_short(const ShortArgs& a, int kind, hipStream_t stream) {
  if (a.rows == 0) return 0;
  const dim3 grid(a.rows, a.heads);
  switch (kind) {
    case kShortMimi:  // an even T: a session's rows in pairs, unless the call is small
      if (a.context <= 8 * kMimiLoads)
        mimi_attend64<1, 1><<<grid, 64, 0, stream>>>(a);
      else if (a.T % 2 == 0 && (int64_t)a.rows * a.heads > kMimiAlone)
        mimi_attend64<2><<<dim3((a.rows + 1) / 2, a.heads), 64 * kMimiWaves, 0, stream>>>(a);
      else
        mimi_attend64<1><<<grid, 64 * kMimiWaves, 0, stream>>>(a);
      break;
    case kShortCodec: codec_attention64<<<grid, 64, 0, stream>>>(a); break;
    case kShortDep: dep_kv_attend64<<<grid, 64, 0, stream>>>(a); break;
    case kShortMimiRope: mimi_rope_kv64<<<a.rows, 256, 0, stream>>>(a); break;
    default: return -2;
  }
  return check_launch();
}

}  // namespace omni
