// One decoder token through every layer in one launch.
//
// The token step is a chain of ~95 dependent row-vector phases (per layer:
// qkv product, attention over the list's entries, merge, output projection,
// MLP up, MLP down), each a few microseconds of work spread over the chip.
// As one kernel per phase (six launches a layer) a step took 0.60 ms, of
// which the weights' 490 MB at the HBM rate are 0.1: the rest was launch gaps
// and, in every launch, the latency of weights that could have been read
// before their input was ready.  Here 256 resident workgroups run the whole
// chain, and
//  * phases hand their vectors over through memory without a grid barrier:
//    every published word carries a tag (bf16 value | 16-bit tag, or fp32
//    value | 32-bit tag), the step's number, so a reader polls the data
//    itself until every word has the tag.  Each vector of each layer has a
//    buffer of its own, rewritten once per step, so a word holds this step's
//    tag or the previous step's.  Words are read and written by relaxed
//    agent-scope atomics (they bypass the per-XCD caches); a bare hand-over
//    takes 2.2 us from store to the last of 256 workgroups' readers;
//  * the weights of a phase are loaded into registers a layer ahead, and the
//    K and V rows of a list entry while the qkv vector is still on its way.
//
// Workgroup w owns rows 12w.. of qkv, 4w.. of both residual outputs and
// 16w.. of the MLP's hidden layer; one (head, list entry) of the attention
// sits on every third workgroup or so.  Its eight wavefronts poll and norm an
// eighth of a phase's input each (a wavefront of its own for that, and for
// publishing, made a phase no faster: it issues an instruction about every
// five cycles).
//
// Measured: 0.30 ms for the sixteen layers (0.58 with the launches per layer),
// 0.26 without the weights' loads: the hand-overs, 93 in a chain, bound it.
// Rows published by the wavefronts one by one, not as one store per workgroup,
// took 0.40 ms: each was a write of its own to the same memory line.
//
// The workgroups of a step wait for each other, so only workgroups that are
// there may take part: each adds itself to a counter as it starts, and the step
// begins when all 256 have, or when one has waited gang_ticks for the rest and
// closes the counter: those that are there then share all the work (the same
// sums in the same order, the weights loaded as they are used), later ones
// leave at once.  So a step ends whatever else holds the device: kernels of
// other streams, another process's step that got the other half of the chip.
// The sixteen layers on 256 workgroups take 0.31 ms with the launches, on 255
// or 128 0.40, on 64 0.57, on 16 1.6, on one 22: with gang_ticks about a step's
// own time the wait costs no more than the step that follows it.
// (Without it two processes whose steps started together, each half-resident,
// waited for each other.)  Within a process a lock in device memory, taken by a
// one-wavefront launch before, lets one step run at a time; a lock that is not
// free within 2 ms is not waited for any longer.
// Every other wait ends too: after spin_ticks the waiter sets the status word
// and goes on with NaN, which reaches every row through the tagged words.
#include <math.h>

#include <mutex>

#include "common.h"

namespace scope {

namespace {
constexpr int kG = 256;              // workgroups
constexpr int kCW = 8;               // wavefronts
constexpr int kThreads = kCW * 64;
constexpr int kDm = 1024, kMlp = 4096, kHd = 128, kHeads = 8, kBs = 128;
constexpr int kMaxSkip = 16;         // U-net skips held in LDS
constexpr int kMaxKv = 32;           // list entries per head
constexpr float kStepLog2e = 1.4426950408889634f;
constexpr uint32_t kNanBf16 = 0x7fc0u;

// workspace: 64 words of header (0: steps done, 1: status, 2: the step's workgroups,
// 3: whether the step holds the lock), then per layer the tagged vectors
constexpr int64_t kHeadWords = 64;
constexpr int kGangWord = 2, kLockWord = 3;
constexpr uint32_t kClosed = 0x80000000u;
constexpr uint64_t kLockTicks = 200000;  // 2 ms: what six steps take
constexpr int64_t kQkvOff = 0, kYOff = kQkvOff + 3 * kDm, kX1Off = kYOff + kDm, kHOff = kX1Off + kDm,
                  kX2Off = kHOff + kMlp, kPartOff = kX2Off + kDm;  // 32-bit words
constexpr int kPartWords = (kHd + 2) * 2;                          // one entry's o, m, l as 64-bit words
}  // namespace

__device__ int g_step_lock;

struct StepArgs {
  scope_decoder_step_params p;
  const scope_decoder_layer* layers;
  const int64_t* tok;
  int64_t* t_dev;
  int64_t* tokens;
  int32_t* docs;
  const uint16_t* embed;
  const uint16_t* ve[3];
  const float* cos_t;
  const float* sin_t;
  uint16_t* x_out;
  uint32_t* work;
  int32_t* host_status;
};

__host__ __device__ __forceinline__ int64_t step_layer_words(int maxkv) {
  return kPartOff + static_cast<int64_t>(kHeads) * maxkv * kPartWords;
}

// sum over the 64 lanes, in every lane (DPP adds, no LDS round trips)
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float step_wave_sum(float x) {
  x = dpp_add<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8: lane 15 of each row of 16 holds the row's sum
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  x = dpp_add<0x118, 0xf>(x);
  x = dpp_add<0x142, 0xa>(x);  // row_bcast15 into rows 1 and 3
  x = dpp_add<0x143, 0xc>(x);  // row_bcast31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
// sum over each row of 16 lanes, in every lane
__device__ __forceinline__ float row_sum16(float x) {
  x = dpp_add<0x128, 0xf>(x);  // row_ror 8, 4, 2, 1
  x = dpp_add<0x124, 0xf>(x);
  x = dpp_add<0x122, 0xf>(x);
  return dpp_add<0x121, 0xf>(x);
}

// a wavefront's waits: when one lasts longer than the limit, it and all later ones end at once with NaN
struct StepWait {
  uint64_t limit;
  uint32_t* status;
  int32_t* host_status;
  bool dead;
};

// Poll `it` of a wait found nothing: whether the wait ends.  The time counts from
// the wait's 64th poll (t0), not from the kernel's start: a kernel that was held
// up between its waits has not waited.
__device__ __forceinline__ bool step_expired(StepWait& w, int it, uint64_t& t0) {
  if (w.dead || (it & 63) != 63) return w.dead;
  const uint64_t now = static_cast<uint64_t>(wall_clock64());
  if (it == 63) {
    t0 = now;
  } else if (now - t0 > w.limit) {
    w.dead = true;
    __hip_atomic_store(w.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (w.host_status) __hip_atomic_store(w.host_status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return w.dead;
}

// 2·N tagged bf16 words of this lane at p[stride·j], j < N (64-bit loads)
template <int N>
__device__ __forceinline__ void poll_bf16(const uint64_t* p, int stride, uint32_t tag, uint64_t (&v)[N], StepWait& w) {
  const uint64_t want = (static_cast<uint64_t>(tag) << 48) | (static_cast<uint64_t>(tag) << 16);
  uint64_t t0 = 0;
  for (int it = 0;; ++it) {
#pragma unroll
    for (int j = 0; j < N; ++j)
      v[j] = __hip_atomic_load(p + static_cast<int64_t>(j) * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t diff = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) diff |= (v[j] ^ want) & 0xffff0000ffff0000ull;
    if (__all(diff == 0)) return;
    if (step_expired(w, it, t0)) break;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = kNanBf16 | (static_cast<uint64_t>(kNanBf16) << 32);
}

// N tagged fp32 words of this lane at q[j]
template <int N>
__device__ __forceinline__ void poll_f32(const uint64_t* const (&q)[N], uint32_t seq, float (&f)[N], StepWait& w) {
  uint64_t t0 = 0;
  for (int it = 0;; ++it) {
    uint64_t v[N];
    uint32_t diff = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = __hip_atomic_load(q[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      diff |= static_cast<uint32_t>(v[j] >> 32) ^ seq;
      f[j] = __uint_as_float(static_cast<uint32_t>(v[j]));
    }
    if (__all(diff == 0)) return;
    if (step_expired(w, it, t0)) break;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) f[j] = __builtin_nanf("");
}

__device__ __forceinline__ float word_lo(uint64_t v) { return bf16_to_f32(static_cast<uint16_t>(v)); }
__device__ __forceinline__ float word_hi(uint64_t v) { return bf16_to_f32(static_cast<uint16_t>(v >> 32)); }
__device__ __forceinline__ void publish(uint32_t* p, uint16_t x, uint32_t tag) {
  __hip_atomic_store(p, (tag << 16) | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish_f32(uint64_t* p, float x, uint32_t seq) {
  __hip_atomic_store(p, (static_cast<uint64_t>(seq) << 32) | __float_as_uint(x), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

struct StepShared {
  __attribute__((aligned(16))) uint16_t xs[2][kDm];  // the phase's input, two phases alternating
  float ss[2][kCW];                                  // the wavefronts' sums of squares
  float part[2][4][kCW];                             // MLP output: (row, segment) sums, two parts alternating
  uint32_t rows[2][16];                              // output words to publish, two phases alternating
  uint16_t xraw[2][kDm];                             // the residual stream before the attention and before the MLP
  uint16_t skip[kMaxSkip][kDm];                      // layer outputs for the U-net skips (each lane its own features)
  float gq[kHd];                                     // attention: the rotated query, and the token's k and v rows
  __attribute__((aligned(16))) uint16_t gk[kHd], gv[kHd];
  float o[2][kCW][kHd], m[2][kCW], l[2][kCW];        // the wavefronts' attention sums and their merged entries
  int gang;                                          // the step's workgroups
  uint32_t rank;                                     // the gang word as this workgroup's arrival found it
};

__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {  // round to nearest even
  typedef __bf16 v2 __attribute__((ext_vector_type(2)));
  v2 v;
  v[0] = static_cast<__bf16>(lo), v[1] = static_cast<__bf16>(hi);
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint16_t r_bf16(float x) { return static_cast<uint16_t>(pk_bf16(x, 0.f)); }
__device__ __forceinline__ float rf_bf16(float x) { return __uint_as_float(pk_bf16(x, 0.f) << 16); }
__device__ __forceinline__ float lo_f(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

__device__ __forceinline__ float relu_nan(float x) { return x < 0.f ? 0.f : x; }  // keeps a NaN

// acc += the product of eight bf16 weights and eight inputs
__device__ __forceinline__ float dot8(const uint4& w, const float* x, float acc) {
  const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc = fmaf(lo_f(q[i]), x[2 * i], acc);
    acc = fmaf(hi_f(q[i]), x[2 * i + 1], acc);
  }
  return acc;
}

__device__ __forceinline__ void lds_x8(const uint16_t* p, float* x) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  const uint32_t q[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) x[2 * i] = lo_f(q[i]), x[2 * i + 1] = hi_f(q[i]);
}

// R whole rows of 1024 of one wavefront: rows row0 + j·stride, columns 8·lane.. of both halves
template <int R>
struct Rows {
  uint4 w[R][2];
  __device__ __forceinline__ void load(const uint16_t* W, int row0, int stride, int lane) {
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        w[j][c] = *reinterpret_cast<const uint4*>(W + static_cast<int64_t>(row0 + j * stride) * kDm + c * 512 + 8 * lane);
  }
  // the bf16 output of row j, in every lane
  __device__ __forceinline__ float run(int j, const float (&x)[16]) const {
    return rf_bf16(step_wave_sum(dot8(w[j][1], x + 8, dot8(w[j][0], x, 0.f))));
  }
};

// Merge of eight wavefronts' (o, m, l) at features lane and lane + 64:
// log2-domain maxima, entries without a key have m = -inf and l = 0.  A NaN
// in l stays, here and in the merges after it, whatever its m.
struct Merged {
  float M, L, O0, O1;
};
__device__ __forceinline__ Merged merge_waves(const float (&o)[kCW][kHd], const float (&m)[kCW], const float (&l)[kCW],
                                              int lane) {
  Merged r{-INFINITY, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kCW; ++w) r.M = fmaxf(r.M, m[w]);
#pragma unroll
  for (int w = 0; w < kCW; ++w) {
    if (m[w] == -INFINITY && l[w] == 0.f) continue;
    const float s = __builtin_amdgcn_exp2f(m[w] - r.M);
    r.L = fmaf(l[w], s, r.L);
    r.O0 = fmaf(o[w][lane], s, r.O0);
    r.O1 = fmaf(o[w][lane + 64], s, r.O1);
  }
  return r;
}

__device__ __forceinline__ int step_next_att(const StepArgs& a, int i) {  // layer i or the next one with attention
  while (i < a.p.layers && !a.layers[i].qkv) ++i;
  return i;
}

// Before a step: the gang word is cleared, and the process's step lock taken, or
// not within kLockTicks (whether it was is kept for the release).
__global__ __launch_bounds__(64) void step_begin_kernel(uint32_t* work) {
  if (threadIdx.x != 0) return;
  __hip_atomic_store(work + kGangWord, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint64_t t0 = static_cast<uint64_t>(wall_clock64());
  uint32_t took = 0;
  do {
    int free_ = 0;
    took = __hip_atomic_compare_exchange_strong(&g_step_lock, &free_, 1, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    if (!took) __builtin_amdgcn_s_sleep(8);
  } while (!took && static_cast<uint64_t>(wall_clock64()) - t0 < kLockTicks);
  __hip_atomic_store(work + kLockWord, took, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The number of workgroups a step runs on, for one of them.  Each adds itself to
// the gang word as it starts: arrivals in the low 16 bits, and once it is closed
// kClosed and the size at that moment in bits 16-30.  Ends when all kG have
// arrived or when a workgroup that waited longer than the limit closes the gang
// with those that are there; a closing and a full gang exclude each other (the
// compare-and-swap expects fewer arrivals).
__device__ __forceinline__ int step_gang(uint32_t* word, uint64_t limit) {
  uint64_t t0 = 0;
  for (bool first = true;; first = false) {
    uint32_t w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (w & kClosed) return static_cast<int>((w & ~kClosed) >> 16);
    if (w == kG) return kG;
    const uint64_t now = static_cast<uint64_t>(wall_clock64());
    if (first) t0 = now;
    if (now - t0 >= limit &&
        __hip_atomic_compare_exchange_strong(word, &w, kClosed | (w << 16) | w, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return static_cast<int>(w);
  }
}

// the weights a workgroup holds in registers: rows of part v of every product
struct StepWeights {
  Rows<2> qkv, fc;  // qkv rows wave and, below wave 4, wave + 8 of the part's twelve
  Rows<1> proj;     // wavefronts 0-3
  uint4 mp[4];      // MLP output: segment `wave` of the four rows
  __device__ __forceinline__ void load_qkv(const scope_decoder_layer& l, int v, int wave, int lane) {
    qkv.load(l.qkv, 12 * v + wave, wave < 4 ? 8 : 0, lane);
  }
  __device__ __forceinline__ void load_proj(const scope_decoder_layer& l, int v, int wave, int lane) {
    proj.load(l.proj, 4 * v + (wave & 3), 0, lane);
  }
  __device__ __forceinline__ void load_fc(const scope_decoder_layer& l, int v, int wave, int lane) {
    fc.load(l.mlp_fc, 16 * v + 2 * wave, 1, lane);
  }
  __device__ __forceinline__ void load_mp(const scope_decoder_layer& l, int v, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      mp[j] = *reinterpret_cast<const uint4*>(l.mlp_proj + static_cast<int64_t>(4 * v + j) * kMlp + wave * 512 + 8 * lane);
  }
};

// The step on n workgroups, of which this is number wg.  FULL: n = kG, part wg
// is this workgroup's, its weights in registers a layer ahead; whether all are
// there is looked at after its first rows are published, when the answer is
// ready: false if not, before anything but those rows (which are the same on any
// number of workgroups) is written.  Otherwise each workgroup takes the parts
// wg, wg + n, .. of every phase, weights loaded as they are used: the same sums
// in the same order.
template <bool FULL>
__device__ __forceinline__ bool step_run(const StepArgs& a, StepShared& sh, StepWeights& W, const int wg, const int n) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const scope_decoder_step_params& p = a.p;
  const int L = p.layers, nskip = L / 2, maxkv = p.maxkv;
  // (atomic loads: workgroup 0 writes the counter and the position at its end)
  const uint32_t seq = __hip_atomic_load(a.work, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1, tag = seq & 0xffffu;
  const bool dead0 = __hip_atomic_load(a.work + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  StepWait wt{p.spin_ticks, a.work + 1, a.host_status, dead0};
  if (dead0 && wg == 0 && tid == 0 && a.host_status)  // the host's copy follows the status
    __hip_atomic_store(a.host_status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const int64_t tok = *a.tok, t = __hip_atomic_load(a.t_dev, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool ok = tok >= 0 && tok < p.vocab && t >= 0 && t < p.T_cap;
  const bool pos_ok = t >= 0 && t < p.T_cap && t < p.rot_rows;
  uint32_t* const vec = a.work + kHeadWords;
  const int64_t lw = step_layer_words(maxkv);
  const int ntask = kHeads * maxkv, every = kG / ntask;  // tasks: (head, list entry), the entries of a head in a row
  // a token outside the vocabulary leaves docs[t] as it is and attends to that document
  const int32_t doc_t = ok    ? (t > 0 ? a.docs[t - 1] : 0) + (tok == p.eot ? 1 : 0)
                        : t >= 0 && t < p.T_cap ? a.docs[t]
                                                : 0;
  auto parts_of = [&](auto&& f) {  // f(v) for this workgroup's parts of a product
    if constexpr (FULL) {
      f(wg);
    } else {
      for (int v = wg; v < kG; v += n) f(v);
    }
  };

  const int sub = lane >> 4, ch = lane & 15, f0 = 128 * wave + 2 * lane;  // f0: this lane's two features of a vector
  int pb = 0, pp = 0;  // which of the two buffers: xs and ss, part
  float x0, x1;   // features f0, f0 + 1
  float x[16];    // inputs of whole rows: columns 8·lane.. of both halves
  auto poll_x = [&](const uint32_t* src) {
    uint64_t v[1];
    poll_bf16<1>(reinterpret_cast<const uint64_t*>(src + f0), 1, tag, v, wt);
    x0 = word_lo(v[0]), x1 = word_hi(v[0]);
  };
  // 1 / rms of the vector (a barrier)
  auto rms = [&]() {
    const float s = step_wave_sum(fmaf(x0, x0, x1 * x1));
    if (lane == 0) sh.ss[pb][wave] = s;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < kCW; ++w) tot += sh.ss[pb][w];
    return 1.f / sqrtf(tot / kDm + p.eps);
  };
  // the phase's input into LDS, and from there to the lanes (a barrier)
  // Publish the workgroup's n rows (sh.rows, a barrier) as one store: separate
  // stores of each row are separate writes of the same memory line.
  int pr = 0;
  auto publish_rows = [&](uint32_t* dst, int n) {
    __syncthreads();
    if (wave == 0 && lane < n)
      __hip_atomic_store(dst + lane, (tag << 16) | sh.rows[pr][lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    pr ^= 1;
  };
  auto spread = [&](float r) {
    *reinterpret_cast<uint32_t*>(&sh.xs[pb][f0]) = pk_bf16(__fmul_rn(x0, r), __fmul_rn(x1, r));
    __syncthreads();
    lds_x8(&sh.xs[pb][8 * lane], x);
    lds_x8(&sh.xs[pb][512 + 8 * lane], x + 8);
    pb ^= 1;
  };

  auto all_there = [&]() {
    if (tid == 0) sh.gang = step_gang(a.work + kGangWord, p.gang_ticks);
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sh.gang) == kG;
  };
  for (int i = 0; i < L; ++i) {
    const scope_decoder_layer lay = a.layers[i];
    uint32_t* const lv = vec + i * lw;
    // ---- the layer's input
    if (i == 0) {
      x0 = x1 = 0.f;
      if (ok) {
        const uint32_t u = *reinterpret_cast<const uint32_t*>(a.embed + tok * kDm + f0);
        x0 = lo_f(u), x1 = hi_f(u);
      }
      const float r = rms();
      pb ^= 1;
      x0 = rf_bf16(__fmul_rn(x0, r)), x1 = rf_bf16(__fmul_rn(x1, r));
    } else {
      poll_x(lv - lw + kX2Off);
      if (i - 1 < nskip) *reinterpret_cast<uint32_t*>(&sh.skip[i - 1][f0]) = pk_bf16(x0, x1);
      if (i >= nskip) {
        const uint32_t u = *reinterpret_cast<const uint32_t*>(&sh.skip[L - 1 - i][f0]);
        x0 = rf_bf16(__fadd_rn(x0, lo_f(u))), x1 = rf_bf16(__fadd_rn(x1, hi_f(u)));
      }
    }
    *reinterpret_cast<uint32_t*>(&sh.xraw[0][f0]) = pk_bf16(x0, x1);
    spread(rms());
    int res = 0;
    if (lay.qkv) {
      const int nx = FULL ? step_next_att(a, i + 1) : L;
      // ---- qkv
      parts_of([&](int v) {
        if (!FULL) W.load_qkv(lay, v, wave, lane);
        const float z0 = W.qkv.run(0, x), z1 = W.qkv.run(1, x);
        if (lane == 0) {
          sh.rows[pr][wave] = r_bf16(z0);
          if (wave < 4) sh.rows[pr][wave + 8] = r_bf16(z1);
        }
        publish_rows(lv + kQkvOff + 12 * v, 12);
      });
      if (FULL && i == 0 && !all_there()) return false;
      if (nx < L) W.load_qkv(a.layers[nx], wg, wave, lane);
      // ---- attention: one (head, list entry)
      uint64_t* const parts = reinterpret_cast<uint64_t*>(lv + kPartOff);
      auto attend = [&](int task) __attribute__((always_inline)) {
        const int head = task / maxkv, ent = task % maxkv;
        // keys 16·wave .. +15 of the entry's block: sixteen lanes per row, four
        // rows at a time; the rows are loaded while the qkv vector is on its way
        const int64_t kblk = ent < lay.kv_num[head] ? lay.kv_idx[static_cast<int64_t>(head) * maxkv + ent] : -1;
        const int64_t k0 = kblk * kBs;
        const bool use = kblk >= 0 && k0 <= t && k0 + kBs <= p.T_cap && pos_ok;
        uint4 ku[4], vu[4];
        int dj[4];
        if (use) {
          const uint16_t* kr = lay.k_cache + head * p.k_sh + 8 * ch;
          const uint16_t* vr = lay.v_cache + head * p.v_sh + 8 * ch;
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const int64_t j = k0 + 16 * wave + 4 * it + sub;
            ku[it] = *reinterpret_cast<const uint4*>(kr + j * p.k_st);
            vu[it] = *reinterpret_cast<const uint4*>(vr + j * p.v_st);
            dj[it] = j < t ? a.docs[j] : doc_t;  // docs[t] is written at the end
          }
        }
        // the token's q (wavefront 0), k (1) and v (2) of the head: lane l holds features 2l and 2l + 1
        if (wave < 3 && pos_ok) {
          uint64_t v[1];
          poll_bf16<1>(reinterpret_cast<const uint64_t*>(lv + kQkvOff + (wave * kHeads + head) * kHd) + lane, 1, tag, v, wt);
          float y0 = word_lo(v[0]), y1 = word_hi(v[0]);
          if (wave < 2) {
            const float r = 1.f / sqrtf(step_wave_sum(fmaf(y0, y0, y1 * y1)) / kHd + p.eps);
            const int d2 = (2 * lane) % (kHd / 2);
            const float2 c = *reinterpret_cast<const float2*>(a.cos_t + t * p.rot_st + d2);
            const float2 sn = *reinterpret_cast<const float2*>(a.sin_t + t * p.rot_st + d2);
            y0 = rf_bf16(__fmul_rn(y0, r)), y1 = rf_bf16(__fmul_rn(y1, r));
            const float o0 = __shfl_xor(y0, 32, kWave), o1 = __shfl_xor(y1, 32, kWave);  // features d ± 64
            if (lane < 32) {
              y0 = __fadd_rn(__fmul_rn(y0, c.x), __fmul_rn(o0, sn.x));
              y1 = __fadd_rn(__fmul_rn(y1, c.y), __fmul_rn(o1, sn.y));
            } else {
              y0 = __fadd_rn(__fmul_rn(o0, -sn.x), __fmul_rn(y0, c.x));
              y1 = __fadd_rn(__fmul_rn(o1, -sn.y), __fmul_rn(y1, c.y));
            }
          } else {
            y0 = rf_bf16(__fmul_rn(lay.va, y0)), y1 = rf_bf16(__fmul_rn(lay.va, y1));
            if (lay.ve >= 0) {
              uint32_t e = 0;
              if (ok) e = *reinterpret_cast<const uint32_t*>(a.ve[lay.ve] + tok * kDm + head * kHd + 2 * lane);
              y0 = __fadd_rn(y0, rf_bf16(__fmul_rn(lay.vb, lo_f(e))));
              y1 = __fadd_rn(y1, rf_bf16(__fmul_rn(lay.vb, hi_f(e))));
            }
          }
          const uint32_t yw = pk_bf16(y0, y1);
          if (wave == 0) {
            *reinterpret_cast<float2*>(&sh.gq[2 * lane]) = make_float2(lo_f(yw), hi_f(yw));
          } else {
            *reinterpret_cast<uint32_t*>(wave == 1 ? &sh.gk[2 * lane] : &sh.gv[2 * lane]) = yw;
            if (ent == 0)  // cache row t, once per head
              *reinterpret_cast<uint32_t*>((wave == 1 ? lay.k_cache + head * p.k_sh + t * p.k_st
                                                      : lay.v_cache + head * p.v_sh + t * p.v_st) + 2 * lane) = yw;
          }
        }
        __syncthreads();  // q, k, v
        float m = -INFINITY, l = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (use) {
          float qv[8], s[4];
#pragma unroll
          for (int c = 0; c < 8; ++c) qv[c] = sh.gq[8 * ch + c] * p.scale * kStepLog2e;
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const int64_t j = k0 + 16 * wave + 4 * it + sub;
            if (j == t) {  // the token's own row
              ku[it] = *reinterpret_cast<const uint4*>(&sh.gk[8 * ch]);
              vu[it] = *reinterpret_cast<const uint4*>(&sh.gv[8 * ch]);
            }
            const float acc = row_sum16(dot8(ku[it], qv, 0.f));
            s[it] = j <= t && dj[it] == doc_t ? acc : -INFINITY;
            m = fmaxf(m, s[it]);
          }
          m = fmaxf(m, __shfl_xor(m, 16, kWave));
          m = fmaxf(m, __shfl_xor(m, 32, kWave));
          // fmaxf skips NaN scores: with nothing but them, any offset keeps them in l and o
          if (m == -INFINITY && __any(s[0] != s[0] || s[1] != s[1] || s[2] != s[2] || s[3] != s[3])) m = 0.f;
          if (m != -INFINITY) {  // wavefront-uniform
#pragma unroll
            for (int it = 0; it < 4; ++it) {
              const float pj = exp2f(s[it] - m);
              l += pj;
              const uint32_t wv[4] = {vu[it].x, vu[it].y, vu[it].z, vu[it].w};
              // a masked key adds nothing whatever its cache row holds
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                o[2 * c] = pj != 0.f ? fmaf(pj, lo_f(wv[c]), o[2 * c]) : o[2 * c];
                o[2 * c + 1] = pj != 0.f ? fmaf(pj, hi_f(wv[c]), o[2 * c + 1]) : o[2 * c + 1];
              }
            }
            l += __shfl_xor(l, 16, kWave);
            l += __shfl_xor(l, 32, kWave);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              o[c] += __shfl_xor(o[c], 16, kWave);
              o[c] += __shfl_xor(o[c], 32, kWave);
            }
          }
        }
        if (sub == 0) {
          *reinterpret_cast<float4*>(&sh.o[0][wave][8 * ch]) = make_float4(o[0], o[1], o[2], o[3]);
          *reinterpret_cast<float4*>(&sh.o[0][wave][8 * ch + 4]) = make_float4(o[4], o[5], o[6], o[7]);
        }
        if (lane == 0) sh.m[0][wave] = m, sh.l[0][wave] = l;
        __syncthreads();  // the wavefronts' sums
        if (wave == 0) {
          const Merged r = merge_waves(sh.o[0], sh.m[0], sh.l[0], lane);
          uint64_t* pp = parts + static_cast<int64_t>(task) * (kHd + 2);
          publish_f32(pp + lane, r.O0, seq);
          publish_f32(pp + lane + 64, r.O1, seq);
          if (lane == 0) {
            publish_f32(pp + kHd, r.M, seq);
            publish_f32(pp + kHd + 1, r.L, seq);
          }
        }
      };
      // merges the head's entries, wavefront w the entries w, w + 8, ..
      auto merge_head = [&](int head) __attribute__((always_inline)) {
        Merged r{-INFINITY, 0.f, 0.f, 0.f};
        for (int e = wave; e < maxkv; e += kCW) {
          const uint64_t* pe = parts + (static_cast<int64_t>(head) * maxkv + e) * (kHd + 2);
          const uint64_t* const q[4] = {pe + lane, pe + lane + 64, pe + kHd, pe + kHd + 1};
          float f[4];
          poll_f32<4>(q, seq, f, wt);
          if (f[2] == -INFINITY && f[3] == 0.f) continue;
          const float Mn = fmaxf(r.M, f[2]);
          const float sa = r.M == Mn ? 1.f : __builtin_amdgcn_exp2f(r.M - Mn), sb = __builtin_amdgcn_exp2f(f[2] - Mn);
          r = Merged{Mn, fmaf(f[3], sb, r.L * sa), fmaf(f[0], sb, r.O0 * sa), fmaf(f[1], sb, r.O1 * sa)};
        }
        sh.o[1][wave][lane] = r.O0, sh.o[1][wave][lane + 64] = r.O1;
        if (lane == 0) sh.m[1][wave] = r.M, sh.l[1][wave] = r.L;
        __syncthreads();  // the merged entries
        if (wave == 0) {
          const Merged y = merge_waves(sh.o[1], sh.m[1], sh.l[1], lane);
          const float inv = 1.f / y.L;  // (L = 0: no key)
          uint32_t* py = lv + kYOff + head * kHd + lane;
          publish(py, r_bf16(y.L == 0.f ? 0.f : y.O0 * inv), tag);
          publish(py + 64, r_bf16(y.L == 0.f ? 0.f : y.O1 * inv), tag);
        }
      };
      if constexpr (FULL) {  // a task on every third workgroup or so
        if (wg % every == 0 && wg / every < ntask) {
          attend(wg / every);
          if (wg / every % maxkv == 0) merge_head(wg / every / maxkv);
        }
      } else {  // (every entry of this workgroup's before it waits for another's)
        for (int task = wg; task < ntask; task += n) attend(task);
        for (int task = wg; task < ntask; task += n) {
          if (task % maxkv) continue;
          merge_head(task / maxkv);
          __syncthreads();  // the merged entries are read
        }
      }
      // ---- output projection and residual
      poll_x(lv + kYOff);
      spread(1.f);
      parts_of([&](int v) {
        if (!FULL) W.load_proj(lay, v, wave, lane);
        if (wave < 4) {
          const float z = W.proj.run(0, x);
          if (lane == 0) sh.rows[pr][wave] = r_bf16(__fadd_rn(bf16_to_f32(sh.xraw[0][4 * v + wave]), z));
        }
        publish_rows(lv + kX1Off + 4 * v, 4);
      });
      if (nx < L) W.load_proj(a.layers[nx], wg, wave, lane);
      poll_x(lv + kX1Off);
      *reinterpret_cast<uint32_t*>(&sh.xraw[1][f0]) = pk_bf16(x0, x1);
      res = 1;
      spread(rms());
    }
    // ---- MLP
    parts_of([&](int v) {
      if (!FULL) W.load_fc(lay, v, wave, lane);
      const float h0 = relu_nan(W.fc.run(0, x)), h1 = relu_nan(W.fc.run(1, x));
      if (lane == 0) {
        sh.rows[pr][2 * wave] = r_bf16(__fmul_rn(h0, h0));
        sh.rows[pr][2 * wave + 1] = r_bf16(__fmul_rn(h1, h1));
      }
      publish_rows(lv + kHOff + 16 * v, 16);
    });
    if (FULL && i == 0 && !lay.qkv && !all_there()) return false;
    {
      // this lane's eight inputs of segment `wave`, straight from the published words
      uint64_t v[4];
      poll_bf16<4>(reinterpret_cast<const uint64_t*>(lv + kHOff + wave * 512 + 8 * lane), 1, tag, v, wt);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[2 * j] = word_lo(v[j]), x[2 * j + 1] = word_hi(v[j]);
    }
    // Loads return in order, so a poll also waits for every load before it: these
    // are issued after the poll.  (The MLP's weights a layer ahead but loaded
    // during the attention, and qkv's during the MLP: 350 instead of 314 us.)
    if (FULL && i + 1 < L) W.load_fc(a.layers[i + 1], wg, wave, lane);
    parts_of([&](int v) {
      if (!FULL) W.load_mp(lay, v, wave, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float z = step_wave_sum(dot8(W.mp[j], x, 0.f));
        if (lane == 0) sh.part[pp][j][wave] = z;
      }
      if (FULL && i + 1 < L) W.load_mp(a.layers[i + 1], wg, wave, lane);
      __syncthreads();  // MLP output sums
      if (wave == 0 && lane < 4) {
        float z = 0.f;
#pragma unroll
        for (int w = 0; w < kCW; ++w) z += sh.part[pp][lane][w];
        const uint16_t y = r_bf16(__fadd_rn(bf16_to_f32(sh.xraw[res][4 * v + lane]), rf_bf16(z)));
        if (i + 1 < L) publish(lv + kX2Off + 4 * v + lane, y, tag);
        else a.x_out[4 * v + lane] = wt.dead ? static_cast<uint16_t>(kNanBf16) : y;
      }
      pp ^= 1;
    });
  }
  // workgroup 0 has read what every workgroup of the step published: all have read the position and the counter
  if (wg == 0 && tid == 0) {
    if (ok) {
      a.tokens[t] = tok;
      a.docs[t] = doc_t;
    }
    *a.t_dev = t + 1;
    a.work[0] = seq;
    if (__hip_atomic_load(a.work + kLockWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      __hip_atomic_store(&g_step_lock, 0, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
  }
  return true;
}

__global__ __launch_bounds__(kThreads) void decoder_step_kernel(StepArgs a) {
  __shared__ StepShared sh;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t old = 0;
  if (tid == 0) old = __hip_atomic_fetch_add(a.work + kGangWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the first weights, as the full gang needs them
  StepWeights W;
  const int i0 = step_next_att(a, 0);
  if (i0 < a.p.layers) {
    W.load_qkv(a.layers[i0], blockIdx.x, wave, lane);
    W.load_proj(a.layers[i0], blockIdx.x, wave, lane);
  }
  W.load_fc(a.layers[0], blockIdx.x, wave, lane);
  W.load_mp(a.layers[0], blockIdx.x, wave, lane);
  if (tid == 0) sh.rank = old;
  __syncthreads();
  const uint32_t rank = __builtin_amdgcn_readfirstlane(sh.rank);
  if (rank & kClosed) return;  // the step runs without this workgroup
  if (step_run<true>(a, sh, W, blockIdx.x, kG)) return;
  const int n = __builtin_amdgcn_readfirstlane(sh.gang);
  __syncthreads();
  step_run<false>(a, sh, W, rank & 0xffffu, n);
}

}  // namespace scope

using namespace scope;

static int step_shape_ok(const scope_decoder_step_params* p) {
  return p && p->layers >= 2 && p->layers % 2 == 0 && p->layers / 2 <= kMaxSkip && p->H == kHeads && p->D == kHd &&
         p->dm == kDm && p->mlp == kMlp && p->bs == kBs && p->maxkv >= 1 && p->maxkv <= kMaxKv && p->T_cap >= kBs &&
         p->T_cap % kBs == 0 && p->workgroups >= 0 && p->workgroups <= kG;
}

extern "C" int scope_decoder_step_supported(const scope_decoder_step_params* p) {
  if (!step_shape_ok(p)) return 0;
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, decoder_step_kernel, kThreads, 0) != hipSuccess)
    return 0;
  return static_cast<int64_t>(cus) * per >= kG;
}

extern "C" int64_t scope_decoder_step_workspace_bytes(const scope_decoder_step_params* p) {
  if (!step_shape_ok(p)) return 0;
  return 4 * (kHeadWords + p->layers * step_layer_words(p->maxkv));
}

extern "C" int scope_decoder_step(const scope_decoder_step_params* p, const scope_decoder_layer* layers,
                                  const int64_t* tok, int64_t* t_dev, int64_t* tokens, int32_t* docs,
                                  const uint16_t* embed, const uint16_t* ve0, const uint16_t* ve1, const uint16_t* ve2,
                                  const float* cos_t, const float* sin_t, uint16_t* x_out, void* work,
                                  int32_t* host_status, void* stream) {
  SCOPE_REQUIRE(p && layers && tok && t_dev && tokens && docs && embed && cos_t && sin_t && x_out && work,
                "scope_decoder_step: null pointer");
  SCOPE_REQUIRE(step_shape_ok(p),
                "scope_decoder_step: supported are an even number of layers (2..%d), %d heads of %d, width %d, MLP %d, "
                "blocks of %d and lists of at most %d entries",
                2 * kMaxSkip, kHeads, kHd, kDm, kMlp, kBs, kMaxKv);
  SCOPE_REQUIRE(scope_decoder_step_supported(p), "scope_decoder_step: the device cannot hold %d workgroups at once", kG);
  SCOPE_REQUIRE(p->vocab >= 1 && p->rot_rows >= 1 && p->rot_st >= kHd / 2 && p->rot_st % 2 == 0,
                "scope_decoder_step: vocab=%lld / rotary table", (long long)p->vocab);
  SCOPE_REQUIRE(p->k_st % 8 == 0 && p->k_sh % 8 == 0 && p->v_st % 8 == 0 && p->v_sh % 8 == 0,
                "scope_decoder_step: cache rows must be 16-byte aligned");
  const auto al = [](const void* x, uintptr_t n) { return (reinterpret_cast<uintptr_t>(x) & (n - 1)) == 0; };
  SCOPE_REQUIRE(al(embed, 16) && al(cos_t, 8) && al(sin_t, 8) && al(work, 8),
                "scope_decoder_step: misaligned embedding, rotary table or workspace");
  StepArgs a{*p, layers, tok, t_dev, tokens, docs, embed, {ve0, ve1, ve2}, cos_t, sin_t, x_out,
             static_cast<uint32_t*>(work), host_status};
  hipStream_t s = as_stream(stream);
  // both launches in a row, also where streams share a hardware queue: a lock that is waited
  // for in front of its holder's step would wait until its limit
  static std::mutex order;
  const std::lock_guard<std::mutex> hold(order);
  hipLaunchKernelGGL(step_begin_kernel, dim3(1), dim3(64), 0, s, a.work);
  int rc = check_launch("step_begin_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(decoder_step_kernel, dim3(p->workgroups ? p->workgroups : kG), dim3(kThreads), 0, s, a);
  return check_launch("decoder_step_kernel");
}
