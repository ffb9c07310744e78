// GQA/MHA query blocks on MFMA with fp32-precise probabilities: packed (TND / NTD) and batched queries over
// paged or dense keys, band masks, a sink. The calls packed_takes() names come from the general kernel, whose
// arguments and meaning these are: scores, row sums, O and partials in fp32, P in the P.V MFMA as a 16-bit pair
// (hi = half(p), lo = half(p - hi)).
//
// Item: (sequence, kv head, block of 256 columns); a column is one (query row, head of the kv head's group), row
// major, so a block holds 256 / g rows of g heads and a single decode row fills g columns of one wave. A
// workgroup of 8 waves takes 32 columns each and streams the block's K/V tiles of 64 tokens through a four-slot
// LDS ring, two tiles ahead (the tile layout and fragment reads of the prefill kernel).
//
// Sequence lengths are on the device, so the launch is one workgroup per CU over equal ranges of the items' cost
// (planned by the kernel itself, or by packed_plan_kernel where sequences are many or long): long prompts, short
// chunks and single tokens fill the chip alike. An item cut by a range's end leaves fp32 partials, which
// packed_merge_kernel joins.
//
// Measured (6 chunks of 128-512 tokens and 24 single tokens over contexts up to 4096, 32 / 8 heads of 128):
// 26.1 ms on the general kernel (each row and head read its keys and values alone), 0.202 ms here: plan 6 us, merge
// 14, the rest this kernel. Its MFMAs (48 per wave and tile, a third of them for lo) take about 100 us; they are 27%
// busy, the vector units 31%, HBM at 2.2 TB/s: score, softmax and P.V of a tile follow one another.
#include "attention_common.h"

namespace tai {
namespace {

constexpr int kKWgs = 256;       // most ranges: one workgroup per CU
constexpr int kKCols = 256;      // columns per item
// Cost of an item: kKItem units for its start (query load, ring fill, output) and per tile 2 units with up to
// one wave per SIMD, 3 with two.
constexpr int kKItem = 5;

struct PackedArgs {
  tai_fia_general_args a;
  int g;              // query heads per kv head
  int64_t kv_cap;
  float scale_log2;   // |scale| * log2(e), > 0
  int neg_scale;      // the scale is negative: Q is negated on load
  int64_t* pref;      // [b + 1] cost of the sequences before
  int4* rec;          // [ranges] the item each range leaves unfinished: {b, kv head, block, last range} (last = 0: none)
  int cap;            // most ranges this call can have
  int waves;          // waves of a workgroup that can hold columns: 32 each of a block's at most 256
  float* part_o;      // [2 * cap][waves][D / 32][4][64 lanes][4]; slot 2r: the item range r continues, 2r + 1: leaves
  float* part_ml;     // [2 * cap][32 * waves][2]
  bool plan_here;     // few sequences of few blocks: the main kernel plans by itself
};
constexpr int kKPlanSeqs = 512;  // the main kernel's threads
constexpr int kKPlanBlocks = 8;

struct SeqInfo {
  int64_t q_start, lq, lk, kv_base, off;
};

__device__ __forceinline__ SeqInfo seq_info(const PackedArgs& p, int64_t b) {
  const tai_fia_general_args& a = p.a;
  SeqInfo s;
  if (a.q_cum) {
    const int64_t end = clamp_len(a.q_cum[b], a.s_q);
    s.q_start = b ? imin64(clamp_len(a.q_cum[b - 1], a.s_q), end) : 0;
    s.lq = end - s.q_start;
  } else {
    s.q_start = 0;
    s.lq = a.seq_lens_q ? clamp_len(a.seq_lens_q[b], a.s_q) : a.s_q;
  }
  s.kv_base = 0;
  if (a.kv_cum) {
    const int64_t end = clamp_len(a.kv_cum[b], a.s_kv);
    s.kv_base = b ? imin64(clamp_len(a.kv_cum[b - 1], a.s_kv), end) : 0;
    s.lk = end - s.kv_base;
  } else {
    s.lk = a.seq_lens_kv ? clamp_len(a.seq_lens_kv[b], p.kv_cap) : a.s_kv;
  }
  s.off = a.mask_origin ? s.lk - s.lq : 0;
  return s;
}
// kv positions [lo, hi) that query row i sees (empty when lo >= hi)
__device__ __forceinline__ int64_t vis_hi(const PackedArgs& p, const SeqInfo& s, int64_t i) {
  return imin64(s.lk, i + s.off + p.a.next_tokens + 1);
}
__device__ __forceinline__ int64_t vis_lo(const PackedArgs& p, const SeqInfo& s, int64_t i) {
  return imax64(0, i + s.off - p.a.pre_tokens);
}

struct Block {
  int64_t kv0;  // first token of its first tile
  int tiles, unit;
};
__device__ __forceinline__ int seq_blocks(const PackedArgs& p, const SeqInfo& s) {
  return static_cast<int>((s.lq * p.g + kKCols - 1) / kKCols);
}
__device__ __forceinline__ Block block_of(const PackedArgs& p, const SeqInfo& s, int j) {
  const uint32_t cols = static_cast<uint32_t>(s.lq * p.g), c0 = static_cast<uint32_t>(j) * kKCols;
  const uint32_t c1 = min(c0 + kKCols, cols) - 1;
  const int64_t hi = vis_hi(p, s, c1 / static_cast<uint32_t>(p.g)), lo = vis_lo(p, s, c0 / static_cast<uint32_t>(p.g));
  Block b;
  b.kv0 = lo / kPKV * kPKV;
  b.tiles = hi > lo ? static_cast<int>((hi - b.kv0 + kPKV - 1) / kPKV) : 0;
  b.unit = c1 - c0 >= 4 * 32 ? 3 : 2;
  return b;
}
__device__ __forceinline__ int64_t block_cost(const Block& b) { return kKItem + static_cast<int64_t>(b.tiles) * b.unit; }
// tiles of an item that lie before its unit u
__device__ __forceinline__ int tiles_before(const Block& b, int64_t u) {
  return static_cast<int>((imax64(u, kKItem) - kKItem + b.unit - 1) / b.unit);
}

// Cost of sequence b's blocks, by one thread.
__device__ __forceinline__ int64_t seq_cost(const PackedArgs& p, int64_t b) {
  const SeqInfo s = seq_info(p, b);
  const int n = seq_blocks(p, s);
  int64_t c = 0;
  for (int j = 0; j < n; ++j) c += block_cost(block_of(p, s, j));
  return c;
}

// A lane per sequence, so that many short ones are planned at once (a wave each took 23 us for 256 single tokens,
// beside 39 of the main kernel); a sequence of many blocks is summed by its whole wave. Neighbouring sequences go to
// different waves.
__global__ __launch_bounds__(1024) void packed_plan_kernel(PackedArgs p) {
  __shared__ int64_t red[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t b0 = 0; b0 < p.a.b; b0 += 1024) {
    const int64_t b = b0 + 16 * lane + w;
    const bool wide = b < p.a.b && seq_blocks(p, seq_info(p, b)) > kKPlanBlocks;
    int64_t c = b < p.a.b && !wide ? seq_cost(p, b) : 0;
    for (uint64_t todo = __ballot(wide); todo; todo &= todo - 1) {
      const int k = __ffsll(static_cast<unsigned long long>(todo)) - 1;
      const SeqInfo s = seq_info(p, b0 + 16 * k + w);
      const int n = seq_blocks(p, s);
      int64_t x = 0;
      for (int j = lane; j < n; j += 64) x += block_cost(block_of(p, s, j));
      x = wave_sum64(x);
      if (lane == k) c = x;
    }
    if (b < p.a.b) p.pref[b + 1] = c * p.a.hkv;
  }
  __threadfence_block();
  __syncthreads();
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < p.a.b; b0 += 1024) {
    const int64_t b = b0 + threadIdx.x;
    const int64_t incl = block_incl_scan<false>(b < p.a.b ? p.pref[b + 1] : int64_t(0), red) + carry;
    if (b < p.a.b) p.pref[b + 1] = incl;
    __syncthreads();
    if (threadIdx.x == 1023) red[0] = incl;
    __syncthreads();
    carry = red[0];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.pref[0] = 0;
}

__device__ __forceinline__ int64_t q_offset(const PackedArgs& p, const int64_t* st, const SeqInfo& s, int64_t b, int64_t i,
                                            int head) {
  const int64_t qb = p.a.q_cum ? 0 : b;
  return qb * st[0] + (s.q_start + i) * st[1] + head * st[2];
}
__device__ __forceinline__ int64_t kv_offset(const PackedArgs& p, const int64_t* st, const SeqInfo& s, int64_t b, int64_t t,
                                             int kvh) {
  if (p.a.block_table) {
    const uint32_t bs = static_cast<uint32_t>(p.a.block_size), pg = static_cast<uint32_t>(t) / bs;
    return p.a.block_table[b * p.a.max_blocks + pg] * st[0] + (static_cast<uint32_t>(t) - pg * bs) * st[1] + kvh * st[2];
  }
  return (p.a.kv_cum ? 0 : b) * st[0] + (s.kv_base + t) * st[1] + kvh * st[2];
}

// One wave's column c of the item over tokens [t0, t1), in plain fp32 as the general kernel computes it: for the
// blocks whose MFMA result is not finite. A causal row's masked tokens enter the MFMA as 0 * v, which is NaN
// where a later token's value is infinite or NaN; here a row reads the tokens it sees only. Returns (m, l) in the
// log2 domain and this lane's dims lane, lane + 64.
template <int D, bool F16>
__device__ __forceinline__ void column_plain(const PackedArgs& p, const SeqInfo& s, int64_t b, int kvh, int64_t i, int head,
                                             int64_t t0, int64_t t1, int lane, float& m, float& l, float (&o)[D / 64]) {
  auto f32 = [](uint16_t x) { return F16 ? f16_to_f32(x) : bf16_to_f32(x); };
  const uint16_t* q = static_cast<const uint16_t*>(p.a.q1) + q_offset(p, p.a.q1_strides, s, b, i, head);
  const uint16_t* k = static_cast<const uint16_t*>(p.a.k1);
  const uint16_t* v = static_cast<const uint16_t*>(p.a.v);
  m = -INFINITY;
  l = 0.0f;
#pragma unroll
  for (int e = 0; e < D / 64; ++e) o[e] = 0.0f;
#pragma unroll 1
  for (int64_t c = t0; c < t1; c += 64) {
    const int64_t t = c + lane;
    const bool ok = t < t1;
    const uint16_t* kr = k + kv_offset(p, p.a.k1_strides, s, b, ok ? t : t1 - 1, kvh);
    float x = 0.0f;
#pragma unroll 1
    for (int d = 0; d < D; ++d) x += f32(kr[d]) * f32(q[d]);
    x = ok ? x * (p.neg_scale ? -p.scale_log2 : p.scale_log2) : -INFINITY;
    const float mc = wave_max(x);
    if (mc == -INFINITY) continue;
    const float mn = fmaxf(m, mc);
    const float al = m == -INFINITY ? 0.0f : exp2f(m - mn);
    const float pr = ok ? exp2f(x - mn) : 0.0f;
    l = l * al + wave_sum(pr);
#pragma unroll
    for (int e = 0; e < D / 64; ++e) o[e] *= al;
    const int n = static_cast<int>(imin64(64, t1 - c));
#pragma unroll 1
    for (int u = 0; u < n; ++u) {
      const float pu = __shfl(pr, u, 64);
      const uint16_t* vr = v + kv_offset(p, p.a.v_strides, s, b, c + u, kvh);
#pragma unroll
      for (int e = 0; e < D / 64; ++e) o[e] += pu * f32(vr[lane + 64 * e]);
    }
    m = mn;
  }
}

// Tiles [s0, s0 + n) of item (b, kvh, block j), whose first tile starts at token kv0. whole: the item's only
// segment, written out; else its partial goes to `slot`.
template <int D, bool F16>
__device__ __forceinline__ void packed_segment(const PackedArgs& p, char* smem, const SeqInfo& s, int b, int kvh, int j,
                                               int64_t kv0, int s0, int n, bool whole, int slot) {
  using T = PrefillTile<D>;
  using H = Half<F16>;
  using hv8 = typename H::v8;
  // fp16 has 2^-24 as its smallest step: P is kept 2^8 above 1 (the factor cancels in O / l), so that what is
  // rounded away lies 2^-32 below the row's largest term
  constexpr float kBias = F16 ? 8.0f : 0.0f;
  constexpr float kSlackUp = F16 ? 6.0f : 8.0f;  // how far a max may rise above the reference before it is raised
  const tai_fia_general_args& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, grp = lane >> 5;
  const uint32_t g = static_cast<uint32_t>(p.g);
  const uint32_t cols = static_cast<uint32_t>(s.lq * p.g);
  const uint32_t cw = static_cast<uint32_t>(j) * kKCols + 32 * w;  // the wave's first column
  const bool wave_ok = cw < cols;
  const bool ok = cw + col < cols;
  const uint32_t c = wave_ok ? min(cw + col, cols - 1) : 0;
  const uint32_t row = c / g;
  const int head = kvh * p.g + static_cast<int>(c - row * g);
  const uint32_t row_first = wave_ok ? cw / g : 0, row_last = wave_ok ? min(cw + 31, cols - 1) / g : 0;
  // this lane's visible tokens, and the wave's, relative to the segment's first tile
  const int64_t base = kv0 + static_cast<int64_t>(s0) * kPKV;
  auto rel = [&](int64_t t) { return static_cast<int>(imin64(imax64(t - base, 0), int64_t(1) << 30)); };
  const int qend = rel(vis_hi(p, s, row)), qbeg = min(rel(vis_lo(p, s, row)), qend);
  const int wave_hi = rel(vis_hi(p, s, row_last)), wave_lo = rel(vis_lo(p, s, row_first));
  const int clean_hi = rel(vis_hi(p, s, row_first)), clean_lo = rel(vis_lo(p, s, row_last));

  hv8 qf[D / 16];
  {
    const uint32_t sign = p.neg_scale ? 0x80008000u : 0u;
    const uint16_t* qp = static_cast<const uint16_t*>(a.q1) + q_offset(p, a.q1_strides, s, b, row, head) + 8 * grp;
#pragma unroll
    for (int kd = 0; kd < D / 16; ++kd) {
      uint4 u = *reinterpret_cast<const uint4*>(qp + 16 * kd);
      u.x ^= sign; u.y ^= sign; u.z ^= sign; u.w ^= sign;
      qf[kd] = __builtin_bit_cast(hv8, u);
    }
  }
  f32x16 acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) acc[i] = f32x16{};
  float m_run = -INFINITY, l_run = 0.0f;

  uint32_t koff[D / 16], voff[2][D / 32];
#pragma unroll
  for (int kd = 0; kd < D / 16; ++kd) koff[kd] = T::off(col, 2 * kd + grp);
  {
    const int h16 = lane >> 4, j16 = lane & 15;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      const int nb = 32 * dt + 16 * (h16 & 1) + 4 * (j16 & 3);
      const int r_lo = 4 * grp + (j16 >> 2);
      voff[0][dt] = T::kTile + T::off(r_lo, nb >> 3) + 2 * (nb & 7);
      voff[1][dt] = T::kTile + T::off(r_lo + 8, nb >> 3) + 2 * (nb & 7);
    }
  }
  const uint32_t lds0 = lds_u32(smem);

  const uint16_t* kbase = static_cast<const uint16_t*>(a.k1) + kvh * a.k1_strides[2];
  const uint16_t* vbase = static_cast<const uint16_t*>(a.v) + kvh * a.v_strides[2];
  if (!a.block_table) {
    const int64_t kb = a.kv_cum ? 0 : b;
    kbase += kb * a.k1_strides[0] + s.kv_base * a.k1_strides[1];
    vbase += kb * a.v_strides[0] + s.kv_base * a.v_strides[1];
  }
  const int32_t* btrow = a.block_table ? a.block_table + static_cast<int64_t>(b) * a.max_blocks : nullptr;
  const int bs = static_cast<int>(a.block_size);
  const int kstr = static_cast<int>(a.k1_strides[1]), vstr = static_cast<int>(a.v_strides[1]);
  const int lk = static_cast<int>(s.lk);
  const int lowest = rel(vis_lo(p, s, static_cast<uint32_t>(j) * kKCols / g));  // the block's lowest visible token
  // tile u of the segment -> ring slot u % 4; rows past the sequence's end load its last row, rows below the band
  // the lowest token that the block sees
  auto issue = [&](int u) __attribute__((always_inline)) {
    char* kst = smem + (u % kPStages) * 2 * T::kTile;
    const int t0 = static_cast<int>(base) + u * kPKV, first = max(0, lowest - u * kPKV);
    // a tile spans at most two pages (block_size >= 32, a multiple of 32): page ids through the scalar cache, whose
    // wait leaves the ring's loads alone
    int split = kPKV;  // rows from here on lie in the second page
    int64_t k0 = 0, v0 = 0, k1 = 0, v1 = 0;
    if (btrow) {
      const int pg = t0 / bs, slot0 = t0 - pg * bs;
      const bool two = slot0 + kPKV > bs && t0 + (bs - slot0) < lk;
      if (two) split = bs - slot0;
      if (first < split) {  // (a page wholly below the band may have left the table)
        const int64_t id0 = sload_i32(btrow + pg);
        k0 = id0 * a.k1_strides[0] + static_cast<int64_t>(slot0) * kstr;
        v0 = id0 * a.v_strides[0] + static_cast<int64_t>(slot0) * vstr;
      }
      if (two) {
        const int64_t id1 = sload_i32(btrow + pg + 1);
        k1 = id1 * a.k1_strides[0] - static_cast<int64_t>(split) * kstr;
        v1 = id1 * a.v_strides[0] - static_cast<int64_t>(split) * vstr;
      }
    } else {
      k0 = static_cast<int64_t>(t0) * kstr;
      v0 = static_cast<int64_t>(t0) * vstr;
    }
    const int last = lk - 1 - t0;
#pragma unroll
    for (int i = 0; i < T::kLoadsPerWave; ++i) {
      const int q = w * T::kLoadsPerWave + i;
      const int r = q * T::kRpi + lane / T::kCpr;
      const int ch = (lane % T::kCpr) ^ T::swz(r);
      const int rr = min(max(r, first), last);
      const int64_t ko = (rr < split ? k0 : k1) + static_cast<int64_t>(rr * kstr + 8 * ch);
      const int64_t vo = (rr < split ? v0 : v1) + static_cast<int64_t>(rr * vstr + 8 * ch);
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(kbase + ko), (lds_void_t*)(kst + q * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(vbase + vo), (lds_void_t*)(kst + T::kTile + q * 1024), 16, 0, 0);
    }
  };
  auto publish = [&](int u) __attribute__((always_inline)) {
    if (u + 1 < n) __builtin_amdgcn_s_waitcnt((T::kLoadsPerTile & 0xF) | ((T::kLoadsPerTile >> 4) << 14) | 0x70 | 0xF00);
    else __builtin_amdgcn_s_waitcnt(0x70 | 0xF00);
    const int left = lk - (static_cast<int>(base) + u * kPKV);
    if (left < kPKV) {  // rows past the sequence's end become zeros: a masked token adds 0 * 0
      const v4i_t z = {0, 0, 0, 0};
      const uint32_t kst = lds0 + (u % kPStages) * 2 * T::kTile;
#pragma unroll
      for (int i = 0; i < T::kLoadsPerWave; ++i) {
        const int q = w * T::kLoadsPerWave + i;
        if (q * T::kRpi + lane / T::kCpr >= left) {
          lds_write_b128<0>(kst + q * 1024 + 16 * lane, z);
          lds_write_b128<T::kTile>(kst + q * 1024 + 16 * lane, z);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  auto step = [&](uint32_t st, auto hc, int nstep) __attribute__((always_inline)) {
    constexpr int HALF = decltype(hc)::value;  // which 32 tokens of the tile
    v4i_t kf[D / 16];
    static_for<D / 16>([&](auto kdc) {
      lds_read_b128<HALF * 32 * T::kRowBytes>(kf[decltype(kdc)::value], st + koff[decltype(kdc)::value]);
    });
    lds_wait<0>();
#pragma unroll
    for (int kd = 0; kd < D / 16; ++kd) asm volatile("" : "+v"(kf[kd]));
    f32x16 sd = H::mfma32(__builtin_bit_cast(hv8, kf[0]), qf[0], f32x16{});
#pragma unroll
    for (int kd = 1; kd < D / 16; ++kd) sd = H::mfma32(__builtin_bit_cast(hv8, kf[kd]), qf[kd], sd);
    // V fragments of both 16-token blocks are read under the softmax
    v2i_t lo[2][D / 32], hi[2][D / 32];
    static_for<2>([&](auto kbc) {
      constexpr int kb = decltype(kbc)::value;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        lds_read_tr16<(2 * HALF + kb) * 16 * T::kRowBytes>(lo[kb][dt], st + voff[0][dt]);
        lds_read_tr16<(2 * HALF + kb) * 16 * T::kRowBytes>(hi[kb][dt], st + voff[1][dt]);
      }
    });
    const int t = 32 * nstep;
    if (t < clean_lo || t + 32 > clean_hi) {
      const int beg = min(32, max(0, qbeg - t)), lim = min(32, max(beg, qend - t));
      const uint32_t span = static_cast<uint32_t>(lim - beg);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int x = 8 * (r >> 2) + 4 * grp + (r & 3);
        sd[r] = static_cast<uint32_t>(x - beg) < span ? sd[r] : -INFINITY;
      }
    }
    float mx = sd[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sd[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * p.scale_log2 - kBias;
    if (__any(mx > m_run + kSlackUp)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= alpha;
      m_run = m_new;
    }
    const float neg_m = m_run == -INFINITY ? 0.0f : -m_run;
    hv8 ph[2], pl[2];
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sd[e], p.scale_log2, neg_m));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sd[e + 1], p.scale_log2, neg_m));
      l_run += p0 + p1;  // this lane's half of the row sum
      const typename H::v2 h = H::pack(p0, p1);
      const typename H::v2 r = H::pack(p0 - static_cast<float>(h[0]), p1 - static_cast<float>(h[1]));
      ph[e >> 3][e & 7] = h[0]; ph[e >> 3][(e & 7) + 1] = h[1];
      pl[e >> 3][e & 7] = r[0]; pl[e >> 3][(e & 7) + 1] = r[1];
    }
    lds_wait<0>();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) asm volatile("" : "+v"(lo[kb][dt]), "+v"(hi[kb][dt]));
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        const hv8 vv = __builtin_bit_cast(hv8, (v4i_t{lo[kb][dt][0], lo[kb][dt][1], hi[kb][dt][0], hi[kb][dt][1]}));
        acc[dt] = H::mfma32(vv, ph[kb], acc[dt]);
        acc[dt] = H::mfma32(vv, pl[kb], acc[dt]);
      }
    }
  };

  // every wave is done with the previous segment's ring
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (n > 0) issue(0);
  if (n > 1) issue(1);
  for (int u = 0; u < n; ++u) {
    publish(u);
    if (u + 2 < n) issue(u + 2);
    const int t = kPKV * u;
    if (!wave_ok || t >= wave_hi || t + kPKV <= wave_lo) continue;
    const uint32_t st = lds0 + static_cast<uint32_t>(u % kPStages) * 2 * T::kTile;
    if (t + 32 > wave_lo) step(st, std::integral_constant<int, 0>{}, 2 * u);
    if (t + 32 < wave_hi) step(st, std::integral_constant<int, 1>{}, 2 * u + 1);
  }
  if (!wave_ok) return;
  l_run += __shfl_xor(l_run, 32, 64);
  float* po = p.part_o + (static_cast<int64_t>(slot) * p.waves + w) * 32 * D;
  float* ml = p.part_ml + (static_cast<int64_t>(slot) * p.waves + w) * 32 * 2;
  const int64_t out_off = q_offset(p, a.out_strides, s, b, row, head);
  uint16_t* op = static_cast<uint16_t*>(a.out);
  float* lse = nullptr;
  if (a.lse) lse = a.lse + (a.q_cum ? (s.q_start + row) * a.hq + head : (static_cast<int64_t>(b) * a.hq + head) * a.s_q + row);

  bool odd = false;  // something infinite or NaN
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) odd = odd || !(fabsf(acc[i][r]) < INFINITY);
  if (__builtin_expect(__any(odd), 0)) {
    const int live_cols = static_cast<int>(min(32u, cols - cw));
#pragma unroll 1
    for (int x = 0; x < live_cols; ++x) {
      const int64_t i = __shfl(static_cast<int>(row), x, 64);
      const int hd = __shfl(head, x, 64);
      float m, l, o[D / 64];
      const int64_t t1 = imin64(vis_hi(p, s, i), base + static_cast<int64_t>(n) * kPKV);
      column_plain<D, F16>(p, s, b, kvh, i, hd, imax64(vis_lo(p, s, i), base), t1, lane, m, l, o);
      float f = 1.0f;
      if (whole) f = join_sink(a.sink, hd, m, l);
      const bool live = l > 0.0f;
#pragma unroll
      for (int e = 0; e < D / 64; ++e) {
        const int d = lane + 64 * e;
        if (whole) op[q_offset(p, a.out_strides, s, b, i, hd) + d] = H::bits(o[e] * (live ? f / l : 0.0f));
        else po[((d >> 3) * 64 + ((d >> 2) & 1) * 32 + x) * 4 + (d & 3)] = o[e];
      }
      if (lane == x) {
        if (!whole) { ml[2 * x] = m; ml[2 * x + 1] = l; }
        else if (lse) *lse = live ? (m + log2f(l)) * kLn2 : -INFINITY;
      }
    }
    return;
  }
  if (!whole) {
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *reinterpret_cast<f32x4*>(po + ((4 * i + r4) * 64 + lane) * 4) =
            f32x4{acc[i][4 * r4], acc[i][4 * r4 + 1], acc[i][4 * r4 + 2], acc[i][4 * r4 + 3]};
    if (grp == 0) {
      ml[2 * col] = m_run;
      ml[2 * col + 1] = l_run;
    }
    return;
  }
  if (!ok) return;
  const float f = join_sink(a.sink, head, m_run, l_run);
  const bool live = l_run > 0.0f;
  const float inv = live ? f / l_run : 0.0f;
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const typename H::v2 y0 = H::pack(acc[i][4 * r4] * inv, acc[i][4 * r4 + 1] * inv);
      const typename H::v2 y1 = H::pack(acc[i][4 * r4 + 2] * inv, acc[i][4 * r4 + 3] * inv);
      *reinterpret_cast<uint2*>(op + out_off + 32 * i + 8 * r4 + 4 * grp) =
          make_uint2(__builtin_bit_cast(uint32_t, y0), __builtin_bit_cast(uint32_t, y1));
    }
  if (lse && grp == 0) *lse = live ? (m_run + log2f(l_run)) * kLn2 : -INFINITY;
}

// Ranges of a launch of W units: at least 6 units each, so that every range inside an item holds a tile's first
// unit (a partial exists for each of them) and no workgroup starts for less than two tiles.
__device__ __forceinline__ int64_t ranges_of(const PackedArgs& p, int64_t W) { return imax64(W > 0 ? 1 : 0, imin64(p.cap, W / 6)); }
// The range a unit x of the launch's W belongs to, of R equal ones.
__device__ __forceinline__ int64_t range_of(int64_t x, int64_t W, int64_t R) { return ((x + 1) * R - 1) / W; }

template <int D, bool F16>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void packed_kernel(PackedArgs p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int64_t s_pref[kKPlanSeqs + 1];
  __shared__ int64_t red[16];
  const int lane = threadIdx.x & 63;
  const int64_t* pref = p.pref;
  if (p.plan_here) {
    // a thread per sequence; the plan kernel and its launch cost small calls more (4 tokens over 64: 15.8 us with it,
    // 13.1 without; 256 single tokens over 64, 16 / 8 heads of 64: 64 and 41 us). Up to 64 sequences one wave does
    // it, which saves the others' part of the scan, 0.4 us.
    if (p.a.b > 64 || threadIdx.x < 64) {
      const int64_t c = threadIdx.x < p.a.b ? seq_cost(p, threadIdx.x) * p.a.hkv : 0;
      const int64_t incl = p.a.b > 64 ? block_incl_scan<false>(c, red) : wave_incl_scan64(c, lane);
      s_pref[threadIdx.x + 1] = incl;
      if (threadIdx.x == 0) s_pref[0] = 0;
      if (blockIdx.x == 0) {  // for the merge
        if (threadIdx.x < p.a.b) p.pref[threadIdx.x + 1] = incl;
        if (threadIdx.x == 0) p.pref[0] = 0;
      }
    }
    __syncthreads();
    pref = s_pref;
  }
  // consecutive ranges, which share a kv head's tiles, run on one XCD
  const int64_t W = uniform64(pref[p.a.b]), R = ranges_of(p, W), per = (R + 7) / 8;
  const int64_t r = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || r >= R) return;
  const int64_t u0 = uniform64(r * W / R), u1 = uniform64((r + 1) * W / R);
  // the sequence of unit u0: 64 prefixes a look
  int64_t b = 0, cnt = p.a.b;
  while (cnt > 1) {
    const int64_t stride = (cnt + 63) / 64, idx = b + lane * stride;
    const uint64_t le = __ballot(lane * stride < cnt && pref[idx] <= u0);
    const int k = __popcll(le) - 1;
    b += k * stride;
    cnt = imin64(stride, cnt - k * stride);
  }
  b = uniform64(b);
  SeqInfo s = seq_info(p, b);
  int nblk = seq_blocks(p, s);
  int64_t x = uniform64(pref[b]);  // first unit of the item (b, kvh, j)
  const int64_t per_head = uniform64((pref[b + 1] - x) / p.a.hkv);
  int kvh = static_cast<int>((u0 - x) / per_head), j = 0;
  x += kvh * per_head;
  for (int j0 = 0;; j0 += 64) {
    const int64_t c = j0 + lane < nblk ? block_cost(block_of(p, s, j0 + lane)) : 0;
    const int64_t incl = wave_incl_scan64(c, lane);
    const uint64_t past = __ballot(x + incl > u0);
    if (past) {
      const int k = __ffsll(static_cast<unsigned long long>(past)) - 1;
      j = j0 + k;
      x += uniform64(__shfl(incl - c, k, 64));
      break;
    }
    x += uniform64(__shfl(incl, 63, 64));
  }
  kvh = __builtin_amdgcn_readfirstlane(kvh);
  j = __builtin_amdgcn_readfirstlane(j);
  int4 rec = make_int4(0, 0, 0, 0);
  for (;;) {
    const Block bl = block_of(p, s, j);
    const int64_t x1 = x + block_cost(bl);
    const int s0 = __builtin_amdgcn_readfirstlane(tiles_before(bl, imax64(u0 - x, 0)));
    const int s1 = __builtin_amdgcn_readfirstlane(u1 < x1 ? tiles_before(bl, u1 - x) : bl.tiles);
    const bool empty = bl.tiles == 0 && u0 <= x;  // nothing visible: its rows are written here
    if (s1 > s0 || empty) {
      const bool whole = s0 == 0 && s1 == bl.tiles, starts = s0 == 0 && !whole;
      const int rr = __builtin_amdgcn_readfirstlane(static_cast<int>(r));
      packed_segment<D, F16>(p, smem, s, __builtin_amdgcn_readfirstlane(static_cast<int>(b)), kvh, j, uniform64(bl.kv0), s0,
                             s1 - s0, __builtin_amdgcn_readfirstlane(whole) != 0,
                             2 * rr + __builtin_amdgcn_readfirstlane(starts));
      if (starts)
        rec = make_int4(static_cast<int>(b), kvh, j,
                        static_cast<int>(range_of(x + kKItem + static_cast<int64_t>(bl.tiles - 1) * bl.unit, W, R)));
    }
    x = x1;
    if (x >= u1) break;  // (an item left unfinished is the range's last)
    if (++j == nblk) {
      j = 0;
      if (++kvh == p.a.hkv) {
        kvh = 0;
        do {
          ++b;
          s = seq_info(p, b);
          nblk = seq_blocks(p, s);
        } while (nblk == 0);
      }
    }
  }
  if (threadIdx.x == 0) p.rec[r] = rec;
}

// Blocks 0 .. waves * cap - 1: 32 columns (wave w) of the item range r leaves unfinished, over its partials. The
// blocks after them write the rows that belong to no sequence (64 rows each).
template <int D, bool F16>
__global__ __launch_bounds__(256) void packed_merge_kernel(PackedArgs p) {
  using H = Half<F16>;
  const tai_fia_general_args& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t joins = static_cast<uint32_t>(p.waves) * p.cap;
  if (blockIdx.x >= joins) {
    // a lane looks at each of the 64 rows (one after another they took 5 us where all belonged to a sequence: 64
    // single tokens over 500 keys, 16 / 8 heads of 64, 42.1 us then, 36.8 now)
    const int64_t rows = a.q_cum ? a.s_q : a.b * a.s_q, v0 = static_cast<int64_t>(blockIdx.x - joins) * 64;
    const int64_t vl = v0 + lane, bl = a.q_cum ? 0 : vl / a.s_q;
    const bool spare = vl < rows && (a.q_cum ? vl >= a.q_cum[a.b - 1] : a.seq_lens_q && vl - bl * a.s_q >= a.seq_lens_q[bl]);
    for (uint64_t todo = __ballot(spare); todo; todo &= todo - 1) {
      const int64_t v = v0 + __ffsll(static_cast<unsigned long long>(todo)) - 1;
      const int64_t b = a.q_cum ? 0 : v / a.s_q, i = v - b * a.s_q;
      for (int e = 4 * tid; e < a.hq * D; e += 1024) {
        const int head = e / D;
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + b * a.out_strides[0] + i * a.out_strides[1] +
                                  head * a.out_strides[2] + (e - head * D)) = make_uint2(0, 0);
      }
      if (a.lse)
        for (int h = tid; h < a.hq; h += 256) a.lse[a.q_cum ? v * a.hq + h : (b * a.hq + h) * a.s_q + i] = -INFINITY;
    }
    return;
  }
  const int r = static_cast<int>(blockIdx.x / static_cast<uint32_t>(p.waves)), w = static_cast<int>(blockIdx.x) - r * p.waves;
  if (r >= ranges_of(p, p.pref[a.b])) return;
  const int4 rec = p.rec[r];
  if (rec.w == 0) return;
  const SeqInfo s = seq_info(p, rec.x);
  const uint32_t cols = static_cast<uint32_t>(s.lq * p.g), c = static_cast<uint32_t>(rec.z) * kKCols + 32 * w + (lane & 31);
  if (static_cast<uint32_t>(rec.z) * kKCols + 32 * w >= cols) return;
  constexpr int E = D / 32;  // 16-byte groups of a thread: groups (tid / 64) + 4e of the wave's D / 8
  float m = -INFINITY, l = 0.0f;
  f32x4 o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = f32x4{};
#pragma unroll 2
  for (int q = r; q <= rec.w; ++q) {
    const int64_t slot = 2 * q + (q == r ? 1 : 0);
    const float* po = p.part_o + (slot * p.waves + w) * 32 * D;
    f32x4 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = *reinterpret_cast<const f32x4*>(po + ((4 * e + (tid >> 6)) * 64 + lane) * 4);
    const float2 st = *reinterpret_cast<const float2*>(p.part_ml + ((slot * p.waves + w) * 32 + (lane & 31)) * 2);
    const float mn = fmaxf(m, st.x);
    const float c0 = m == -INFINITY ? 0.0f : exp2f(m - mn), c1 = st.x == -INFINITY ? 0.0f : exp2f(st.x - mn);
    l = l * c0 + st.y * c1;
#pragma unroll
    for (int e = 0; e < E; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[e][i] = o[e][i] * c0 + v[e][i] * c1;
    m = mn;
  }
  if (c >= cols) return;
  const uint32_t row = c / static_cast<uint32_t>(p.g);
  const int head = rec.y * p.g + static_cast<int>(c - row * p.g);
  const float f = join_sink(a.sink, head, m, l);
  const bool live = l > 0.0f;
  const float inv = live ? f / l : 0.0f;
  uint16_t* op = static_cast<uint16_t*>(a.out) + q_offset(p, a.out_strides, s, rec.x, row, head);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    f32x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = o[e][i] * inv;
    const typename H::v2 y0 = H::pack(y[0], y[1]), y1 = H::pack(y[2], y[3]);
    *reinterpret_cast<uint2*>(op + 8 * (4 * e + (tid >> 6)) + 4 * (lane >> 5)) =
        make_uint2(__builtin_bit_cast(uint32_t, y0), __builtin_bit_cast(uint32_t, y1));
  }
  if (a.lse && tid < 32)
    a.lse[a.q_cum ? (s.q_start + row) * a.hq + head : (static_cast<int64_t>(rec.x) * a.hq + head) * a.s_q + row] =
        live ? (m + log2f(l)) * kLn2 : -INFINITY;
}

// What the call can have at most, from what the host knows of it. A range has at least 6 units, so small calls have
// few ranges, and few rows fill few waves: the partials take 2 MB for 4 tokens over pages of 128 keys where 256
// ranges of 256 columns take 64 MB.
int packed_waves(const tai_fia_general_args& a) {
  return static_cast<int>(cdiv(imin64(a.s_q * (a.hq / a.hkv), kKCols), 32));
}
int packed_cap(const tai_fia_general_args& a) {
  const int64_t blocks = cdiv(a.s_q * (a.hq / a.hkv), kKCols);  // of a sequence; packed ones share them, each with a rest
  const int64_t items = a.hkv * (a.q_cum ? blocks + a.b : blocks * a.b);
  if (items >= 2 * kKWgs) return kKWgs;
  const int64_t tiles = cdiv(a.block_table ? a.max_blocks * a.block_size : a.s_kv, kPKV);
  return static_cast<int>(imax64(1, imin64(kKWgs, items * (kKItem + tiles * (packed_waves(a) > 4 ? 3 : 2)) / 6)));
}

struct PackedWs {
  size_t rec, part_o, part_ml, total;
};
PackedWs packed_ws(const tai_fia_general_args& a) {
  const size_t waves = 2 * static_cast<size_t>(packed_cap(a)) * packed_waves(a);
  PackedWs w;
  w.rec = (static_cast<size_t>(a.b + 1) * sizeof(int64_t) + 255) / 256 * 256;
  w.part_o = (w.rec + packed_cap(a) * sizeof(int4) + 255) / 256 * 256;
  w.part_ml = w.part_o + waves * 32 * a.dv * sizeof(float);
  w.total = w.part_ml + waves * 32 * 2 * sizeof(float);
  return w;
}

}  // namespace

// 16-bit q/k/v of head dim 64 or 128 with 16-byte rows, no explicit mask, pse, shared prefix or int8 anything;
// paged keys in pages of whole 32-token steps. 64 rows of K/V and all positions and columns stay in 32 bits.
bool packed_takes(const tai_fia_general_args& a) {
  const int64_t rows = a.q_cum ? a.s_q : a.b * a.s_q;
  return (a.dtype == TAI_DT_BF16 || a.dtype == TAI_DT_FP16) && a.kv_dtype == 0 && a.q_dtype == 0 && a.out_dtype == 0 &&
         (a.dk1 == 64 || a.dk1 == 128) && a.dv == a.dk1 && a.dk2 == 0 && a.hkv > 0 && a.hq > 0 && a.hq % a.hkv == 0 &&
         a.b > 0 && a.b < (int64_t(1) << 24) && a.s_q > 0 && a.s_kv > 0 && !a.mask && !a.pse && !a.k_prefix &&
         (a.mask_origin == 0 || a.mask_origin == 1) &&
         (a.block_table ? a.block_size >= 32 && a.block_size % 32 == 0 && a.max_blocks > 0 && a.seq_lens_kv && !a.kv_cum &&
                              a.block_size * a.max_blocks < (int64_t(1) << 30)
                        : (a.kv_cum != nullptr) == (a.q_cum != nullptr) && a.s_kv < (int64_t(1) << 30)) &&
         rows < (int64_t(1) << 30) && a.s_q * (a.hq / a.hkv) < (int64_t(1) << 30) && a.q1 && a.k1 && a.v && a.out &&
         aligned(a.q1, 16) && aligned(a.k1, 16) && aligned(a.v, 16) && aligned(a.out, 8) && rows_aligned(a.q1_strides, 8) &&
         rows_aligned(a.k1_strides, 8) && rows_aligned(a.v_strides, 8) && rows_aligned(a.out_strides, 4) &&
         a.k1_strides[1] >= 0 && a.k1_strides[1] < (int64_t(1) << 24) && a.v_strides[1] >= 0 &&
         a.v_strides[1] < (int64_t(1) << 24);
}

size_t packed_workspace(const tai_fia_general_args& a) { return packed_ws(a).total; }

int packed_run(const tai_fia_general_args& a, void* workspace, size_t ws_bytes, hipStream_t st) {
  const PackedWs w = packed_ws(a);
  if (workspace == nullptr || ws_bytes < w.total) {
    set_error("tai_fia_tiled: workspace of %zu bytes, need %zu", ws_bytes, w.total);
    return TAI_ERR_WORKSPACE;
  }
  PackedArgs p{};
  p.a = a;
  p.a.pre_tokens = imin64(imax64(a.pre_tokens, -kNoBound), kNoBound);
  p.a.next_tokens = imin64(imax64(a.next_tokens, -kNoBound), kNoBound);
  p.g = a.hq / a.hkv;
  p.cap = packed_cap(a);
  p.waves = packed_waves(a);
  p.kv_cap = a.block_table ? a.max_blocks * a.block_size : a.s_kv;
  // a zero scale makes every score zero, which the smallest normal scale gives up to rounding far below the output's
  // (written so that a NaN stays one)
  p.scale_log2 = fabsf(a.scale) * kLog2e;
  if (p.scale_log2 < 1.17549435e-38f) p.scale_log2 = 1.17549435e-38f;
  p.neg_scale = a.scale < 0.0f;
  char* ws = static_cast<char*>(workspace);
  p.pref = reinterpret_cast<int64_t*>(ws);
  p.rec = reinterpret_cast<int4*>(ws + w.rec);
  p.part_o = reinterpret_cast<float*>(ws + w.part_o);
  p.part_ml = reinterpret_cast<float*>(ws + w.part_ml);
  static const bool lds_ok = [] {
    auto set = [](const void* f, int bytes) {
      return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
    };
    const bool ok = set(reinterpret_cast<const void*>(&packed_kernel<64, false>), PrefillTile<64>::kLds) &&
                    set(reinterpret_cast<const void*>(&packed_kernel<64, true>), PrefillTile<64>::kLds) &&
                    set(reinterpret_cast<const void*>(&packed_kernel<128, false>), PrefillTile<128>::kLds) &&
                    set(reinterpret_cast<const void*>(&packed_kernel<128, true>), PrefillTile<128>::kLds);
    (void)hipGetLastError();
    return ok;
  }();
  if (!lds_ok) {
    set_error("tai_fia_tiled: the device cannot give a workgroup %d bytes of LDS", PrefillTile<128>::kLds);
    return TAI_ERR_LAUNCH;
  }
  p.plan_here = a.b <= kKPlanSeqs && cdiv(a.s_q * p.g, kKCols) <= kKPlanBlocks;
  if (!p.plan_here) packed_plan_kernel<<<1, 1024, 0, st>>>(p);
  const int64_t rows = a.q_cum ? a.s_q : a.b * a.s_q;
  const unsigned mgrid = static_cast<unsigned>(p.waves * p.cap + cdiv(rows, 64));
  const unsigned grid = static_cast<unsigned>(8 * cdiv(p.cap, 8));
  auto launch = [&](auto f16c) {
    constexpr bool F16 = decltype(f16c)::value;
    if (a.dk1 == 64) {
      packed_kernel<64, F16><<<grid, 512, PrefillTile<64>::kLds, st>>>(p);
      packed_merge_kernel<64, F16><<<mgrid, 256, 0, st>>>(p);
    } else {
      packed_kernel<128, F16><<<grid, 512, PrefillTile<128>::kLds, st>>>(p);
      packed_merge_kernel<128, F16><<<mgrid, 256, 0, st>>>(p);
    }
  };
  if (a.dtype == TAI_DT_FP16) launch(std::true_type());
  else launch(std::false_type());
  return launch_status("tai_fia_tiled");
}

}  // namespace tai
