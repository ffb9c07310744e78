// Tiled MFMA kernels for attention whose probabilities stay in fp32 precision: the MLA latent cache in
// bf16 (here), and GQA/MHA query blocks (attention_packed.hip). They take over from the general kernel
// (attention_general.hip) the calls tai_fia_tiled_workspace_size() names; the arguments and the meaning of
// every field are that kernel's.
//
// P enters the P.V MFMA as a bf16 pair, hi = bf16(p) and lo = bf16(p - hi): hi + lo carries 16 bits of p's
// mantissa, so the products' error is 2^-17 of a term, below the output's own rounding (2^-8). Scores, row
// sums, O and the partial results are fp32, as in the general kernel.
#include "attention_common.h"

namespace tai {

// attention_packed.hip: GQA/MHA query blocks of any layout
bool packed_takes(const tai_fia_general_args& a);
size_t packed_workspace(const tai_fia_general_args& a);
int packed_run(const tai_fia_general_args& a, void* workspace, size_t ws_bytes, hipStream_t st);

namespace {

// A query row of the call: its sequence and how many of its sequence's keys it sees (from the first on).
struct RowInfo {
  int64_t b, len;
  bool real;  // a row inside its sequence (padding rows write zeros and lse -inf)
};
__device__ __forceinline__ RowInfo row_info(const tai_fia_general_args& a, int64_t v) {
  int64_t b, i, lq;
  if (a.q_cum) {
    int64_t lo = 0, hi = a.b;  // the first sequence whose end lies past row v
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (a.q_cum[mid] > v) hi = mid; else lo = mid + 1;
    }
    if (lo >= a.b) return {0, 0, false};
    const int64_t end = imin64(a.q_cum[lo], a.s_q);
    const int64_t start = lo ? imax64(0, imin64(a.q_cum[lo - 1], end)) : 0;
    b = lo; i = v - start; lq = end - start;
  } else {
    // (both fit 32 bits: a call has at most 2^18 rows)
    b = static_cast<uint32_t>(v) / static_cast<uint32_t>(a.s_q); i = v - b * a.s_q;
    lq = a.seq_lens_q ? clamp_len(a.seq_lens_q[b], a.s_q) : a.s_q;
  }
  if (i >= lq) return {b, 0, false};
  const int64_t lk = clamp_len(a.seq_lens_kv[b], a.max_blocks * a.block_size);
  const int64_t off = a.mask_origin ? lk - lq : 0;
  return {b, imax64(0, imin64(lk, i + off + a.next_tokens + 1)), true};
}

// ============================================================================ MLA, bf16 latent
// One workgroup of 8 waves (2 per SIMD) owns 128 heads of one query row at a time: wave w holds heads
// 32 (w & 3) .. + 31 and half (w >> 2) of the latent dims, so its Q^T fragments (18 x 4 registers) and O^T
// accumulators (8 x 16) fit 256 registers and each SIMD has a second wave to run while one waits on LDS.
// Per 32-token step:
//   - the step's rows (1 KB latent + 128 B rope key) come global -> LDS by global_load_lds, already in bf16
//     and so without a conversion pass, through a ring of 3 stages, two steps ahead;
//   - each wave forms S^T over its half of the dims (v_mfma_f32_32x32x16_bf16), the two waves of a head
//     block swap their partial sums through LDS, and both run the softmax;
//   - O^T += C^T P^T over the wave's half of the latent, P as hi + lo.
// Query rows are independent items: a row's keys are the first len of its sequence, so several query tokens
// (and packed ones) need no mask. The rows' steps are cut into one equal range per workgroup; a row cut by a
// range's end leaves fp32 partials that mla_rows_merge_kernel joins, any other row is written here.
//
// Measured (32 sequences of 512-4096 tokens, 128 heads): 5.2 ms on the general kernel (a wave per row and head,
// nothing shared), 67 us here, of which the merge 13. A step takes 3.4 us against 1.4 us of MFMAs (100 per
// SIMD: 36 score, 64 P.V) because its score, softmax and P.V phases follow one another between the barriers;
// a segment costs about 25 us on top (query fragments, ring fill, 256 KB of partial per workgroup).
constexpr int kRStep = 32;
constexpr int kRWgs = 256;    // at most: one workgroup per CU
constexpr int kRHeads = 128;
constexpr int kRRing = 3;
constexpr int kRRope = kRStep * 1024;            // rope rows behind the latent rows of a stage
constexpr int kRStage = kRRope + kRStep * 128;
constexpr int kRSwap = kRRing * kRStage;         // [wave][4 KB] partial scores
constexpr int kRQr = kRSwap + 8 * 4096;          // [wave][2 KB] rope query fragments
constexpr int kRLds = kRQr + 8 * 2048;
constexpr int kRLoads = 5;                       // global_load_lds per wave and step
constexpr int kRScan = 256;                      // rows whose step prefix a workgroup scans by itself
constexpr float kRSlack = 8.0f;                  // log2 headroom of the lazily raised softmax max

struct MlaRowsArgs {
  tai_fia_general_args a;
  int64_t nv;     // query rows
  int hgroups, hcap;
  int64_t* pref;  // [nv + 1] balance units before each row
  float* part_o;  // [2 * ranges][hcap][512]: slot 2w of the row range w continues, 2w + 1 of the row it leaves unfinished
  float* part_ml; // [2 * ranges][hcap][2]
  float scale_log2;
  bool pref_ready;
};

// Balance units of a row: its 32-token steps, and SC for its start (see mla_rows; a template argument, as the
// kernel has no register left to hold it).
template <int SC>
__device__ __forceinline__ int64_t row_units(int64_t len) { return len > 0 ? (len + kRStep - 1) / kRStep + SC : 0; }
// Chunk c of tile row r sits at chunk c ^ X(r): 16 rows at one chunk hit 16 distinct 16-byte bank groups
// (score reads), and 4 consecutive rows x 4 chunks do too (transposing value reads). X(r + 16) = X(r).
__device__ __forceinline__ int row_x(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

template <int SC>
__global__ __launch_bounds__(1024) void mla_rows_prefix_kernel(MlaRowsArgs g) {
  __shared__ int64_t red[16];
  int64_t carry = 0;
  for (int64_t v0 = 0; v0 < g.nv; v0 += 1024) {
    const int64_t v = v0 + threadIdx.x;
    const int64_t n = v < g.nv ? row_units<SC>(row_info(g.a, v).len) : 0;
    const int64_t incl = block_incl_scan<false>(n, red) + carry;
    if (v < g.nv) g.pref[v + 1] = incl;
    __syncthreads();
    if (threadIdx.x == 1023) red[0] = incl;
    __syncthreads();
    carry = red[0];
    __syncthreads();
  }
  if (threadIdx.x == 0) g.pref[0] = 0;
}

// Where query row v's head writes its dims, and its lse.
__device__ __forceinline__ uint16_t* out_row(const tai_fia_general_args& a, int64_t qb, int64_t qt, int head) {
  return static_cast<uint16_t*>(a.out) + qb * a.out_strides[0] + qt * a.out_strides[1] + head * a.out_strides[2];
}
__device__ __forceinline__ void store_lse(const tai_fia_general_args& a, int64_t qb, int64_t qt, int head, float x) {
  if (a.lse) a.lse[a.q_cum ? qt * a.hq + head : (qb * a.hq + head) * a.s_q + qt] = x;
}
__device__ __forceinline__ void store4(uint16_t* p, f32x4 o, float inv) {
  const bf16x2_t y0 = __builtin_convertvector((f32x2_t){o[0] * inv, o[1] * inv}, bf16x2_t);
  const bf16x2_t y1 = __builtin_convertvector((f32x2_t){o[2] * inv, o[3] * inv}, bf16x2_t);
  *reinterpret_cast<uint2*>(p) = make_uint2(__builtin_bit_cast(uint32_t, y0), __builtin_bit_cast(uint32_t, y1));
}
// Steps [s0, s0 + nsteps) of query row v for head group hg; `whole`: the row's only segment, written out.
__device__ __forceinline__ void mla_rows_segment(const MlaRowsArgs& g, char* smem, int v, int b, int64_t len, int hg,
                                                 int64_t s0, int nsteps, bool whole, int slot) {
  const tai_fia_general_args& a = g.a;
  constexpr int NF = 18;  // K fragments of 16 dims per wave: 16 latent, 2 rope
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hb = w & 3, half = w >> 2;
  const int col = lane & 31, h = lane >> 5;
  const int hl = 32 * hb + col;
  const int head = hg * kRHeads + hl;
  const bool head_ok = head < a.hq;
  const bool wave_ok = hg * kRHeads + 32 * hb < a.hq;  // a wave without heads loads and keeps the barriers only

  const int64_t qb = a.q_cum ? 0 : b, qt = a.q_cum ? v : v - static_cast<int64_t>(b) * a.s_q;
  const uint32_t lds0 = lds_u32(smem);
  // a copy of the lane id the compiler cannot see through: what is derived from it is formed where it is used
  // and not kept in registers across the loop (the loop runs at the limit of 256, and the reload of a spilled
  // register waits for the ring's loads)
  auto here = [&]() __attribute__((always_inline)) {
    int ln;
    asm volatile("v_mov_b32 %0, %1" : "=v"(ln) : "v"(lane));
    return ln;
  };

  bf16x8 qf[NF - 2];  // (the two rope fragments live in LDS: all 18 would pass 256 registers)
  {
    const int hh = head_ok ? head : 0;
    const uint16_t* q1 = static_cast<const uint16_t*>(a.q1) + qb * a.q1_strides[0] + qt * a.q1_strides[1] +
                         hh * a.q1_strides[2] + 256 * half + 8 * h;
    const uint16_t* q2 = static_cast<const uint16_t*>(a.q2) + qb * a.q2_strides[0] + qt * a.q2_strides[1] +
                         hh * a.q2_strides[2] + 32 * half + 8 * h;
    // (lanes past the last head compute on head 0 and store nothing)
#pragma unroll
    for (int m = 0; m < NF - 2; ++m) qf[m] = as_bf16x8(*reinterpret_cast<const uint4*>(q1 + 16 * m));
#pragma unroll
    for (int m = 0; m < 2; ++m)
      lds_write_b128<0>(lds0 + kRQr + w * 2048 + m * 1024 + 16 * lane,
                        __builtin_bit_cast(v4i_t, *reinterpret_cast<const uint4*>(q2 + 16 * m)));
  }
  f32x16 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = f32x16{};
  float m_run = -INFINITY, l_run = 0.0f;

  const int64_t t_begin = s0 * kRStep;
  const int n_local = static_cast<int>(imin64(len - t_begin, static_cast<int64_t>(nsteps) * kRStep));
  // A step lies inside one page (block_size % 32 == 0). 64 page ids are held one per lane.
  const int32_t* btrow = a.block_table + static_cast<int64_t>(b) * a.max_blocks;
  const int bs = static_cast<int>(a.block_size);
  const int64_t pg_first = uniform64(t_begin / bs), pg_last = uniform64((t_begin + n_local - 1) / bs);
  int64_t win = pg_first;
  int my_page = lane <= pg_last - win ? btrow[win + lane] : 0;
  int cur_pg = 0, cur_slot = static_cast<int>(t_begin - pg_first * bs);
  const uint16_t* kc = static_cast<const uint16_t*>(a.k1);
  const uint16_t* kr = static_cast<const uint16_t*>(a.k2);
  const uint32_t lat_bytes = static_cast<uint32_t>(2 * a.k1_strides[1]), rope_bytes = static_cast<uint32_t>(2 * a.k2_strides[1]);

  // Every wave issues 5 loads a step: 4 latent rows of 1 KB and 8 rope rows of 128 B (waves 4-7 repeat the
  // rope rows of waves 0-3, the same bytes to the same place, so that one wait count fits all).
  auto issue = [&](int s) __attribute__((always_inline)) {
    char* st = smem + (s % kRRing) * kRStage;
    if (cur_pg == 64) {  // rare: the next 64 pages
      win += 64;
      cur_pg = 0;
      my_page = lane <= pg_last - win ? btrow[win + lane] : 0;
      __builtin_amdgcn_s_waitcnt(0x70 | 0xF00);  // here, so that the common path waits for nothing
    }
    const int page = __builtin_amdgcn_readfirstlane(__shfl(my_page, cur_pg, 64));
    const int slot0 = cur_slot;
    cur_slot += kRStep;
    if (cur_slot >= bs) { cur_slot = 0; ++cur_pg; }
    const int last = n_local - 1 - s * kRStep;  // rows past it load the last row, and are zeroed in LDS
    const char* lat = reinterpret_cast<const char*>(kc + page * a.k1_strides[0] + slot0 * a.k1_strides[1]);
    const char* rope = reinterpret_cast<const char*>(kr + page * a.k2_strides[0] + slot0 * a.k2_strides[1]);
    const int ln = here();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * w + i;
      const uint32_t off = static_cast<uint32_t>(min(row, last)) * lat_bytes + 16 * (ln ^ row_x(row));
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(lat + off), (lds_void_t*)(st + row * 1024), 16, 0, kCpolNt);
    }
    const int r8 = 8 * (w & 3), row = r8 + (ln >> 3);
    const uint32_t off = static_cast<uint32_t>(min(row, last)) * rope_bytes + 16 * ((ln & 7) ^ ((row >> 1) & 7));
    __builtin_amdgcn_global_load_lds((gbl_void_t*)(rope + off), (lds_void_t*)(st + kRRope + r8 * 128), 16, 0, kCpolNt);
  };
  // Rows of the sequence's last step past its end become zeros (each wave its own rows, once they have landed),
  // so that a masked token adds 0 * 0 whatever the cache holds there.
  auto zero_tail = [&](int s) __attribute__((always_inline)) {
    const int left = n_local - s * kRStep;
    const uint32_t st = lds0 + static_cast<uint32_t>(s % kRRing) * kRStage;
    const int ln = here();
    const v4i_t z = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * w + i >= left) lds_write_b128<0>(st + (4 * w + i) * 1024 + 16 * ln, z);
    if (8 * (w & 3) + (ln >> 3) >= left) lds_write_b128<0>(st + kRRope + 1024 * (w & 3) + 16 * ln, z);
  };

  // every wave is done with the previous segment's stages and swap area
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  issue(0);
  if (nsteps > 1) issue(1);
  auto publish = [&](int s) __attribute__((always_inline)) {
    // step s has landed once only step s + 1's loads are outstanding
    if (s + 1 < nsteps) __builtin_amdgcn_s_waitcnt(kRLoads | 0x70 | 0xF00);
    else __builtin_amdgcn_s_waitcnt(0x70 | 0xF00);
    if (n_local - s * kRStep < kRStep) zero_tail(s);
    // ... for every wave, and every wave is done with step s - 1 (its stage is refilled next)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + 2 < nsteps) issue(s + 2);
  };
  if (!wave_ok) {  // loads and barriers only
    for (int s = 0; s < nsteps; ++s) {
      publish(s);
      asm volatile("s_barrier" ::: "memory");
    }
    return;
  }
  for (int s = 0; s < nsteps; ++s) {
    publish(s);
    const uint32_t st = lds0 + static_cast<uint32_t>(s % kRRing) * kRStage;
    f32x16 sn = {};
    {
      // score fragment m: row col of the tile, dims 16m + 8h of the wave's half (16-byte chunks, see row_x)
      const int ln = here(), c32 = ln & 31, hh = ln >> 5;
      const uint32_t k_row = st + c32 * 1024 + 512 * half, k_pat = 16 * (hh ^ row_x(c32));
      const uint32_t r_row = st + kRRope + c32 * 128, r_pat = 16 * ((4 * half + hh) ^ ((c32 >> 1) & 7));
      // K fragments in batches of 2, the next batch's reads in flight
      constexpr int KB = 2, NKB = NF / KB;
      v4i_t kf[2][KB];
      auto kread = [&](auto mc, v4i_t& d) __attribute__((always_inline)) {
        constexpr int f = decltype(mc)::value, m = f - 2;  // rope first, so that its query fragments are free soon
        if constexpr (f >= 2) lds_read_b128<256 * (m >> 3)>(d, k_row + (k_pat ^ (32u * (m & 7))));
        else lds_read_b128<0>(d, r_row + (r_pat ^ (32u * f)));
      };
      v4i_t qr[2];
      static_for<2>([&](auto i) {
        lds_read_b128<1024 * decltype(i)::value>(qr[decltype(i)::value], lds0 + kRQr + w * 2048 + 16 * ln);
      });
      static_for<KB>([&](auto i) { kread(i, kf[0][decltype(i)::value]); });
      static_for<NKB>([&](auto bc) {
        constexpr int bi = decltype(bc)::value, cur = bi & 1;
        if constexpr (bi + 1 < NKB) {
          static_for<KB>([&](auto i) {
            kread(std::integral_constant<int, (bi + 1) * KB + decltype(i)::value>{}, kf[cur ^ 1][decltype(i)::value]);
          });
          lds_wait<KB>();
        } else {
          lds_wait<0>();
        }
        static_for<KB>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          asm volatile("" : "+v"(kf[cur][i]));
          constexpr int f = bi * KB + i;
          bf16x8 q;
          if constexpr (f >= 2) {
            q = qf[f - 2];
          } else {
            asm volatile("" : "+v"(qr[f]));  // (read before any K fragment: complete with the first)
            q = __builtin_bit_cast(bf16x8, qr[f]);
          }
          sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[cur][i]), q, sn, 0, 0, 0);
        });
      });
      // the LDS writes are inline asm, into which the compiler tracks no MFMA latency (18 wait states)
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(sn));
      static_for<4>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const f32x4 x = {sn[4 * i], sn[4 * i + 1], sn[4 * i + 2], sn[4 * i + 3]};
        lds_write_b128<1024 * i>(lds0 + kRSwap + w * 4096 + 16 * ln, __builtin_bit_cast(v4i_t, x));
      });
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    {
      v4i_t x[4];
      const uint32_t swap_in = lds0 + kRSwap + (w ^ 4) * 4096 + 16 * here();
      static_for<4>([&](auto ic) { lds_read_b128<1024 * decltype(ic)::value>(x[decltype(ic)::value], swap_in); });
      lds_wait<0>();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        asm volatile("" : "+v"(x[i]));
        const f32x4 o = __builtin_bit_cast(f32x4, x[i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) sn[4 * i + r] += o[r];  // (commutes: both waves hold the same sums)
      }
    }
    // ---- softmax of the step: this lane's tokens are 8i + 4h + r of head col
    float mx = -INFINITY;
    const int left = n_local - s * kRStep;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float x = 8 * (e >> 2) + 4 * h + (e & 3) < left ? sn[e] * g.scale_log2 : -INFINITY;
      sn[e] = x;
      mx = fmaxf(mx, x);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m_run + kRSlack)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= alpha;
      m_run = m_new;
    }
    const float neg_m = m_run == -INFINITY ? 0.0f : -m_run;
    bf16x8 ph[2], pl[2];
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float p0 = __builtin_amdgcn_exp2f(sn[e] + neg_m), p1 = __builtin_amdgcn_exp2f(sn[e + 1] + neg_m);
      l_run += p0 + p1;  // this lane's half of the row sum
      const bf16x2_t hi = __builtin_convertvector((f32x2_t){p0, p1}, bf16x2_t);
      const bf16x2_t lo = __builtin_convertvector(
          (f32x2_t){p0 - static_cast<float>(hi[0]), p1 - static_cast<float>(hi[1])}, bf16x2_t);
      ph[e >> 3][e & 7] = hi[0]; ph[e >> 3][(e & 7) + 1] = hi[1];
      pl[e >> 3][e & 7] = lo[0]; pl[e >> 3][(e & 7) + 1] = lo[1];
    }
    // ---- O^T += C^T P^T: fragment f = 8 kk + dt (32 dims of the wave's half, 16 tokens; two transposing reads),
    //      in batches of 2 with the next batch's reads in flight
    uint32_t v_row[2], v_pat[2];
    {
      const int ln = here(), gq = ln >> 4, j = ln & 15;
      const int cp = 2 * (gq & 1) + ((j >> 1) & 1);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int row = 4 * (ln >> 5) + (j >> 2) + 8 * u;
        v_row[u] = st + row * 1024 + 512 * half + 8 * (j & 1);
        v_pat[u] = 16 * (cp ^ row_x(row));
      }
    }
    constexpr int VB = 2, NVB = 16 / VB;
    v2i_t vlo[2][VB], vhi[2][VB];
    auto vread = [&](auto fc, v2i_t& lo, v2i_t& hi) __attribute__((always_inline)) {
      constexpr int f = decltype(fc)::value, kk = f / 8, dt = f % 8;
      lds_read_tr16<256 * (dt >> 2) + 16384 * kk>(lo, v_row[0] + (v_pat[0] ^ (64u * (dt & 3))));
      lds_read_tr16<256 * (dt >> 2) + 16384 * kk>(hi, v_row[1] + (v_pat[1] ^ (64u * (dt & 3))));
    };
    static_for<VB>([&](auto i) { vread(i, vlo[0][decltype(i)::value], vhi[0][decltype(i)::value]); });
    static_for<NVB>([&](auto bc) {
      constexpr int bi = decltype(bc)::value, cur = bi & 1;
      if constexpr (bi + 1 < NVB) {
        static_for<VB>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          vread(std::integral_constant<int, (bi + 1) * VB + i>{}, vlo[cur ^ 1][i], vhi[cur ^ 1][i]);
        });
        lds_wait<2 * VB>();
      } else {
        lds_wait<0>();
      }
      static_for<VB>([&](auto ic) {
        constexpr int i = decltype(ic)::value, f = bi * VB + i, kk = f / 8, dt = f % 8;
        asm volatile("" : "+v"(vlo[cur][i]), "+v"(vhi[cur][i]));
        const bf16x8 vv = __builtin_bit_cast(bf16x8, v4i_t{vlo[cur][i][0], vlo[cur][i][1], vhi[cur][i][0], vhi[cur][i][1]});
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, ph[kk], acc[dt], 0, 0, 0);
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, pl[kk], acc[dt], 0, 0, 0);
      });
    });
  }
  if (!head_ok) return;
  l_run += __shfl_xor(l_run, 32, 64);
  if (whole) {
    const float f = join_sink(a.sink, head, m_run, l_run);
    const bool live = l_run > 0.0f;
    const float inv = live ? f / l_run : 0.0f;
    uint16_t* po = out_row(a, qb, qt, head) + 256 * half + 4 * h;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = acc[dt][4 * i + r];
        store4(po + 32 * dt + 8 * i, o, inv);
      }
    if (half == 0 && h == 0) store_lse(a, qb, qt, head, live ? (m_run + log2f(l_run)) * kLn2 : -INFINITY);
    return;
  }
  float* po = g.part_o + (static_cast<int64_t>(slot) * g.hcap + hl) * 512 + 256 * half + 4 * h;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(po + 32 * dt + 8 * i) =
          f32x4{acc[dt][4 * i], acc[dt][4 * i + 1], acc[dt][4 * i + 2], acc[dt][4 * i + 3]};
  if (half == 0 && h == 0) {
    g.part_ml[(static_cast<int64_t>(slot) * g.hcap + hl) * 2] = m_run;
    g.part_ml[(static_cast<int64_t>(slot) * g.hcap + hl) * 2 + 1] = l_run;
  }
}

template <int SC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mla_rows_kernel(MlaRowsArgs g) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int64_t s_pref[kRScan + 1];
  __shared__ int64_t red[16];
  const int64_t nv = g.nv;
  if (!g.pref_ready) {  // nv <= kRScan: every workgroup scans the rows, the first keeps the prefix for the merge
    const int64_t n = threadIdx.x < nv ? row_units<SC>(row_info(g.a, threadIdx.x).len) : 0;
    const int64_t incl = block_incl_scan<false>(n, red);
    if (threadIdx.x == 0) s_pref[0] = 0;
    if (threadIdx.x < kRScan) s_pref[threadIdx.x + 1] = incl;
    __syncthreads();
    if (blockIdx.x == 0)
      for (int64_t i = threadIdx.x; i <= nv; i += 512) g.pref[i] = s_pref[i];
  }
  const int64_t* pref = g.pref_ready ? g.pref : s_pref;
  const int64_t S = uniform64(pref[nv]), W = S * g.hgroups;
  const int64_t R = imin64(kRWgs, W), wg = blockIdx.x;
  if (wg >= R) return;
  const int64_t g0 = wg * W / R, g1 = (wg + 1) * W / R;
  int hg = static_cast<int>(g0 / S);
  int64_t x = g0 - hg * S, v;
  {
    int64_t lo = 0, hi = nv;  // the last row with pref <= x (it has steps, since x < S)
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (pref[mid] <= x) lo = mid; else hi = mid;
    }
    v = uniform64(lo);
  }
  for (int64_t p = g0; p < g1;) {
    const int64_t p0 = uniform64(pref[v]), p1 = uniform64(pref[v + 1]);
    const int64_t seg = imin64(g1 - p, p1 - x);
    // units [u0, u0 + seg) of the row; the first SC carry no tokens
    const int64_t u0 = x - p0;
    const int64_t s0 = imax64(u0, SC) - SC, s1 = imax64(u0 + seg, SC) - SC;
    if (s1 > s0) {
      const RowInfo ri = row_info(g.a, v);
      // wave-uniform values, told to be: 64-bit divisions leave theirs in vector registers
      auto u32 = [](int64_t n) { return __builtin_amdgcn_readfirstlane(static_cast<int>(n)); };
      mla_rows_segment(g, smem, u32(v), u32(ri.b), uniform64(ri.len), u32(hg), uniform64(s0), u32(s1 - s0),
                       u32(s0 == 0 && s1 == p1 - p0 - SC) != 0, u32(2 * wg + (s0 == 0 ? 1 : 0)));
    }
    p += seg;
    x += seg;
    if (x == p1 && ++v == nv) { v = 0; x = 0; ++hg; }
  }
}

// Joins the partials of the rows that ranges cut, and writes the rows that see no key: one workgroup per
// (row, head), its four waves take every fourth partial (a long row of a small batch has hundreds), a lane
// owns 8 of the 512 dims.
template <int SC>
__global__ __launch_bounds__(256) void mla_rows_merge_kernel(MlaRowsArgs g) {
  const tai_fia_general_args& a = g.a;
  __shared__ float s_o[4][512];
  __shared__ float s_ml[4][2];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t v = blockIdx.x / a.hq;
  const int head = static_cast<int>(blockIdx.x - v * a.hq);
  const int hg = head / kRHeads, hl = head % kRHeads;
  const int64_t qb = a.q_cum ? 0 : v / a.s_q, qt = v - qb * a.s_q;
  uint16_t* po = out_row(a, qb, qt, head);
  const int64_t S = g.pref[g.nv], p0 = g.pref[v], p1 = g.pref[v + 1];
  if (p1 == p0) {
    if (wv == 0) {
      const bool real = row_info(a, v).real;
      float m = -INFINITY, l = 0.0f;
      if (real) (void)join_sink(a.sink, head, m, l);
      store4(po + 8 * lane, f32x4{}, 0.0f);
      store4(po + 8 * lane + 4, f32x4{}, 0.0f);
      if (lane == 0) store_lse(a, qb, qt, head, l > 0.0f ? (m + log2f(l)) * kLn2 : -INFINITY);
    }
    return;
  }
  const int64_t W = S * g.hgroups, R = imin64(kRWgs, W);
  const int64_t x0 = hg * S + p0 + SC, x1 = hg * S + p1;  // units of its steps
  const int64_t w0 = ((x0 + 1) * R - 1) / W, w1 = (x1 * R - 1) / W;  // ranges of the row's first and last step
  if (w0 == w1) return;  // written by its range
  float m = -INFINITY, l = 0.0f, o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = 0.0f;
#pragma unroll 2
  for (int64_t w = w0 + wv; w <= w1; w += 4) {
    const int64_t row = (2 * w + (w == w0 ? 1 : 0)) * g.hcap + hl;
    const f32x4 a0 = *reinterpret_cast<const f32x4*>(g.part_o + row * 512 + 8 * lane);
    const f32x4 a1 = *reinterpret_cast<const f32x4*>(g.part_o + row * 512 + 8 * lane + 4);
    const float pm = g.part_ml[2 * row], pl = g.part_ml[2 * row + 1];
    const float mn = fmaxf(m, pm);
    const float c = m == -INFINITY ? 0.0f : exp2f(m - mn), f = pm == -INFINITY ? 0.0f : exp2f(pm - mn);
    l = l * c + pl * f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = o[i] * c + a0[i] * f;
      o[4 + i] = o[4 + i] * c + a1[i] * f;
    }
    m = mn;
  }
  if (lane == 0) {
    s_ml[wv][0] = m;
    s_ml[wv][1] = l;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) s_o[wv][8 * lane + i] = o[i];
  __syncthreads();
  if (wv >= 2) return;
  // 128 threads, 4 dims each
  const int d = 4 * (64 * wv + lane);
  float M = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) M = fmaxf(M, s_ml[i][0]);
  float L = 0.0f;
  f32x4 r = {};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float f = s_ml[i][0] == -INFINITY ? 0.0f : exp2f(s_ml[i][0] - M);
    L += s_ml[i][1] * f;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] += s_o[i][d + q] * f;
  }
  const float f = join_sink(a.sink, head, M, L);
  const bool live = L > 0.0f;
  store4(po + d, r, live ? f / L : 0.0f);
  if (wv == 0 && lane == 0) store_lse(a, qb, qt, head, live ? (M + log2f(L)) * kLn2 : -INFINITY);
}

int64_t query_rows(const tai_fia_general_args& a) { return a.q_cum ? a.s_q : a.b * a.s_q; }

// A workgroup whose range begins another row loads query fragments, fills the ring and writes a partial again:
// about 7 steps' worth with 128 heads (32 sequences of 512-4096 tokens: 85 us with steps alone, 75 / 65 / 67 us
// with 4 / 7 / 10), less with few heads (100 sequences, 16 heads: 61, then 58 / 60 / 65 us).
int mla_rows_seg_cost(int64_t hq) { return hq > 64 ? 7 : 4; }

// The most ranges the call can have: one per unit, from the rows and the keys a block-table row can hold (no row is
// longer, see row_info). One sequence of up to 128 keys takes 6 MB of partials, not 128.
int mla_rows_cap(const tai_fia_general_args& a) {
  const int64_t rows = query_rows(a) * cdiv(a.hq, kRHeads);
  if (rows >= kRWgs || a.max_blocks >= kRWgs) return kRWgs;
  const int64_t steps = imin64(a.block_size / kRStep, kRWgs) * a.max_blocks;
  return static_cast<int>(imin64(kRWgs, rows * (steps + mla_rows_seg_cost(a.hq))));
}

struct MlaRowsWs {
  size_t part_o, part_ml, total;
};
MlaRowsWs mla_rows_ws(const tai_fia_general_args& a) {
  const size_t heads = 2 * static_cast<size_t>(mla_rows_cap(a)) * static_cast<size_t>(imin64(a.hq, kRHeads));
  MlaRowsWs w;
  w.part_o = (static_cast<size_t>(query_rows(a) + 1) * sizeof(int64_t) + 255) / 256 * 256;
  w.part_ml = w.part_o + heads * 512 * sizeof(float);
  w.total = w.part_ml + heads * 2 * sizeof(float);
  return w;
}

// 32 rows of a tile stay below 2^31 bytes
bool small_row(int64_t stride) { return stride >= 0 && stride < (int64_t(1) << 24); }

// The bf16 MLA calls: one kv head with a 512-wide latent that is key and value, a 64-wide rope key, pages of
// whole 32-token steps and 16-byte rows; no lower bound on the visible keys and no explicit mask (a row's keys
// are a prefix of its sequence).
bool mla_rows_takes(const tai_fia_general_args& a) {
  return a.dtype == TAI_DT_BF16 && a.kv_dtype == 0 && a.q_dtype == 0 && a.out_dtype == 0 && a.dk1 == 512 && a.dk2 == 64 &&
         a.dv == 512 && a.hkv == 1 && a.hq > 0 && a.hq <= 4096 && a.b > 0 && a.s_q > 0 && a.block_table && a.seq_lens_kv &&
         a.block_size > 0 && a.block_size % kRStep == 0 && a.block_size < (int64_t(1) << 30) && a.max_blocks > 0 &&
         !a.mask && !a.pse && !a.k_prefix && !a.kv_cum && a.v == a.k1 && a.v_strides[0] == a.k1_strides[0] &&
         a.v_strides[1] == a.k1_strides[1] && a.pre_tokens >= (int64_t(1) << 31) - 1 && a.q1 && a.q2 && a.k1 && a.k2 &&
         a.out && aligned(a.q1, 16) && aligned(a.q2, 16) && aligned(a.k1, 16) && aligned(a.k2, 16) && aligned(a.out, 8) &&
         rows_aligned(a.q1_strides, 8) && rows_aligned(a.q2_strides, 8) && rows_aligned(a.k1_strides, 8) &&
         rows_aligned(a.k2_strides, 8) && small_row(a.k1_strides[1]) && small_row(a.k2_strides[1]) &&
         rows_aligned(a.out_strides, 4) && query_rows(a) <= (int64_t(1) << 18) &&
         query_rows(a) * a.hq < (int64_t(1) << 31);
}

int mla_rows(const tai_fia_general_args& a, void* workspace, size_t ws_bytes, hipStream_t st) {
  MlaRowsArgs g{};
  g.a = a;
  g.a.next_tokens = imin64(imax64(a.next_tokens, -kNoBound), kNoBound);
  g.nv = query_rows(a);
  const MlaRowsWs w = mla_rows_ws(a);
  if (workspace == nullptr || ws_bytes < w.total) {
    set_error("tai_fia_tiled: workspace of %zu bytes, need %zu", ws_bytes, w.total);
    return TAI_ERR_WORKSPACE;
  }
  g.hgroups = static_cast<int>(cdiv(a.hq, kRHeads));
  g.hcap = static_cast<int>(imin64(a.hq, kRHeads));
  char* ws = static_cast<char*>(workspace);
  g.pref = reinterpret_cast<int64_t*>(ws);
  g.part_o = reinterpret_cast<float*>(ws + w.part_o);
  g.part_ml = reinterpret_cast<float*>(ws + w.part_ml);
  g.scale_log2 = a.scale * kLog2e;
  g.pref_ready = g.nv > kRScan;
  static const bool lds_ok = [] {
    auto set = [](const void* f) {
      return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kRLds) == hipSuccess;
    };
    const bool ok = set(reinterpret_cast<const void*>(&mla_rows_kernel<4>)) &&
                    set(reinterpret_cast<const void*>(&mla_rows_kernel<7>));
    (void)hipGetLastError();
    return ok;
  }();
  if (!lds_ok) {
    set_error("tai_fia_tiled: the device cannot give a workgroup %d bytes of LDS", kRLds);
    return TAI_ERR_LAUNCH;
  }
  auto launch = [&](auto sc) {
    constexpr int SC = decltype(sc)::value;
    if (g.pref_ready) mla_rows_prefix_kernel<SC><<<1, 1024, 0, st>>>(g);
    mla_rows_kernel<SC><<<mla_rows_cap(a), 512, kRLds, st>>>(g);
    mla_rows_merge_kernel<SC><<<static_cast<unsigned>(g.nv * a.hq), 256, 0, st>>>(g);
  };
  if (mla_rows_seg_cost(a.hq) == 7) launch(std::integral_constant<int, 7>());
  else launch(std::integral_constant<int, 4>());
  return launch_status("tai_fia_tiled");
}

}  // namespace
}  // namespace tai

using namespace tai;

extern "C" size_t tai_fia_tiled_workspace_size(const tai_fia_general_args* args) {
  if (!args) return 0;
  if (mla_rows_takes(*args)) return mla_rows_ws(*args).total;
  return packed_takes(*args) ? packed_workspace(*args) : 0;
}

extern "C" int tai_fia_tiled(const tai_fia_general_args* args, void* workspace, size_t ws_bytes, void* stream) {
  TAI_CHECK_ARG(args != nullptr, "tai_fia_tiled: null arguments");
  if (mla_rows_takes(*args)) return mla_rows(*args, workspace, ws_bytes, static_cast<hipStream_t>(stream));
  TAI_UNSUPPORTED(!packed_takes(*args), "tai_fia_tiled: a call tai_fia_tiled_workspace_size does not name");
  return packed_run(*args, workspace, ws_bytes, static_cast<hipStream_t>(stream));
}
