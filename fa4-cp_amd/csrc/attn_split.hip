// Split ring sweep: the fused sweep of attn_kernels.h with a row tile's keys shared out.
//
// A sweep of few row tiles leaves most of the chip idle: one workgroup walks all keys of 256
// (row, head) pairs, so a 2048-token ring of 8 heads is 16 workgroups, and 16384 tokens at 32
// heads are one workgroup per CU of which the back-half ones last four times as long as the
// front-half ones.  The split form hands a row tile's key tiles to up to ns_back / ns_front
// workgroups (about `chunk` tiles each, equal shares); each writes its rows' normalised fp32
// output and LSE to a slot of the workspace, and the last of a row tile's to finish merges its
// slots.  Shares are cut at tile granularity from the flattened segment list, alike for contiguous
// and paged K, so the two stay bit-identical.  split_plan (attn_plan.h) says how many.
#include "attn_kernels.h"
#include "attn_split.h"

namespace fa4cp {
namespace {

struct SweepSplit {
  SweepParams p;
  unsigned* done;  // [head group][row tile of the order]: shares finished; zero between launches
  float* po;       // [slots][256 (row, head) pairs x d], in Share::merge's order
  float* pl;       // [slots][256]
  int chunk;       // key tiles aimed at per workgroup
  int ns_back;     // grid workgroups of each row tile from n_front on
  int ns_front;    // of the row tiles before n_front (one sequence)
  int n_front;     // row tiles that meet no later source (one sequence; 0 when packed)
  int n_row;       // row tiles of a head group in the grid
  int per_hg;      // slots of a head group: a multiple of 8
};

// Slot (head group, r) of workgroup b.  Every XCD takes whole head groups, or every k-th slot
// of one where there are fewer head groups than XCDs, so that its L2 serves few kv heads; where
// the head groups do not divide over the XCDs they take turns.  Longest first on each.
__device__ __forceinline__ void split_slot(const SweepSplit& sp, int b, int& hg, int& r) {
  const int n_hg = sp.p.n_hg, x = b & 7, i = b >> 3;
  if (n_hg < 8 && 8 % n_hg == 0) {
    const int k = 8 / n_hg;
    hg = x / k;
    r = x % k + k * i;
  } else if (n_hg % 8 == 0) {
    const int m = n_hg >> 3;
    hg = x * m + i % m;
    r = i / m;
  } else {
    hg = b % n_hg;
    r = b / n_hg;
  }
}

// Cache policy sc1 (agent scope): stores go through to the memory that every XCD sees, loads
// are not served from a stale line of this XCD's L2.
constexpr int kAgent = 16;

// One workgroup's share of a row tile: tiles [lo, hi) of its flattened segment list, lo < hi.
template <int D, int BN, bool PAGED>
struct Share : RingSegments<BN, PAGED> {
  using Base = RingSegments<BN, PAGED>;
  static constexpr bool kSplit = true;
  static constexpr int kRows = 32 * kPPWaves;  // (row, head) pairs of a row tile
  int s_lo, t_lo, s_hi, t_hi, n;
  int shares, own;  // workgroups of the row tile, and which of them this one is
  float* po;        // the row tile's first slot
  float* pl;
  unsigned* done;
  // Takes share r - first of the at most ns; false: the row tile has fewer.  own_t, step_t,
  // late_t: key tiles of step 0, of a step <= rank, of a step > rank.
  __device__ __forceinline__ bool cut(const SweepSplit& sp, int i, int ns) {
    const SweepParams& p = sp.p;
    const int half = this->L >> 1, late = p.S - 1 - p.rank;
    const int last_row = min(this->row_tile0 + this->rows, this->L) - 1;
    const int own_t = last_row / BN + 1;
    const int step_t = (half + BN - 1) / BN;
    const int late_t = this->row_tile0 + this->rows > half ? (this->L + BN - 1) / BN : 0;
    const int total = own_t + p.rank * step_t + late * late_t;
    shares = max(1, min(ns, (total + sp.chunk - 1) / sp.chunk));
    own = i;
    if (i >= shares) return false;
    const int lo = total * i / shares, hi = total * (i + 1) / shares;
    n = hi - lo;
    auto find = [&](int x, int& s, int& t) __attribute__((always_inline)) {
      s = 0;
      t = x;
      if (t < own_t) return;
      t -= own_t;
      s = 1;
      if (t >= p.rank * step_t) {
        t -= p.rank * step_t;
        s = 1 + p.rank;
      }
      const int per = s == 1 && p.rank > 0 ? step_t : late_t;
      const int k = t / per;
      s += k;
      t -= k * per;
    };
    find(lo, s_lo, t_lo);
    find(hi - 1, s_hi, t_hi);
    ++t_hi;
    return true;
  }
  __device__ __forceinline__ int first() const { return t_lo; }
  __device__ __forceinline__ int nseg() const { return s_hi - s_lo + 1; }
  __device__ __forceinline__ int n_tiles() const { return n; }
  __device__ __forceinline__ StepSeg seg(int i) const {
    StepSeg g = Base::seg(s_lo + i);
    if (s_lo + i == s_hi) {
      g.tiles = min(g.tiles, t_hi);
      g.first_mask = min(g.first_mask, t_hi);
    }
    return g;
  }
  // The shares of a row tile meet here: each leaves its rows' normalised fp32 output and LSE in
  // its slot, and the last one to finish merges them all, in order (the same bits whoever is
  // last): out = sum_i a_i o_i / sum_i a_i with a_i = e^(lse_i - m), m the largest lse_i, lse = m +
  // log of that sum.  A share without a visible key has LSE -inf and adds nothing.  Returns
  // whether this workgroup is the last: o, inv and lse then hold the merged row.  Slot layout:
  // f32x4 16 dt .. of a wavefront's lanes side by side, so stores and loads are 1 KB runs.
  template <int NDT>
  __device__ __forceinline__ bool merge(f32x16 (&o)[NDT], float& inv, float& lse) const {
    if (shares == 1) return true;
    __shared__ int last;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int row = 4 * (32 * wave + (lane & 31)), at = 128 * D * wave + 16 * lane;  // bytes
    {
      const auto ro = make_rsrc32(po + (int64_t)own * kRows * D, 4 * kRows * D);
      const auto rl = make_rsrc32(pl + own * kRows, 4 * kRows);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = {o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv, o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv};
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ro, at + 1024 * (4 * dt + g), 0, kAgent);
        }
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(lse), rl, row, 0, kAgent);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      last = atomicAdd(done, 1u) == (unsigned)shares - 1u;
      if (last) atomicExch(done, 0u);
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(last) == 0) return false;
    const auto rl = make_rsrc32(pl, 4 * kRows * shares);
    float m = -INFINITY;
    for (int i = 0; i < shares; ++i)
      m = fmaxf(m, __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rl, row + 4 * kRows * i, 0, kAgent)));
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x16{};
    float sum = 0.f;
    for (int i = 0; i < shares; ++i) {
      const float l = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rl, row + 4 * kRows * i, 0, kAgent));
      const float a = l == -INFINITY ? 0.f : fast_exp2((l - m) * kLog2e);
      sum += a;
      const auto ro = make_rsrc32(po + (int64_t)i * kRows * D, 4 * kRows * D);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(ro, at + 1024 * (4 * dt + g), 0, kAgent));
#pragma unroll
          for (int e = 0; e < 4; ++e) o[dt][4 * g + e] = fmaf(a, v[e], o[dt][4 * g + e]);
        }
    }
    inv = sum > 0.f ? 1.f / sum : 0.f;
    lse = sum > 0.f ? m + logf(sum) : -INFINITY;
    return true;
  }
};

// What a split workgroup works on; false: nothing (past the grid's row tiles or its tile's shares).
template <int D, int HP, int BN, int ESZ, bool PAGED>
struct SplitWork {
  Share<D, BN, PAGED> geo;
  int head, r0, qs, L;
  __device__ __forceinline__ bool start(const SweepSplit& sp) {
    constexpr int RB = kPPWaves / HP;
    const SweepParams& p = sp.p;
    int hg, r, ns, first;
    split_slot(sp, (int)blockIdx.x, hg, r);
    const int back = (sp.n_row - sp.n_front) * sp.ns_back;  // slots of the first class
    int ri;
    if (r < back) {
      ns = sp.ns_back;
      ri = r / ns;
      first = ri * ns;
    } else {
      ns = sp.ns_front;
      ri = (r - back) / ns;
      first = back + ri * ns;
      ri += sp.n_row - sp.n_front;
    }
    if (ri >= sp.n_row) return false;
    int rt;
    int64_t vt_pos;
    if (p.nseq > 1) {
      if (!packed_row_tile(p, RB * 32, ri, geo.seq, rt, qs, L, vt_pos)) return false;
    } else {
      geo.seq = 0;
      rt = sp.n_row - 1 - ri;
      vt_pos = 0;
      seq_range(p.cu, 0, p.total, FA4CP_SEL_ALL, qs, L);
      if (rt * RB * 32 >= L) return false;
    }
    if (vt_pos + (L + kVtPad - 1) / kVtPad * kVtPad > p.vt_ds) return false;  // malformed cu: outside V^T
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int groups_per_kv = p.group / HP;
    const int kvh = hg / groups_per_kv;
    head = kvh * p.group + (hg - kvh * groups_per_kv) * HP + (wave % HP);
    geo.p = &p;
    geo.L = L;
    geo.row_tile0 = rt * RB * 32;
    geo.rows = RB * 32;
    geo.kvh = kvh;
    geo.k_off = ((PAGED ? 0 : (int64_t)qs * p.k_rs) + (int64_t)kvh * p.k_hs) * ESZ;
    geo.v_off = ((int64_t)kvh * D * p.vt_ds + vt_pos) * ESZ;
    r0 = geo.row_tile0 + (wave / HP) * 32;
    const int64_t row = ((int64_t)hg * sp.per_hg + first) * (32 * kPPWaves);
    geo.po = sp.po + row * D;
    geo.pl = sp.pl + row;
    geo.done = sp.done + (int64_t)hg * sp.n_row + ri;
    return geo.cut(sp, p.nseq > 1 ? turned_share(r - first, ri, ns) : r - first, ns);
  }
};

template <typename T, int D, int HP, bool PAGED, int WGS = 1>
__global__ __launch_bounds__(kPPThreads, 2 * WGS) void attn_fwd_16bit_sweep_split(SweepSplit sp) {
  const SweepParams& p = sp.p;
  SplitWork<D, HP, vt_bn<D>(), (int)sizeof(T), PAGED> w;
  if (!w.start(sp)) return;
  const T* q = reinterpret_cast<const T*>(p.q) + (int64_t)(w.qs + w.r0) * p.q_rs + (int64_t)w.head * p.q_hs;
  T* out = reinterpret_cast<T*>(p.out) + (int64_t)(w.qs + w.r0) * p.o_rs + (int64_t)w.head * p.o_hs;
  float* lse = p.lse + (int64_t)(w.qs + w.r0) * p.lse_rs + w.head;
  vt_pipeline<T, D, HP>(w.geo, q, p.q_rs, min(w.L - w.r0, 32), out, p.o_rs, lse, p.lse_rs, w.r0, w.L,
                        (int)(p.k_rs * (int64_t)sizeof(T)), (int)(p.vt_ds * (int64_t)sizeof(T)), p.scale);
}

// The split form of the e4m3 sweep, with the precision rules of attn_fwd_e4m3_sweep (they go by
// all keys of the row tile, so every share of it takes the same ones).
template <int D, int HP, bool PAGED>
__global__ __launch_bounds__(kPPThreads, 2) void attn_fwd_e4m3_sweep_split(SweepSplit sp) {
  const SweepParams& p = sp.p;
  SplitWork<D, HP, e8_bn<D>(), 1, PAGED> w;
  if (!w.start(sp)) return;
  const uint8_t* q = reinterpret_cast<const uint8_t*>(p.q) + (int64_t)(w.qs + w.r0) * p.q_rs + (int64_t)w.head * p.q_hs;
  __bf16* out = reinterpret_cast<__bf16*>(p.out) + (int64_t)(w.qs + w.r0) * p.o_rs + (int64_t)w.head * p.o_hs;
  float* lse = p.lse + (int64_t)(w.qs + w.r0) * p.lse_rs + w.head;
  const float c_q = p.scale * (p.qd ? p.qd[w.geo.kvh] : 1.f);
  const int k_rsb = (int)p.k_rs, vt_rsb = (int)p.vt_ds;
  const int qv = min(w.L - w.r0, 32), r0 = w.r0, L = w.L;
  const bool with_keys = (p.rank > 0 && (L >> 1) > 0) || (p.S - 1 > p.rank && w.geo.row_tile0 + w.geo.rows > (L >> 1));
  __shared__ E8Lds<D> lds;
  if (with_keys)
    e8_pipeline<D, HP, 0>(lds, w.geo, q, p.q_rs, qv, out, p.o_rs, lse, p.lse_rs, r0, L, k_rsb, vt_rsb, c_q);
  else if constexpr (D == 128) {
    if (r0 >= kPreciseRows)
      e8_pipeline<D, HP, 1>(lds, w.geo, q, p.q_rs, qv, out, p.o_rs, lse, p.lse_rs, r0, L, k_rsb, vt_rsb, c_q);
    else
      e8_pipeline<D, HP, 2>(lds, w.geo, q, p.q_rs, qv, out, p.o_rs, lse, p.lse_rs, r0, L, k_rsb, vt_rsb, c_q);
  } else {
    e8_pipeline<D, HP, 2>(lds, w.geo, q, p.q_rs, qv, out, p.o_rs, lse, p.lse_rs, r0, L, k_rsb, vt_rsb, c_q);
  }
}

int64_t split_rows(const SplitPlan& pl, int n_hg) { return (int64_t)n_hg * pl.per_hg * 32 * kPPWaves; }
int64_t done_bytes(int64_t words) { return (words * 4 + 255) / 256 * 256; }

}  // namespace

int64_t split_words(const SplitPlan& pl, int n_hg) { return (int64_t)n_hg * pl.n_row; }
int64_t split_bytes(const SplitPlan& pl, int n_hg, int d) {
  return done_bytes(split_words(pl, n_hg)) + split_rows(pl, n_hg) * (d + 1) * 4;
}

int launch_split(const SweepParams& p, const SplitPlan& pl, void* ws, int dtype, int d, int hp, bool paged,
                 hipStream_t st) {
  SweepSplit sp;
  sp.p = p;
  sp.p.claim = nullptr;
  sp.done = reinterpret_cast<unsigned*>(ws);
  sp.po = reinterpret_cast<float*>(reinterpret_cast<char*>(ws) + done_bytes(split_words(pl, p.n_hg)));
  sp.pl = sp.po + split_rows(pl, p.n_hg) * d;
  sp.chunk = pl.shares.chunk;
  sp.ns_back = pl.ns_back;
  sp.ns_front = pl.ns_front;
  sp.n_front = pl.n_front;
  sp.n_row = pl.n_row;
  sp.per_hg = pl.per_hg;
  void (*fn)(SweepSplit) = nullptr;
  const int64_t slots = (int64_t)p.n_hg * ((pl.n_row - pl.n_front) * pl.ns_back + pl.n_front * pl.ns_front);
  const bool two = two_per_cu(d, slots, kCus);
#define FA4CP_PICK_HP(KERNEL, ...)                                                          \
  {                                                                                         \
    if (hp == 4) fn = paged ? KERNEL<__VA_ARGS__, 4, true> : KERNEL<__VA_ARGS__, 4, false>; \
    else if (hp == 2) fn = paged ? KERNEL<__VA_ARGS__, 2, true> : KERNEL<__VA_ARGS__, 2, false>; \
    else fn = paged ? KERNEL<__VA_ARGS__, 1, true> : KERNEL<__VA_ARGS__, 1, false>;         \
  }
#define FA4CP_PICK_TWO(T, H) \
  fn = paged ? attn_fwd_16bit_sweep_split<T, 64, H, true, 2> : attn_fwd_16bit_sweep_split<T, 64, H, false, 2>;
#define FA4CP_PICK_16(T)                                               \
  {                                                                    \
    if (two && hp == 4) FA4CP_PICK_TWO(T, 4)                             \
    else if (two && hp == 2) FA4CP_PICK_TWO(T, 2)                        \
    else if (two) FA4CP_PICK_TWO(T, 1)                                   \
    else if (d == 64) FA4CP_PICK_HP(attn_fwd_16bit_sweep_split, T, 64)   \
    else if (d == 128) FA4CP_PICK_HP(attn_fwd_16bit_sweep_split, T, 128) \
    else FA4CP_PICK_HP(attn_fwd_16bit_sweep_split, T, 256)               \
  }
  if (dtype == FA4CP_E4M3) {
    if (d == 128) FA4CP_PICK_HP(attn_fwd_e4m3_sweep_split, 128)
    else FA4CP_PICK_HP(attn_fwd_e4m3_sweep_split, 256)
  } else if (dtype == FA4CP_BF16) {
    FA4CP_PICK_16(__bf16)
  } else {
    FA4CP_PICK_16(_Float16)
  }
#undef FA4CP_PICK_16
#undef FA4CP_PICK_TWO
#undef FA4CP_PICK_HP
  hipLaunchKernelGGL(fn, dim3((unsigned)(p.n_hg * pl.per_hg)), dim3(kPPThreads), 0, st, sp);
  return check_launch("ring_sweep_fwd_ws");
}

}  // namespace fa4cp

using namespace fa4cp;

extern "C" int64_t fa4cp_ring_sweep_workspace_bytes(const fa4cp_sweep_args* a, int32_t* clear_words) {
  clear_error();
  if (clear_words != nullptr) *clear_words = 0;
  if (a == nullptr) return set_error(FA4CP_EINVAL, "ring_sweep_workspace_bytes: null args");
  if (a->h_q <= 0 || a->h_kv <= 0 || a->h_q % a->h_kv != 0 || a->total < 0 || (a->cu != nullptr && (a->nseq < 1 || a->max_seqlen < 0)) ||
      a->cp_size < 1 || a->cp_size > FA4CP_MAX_CP || a->cp_rank < 0 || a->cp_rank >= a->cp_size || a->d <= 0)
    return set_error(FA4CP_EINVAL, "ring_sweep_workspace_bytes: bad shape total=%d h_q=%d h_kv=%d d=%d nseq=%d cp_rank=%d "
                     "cp_size=%d", a->total, a->h_q, a->h_kv, a->d, a->nseq, a->cp_rank, a->cp_size);
  const SplitPlan pl = split_plan(a);
  if (!pl.split()) return 0;
  const int n_hg = a->h_q / heads_per_wg(a->h_q / a->h_kv);
  if (clear_words != nullptr) *clear_words = (int32_t)split_words(pl, n_hg);
  return split_bytes(pl, n_hg, a->d);
}
