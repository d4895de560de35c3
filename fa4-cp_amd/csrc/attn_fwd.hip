// Attention forward, host side: fa4cp_attn_fwd (one attention call) and fa4cp_ring_sweep_fwd
// (a whole ring sweep).  The kernels are in attn_kernels.h.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "attn_kernels.h"
#include "attn_split.h"

namespace fa4cp {
namespace {

//--------------------------------------------------------------------------------------
// host dispatch
//--------------------------------------------------------------------------------------
typedef void (*KernelFn)(AttnParams);

struct KernelChoice {
  KernelFn fn = nullptr;
  int threads = 0;   // workgroup size
  int rows = 0;      // query rows per workgroup (per head)
};

template <typename T>
KernelChoice pick16(int d, int hp, bool vt) {
  KernelChoice k;
  if (vt && (d == 64 || d == 128 || d == 256)) {
    k.threads = kPPThreads;
    k.rows = 32 * kPPWaves / hp;
#define FA4CP_PICK(DD)                                  \
  if (d == DD) {                                        \
    if (hp == 4) k.fn = attn_fwd_16bit_vt<T, DD, 4>;    \
    else if (hp == 2) k.fn = attn_fwd_16bit_vt<T, DD, 2>; \
    else k.fn = attn_fwd_16bit_vt<T, DD, 1>;            \
  }
    FA4CP_PICK(64)
    FA4CP_PICK(128)
    FA4CP_PICK(256)
#undef FA4CP_PICK
  } else if (d == 64 || d == 128) {
    k.threads = kPPThreads;
    k.rows = 32 * kPPWaves / hp;
#define FA4CP_PICK(DD)                                  \
  if (d == DD) {                                        \
    if (hp == 4) k.fn = attn_fwd_16bit_pp<T, DD, 4>;    \
    else if (hp == 2) k.fn = attn_fwd_16bit_pp<T, DD, 2>; \
    else k.fn = attn_fwd_16bit_pp<T, DD, 1>;            \
  }
    FA4CP_PICK(64)
    FA4CP_PICK(128)
#undef FA4CP_PICK
  } else if (d == 256) {
    k.threads = kThreads;
    k.rows = 32 * kWaves / hp;
    if (hp == 4) k.fn = attn_fwd_16bit<T, 256, 4>;
    else if (hp == 2) k.fn = attn_fwd_16bit<T, 256, 2>;
    else k.fn = attn_fwd_16bit<T, 256, 1>;
  }
  return k;
}

// The V^T kernel of head dim 64 with two workgroups per CU.
template <typename T>
auto pick_two(int hp) {
  return hp == 4 ? attn_fwd_16bit_vt<T, 64, 4, 2> : hp == 2 ? attn_fwd_16bit_vt<T, 64, 2, 2> : attn_fwd_16bit_vt<T, 64, 1, 2>;
}

KernelChoice pick8(int d, int hp, bool vt) {
  KernelChoice k;
  if (vt && (d == 128 || d == 256)) {
    k.threads = kPPThreads;
    k.rows = 32 * kPPWaves / hp;
    if (d == 128) {
      if (hp == 4) k.fn = attn_fwd_e4m3_vt<128, 4>;
      else if (hp == 2) k.fn = attn_fwd_e4m3_vt<128, 2>;
      else k.fn = attn_fwd_e4m3_vt<128, 1>;
    } else {
      if (hp == 4) k.fn = attn_fwd_e4m3_vt<256, 4>;
      else if (hp == 2) k.fn = attn_fwd_e4m3_vt<256, 2>;
      else k.fn = attn_fwd_e4m3_vt<256, 1>;
    }
  } else if (d == 128) {
    k.threads = kPPThreads;
    k.rows = 32 * kPPWaves / hp;
    if (hp == 4) k.fn = attn_fwd_e4m3_pp<4>;
    else if (hp == 2) k.fn = attn_fwd_e4m3_pp<2>;
    else k.fn = attn_fwd_e4m3_pp<1>;
  } else if (d == 256) {
    k.threads = kThreads;
    k.rows = 32 * kWaves / hp;
    if (hp == 4) k.fn = attn_fwd_e4m3<256, 4>;
    else if (hp == 2) k.fn = attn_fwd_e4m3<256, 2>;
    else k.fn = attn_fwd_e4m3<256, 1>;
  }
  return k;
}

}  // namespace
}  // namespace fa4cp

using namespace fa4cp;

// The kernels address within a tile by 32-bit byte offsets: up to 256 rows of a row-major
// operand, and rows 0..d-1 of V^T.
static bool tile_offsets_fit(int64_t row_stride, int esz, int d, int64_t vt_d_stride) {
  constexpr int64_t kMax = 0x7fffffffLL;
  return 256 * row_stride * esz < kMax && (int64_t)d * vt_d_stride * esz + 256 < kMax;
}

// Counters of the dynamic row tile hand-out (claim_block) of the sweeps and the per-step
// attention kernels: kClaimSlots slots of nine counters kClaimStride words apart, zero at
// module load.  Each launch takes the next slot of its GPU and its last workgroup to claim
// clears it, so a launch must have finished before the kClaimSlots-th launch after it on
// the same GPU (over all streams) starts; on one stream that always holds.  A launch captured
// in a graph keeps its slot: replays of it must not overlap.  In host code the array's name
// is a host-side stand-in: its device address is looked up once per device
// (hipGetSymbolAddress, with the device current).
constexpr int kClaimSlots = 64;
static __device__ __align__(256) unsigned sweep_claims[kClaimSlots * 9 * kClaimStride];

namespace {
constexpr int kClaimDevices = 64;
std::mutex g_claims_mu;
unsigned* g_claims_addr[kClaimDevices] = {};
std::atomic<unsigned> g_claims_next[kClaimDevices];

// The next claim slot of the stream's GPU, or NULL (the fixed order then) when the stream
// belongs to another GPU than the current one or the lookup fails.
unsigned* claim_slot(hipStream_t st) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kClaimDevices) return nullptr;
  if (st != nullptr) {
    int sdev = -1;
    if (hipStreamGetDevice(st, &sdev) != hipSuccess || sdev != dev) return nullptr;
  }
  unsigned* base;
  {
    std::lock_guard<std::mutex> lock(g_claims_mu);
    if (g_claims_addr[dev] == nullptr) {
      void* ptr = nullptr;
      if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(sweep_claims)) != hipSuccess || ptr == nullptr) {
        (void)hipGetLastError();
        return nullptr;
      }
      g_claims_addr[dev] = static_cast<unsigned*>(ptr);
    }
    base = g_claims_addr[dev];
  }
  const unsigned slot = g_claims_next[dev].fetch_add(1u, std::memory_order_relaxed) % kClaimSlots;
  return base + (size_t)slot * 9 * kClaimStride;
}
}  // namespace

extern "C" int fa4cp_attn_fwd(const fa4cp_attn_args* a, void* stream) {
  clear_error();
  if (a == nullptr) return set_error(FA4CP_EINVAL, "attn_fwd: null args");
  if (a->total_q > 0 && (!a->q || !a->k || !a->v || !a->out || !a->lse))  // NULL only with no query rows
    return set_error(FA4CP_EINVAL, "attn_fwd: null tensor pointer");
  if (a->h_q <= 0 || a->h_kv <= 0 || a->h_q % a->h_kv != 0)
    return set_error(FA4CP_EINVAL, "attn_fwd: h_q=%d must be a positive multiple of h_kv=%d",
                     a->h_q, a->h_kv);
  if (a->total_q < 0 || a->total_k < 0) return set_error(FA4CP_EINVAL, "attn_fwd: negative rows");
  if ((a->cu_q == nullptr) != (a->cu_k == nullptr))
    return set_error(FA4CP_EINVAL, "attn_fwd: cu_q and cu_k must both be given or both be NULL");
  const int nseq = a->cu_q ? a->nseq : 1;
  if (nseq < 1) return set_error(FA4CP_EINVAL, "attn_fwd: nseq must be >= 1");
  if (a->q_sel != FA4CP_SEL_ALL && a->q_sel != FA4CP_SEL_BACK_HALF &&
      a->q_sel != FA4CP_SEL_FRONT_HALF)
    return set_error(FA4CP_EINVAL, "attn_fwd: bad q_sel %d", a->q_sel);
  if (a->k_sel != FA4CP_SEL_ALL && a->k_sel != FA4CP_SEL_BACK_HALF &&
      a->k_sel != FA4CP_SEL_FRONT_HALF)
    return set_error(FA4CP_EINVAL, "attn_fwd: bad k_sel %d", a->k_sel);
  const int max_q_full = a->cu_q ? a->max_seqlen_q : a->total_q;
  if (max_q_full < 0) return set_error(FA4CP_EINVAL, "attn_fwd: bad max_seqlen_q");
  const int max_q = (a->q_sel == FA4CP_SEL_ALL) ? max_q_full : (max_q_full + 1) / 2;
  const int group = a->h_q / a->h_kv;
  const int hp = heads_per_wg(group);
  const int d = a->d;

  const bool use_vt = a->v_t != nullptr;
  if (use_vt) {
    if (a->vt_d_stride < fa4cp_vt_min_d_stride(a->total_k, nseq) || a->vt_d_stride % kVtPad != 0 ||
        ((uintptr_t)a->v_t % 16) != 0)
      return set_error(FA4CP_EINVAL, "attn_fwd: v_t must be 16-byte aligned with vt_d_stride a multiple "
                       "of %d and >= %lld", kVtPad, (long long)fa4cp_vt_min_d_stride(a->total_k, nseq));
  }
  KernelChoice kc;
  switch (a->dtype) {
    case FA4CP_BF16: kc = pick16<__bf16>(d, hp, use_vt); break;
    case FA4CP_FP16: kc = pick16<_Float16>(d, hp, use_vt); break;
    case FA4CP_E4M3: kc = pick8(d, hp, use_vt); break;
    default: return set_error(FA4CP_EUNSUPPORTED, "attn_fwd: unsupported dtype %d", a->dtype);
  }
  if (kc.fn == nullptr)
    return set_error(FA4CP_EUNSUPPORTED, "attn_fwd: head dim %d not implemented for dtype %d "
                     "(bf16/fp16: 64, 128, 256; e4m3: 128, 256)", d, a->dtype);
  // Fragment loads are 16 bytes wide (8 bytes for e4m3 V) and outputs are written 4
  // elements at a time, so every row / head start must keep that alignment.
  {
    const bool fp8 = a->dtype == FA4CP_E4M3;
    const int64_t qa = fp8 ? 16 : 8, ka = fp8 ? 16 : 8, va = 8;  // elements
    auto ok = [](const void* ptr, int64_t rs, int64_t hs, int64_t al, int esz) {
      return rs > 0 && hs > 0 && rs % al == 0 && hs % al == 0 &&
             ((uintptr_t)ptr % (uintptr_t)(al * esz)) == 0;
    };
    const int esz = fp8 ? 1 : 2;
    if (!ok(a->q, a->q_row_stride, a->q_head_stride, qa, esz) ||
        !ok(a->k, a->k_row_stride, a->k_head_stride, ka, esz) ||
        !ok(a->v, a->v_row_stride, a->v_head_stride, va, esz) ||
        !ok(a->out, a->o_row_stride, a->o_head_stride, 4, 2) || a->lse_row_stride < a->h_q)
      return set_error(FA4CP_EINVAL, "attn_fwd: misaligned pointer or stride (q/k rows and heads "
                       "need 16-byte alignment, v 8-byte for e4m3, out 8-byte; lse_row_stride >= h_q)");
    const int64_t rs = std::max(a->q_row_stride, std::max(a->k_row_stride, a->v_row_stride));
    if (!tile_offsets_fit(rs, esz, use_vt ? d : 0, a->vt_d_stride))
      return set_error(FA4CP_EINVAL, "attn_fwd: row or V^T stride too large for 32-bit tile offsets");
  }
  AttnParams p;
  p.q = a->q; p.k = a->k; p.v = a->v; p.out = a->out; p.lse = a->lse;
  p.q_rs = a->q_row_stride; p.q_hs = a->q_head_stride;
  p.k_rs = a->k_row_stride; p.k_hs = a->k_head_stride;
  p.v_rs = a->v_row_stride; p.v_hs = a->v_head_stride;
  p.o_rs = a->o_row_stride; p.o_hs = a->o_head_stride;
  p.lse_rs = a->lse_row_stride;
  p.cu_q = a->cu_q; p.cu_k = a->cu_k;
  p.nseq = nseq; p.total_q = a->total_q; p.total_k = a->total_k;
  p.h_kv = a->h_kv; p.group = group;
  p.causal = a->causal ? 1 : 0; p.q_sel = a->q_sel; p.k_sel = a->k_sel;
  p.scale = a->softmax_scale;
  p.qd = a->q_descale; p.kd = a->k_descale; p.vd = a->v_descale;
  p.vt = a->v_t; p.vt_ds = a->vt_d_stride;
  p.n_rt = (max_q + kc.rows - 1) / kc.rows;
  p.n_hg = a->h_kv * (group / hp);
  const int64_t blocks = (int64_t)p.n_hg * nseq * p.n_rt;
  if (blocks == 0 || a->total_q == 0) return FA4CP_OK;
  if (blocks > 0x7fffffffLL) return set_error(FA4CP_EINVAL, "attn_fwd: grid too large");
  p.n_blocks = (int)blocks;
  // one sequence: the dynamic hand-out of the row tiles, with a tenth more workgroups
  unsigned grid = (unsigned)blocks;
  p.claim = nullptr;
  const int64_t spare = (blocks / 8 + 9) / 10;
  if (nseq == 1 && blocks % 8 == 0 && blocks + 8 * spare <= 0x7fffffffLL) {
    p.claim = claim_slot((hipStream_t)stream);
    if (p.claim != nullptr) grid = (unsigned)(blocks + 8 * spare);
  }
  if (use_vt && attn_two_per_cu(a)) kc.fn = a->dtype == FA4CP_BF16 ? pick_two<__bf16>(hp) : pick_two<_Float16>(hp);
  hipLaunchKernelGGL(kc.fn, dim3(grid), dim3(kc.threads), 0, (hipStream_t)stream, p);
  return check_launch("attn_fwd");
}


// fa4cp_ring_sweep_fwd (kp == NULL) and fa4cp_ring_sweep_fwd_paged; with a workspace the split
// form where split_plan chooses it.
static int ring_sweep_launch(const fa4cp_sweep_args* a, const fa4cp_sweep_kpages* kp, void* ws, int64_t ws_bytes,
                             void* stream) {
  clear_error();
  if (a == nullptr) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: null args");
  const bool empty = a->total == 0;  // no rows: every pointer may be NULL
  if (!empty && (!a->q || !a->out || !a->lse)) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: null pointer");
  if (a->cp_size < 1 || a->cp_size > FA4CP_MAX_CP || a->cp_rank < 0 || a->cp_rank >= a->cp_size)
    return set_error(FA4CP_EINVAL, "ring_sweep_fwd: cp_rank %d / cp_size %d out of range (cp_size <= %d)",
                     a->cp_rank, a->cp_size, FA4CP_MAX_CP);
  for (int i = 0; i < a->cp_size; ++i)
    if (!empty && (!a->k[i] || !a->v_t[i])) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: null K / V^T of source %d", i);
  if (a->h_q <= 0 || a->h_kv <= 0 || a->h_q % a->h_kv != 0)
    return set_error(FA4CP_EINVAL, "ring_sweep_fwd: h_q=%d must be a positive multiple of h_kv=%d", a->h_q, a->h_kv);
  const int nseq = a->cu ? a->nseq : 1;
  if (nseq < 1 || a->total < 0) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: bad nseq / total");
  if (a->vt_d_stride < fa4cp_vt_min_d_stride(a->total, nseq) || a->vt_d_stride % kVtPad != 0)
    return set_error(FA4CP_EINVAL, "ring_sweep_fwd: vt_d_stride must be a multiple of %d and >= %lld", kVtPad,
                     (long long)fa4cp_vt_min_d_stride(a->total, nseq));
  const int max_len = a->cu ? a->max_seqlen : a->total;
  if (max_len < 0) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: bad max_seqlen %d", max_len);
  const int group = a->h_q / a->h_kv;
  const int hp = heads_per_wg(group);
  const int d = a->d;
  const bool fp8 = a->dtype == FA4CP_E4M3;
  if (a->dtype != FA4CP_BF16 && a->dtype != FA4CP_FP16 && !fp8)
    return set_error(FA4CP_EUNSUPPORTED, "ring_sweep_fwd: dtype %d (BF16 / FP16 / E4M3 only)", a->dtype);
  if (fp8 ? (d != 128 && d != 256) : (d != 64 && d != 128 && d != 256))
    return set_error(FA4CP_EUNSUPPORTED, "ring_sweep_fwd: head dim %d (64 / 128 / 256 for BF16 / FP16, 128 / 256 for E4M3)", d);
  {
    // element sizes: q / k 1 (e4m3) or 2; out 2 (bf16 for e4m3)
    const int esz = fp8 ? 1 : 2;
    auto ok = [](const void* ptr, int64_t rs, int64_t hs, int64_t al, int es) {
      return rs > 0 && hs > 0 && rs % al == 0 && hs % al == 0 && ((uintptr_t)ptr % (uintptr_t)(al * es)) == 0;
    };
    const int64_t qa = 16 / esz;  // 16-byte rows
    bool good = ok(a->q, a->q_row_stride, a->q_head_stride, qa, esz) &&
                ok(a->out, a->o_row_stride, a->o_head_stride, 4, 2) && a->lse_row_stride >= a->h_q;
    for (int i = 0; i < a->cp_size; ++i)
      good = good && ok(a->k[i], a->k_row_stride, a->k_head_stride, qa, esz) && ((uintptr_t)a->v_t[i] % 16) == 0;
    if (!good) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: misaligned pointer or stride");
    if (!tile_offsets_fit(std::max(a->q_row_stride, a->k_row_stride), esz, d, a->vt_d_stride))
      return set_error(FA4CP_EINVAL, "ring_sweep_fwd: row or V^T stride too large for 32-bit tile offsets");
  }
  SweepParams p;
  p.q = a->q; p.out = a->out; p.lse = a->lse;
  p.q_rs = a->q_row_stride; p.q_hs = a->q_head_stride;
  p.o_rs = a->o_row_stride; p.o_hs = a->o_head_stride; p.lse_rs = a->lse_row_stride;
  for (int i = 0; i < FA4CP_MAX_CP; ++i) {
    p.k[i] = i < a->cp_size ? a->k[i] : nullptr;
    p.vt[i] = i < a->cp_size ? a->v_t[i] : nullptr;
  }
  p.k_rs = a->k_row_stride; p.k_hs = a->k_head_stride; p.vt_ds = a->vt_d_stride;
  p.cu = a->cu; p.nseq = nseq; p.total = a->total;
  p.h_kv = a->h_kv; p.group = group;
  p.rank = a->cp_rank; p.S = a->cp_size;
  p.scale = a->softmax_scale;
  p.qd = fp8 ? a->q_descale : nullptr;
  p.kd = fp8 ? a->k_descale : nullptr;
  p.vd = fp8 ? a->v_descale : nullptr;
  for (int i = 0; i < FA4CP_MAX_CP; ++i) p.kpt[i] = nullptr;
  p.kpt_stride = p.page_size = p.num_pages = 0;
  const bool paged = kp != nullptr;
  if (paged) {
    if (kp->page_size <= 0 || kp->page_size % kVtPad != 0)
      return set_error(FA4CP_EINVAL, "ring_sweep_fwd_paged: page_size %d must be a positive multiple of %d",
                       kp->page_size, kVtPad);
    if (kp->num_pages < 0) return set_error(FA4CP_EINVAL, "ring_sweep_fwd_paged: num_pages %d < 0", kp->num_pages);
    if (kp->pt_stride < std::max(1, (max_len + kp->page_size - 1) / kp->page_size) || kp->pt_stride > 0x7fffffffLL)
      return set_error(FA4CP_EINVAL, "ring_sweep_fwd_paged: pt_stride %lld holds fewer pages than a sequence of %d "
                       "rows needs (or exceeds 2^31 - 1)", (long long)kp->pt_stride, max_len);
    for (int i = 0; i < a->cp_size; ++i)
      if (!empty && kp->page_table[i] == nullptr)
        return set_error(FA4CP_EINVAL, "ring_sweep_fwd_paged: page table of source %d is null", i);
    for (int i = 0; i < a->cp_size; ++i) p.kpt[i] = kp->page_table[i];
    p.kpt_stride = (int)kp->pt_stride;
    p.page_size = kp->page_size;
    p.num_pages = kp->num_pages;
  }
  const int rows = 32 * kPPWaves / hp;
  p.n_rt = (max_len + rows - 1) / rows;
  p.n_hg = a->h_kv * (group / hp);
  const int64_t blocks = (int64_t)p.n_hg * nseq * p.n_rt;
  if (blocks == 0 || empty) return FA4CP_OK;
  if (blocks > 0x7fffffffLL) return set_error(FA4CP_EINVAL, "ring_sweep_fwd: grid too large");
  p.n_blocks = (int)blocks;
  if (ws != nullptr) {
    const SplitPlan pl = split_plan(a);
    if (pl.split()) {
      const int64_t need = split_bytes(pl, p.n_hg, d);
      if (ws_bytes < need || ((uintptr_t)ws % 16) != 0)
        return set_error(FA4CP_EINVAL, "ring_sweep_fwd_ws: workspace of %lld bytes at %p; %lld bytes, 16-byte aligned, "
                         "needed", (long long)ws_bytes, ws, (long long)need);
      return launch_split(p, pl, ws, a->dtype, d, hp, paged, (hipStream_t)stream);
    }
  }
  void (*fn)(SweepParams) = nullptr;
  const bool pack = nseq > 1;  // several sequences: the gap-free row tile order
  const bool two = sweep_two_per_cu(a);
#define FA4CP_PICK_PK(KERNEL, H, ...)                                                       \
  {                                                                                         \
    if (paged) fn = pack ? KERNEL<__VA_ARGS__, H, true, true> : KERNEL<__VA_ARGS__, H, true, false>; \
    else fn = pack ? KERNEL<__VA_ARGS__, H, false, true> : KERNEL<__VA_ARGS__, H, false, false>;   \
  }
#define FA4CP_PICK_TWO(T, H)                                                                                     \
  {                                                                                                              \
    if (paged) fn = pack ? attn_fwd_16bit_sweep<T, 64, H, true, true, 2> : attn_fwd_16bit_sweep<T, 64, H, true, false, 2>; \
    else fn = pack ? attn_fwd_16bit_sweep<T, 64, H, false, true, 2> : attn_fwd_16bit_sweep<T, 64, H, false, false, 2>;     \
  }
#define FA4CP_PICK_64(T)                                                   \
  {                                                                        \
    if (two && hp == 4) FA4CP_PICK_TWO(T, 4)                                \
    else if (two && hp == 2) FA4CP_PICK_TWO(T, 2)                           \
    else if (two) FA4CP_PICK_TWO(T, 1)                                      \
    else FA4CP_PICK_HP(attn_fwd_16bit_sweep, T, 64)                         \
  }
#define FA4CP_PICK_HP(KERNEL, ...)                      \
  {                                                     \
    if (hp == 4) FA4CP_PICK_PK(KERNEL, 4, __VA_ARGS__)  \
    else if (hp == 2) FA4CP_PICK_PK(KERNEL, 2, __VA_ARGS__) \
    else FA4CP_PICK_PK(KERNEL, 1, __VA_ARGS__)          \
  }
  if (fp8) {
    if (d == 128) FA4CP_PICK_HP(attn_fwd_e4m3_sweep, 128)
    else FA4CP_PICK_HP(attn_fwd_e4m3_sweep, 256)
  } else if (a->dtype == FA4CP_BF16) {
    if (d == 64) FA4CP_PICK_64(__bf16)
    else if (d == 128) FA4CP_PICK_HP(attn_fwd_16bit_sweep, __bf16, 128)
    else FA4CP_PICK_HP(attn_fwd_16bit_sweep, __bf16, 256)
  } else {
    if (d == 64) FA4CP_PICK_64(_Float16)
    else if (d == 128) FA4CP_PICK_HP(attn_fwd_16bit_sweep, _Float16, 128)
    else FA4CP_PICK_HP(attn_fwd_16bit_sweep, _Float16, 256)
  }
#undef FA4CP_PICK_64
#undef FA4CP_PICK_TWO
#undef FA4CP_PICK_HP
#undef FA4CP_PICK_PK
  // dynamic hand-out of the lists' tails with a tenth more workgroups than row tiles (the
  // spares exit once every XCD's list is used up): one sequence, or up to 64 packed ones
  // where each XCD owns one head group
  unsigned grid = (unsigned)blocks;
  p.claim = nullptr;
  const int64_t per_xcd = blocks / 8;
  const int64_t spare = (per_xcd + 9) / 10;
  if ((!pack || (p.n_hg == 8 && nseq <= 64)) && blocks % 8 == 0 && blocks + 8 * spare <= 0x7fffffffLL) {
    p.claim = claim_slot((hipStream_t)stream);
    if (p.claim != nullptr) grid = (unsigned)(blocks + 8 * spare);
  }
  hipLaunchKernelGGL(fn, dim3(grid), dim3(kPPThreads), 0, (hipStream_t)stream, p);
  return check_launch(paged ? "ring_sweep_fwd_paged" : "ring_sweep_fwd");
}

extern "C" int fa4cp_ring_sweep_fwd(const fa4cp_sweep_args* a, void* stream) {
  return ring_sweep_launch(a, nullptr, nullptr, 0, stream);
}

extern "C" int fa4cp_ring_sweep_fwd_paged(const fa4cp_sweep_args* a, const fa4cp_sweep_kpages* kp, void* stream) {
  if (kp == nullptr) {
    clear_error();
    return set_error(FA4CP_EINVAL, "ring_sweep_fwd_paged: null k_pages");
  }
  return ring_sweep_launch(a, kp, nullptr, 0, stream);
}

extern "C" int fa4cp_ring_sweep_fwd_ws(const fa4cp_sweep_args* a, const fa4cp_sweep_kpages* kp, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  return ring_sweep_launch(a, kp, workspace, workspace_bytes, stream);
}
