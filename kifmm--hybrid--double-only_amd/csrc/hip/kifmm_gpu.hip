/*
 * kifmm_gpu.hip -- create / evaluate / destroy of the MI355X KIFMM evaluator.
 *
 * kifmm_gpu_create is the counterpart of preproc() (fmm/evaluate--cuda.cu:1441-2239):
 * it derives the device work lists from the flattened tree and uploads
 * everything once.  kifmm_gpu_evaluate is the counterpart of run()
 * (fmm/run--cuda.cu:27-345): up (S2M + M2M), V (forward DFT,
 * translation spectra, spectral multiply-add, inverse DFT), W, X, down
 * (L2L + DC2DE + L2T) and the U-list, which writes the potentials to the
 * host as well, in that order on one stream (by default; enqueue_side).
 *
 * Device layout (HBM):
 *   src4 / trg4   gathered points as (x, y, z, w) double4 records
 *   uden/dchk/dden  node-major vectors, ld_e = n_e rounded up to 8 doubles,
 *                 zero padding
 *   chk           UC check potentials of one batch of columns (ld_uc)
 *   X / Y         source / target spectra, slot-major [slot][f][octant]:
 *                 slot 1 + b holds the 8 children of child block b (nodes
 *                 1+8b .. 8+8b); slot 0 is all zero and stands for a missing
 *                 neighbour
 *   T             translation spectra, frequency-major [f][343]
 *   operators     padded column-major, UE2UC and DE2DC stacked by octant
 */
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "kifmm_hip.h"
#include "../host/kifmm_internal.h"
#include "device_pool.hpp"
#include "kernels.hpp"

using namespace kifmm_dev;
using kifmm::set_error;

/* Device scratch of kifmm_gpu_direct_noalloc: the staged coordinates of up
 * to KIFMM_DIRECT_NOALLOC_MAX points, their sums and the chunks' partial
 * sums (direct_plan: at most DIR_ITEMS groups of them).  Every device the
 * library runs on holds its own copy until the process ends.  In host code
 * the array's name is not a device address: the per-device address comes
 * from hipGetSymbolAddress (scratch_address, called by kifmm_gpu_create with
 * the handle's device current) and only that address is passed on. */
constexpr int DIR_ITEMS = 4096;
static __device__ __align__(256) double scratch[4 * KIFMM_DIRECT_NOALLOC_MAX + 2 * DIR_T * DIR_ITEMS];

namespace {

inline int rup(int x, int m) { return (x + m - 1) / m * m; }

struct GemmList {
  int n = 0;
  int* in_off = nullptr;
  int* out_off = nullptr;
  int* sexp = nullptr;
};

struct LevelOps {
  GemmList m2m_a, m2m_b; /* UE2UC stack -> chk, UC2UE -> uden */
  GemmList l2l, dc2de;
};

}  // namespace

struct kifmm_gpu {
  int dev = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev[16] = {};
  /* an event for the start of the next launch (null: none); the phase being
   * launched (an index of ev) and how its last launch left
   * that event; ev_at[i]: the event that stands for boundary i, an earlier
   * one where a phase launched nothing (phase_end) */
  hipEvent_t start_ev = nullptr;
  int phase = 0, phase_state = 0, ev_at[16] = {};
  /* KIFMM_GPU_OVERLAP: the U-list on a second stream (default priority)
   * alongside up and V; fork / join events and the U-list's own timing */
  int overlap = 0;
  hipStream_t side = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr, su0 = nullptr, su1 = nullptr;
  int np = 0, n_e = 0, n_uc = 0, ld_e = 0, ld_uc = 0, lda_e = 0, lda_uc = 0, lda_l2l = 0, ld_surf = 0;
  int N = 0, H = 0, F = 0;
  int n_nodes = 0, n_src = 0, n_trg = 0, coincident = 0, max_depth = 0, precision = 0;
  DeviceArena mem;
  /* create time only: pinned staging of the uploads, and how much of it
   * copies not yet waited for use (null: straight from the caller's memory) */
  char* up_pin = nullptr;
  size_t up_used = 0;
  /* device data */
  double4 *src4 = nullptr, *trg4 = nullptr, *geo = nullptr;
  double *pot = nullptr, *uden = nullptr, *dchk = nullptr, *dden = nullptr, *chk = nullptr;
  double *UC2UE = nullptr, *UE2UC = nullptr, *DC2DE = nullptr, *DE2DC = nullptr;
  double *surf_ue = nullptr, *surf_uc = nullptr, *surf_de = nullptr, *surf_dc = nullptr;
  double2 *X = nullptr, *Y = nullptr, *T = nullptr, *That = nullptr, *tw = nullptr;
  /* mixed path: FP32 spectra, FP32 unit surfaces, FP32 leaf-local sources */
  float2 *Xf = nullptr, *Yf = nullptr, *Tf = nullptr;
  float *surf_uc32 = nullptr, *surf_de32 = nullptr;
  float4* src32 = nullptr;
  int *cube2surf = nullptr, *surf2cube = nullptr;
  int *snum = nullptr, *sbeg = nullptr, *depth = nullptr, *tag = nullptr;
  int *u_ptr = nullptr, *u_idx = nullptr; /* U-list CSR (node ids), for the close-pair search */
  /* work lists */
  int4* p2p_items = nullptr; int n_p2p = 0;
  int4* p2p_items64 = nullptr; int n_p2p64 = 0;
  int4* p2p_items5 = nullptr; int n_p2p5 = 0; /* <= P2P_MAXT5 targets: the FP64 Gram-form kernels */
  int4* p2p_itemsW = nullptr; int n_p2pW = 0, wave_g = 0; /* <= 8 wave_g targets (none: 0): k_p2p_wave */
  int4* p2p_itemsP = nullptr; int n_p2pP = 0; /* sibling pairs and single leaves: the mixed tau kernel */
  int* rng_ptr = nullptr; int2* rng = nullptr;
  int* p2p_counters = nullptr; /* 8, one per XCD: persistent U-list */
  int persist_grid[2] = {0, 0}; /* blocks of the persistent U-list form: difference, Gram */
  /* launch shapes (kifmm_gpu_set_tuning / kifmm_gpu_autotune) */
  int mix_lpb = 1; /* leaves per block of the mixed S2M / L2T */
  int p2p_form = KIFMM_P2P_STATIC;
  int had_fb = 8, had_auto = 1; /* kifmm_gpu_tuning.hadamard_fb, .hadamard_auto */
  int had_form = KIFMM_HAD_MFMA;
  int up_form = KIFMM_LEVEL_AUTO, down_form = KIFMM_LEVEL_AUTO;
  /* mixed path: per target, the U-list sources closer than MIX_CLOSE h */
  int* cptr = nullptr; int* cidx = nullptr;
  int close_listed = 0;
  int gram_u = 0;              /* the U-list runs on the FP64 Gram form: close pairs listed, FP64 path */
  double4* trg_gram = nullptr; /* (-2t', |t'|^2) per target, for gram_u and the W / X lists */
  double4* dc_gram = nullptr;  /* the same of the DC check surface in its node's frame */
  long long n_close = 0;
  int4* s2m_items = nullptr; int n_s2m = 0;
  GemmList s2m_gemm;
  std::vector<LevelOps> lv;
  int* vblocks = nullptr; int* vslot = nullptr; int n_vblocks = 0;
  int* hslot = nullptr; int n_hpar = 0;
  int4* hgroups = nullptr; int n_hgroups = 0;
  int* huslots = nullptr;
  unsigned char* hloc = nullptr;
  int4* wx_items = nullptr; int n_wx = 0;   /* k_wx items, two int4 each */
  int4* wx_red = nullptr; int n_wxred = 0;  /* k_wx_reduce items, two int4 each */
  int2* wx_rng = nullptr;                   /* their source ranges */
  int4* xs_items = nullptr; int n_xs = 0;   /* mixed path: k_x_surf items, two int4 each */
  int4* xs_red = nullptr; int n_xsred = 0;  /* and the reductions of split ones */
  double* wxpart = nullptr;                 /* chunk sums, WX_T per slot (k_x_surf: 64) */
  bool wx_targets = false;                  /* some item's points are targets */
  double wx_cost[2] = {0.0, 0.0};           /* of the W and of the X items (wx_plan) */
  int4* l2t_items = nullptr; int n_l2t = 0;
  size_t chk_cols = 0;
  double* ws = nullptr;
  size_t ws_len = 0;
  kifmm_work_counts counts{};
  /* wall ms of kifmm_gpu_create: host plan, upload, close-pair search,
   * other device set-up (translation spectra, Gram records), whole call */
  double create_ms[5] = {0, 0, 0, 0, 0};
  /* pinned host buffer of the potentials, and its device address: the last
   * kernels of an evaluation write it themselves */
  double* pinned = nullptr;
  double* pinned_dev = nullptr;
  /* HIP graph of the whole launch sequence (KIFMM_GPU_GRAPH) */
  int use_graph = 0;
  bool capturing = false;
  hipGraph_t graph[2] = {nullptr, nullptr}; /* [0]: the far-field sequence */
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
  /* copy-out: target cuts of the U-list chunks (leaf starts, 0 .. n_trg),
   * the first item of each chunk per item list, whether the items cover every
   * target, and the events that mark a chunk's potentials as on the host */
  std::vector<int> cuts;
  std::vector<int> chunk_beg[5];
  /* the items of list u_order_list over the whole range, in launch order (u_launch_order) */
  int4* u_order = nullptr;
  int u_order_list = -1;
  std::vector<double> u_cost[5]; /* prefix sums of the items' costs, per list */
  bool tiled = false;
  std::vector<hipEvent_t> cd_ev;
  hipEvent_t far_ev = nullptr, sdone_ev = nullptr;
  hipStream_t cstream = nullptr; /* copies of early chunks; taken by the first evaluation with some */
  hipEvent_t copied_ev = nullptr;
  /* the U-list's own sums when it runs on the second stream (overlap layout) */
  double* potU = nullptr;
  /* staging of kifmm_gpu_set_densities */
  double* den_stage = nullptr;
  double *den_pin = nullptr, *den_pin_dev = nullptr; /* pinned, and its device address: kifmm_gpu_set_densities */
  bool den_queued = false; /* a kernel that reads den_pin may not have run */
  /* this device's address of the file-scope scratch array */
  double* scratch = nullptr;
};

namespace {

#define HIP_TRY(expr)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) {                                                                \
      set_error(std::string(#expr) + ": " + hipGetErrorString(e_));                        \
      return KIFMM_EDEVICE;                                                                \
    }                                                                                      \
  } while (0)

/* Uploads of up to UP_STAGED bytes are staged through pinned memory and not
 * waited for: a copy from the caller's memory that is waited for, since the
 * source may be a temporary, took 12 us at 1 KB and 47 at 100 KB, staged 2 and 6.
 * From 1 MB both are bound by the copy. */
constexpr size_t UP_PIN = (size_t)1 << 20, UP_STAGED = (size_t)256 << 10;

template <typename T>
int dev_upload(kifmm_gpu* g, T** dst, const T* src, size_t n) {
  *dst = nullptr;
  const size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
  void* const p = g->mem.get(bytes);
  if (!p) {
    set_error("hipMalloc of " + std::to_string(bytes) + " bytes failed");
    return KIFMM_ENOMEM;
  }
  *dst = (T*)p;
  /* on the handle's (non-blocking) stream, so that the kernels that fill
   * the buffer at create time run after the clear: a null-stream memset is
   * not ordered with them */
  if (!src || !n) {
    HIP_TRY(hipMemsetAsync(p, 0, bytes, g->stream));
  } else if (g->up_pin && bytes <= UP_STAGED) {
    if (g->up_used + bytes > UP_PIN) {
      HIP_TRY(hipStreamSynchronize(g->stream));
      g->up_used = 0;
    }
    char* const stage = g->up_pin + g->up_used;
    g->up_used += (bytes + 63) / 64 * 64;
    std::memcpy(stage, src, bytes);
    HIP_TRY(hipMemcpyAsync(p, stage, bytes, hipMemcpyHostToDevice, g->stream));
  } else {
    HIP_TRY(hipMemcpyAsync(p, src, bytes, hipMemcpyHostToDevice, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream)); /* src may be a temporary */
    g->up_used = 0;
  }
  return KIFMM_OK;
}

template <typename T>
int dev_zero(kifmm_gpu* g, T** dst, size_t n) {
  return dev_upload<T>(g, dst, nullptr, n);
}

#define TRY(expr)            \
  do {                       \
    int r_ = (expr);         \
    if (r_ != KIFMM_OK) return r_; \
  } while (0)

/* boundary nodes of an np^3 grid on [-R,R]^3, x slowest (fmm/trans.cc:31-62):
 * rows x, y, z, then |p|^2 (row 3, for the Gram-form L2T) */
void host_surface(int np, double R, std::vector<double>& xyz, int ld) {
  const double step = 2.0 / (np - 1);
  int cnt = 0;
  for (int i = 0; i < np; i++)
    for (int j = 0; j < np; j++)
      for (int k = 0; k < np; k++) {
        if (!(i == 0 || i == np - 1 || j == 0 || j == np - 1 || k == 0 || k == np - 1)) continue;
        const double x = R * (-1.0 + i * step), y = R * (-1.0 + j * step), z = R * (-1.0 + k * step);
        xyz[cnt] = x;
        xyz[ld + cnt] = y;
        xyz[2 * ld + cnt] = z;
        xyz[3 * ld + cnt] = x * x + y * y + z * z;
        cnt++;
      }
}

int find_box(const kifmm_tree_view* t, int d, const int want[3]) {
  int cur = 0;
  while (t->depth[cur] < d && t->child[cur] != -1) {
    const int sh = d - t->depth[cur] - 1;
    const int o = (((want[0] >> sh) & 1) << 2) | (((want[1] >> sh) & 1) << 1) | ((want[2] >> sh) & 1);
    cur = t->child[cur] + o;
  }
  return cur;
}

/* The per-device address of `scratch`, looked up once per device (the
 * device must be current) and kept. */
int scratch_address(int dev, double** out) {
  static std::mutex mu;
  static std::vector<double*> addr;
  std::lock_guard<std::mutex> lock(mu);
  if (dev < 0) {
    set_error("scratch_address: invalid device");
    return KIFMM_EINVAL;
  }
  if ((size_t)dev >= addr.size()) addr.resize(dev + 1, nullptr);
  if (!addr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
      return KIFMM_EDEVICE;
    }
    addr[dev] = (double*)p;
  }
  *out = addr[dev];
  return KIFMM_OK;
}

/* Structural checks of a caller-supplied tree view: every index a kernel
 * derives from it must land inside the arrays it addresses. */
int check_view(const kifmm_tree_view* t) {
  const int nn = t->n_nodes;
  auto bad = [](const std::string& m) {
    set_error("kifmm_gpu_create: malformed tree view: " + m);
    return KIFMM_EINVAL;
  };
  if (t->n_levels < 2 || t->level_start[0] != 0 || t->level_start[t->n_levels - 1] != nn)
    return bad("level_start");
  for (int i = 0; i < nn; i++) {
    const int c = t->child[i];
    if (c != -1 && (c < 1 || c + 8 > nn || (c - 1) % 8 != 0)) return bad("child index");
    if (t->depth[i] < 0 || t->depth[i] > 30) return bad("depth");
    if (t->depth[i] + 2 > t->n_levels) return bad("depth vs levels");
    const int lim = 1 << t->depth[i];
    for (int k = 0; k < 3; k++)
      if (t->path[3 * i + k] < 0 || t->path[3 * i + k] >= lim) return bad("path");
    if (t->src_num[i] < 0 || t->src_beg[i] < 0 || (long)t->src_beg[i] + t->src_num[i] > t->n_src) return bad("source range");
    if (t->trg_num[i] < 0 || t->trg_beg[i] < 0 || (long)t->trg_beg[i] + t->trg_num[i] > t->n_trg) return bad("target range");
    if ((t->src_num[i] > 0 || t->trg_num[i] > 0) && c != -1) return bad("points on an inner node");
  }
  for (int d = 0; d + 1 < t->n_levels; d++)
    if (t->level_start[d] > t->level_start[d + 1]) return bad("level order");
  const int* ptrs[4] = {t->u_ptr, t->v_ptr, t->w_ptr, t->x_ptr};
  const int* idxs[4] = {t->u_idx, t->v_idx, t->w_idx, t->x_idx};
  for (int L = 0; L < 4; L++) {
    if (ptrs[L][0] != 0) return bad("list pointer");
    for (int i = 0; i < nn; i++)
      if (ptrs[L][i + 1] < ptrs[L][i]) return bad("list pointer order");
    unsigned out = 0; /* no early exit: the loop vectorises */
    for (int k = 0; k < ptrs[L][nn]; k++) out |= (unsigned)((unsigned)idxs[L][k] >= (unsigned)nn);
    if (out) return bad("list entry");
  }
  return KIFMM_OK;
}

/* Parts along K of a level's UE2UC stack: on the FP64 path short levels split
 * it over more blocks, whose waves otherwise run 304 (NP 6) or 112 (NP 4) MFMA
 * steps one after another: with the sum over the parts in UC2UE a level of 64
 * parents takes 11.2 us at NP 4 instead of 14.8.  The mixed path keeps one order of
 * summation. */
constexpr int M2M_PARTS = 4;
inline int m2m_parts(int ncols, bool mixed) { return !mixed && ncols < 1024 ? M2M_PARTS : 1; }
constexpr int LEAF_SPLIT = 8192; /* leaves below which the FP64 leaf UC2UE is a k_level_op */

/* Everything the device needs, derived on the host from the tree view.
 * make_plan() touches no device; upload() copies a checked plan. */
struct HostGemm {
  std::vector<int> in, out, sexp;
};
struct HostLevel {
  HostGemm m2m_a, m2m_b, l2l, dc2de;
};
struct Plan {
  int np = 0, n_e = 0, n_uc = 0, ld_e = 0, ld_uc = 0, lda_e = 0, lda_uc = 0, lda_l2l = 0, ld_surf = 0;
  int N = 0, H = 0, F = 0, nblk = 0, max_depth = 0;
  std::vector<int4> p2p_items, p2p_items64, p2p_items5, p2p_itemsP, p2p_itemsW;
  int wave_g = 0;
  /* copy-out chunks: target cut points (leaf starts, 0 .. n_trg) and, per
   * item list (<= P2P_MAXT, <= P2P_MAXT / 2, <= P2P_MAXT5, pairs), the
   * first item of each chunk */
  std::vector<int> cuts;
  std::vector<int> chunk_beg[5];
  std::vector<double> u_cost[5];
  std::vector<int4> u_order;
  int u_order_list = -1;
  bool tiled = false;
  std::vector<int> rng_ptr;
  std::vector<int2> rng;
  std::vector<int4> s2m_items;
  HostGemm s2m_gemm;
  std::vector<HostLevel> lv;
  size_t chk_cols = 0;
  size_t ws_len = 0;
  std::vector<int> vblocks, vslot, hnbr, hslot, l2t;
  std::vector<int4> wx_items, wx_red, xs_items, xs_red; /* two int4 per item */
  std::vector<int2> wx_rng;
  int wx_slots = 0, xs_slots = 0;
  bool wx_targets = false; /* some W / X item's points are targets */
  double wx_cost[2] = {0.0, 0.0};
  std::vector<int4> l2t_items;
  std::vector<int4> hgroups;
  std::vector<int> huslots;
  std::vector<unsigned char> hloc, hoct; /* union index; octant of the neighbour's position */
  kifmm_work_counts wc{};
};

bool offsets_ok(const std::vector<int>& off, long len_read, long buf_len) {
  for (int o : off)
    if (o < 0 || (long)o + len_read > buf_len) return false;
  return true;
}

/* Targets of a U-list work item: it.z holds n_A | n_B << 16, with n_B = 0
 * but for the sibling pairs of the pair list. */
inline int item_targets(const int4& it) { return (it.z & 0xffff) + (it.z >> 16); }

/* The mixed tau kernel's item list.  Two sibling leaves A and B = A + 1
 * (octants 2m and 2m + 1 of one parent, so adjacent) at one depth, whose
 * targets follow each other and fill at most P2P_MAXT5 / 16 groups of 16
 * (each leaf's own groups), are one item: three source sets follow each
 * other in rng_ptr (the boxes in both U-lists, in A's order; those only in
 * A's; those only in B's) and the item is (first set, A's first target,
 * n_A | n_B << 16, A).  Every other leaf keeps its items of the P2P_MAXT5
 * list (its own set, n_B = 0).  A pair stages each shared source once for
 * the targets of both leaves: 36 boxes of sources instead of 2 x 27 for
 * same-size neighbours. */
int pair_items(const kifmm_tree_view* t, Plan& P) {
  const int nn = t->n_nodes;
  auto trg_leaf = [&](int i) { return i >= 0 && i < nn && t->child[i] == -1 && t->trg_num[i] > 0; };
  std::vector<char> mark(nn, 0);
  std::vector<int> sh, oa, ob;
  auto add_set = [&](const std::vector<int>& boxes) {
    for (int s : boxes) {
      const int b = t->src_beg[s], n = t->src_num[s];
      if (n <= 0) continue;
      if ((int)P.rng.size() > P.rng_ptr.back() && P.rng.back().x + P.rng.back().y == b) P.rng.back().y += n;
      else P.rng.push_back(make_int2(b, n));
    }
    P.rng_ptr.push_back((int)P.rng.size());
  };
  const std::vector<int4>& L5 = P.p2p_items5; /* in leaf order */
  size_t k5 = 0;
  P.p2p_itemsP.clear();
  for (int i = 0; i < nn; i++) {
    if (!trg_leaf(i)) continue;
    const int j = i + 1, nA = t->trg_num[i];
    const bool pair = i >= 1 && (i - 1) % 2 == 0 && trg_leaf(j) && (i - 1) / 8 == (j - 1) / 8 &&
                      t->depth[i] == t->depth[j] && t->trg_beg[j] == t->trg_beg[i] + nA &&
                      (nA + 15) / 16 + (t->trg_num[j] + 15) / 16 <= P2P_MAXT5 / 16;
    while (k5 < L5.size() && L5[k5].w < i) k5++;
    if (!pair) {
      while (k5 < L5.size() && L5[k5].w == i) P.p2p_itemsP.push_back(L5[k5++]);
      continue;
    }
    sh.clear();
    oa.clear();
    ob.clear();
    for (int k = t->u_ptr[j]; k < t->u_ptr[j + 1]; k++) mark[t->u_idx[k]] = 1;
    for (int k = t->u_ptr[i]; k < t->u_ptr[i + 1]; k++) {
      const int s = t->u_idx[k];
      if (mark[s]) {
        sh.push_back(s);
        mark[s] = 2;
      } else {
        oa.push_back(s);
      }
    }
    for (int k = t->u_ptr[j]; k < t->u_ptr[j + 1]; k++) {
      const int s = t->u_idx[k];
      if (mark[s] == 1) ob.push_back(s);
      mark[s] = 0;
    }
    const int set = (int)P.rng_ptr.size() - 1;
    add_set(sh);
    add_set(oa);
    add_set(ob);
    P.p2p_itemsP.push_back(make_int4(set, t->trg_beg[i], nA | (t->trg_num[j] << 16), i));
    P.wc.pair_items += 1.0;
    i = j; /* B is done */
  }
  for (const int4& it : P.p2p_itemsP) {
    const int nA = it.z & 0xffff, nB = it.z >> 16, sets = nB ? 3 : 1;
    if (it.x < 0 || it.x + sets >= (int)P.rng_ptr.size() || nA < 1 ||
        (nA + 15) / 16 + (nB + 15) / 16 > P2P_MAXT5 / 16 || it.y < 0 || (long)it.y + nA + nB > t->n_trg ||
        it.w < 0 || it.w + (nB ? 1 : 0) >= nn) {
      set_error("internal: U-list pair item out of range");
      return KIFMM_EINVAL;
    }
  }
  return KIFMM_OK;
}

/* What a U-list item costs its CU, in steps of 64 sources (16 x 16 tiles on
 * the mixed path) by one target group: its longest wave's steps, and a fixed
 * part (item and range loads, first tile, close pairs, reductions) of about
 * 4 such steps.  set_src: the sources of each range set. */
double item_cost(const int4& it, int group, const std::vector<int>& set_src) {
  const int groups = ((it.z & 0xffff) + group - 1) / group + ((it.z >> 16) + group - 1) / group;
  double src = set_src[it.x];
  if (it.z >> 16) src += 0.5 * ((double)set_src[it.x + 1] + set_src[it.x + 2]); /* of a pair: half the groups each */
  return (groups + 3) / 4 * (src / 64.0 + 1.0) + 4.0;
}

double wave_cost(const int4& it, const std::vector<int>& set_src) { /* of k_p2p_wave's */
  return (it.z + 7) / 8 * (set_src[it.x] / 64.0 + 1.0) + 4.0;
}

constexpr double U_SMALL = 96.0; /* u_list_index */

/* 8-target groups per wave of the U-list's wave kernel (k_p2p_wave), 0: the
 * block kernels.  One up to 8 groups per SIMD of the chip, so that few items
 * spread (16 thousand points, 2752 groups: 16.5 us with one, 20 with two); then two,
 * which share a row's conversion (100 thousand, 14504 groups: 55 and 53); from 65536 on
 * the blocks' shared conversion is as good (300 thousand, 47776: 136 against 138; 1M
 * ellipsoid, 180072: 472 - 495 and 482 - 492; 16M: 12950 and 12770). */
int u_wave_groups(const kifmm_tree_view* t) {
  long groups = 0;
  for (int i = 0; i < t->n_nodes; i++)
    if (t->child[i] == -1) groups += (t->trg_num[i] + 7) / 8;
  return groups < 8192 ? 1 : groups < 65536 ? 2 : 0;
}

/* Items [b, e) of a list cut into 8 runs of about equal cost. */
XcdRuns xcd_runs(const std::vector<double>& cost, int b, int e) {
  XcdRuns r;
  r.beg[0] = b;
  for (int x = 1; x < 8; x++) {
    const double want = cost[b] + (cost[e] - cost[b]) * x / 8;
    const int k = (int)(std::lower_bound(cost.begin() + b, cost.begin() + e, want) - cost.begin());
    r.beg[x] = std::max(k, r.beg[x - 1]);
  }
  r.beg[8] = e;
  return r;
}

/* The indices [b, e) of items, those of more than the mean cost first, in
 * classes of falling cost (factor 1.25), then the others in their order, in
 * which neighbours share data.  An uneven list otherwise ends with its long
 * items on an emptying chip. */
template <typename Cost>
void long_first(int b, int e, double mean, Cost cost, std::vector<int>& out) {
  std::vector<std::vector<int>> cls(1);
  for (int k = b; k < e; k++) {
    const double r = cost(k) / mean;
    const size_t c = r <= 1.0 ? 0 : std::min<size_t>(30, 1 + (size_t)(std::log(r) / std::log(1.25)));
    if (c >= cls.size()) cls.resize(c + 1);
    cls[c].push_back(k);
  }
  for (size_t c = cls.size(); c-- > 0;) out.insert(out.end(), cls[c].begin(), cls[c].end());
}
/* The U-list items of a launch over all of them, long ones first within each
 * XCD's run.  U-list kernel: 53 -> 50.5 us at 100 thousand points, 136 -> 128 at 300
 * thousand, 482 -> 465 at 1M ellipsoid, 5.36 -> 5.28 ms at 4M; mixed 258 -> 238 us at
 * 465 thousand, 32.8 -> 31.8 at 65 thousand, 1.96 -> 1.93 ms at 4M. */
std::vector<int4> u_launch_order(const std::vector<int4>& items, const std::vector<double>& cost) {
  const int n = (int)items.size();
  if (n == 0) return {};
  const XcdRuns runs = xcd_runs(cost, 0, n);
  std::vector<int> order;
  for (int x = 0; x < 8; x++)
    long_first(runs.beg[x], runs.beg[x + 1], cost[n] / n, [&](int k) { return cost[k + 1] - cost[k]; }, order);
  std::vector<int4> out;
  for (int k : order) out.push_back(items[k]);
  return out;
}

/* The W / X items (k_wx) and their reductions.  Per target node and list,
 * the entries' sources as ranges, far ones (Gram form) before near ones,
 * cut into chunks; the node's points in blocks of WX_T; an item per block and
 * chunk with a slot of its own, the slots of a block's chunks consecutive.
 * Chunks hold WX_CAP sources on inputs with plenty of work; below, as many
 * as leave about WX_ITEMS items (16 waves on each of 256 CUs), at least 128:
 * a 4 thousand point input has 33 W blocks, and walking 1024 sources each
 * took 82 us on an otherwise idle chip.  Items run largest first.
 * wx_cost, which splits the launch's time between the lists: in passes of 64
 * sources over 8 points (96 issue slots, twice that on differences), 0.4 for
 * the conversion of 64 sources and 1 for the rest of an item.  W's share by
 * that, and of the two lists run alone: 0.476 and 0.474 at 1M ellipsoid points
 * NP 4, 0.474 and 0.51 at 300 thousand NP 6 (by pairs alone 0.512 and 0.51).  On the
 * mixed path the X sums onto check surfaces are k_x_surf's: blocks of 64
 * points, chunks of XS_CHUNK sources cut at entry boundaries. */
int wx_plan(const kifmm_tree_view* t, int ne, int lde, bool mixed, Plan& P) {
  constexpr long WX_ITEMS = 4096;
  const int nn = t->n_nodes;
  auto w_of = [&](int i) { return t->child[i] == -1 && (t->tag[i] & KIFMM_TRGNODE) && t->w_ptr[i + 1] > t->w_ptr[i]; };
  auto x_of = [&](int i) { return (t->tag[i] & KIFMM_TRGNODE) && t->x_ptr[i + 1] > t->x_ptr[i]; };
  /* a list entry as a range, {0, 0} if it has no sources */
  auto range = [&](int s, bool xl) {
    if (xl || (t->child[s] == -1 && t->src_num[s] < ne))
      return t->src_num[s] > 0 ? make_int2(t->src_beg[s], t->src_num[s]) : make_int2(0, 0);
    return make_int2(~s, ne);
  };
  auto points = [&](int i, bool xl, bool& surf) {
    surf = xl && !(t->child[i] == -1 && t->trg_num[i] < ne);
    return surf ? ne : t->trg_num[i];
  };
  /* whether box s stays WX_FAR h away from box i (h = i's half-width) */
  auto far = [&](int i, int s) {
    const double hi = 1.0 / (1 << t->depth[i]), hs = 1.0 / (1 << t->depth[s]);
    double d2 = 0.0;
    for (int k = 0; k < 3; k++) {
      const double gap = std::fabs((2 * t->path[3 * i + k] + 1) * hi - (2 * t->path[3 * s + k] + 1) * hs) - (hi + hs);
      if (gap > 0.0) d2 += gap * gap;
    }
    return d2 >= WX_FAR * WX_FAR * hi * hi;
  };
  long total = 0; /* sources x blocks */
  for (int i = 0; i < nn; i++)
    for (int xl = 0; xl < 2; xl++) {
      if (!(xl ? x_of(i) : w_of(i))) continue;
      bool surf;
      const long blocks = (points(i, xl, surf) + WX_T - 1) / WX_T;
      if (mixed && surf) continue;
      const int *ptr = xl ? t->x_ptr : t->w_ptr, *idx = xl ? t->x_idx : t->w_idx;
      for (int k = ptr[i]; k < ptr[i + 1]; k++) total += blocks * range(idx[k], xl).y;
    }
  const int chunk = (int)std::min<long>(WX_CAP, std::max<long>(128, (total / WX_ITEMS + 63) / 64 * 64));
  struct Chunk {
    int rb, re, n, flags;
  };
  std::vector<Chunk> chunks;
  std::vector<int2> lists[2]; /* far, near */
  struct Work {
    int cost; /* in steps of 64 sources */
    int4 a, b;
  };
  std::vector<Work> work, xs_work;
  auto sorted = [](const std::vector<Work>& w, std::vector<int4>& out) { /* largest first, stable */
    int most = 0;
    for (const Work& e : w) most = std::max(most, e.cost);
    std::vector<size_t> at((size_t)most + 2, 0);
    for (const Work& e : w) at[most - e.cost + 1]++;
    for (int c = 0; c <= most; c++) at[c + 1] += at[c];
    out.resize(2 * w.size());
    for (const Work& e : w) {
      const size_t k = at[most - e.cost]++;
      out[2 * k] = e.a;
      out[2 * k + 1] = e.b;
    }
  };
  for (int i = 0; i < nn; i++) {
    size_t wred_at = 0; /* the node's W reductions, to which X sums of the same targets are added */
    bool wred = false;
    for (int xl = 0; xl < 2; xl++) {
      if (!(xl ? x_of(i) : w_of(i))) continue;
      bool surf;
      const int npts = points(i, xl, surf);
      const int *ptr = xl ? t->x_ptr : t->w_ptr, *idx = xl ? t->x_idx : t->w_idx;
      if (mixed && surf) { /* one range per entry, chunks as rng index ranges */
        chunks.clear();
        Chunk c{(int)P.wx_rng.size(), 0, 0, 0};
        for (int k = ptr[i]; k < ptr[i + 1]; k++) {
          const int2 r = range(idx[k], true);
          if (r.y <= 0) continue;
          if (c.n > 0 && c.n + r.y > XS_CHUNK) {
            c.re = (int)P.wx_rng.size();
            chunks.push_back(c);
            c = Chunk{(int)P.wx_rng.size(), 0, 0, 0};
          }
          P.wx_rng.push_back(r);
          c.n += r.y;
        }
        c.re = (int)P.wx_rng.size();
        if (c.n > 0) chunks.push_back(c);
        const int nch = (int)chunks.size();
        for (int p = 0; p < npts && nch > 0; p += 64) {
          const int4 a = make_int4(i, p, std::min(64, npts - p), 0);
          for (int h = 0; h < nch; h++)
            xs_work.push_back({(chunks[h].n + 63) / 64, a, make_int4(chunks[h].rb, chunks[h].re, nch > 1 ? P.xs_slots + h : -1, 0)});
          if (nch > 1) {
            P.xs_red.push_back(a);
            P.xs_red.push_back(make_int4(P.xs_slots, nch, 0, 0));
            P.xs_slots += nch;
          }
        }
        continue;
      }
      lists[0].clear();
      lists[1].clear();
      for (int k = ptr[i]; k < ptr[i + 1]; k++) {
        const int2 r = range(idx[k], xl);
        if (r.y <= 0) continue;
        std::vector<int2>& L = lists[far(i, idx[k]) ? 0 : 1];
        if (r.x >= 0 && !L.empty() && L.back().x >= 0 && L.back().x + L.back().y == r.x) L.back().y += r.y;
        else L.push_back(r);
      }
      chunks.clear();
      for (int near = 0; near < 2; near++) {
        Chunk c{(int)P.wx_rng.size(), 0, 0, near ? WX_DIFF : 0};
        auto close = [&] {
          if (c.n > 0) {
            c.re = (int)P.wx_rng.size();
            chunks.push_back(c);
          }
          c.rb = (int)P.wx_rng.size();
          c.n = 0;
        };
        for (int2 r : lists[near]) {
          if (r.x < 0) { /* a surface is never split */
            if (c.n > 0 && c.n + r.y > chunk) close();
            P.wx_rng.push_back(r);
            c.n += r.y;
            continue;
          }
          while (r.y > 0) {
            if (c.n >= chunk) close();
            const int take = std::min(r.y, chunk - c.n);
            P.wx_rng.push_back(make_int2(r.x, take));
            c.n += take;
            r.x += take;
            r.y -= take;
          }
        }
        close();
      }
      if (chunks.empty() || npts <= 0) continue;
      if (!surf) P.wx_targets = true;
      const int out0 = surf ? i * lde : t->trg_beg[i];
      const bool join = xl && !surf && wred;
      if (!xl) {
        wred = true;
        wred_at = P.wx_red.size();
      }
      for (int p = 0, m = 0; p < npts; p += WX_T, m++) {
        const int cnt = std::min(WX_T, npts - p), slot0 = P.wx_slots;
        for (const Chunk& c : chunks) {
          const int steps = (c.n + 63) / 64, groups = (cnt + 7) / 8;
          P.wx_cost[xl] += 1.0 + steps * (0.4 + groups * (c.flags & WX_DIFF ? 2.0 : 1.0));
          work.push_back({steps * groups,
                          make_int4(c.rb, c.re, surf ? p : t->trg_beg[i] + p, cnt),
                          make_int4(i, P.wx_slots++, c.flags | (surf ? WX_SURF : 0) | (xl ? WX_X : WX_W), c.n)});
        }
        const int nch = P.wx_slots - slot0;
        if (join) {
          int4& b = P.wx_red[wred_at + 2 * m + 1];
          b.z = slot0;
          b.w = nch;
        } else {
          P.wx_red.push_back(make_int4(out0 + p, cnt, surf ? 1 : 0, 0));
          P.wx_red.push_back(xl ? make_int4(0, 0, slot0, nch) : make_int4(slot0, nch, 0, 0));
        }
      }
    }
  }
  sorted(work, P.wx_items);
  sorted(xs_work, P.xs_items);
  /* what k_wx, k_x_surf and their reductions index */
  bool ok = true;
  for (const int2& r : P.wx_rng)
    ok = ok && (r.x >= 0 ? r.y >= 1 && (long)r.x + r.y <= t->n_src : ~r.x < nn && r.y == ne);
  for (size_t m = 0; m < P.wx_items.size(); m += 2) {
    const int4 a = P.wx_items[m], b = P.wx_items[m + 1];
    int n = 0;
    for (int k = a.x; k < a.y; k++) n += P.wx_rng[k].y;
    ok = ok && a.x >= 0 && a.y <= (int)P.wx_rng.size() && a.w >= 1 && a.w <= WX_T && a.z >= 0 &&
         (long)a.z + a.w <= (b.z & WX_SURF ? ne : t->n_trg) && b.x >= 0 && b.x < nn && b.y >= 0 && b.y < P.wx_slots &&
         b.w == n && n >= 1 && n <= WX_CAP;
  }
  for (size_t m = 0; m < P.wx_red.size(); m += 2) {
    const int4 a = P.wx_red[m], b = P.wx_red[m + 1];
    ok = ok && a.x >= 0 && a.y >= 1 && a.y <= WX_T && (long)a.x + a.y <= (a.z ? (long)nn * lde : (long)t->n_trg) &&
         b.x >= 0 && b.x + b.y <= P.wx_slots && b.z >= 0 && b.z + b.w <= P.wx_slots;
  }
  for (size_t m = 0; m < P.xs_items.size(); m += 2) {
    const int4 a = P.xs_items[m], b = P.xs_items[m + 1];
    ok = ok && a.x >= 0 && a.x < nn && a.y >= 0 && a.z >= 1 && a.z <= 64 && a.y + a.z <= ne && b.x >= 0 && b.x < b.y &&
         b.y <= (int)P.wx_rng.size() && b.z < P.xs_slots;
    for (int k = b.x; ok && k < b.y; k++) ok = P.wx_rng[k].x >= 0;
  }
  for (size_t m = 0; m < P.xs_red.size(); m += 2) {
    const int4 a = P.xs_red[m], b = P.xs_red[m + 1];
    ok = ok && a.x >= 0 && a.x < nn && a.y >= 0 && a.z >= 1 && a.z <= 64 && a.y + a.z <= ne && b.x >= 0 && b.y >= 2 &&
         b.x + b.y <= P.xs_slots;
  }
  if (!ok) {
    set_error("internal: W / X work item out of range");
    return KIFMM_EINVAL;
  }
  return KIFMM_OK;
}

/* Hadamard groups: runs of at most 64 consecutive parents (a lane each) whose
 * neighbour-slot union fits the LDS staging area.  The runs are put together
 * from whole 4 x 4 x 4 blocks of parents (the same box two levels up) where
 * they fit: such a block's union is at most 6 x 6 x 6, while 64 parents
 * across two blocks overrun the area.  (Runs cut blindly every 64 parents
 * are out of step with the blocks from the second level on: 876 groups
 * instead of 586 at 16M uniform points.)  A block too large by itself is
 * cut between siblings.
 * The union is laid out by octant, a position of octant r (of its own
 * sibling group) at an index of residue r mod 8, missing neighbours (slot 0)
 * included, so that a group's neighbours in any direction spread evenly over
 * the LDS banks (k_hadamard_fact). */
int had_groups(const kifmm_tree_view* t, Plan& P) {
  const int np_ = (int)P.hslot.size();
  P.hloc.assign((size_t)np_ * 27, 0);
  std::vector<int> node(np_); /* the parents' nodes */
  for (int p = 0; p < np_; p++) node[p] = t->parent[P.vblocks[p]];
  auto same_box = [&](int p, int q, int up) {
    if (t->depth[node[p]] != t->depth[node[q]]) return false;
    for (int k = 0; k < 3; k++)
      if ((t->path[3 * node[p] + k] >> up) != (t->path[3 * node[q] + k] >> up)) return false;
    return true;
  };
  /* per class (octant) the slots in the open group; mark[slot] = the group
   * that holds it, index[slot] its place among its class.  A slot has one
   * octant, but for slot 0, which each class holds once when it needs it. */
  std::vector<int> mark(P.nblk + 1, -1), index(P.nblk + 1, 0), cls[8];
  int zero[8], group = 0, first = 0, cnt = 0;
  auto open = [&](int p) {
    first = p;
    cnt = 0;
    group++;
    for (int r = 0; r < 8; r++) {
      cls[r].clear();
      zero[r] = -1;
    }
  };
  /* adds the parents [p, e) if they fit; else leaves the group as it was */
  auto add = [&](int p, int e) {
    if (cnt + (e - p) > 64) return false;
    size_t was[8];
    int wz[8];
    for (int r = 0; r < 8; r++) {
      was[r] = cls[r].size();
      wz[r] = zero[r];
    }
    size_t most = 0;
    for (size_t k = (size_t)p * 27; k < (size_t)e * 27; k++) {
      const int slot = P.hnbr[k], r = P.hoct[k];
      if (slot == 0 ? zero[r] >= 0 : mark[slot] == group) continue;
      if (slot == 0) {
        zero[r] = (int)cls[r].size();
      } else {
        mark[slot] = group;
        index[slot] = (int)cls[r].size();
      }
      cls[r].push_back(slot);
      most = std::max(most, cls[r].size());
    }
    if (8 * most > (size_t)HAD_CAP) {
      for (int r = 0; r < 8; r++) {
        for (size_t j = was[r]; j < cls[r].size(); j++)
          if (cls[r][j] != 0) mark[cls[r][j]] = -1;
        cls[r].resize(was[r]);
        zero[r] = wz[r];
      }
      return false;
    }
    cnt += e - p;
    return true;
  };
  auto close = [&] {
    if (cnt == 0) return;
    size_t most = 0;
    for (auto& c : cls) most = std::max(most, c.size());
    P.hgroups.push_back(make_int4(first, cnt, (int)P.huslots.size(), (int)(8 * most)));
    for (size_t k = (size_t)first * 27; k < (size_t)(first + cnt) * 27; k++)
      P.hloc[k] = (unsigned char)(8 * (P.hnbr[k] ? index[P.hnbr[k]] : zero[P.hoct[k]]) + P.hoct[k]);
    for (size_t j = 0; j < most; j++)
      for (int r = 0; r < 8; r++) P.huslots.push_back(j < cls[r].size() ? cls[r][j] : 0);
  };
  open(0);
  for (int p = 0; p < np_;) {
    int e = p + 1;
    while (e < np_ && same_box(p, e, 2)) e++;
    if (!add(p, e)) {
      close();
      open(p);
      if (!add(p, e)) { /* a block larger than a group: sibling sets one by one */
        for (int a = p; a < e;) {
          int b = a + 1;
          while (b < e && b - a < 8 && same_box(a, b, 1)) b++;
          if (!add(a, b)) {
            close();
            open(a);
            if (!add(a, b)) {
              set_error("internal: Hadamard neighbour union exceeds the LDS capacity");
              return KIFMM_EINVAL;
            }
          }
          a = b;
        }
      }
    }
    p = e;
  }
  close();
  return KIFMM_OK;
}

int make_plan(const kifmm_tree_view* t, const kifmm_operators* ops, bool mixed, Plan& P) {
  TRY(check_view(t));
  const int np = t->np;
  P.np = np;
  P.n_e = ops->n_e;
  P.n_uc = ops->n_uc;
  P.ld_e = rup(P.n_e, 8);
  P.ld_uc = rup(P.n_uc, 8);
  P.lda_e = rup(P.n_e, 16);
  P.lda_uc = rup(P.n_uc, 16);
  P.lda_l2l = rup(8 * P.ld_e, 16);
  P.ld_surf = rup(std::max(P.n_uc, P.n_e), 8);
  P.N = 2 * np;
  P.H = np + 1;
  P.F = P.N * P.N * P.H;
  const int nn = t->n_nodes, ne = P.n_e, nuc = P.n_uc, lde = P.ld_e, lduc = P.ld_uc;
  P.nblk = (nn - 1) / 8;
  int maxd = 0;
  for (int i = 0; i < nn; i++) maxd = std::max(maxd, t->depth[i]);
  P.max_depth = maxd;
  kifmm_work_counts& wc = P.wc;
  std::memset(&wc, 0, sizeof wc);
  auto fail = [](const char* m) {
    set_error(std::string("internal: ") + m);
    return KIFMM_EINVAL;
  };

  /* U-list: merged source ranges per target leaf; a leaf's targets split
   * into the fewest items of <= P2P_MAXT, balanced, in multiples of 16
   * (also of <= P2P_MAXT / 2 and <= P2P_MAXT5 for the other launch shapes) */
  P.rng_ptr.assign(1, 0);
  for (int i = 0; i < nn; i++) {
    if (t->child[i] != -1 || t->trg_num[i] <= 0) continue;
    const int set = (int)P.rng_ptr.size() - 1;
    for (int k = t->u_ptr[i]; k < t->u_ptr[i + 1]; k++) {
      const int s = t->u_idx[k];
      const int b = t->src_beg[s], n = t->src_num[s];
      if (n <= 0) continue;
      wc.u_pairs += (double)n * t->trg_num[i];
      if ((int)P.rng.size() > P.rng_ptr.back() && P.rng.back().x + P.rng.back().y == b) P.rng.back().y += n;
      else P.rng.push_back(make_int2(b, n));
    }
    P.rng_ptr.push_back((int)P.rng.size());
    const int n = t->trg_num[i];
    for (int cap : {P2P_MAXT, P2P_MAXT / 2, P2P_MAXT5}) { /* the item lists of the launch shapes */
      const int nit = (n + cap - 1) / cap;
      const int per = (((n + nit - 1) / nit) + 15) & ~15;
      std::vector<int4>& out = cap == P2P_MAXT ? P.p2p_items : cap == P2P_MAXT5 ? P.p2p_items5 : P.p2p_items64;
      for (int c = 0; c < n; c += per) out.push_back(make_int4(set, t->trg_beg[i] + c, std::min(per, n - c), i));
    }
  }
  /* k_p2p_ulist reads trg4[it.y .. it.y+it.z-1] and src4 inside each range */
  for (int cap : {P2P_MAXT, P2P_MAXT / 2, P2P_MAXT5})
    for (const int4& it : cap == P2P_MAXT ? P.p2p_items : cap == P2P_MAXT5 ? P.p2p_items5 : P.p2p_items64)
      if (it.x < 0 || it.x + 1 >= (int)P.rng_ptr.size() || it.z < 1 || it.z > cap || it.y < 0 ||
          (long)it.y + it.z > t->n_trg || it.w < 0 || it.w >= nn)
        return fail("U-list work item out of range");
  TRY(pair_items(t, P));
  if (!mixed) P.wave_g = u_wave_groups(t);
  for (int i = 0, set = 0; P.wave_g > 0 && i < nn; i++) {
    if (t->child[i] != -1 || t->trg_num[i] <= 0) continue;
    const int n = t->trg_num[i], cap = 8 * P.wave_g, nit = (n + cap - 1) / cap, per = (((n + nit - 1) / nit) + 7) & ~7;
    for (int c = 0; c < n; c += per) P.p2p_itemsW.push_back(make_int4(set, t->trg_beg[i] + c, std::min(per, n - c), i));
    set++;
  }
  for (const int4& it : P.p2p_itemsW)
    if (it.x < 0 || it.x + 1 >= (int)P.rng_ptr.size() || it.z < 1 || it.z > 8 * P.wave_g || it.y < 0 ||
        (long)it.y + it.z > t->n_trg || it.w < 0 || it.w >= nn)
      return fail("U-list wave item out of range");
  for (const int2& r : P.rng)
    if (r.x < 0 || r.y < 1 || (long)r.x + r.y > t->n_src) return fail("U-list source range out of range");
  /* Copy-out chunks.  The U-list runs last, as one launch that writes the
   * device's and the pinned host potentials; it runs chunk by chunk only where
   * the host copies each chunk to a caller's own buffer while the next ones
   * compute, and where some chunks run early on the second stream
   * (early_chunks).  A chunk is a run of whole leaves whose targets are one
   * contiguous range: the item lists cover [0, n_trg) in item order with no
   * gap (checked), and cuts fall at leaf starts, where every list has an item
   * boundary.  The chunks shrink towards the end so that the host's pass left
   * after the last chunk is short.  Small inputs are one chunk. */
  {
    const std::vector<int4>* lists[5] = {&P.p2p_items, &P.p2p_items64, &P.p2p_items5, &P.p2p_itemsP, &P.p2p_itemsW};
    bool tiled = t->n_trg > 0;
    for (const std::vector<int4>* L : lists) {
      if (L == &P.p2p_itemsW && P.wave_g == 0) continue; /* not in use */
      long next = 0;
      for (const int4& it : *L) {
        if (it.y != next) tiled = false;
        next = (long)it.y + item_targets(it);
      }
      if (next != t->n_trg) tiled = false;
    }
    P.tiled = tiled;
    P.cuts.assign(1, 0);
    if (tiled && t->n_trg >= (1 << 18)) {
      static const double frac[] = {0.30, 0.55, 0.75, 0.88, 0.95};
      for (double f : frac) {
        const long want = (long)(f * t->n_trg);
        /* the first leaf start at or after want that starts an item of
         * the pair list (then every list has an item boundary there) */
        int cut = -1;
        for (const int4& it : P.p2p_itemsP)
          if (it.y >= want && it.y == t->trg_beg[it.w]) {
            cut = it.y;
            break;
          }
        if (cut > P.cuts.back() && cut < t->n_trg) P.cuts.push_back(cut);
      }
    }
    P.cuts.push_back(t->n_trg);
    std::vector<int> set_src(P.rng_ptr.size(), 0); /* sources of each range set */
    for (size_t k = 0; k + 1 < P.rng_ptr.size(); k++)
      for (int r = P.rng_ptr[k]; r < P.rng_ptr[k + 1]; r++) set_src[k] += P.rng[r].y;
    for (int l = 0; l < 5; l++) {
      const std::vector<int4>& L = *lists[l];
      std::vector<double>& cost = P.u_cost[l];
      cost.assign(1, 0.0);
      for (const int4& it : L)
        cost.push_back(cost.back() + (l == 4 ? wave_cost(it, set_src) : item_cost(it, l == 3 ? 16 : 8, set_src)));
      P.chunk_beg[l].clear();
      size_t k = 0;
      for (size_t c = 0; c + 1 < P.cuts.size(); c++) {
        while (k < L.size() && L[k].y < P.cuts[c]) k++;
        if (k < L.size() && L[k].y != P.cuts[c] && c > 0) return fail("copy-out chunk does not start an item");
        P.chunk_beg[l].push_back((int)k);
      }
      P.chunk_beg[l].push_back((int)L.size());
    }
    /* the list that the default form launches */
    P.u_order_list = mixed ? 3 : P.wave_g > 0 ? 4 : t->n_trg <= U_SMALL * P.p2p_items5.size() ? 1 : 2;
    P.u_order = u_launch_order(*lists[P.u_order_list], P.u_cost[P.u_order_list]);
  }

  /* S2M + UC2UE over source leaves */
  for (int i = 0; i < nn; i++) {
    if (t->child[i] != -1 || !(t->tag[i] & KIFMM_SRCNODE) || t->src_num[i] <= 0) continue;
    const int col = (int)P.s2m_items.size();
    P.s2m_items.push_back(make_int4(i, t->src_beg[i], t->src_num[i], col));
    P.s2m_gemm.in.push_back(col * lduc);
    P.s2m_gemm.out.push_back(i * lde);
    P.s2m_gemm.sexp.push_back(-t->depth[i]);
    wc.s2m_pairs += (double)nuc * t->src_num[i];
    wc.gemm_flops += 2.0 * ne * nuc;
  }
  P.chk_cols = P.s2m_items.size();
  for (const int4& it : P.s2m_items)
    if (it.y < 0 || it.z < 1 || (long)it.y + it.z > t->n_src) return fail("S2M source range out of range");
  /* FP64: long leaves first, 60 -> 50 us at 300 thousand points NP 6, 14.2 -> 12.8 at 100
   * thousand NP 4, no change at 4M; the mixed kernel, four leaves a block, was
   * slower for it (65 thousand points 16.6 -> 18.1).  The columns stay in leaf order */
  if (!mixed) {
    const int n = (int)P.s2m_items.size();
    const std::vector<int4> by_leaf(P.s2m_items);
    std::vector<int> order;
    long_first(0, n, (double)t->n_src / std::max(n, 1), [&](int k) { return (double)by_leaf[k].z; }, order);
    for (int k = 0; k < n; k++) P.s2m_items[k] = by_leaf[order[k]];
  }

  /* per-level M2M, L2L and DC2DE column lists */
  P.lv.assign(maxd + 1, HostLevel());
  for (int d = 0; d <= maxd; d++) {
    HostLevel& L = P.lv[d];
    int col = 0;
    for (int i = t->level_start[d]; i < t->level_start[d + 1]; i++) {
      if (t->depth[i] != d) return fail("level_start does not match depth");
      /* upward densities of depth 0 and 1 are never read: V-lists start at
       * depth 2 and W-list boxes lie at depth >= 2 */
      if (d >= 2 && t->child[i] != -1 && (t->tag[i] & KIFMM_SRCNODE)) {
        L.m2m_a.in.push_back(t->child[i] * lde); L.m2m_a.out.push_back(col * lduc); L.m2m_a.sexp.push_back(d + 1);
        L.m2m_b.in.push_back(col * lduc); L.m2m_b.out.push_back(i * lde); L.m2m_b.sexp.push_back(-d);
        col++;
        wc.gemm_flops += 2.0 * nuc * 8 * ne + 2.0 * ne * nuc;
      }
      if (d + 1 >= 3 && t->child[i] != -1 && (t->tag[i] & KIFMM_TRGNODE)) {
        L.l2l.in.push_back(i * lde); L.l2l.out.push_back(t->child[i] * lde); L.l2l.sexp.push_back(d);
        wc.gemm_flops += 2.0 * 8 * ne * ne;
      }
      if (d >= 2 && (t->tag[i] & KIFMM_TRGNODE)) {
        L.dc2de.in.push_back(i * lde); L.dc2de.out.push_back(i * lde); L.dc2de.sexp.push_back(-d);
        wc.gemm_flops += 2.0 * ne * ne;
      }
    }
    P.chk_cols = std::max(P.chk_cols, (size_t)col * m2m_parts(col, mixed));
  }
  /* the fused downward kernel (k_l2l_dc2de) of depth d >= 3 runs over the
   * L2L parents at d - 1 and writes the densities of their target
   * children: exactly the DC2DE list of depth d */
  for (int d = 3; d <= maxd; d++) {
    size_t kids = 0;
    for (int off : P.lv[d - 1].l2l.out) {
      const int c0 = off / lde;
      for (int o = 0; o < 8; o++) kids += (t->tag[c0 + o] & KIFMM_TRGNODE) != 0;
    }
    if (kids != P.lv[d].dc2de.in.size()) return fail("L2L parents do not cover the DC2DE nodes of a level");
  }
  /* split-K workspace: the largest nsplit * ncols * ldw of any launch */
  {
    auto need = [&](size_t ncols, int M, int K) {
      if (!ncols) return;
      const GemmShape sh = gemm_shape((int)ncols, M, K);
      if (sh.nsplit > 1) P.ws_len = std::max(P.ws_len, (size_t)sh.nsplit * ncols * sh.ldw);
    };
    need(P.s2m_gemm.in.size(), ne, lduc);
    for (const HostLevel& L : P.lv) {
      need(L.m2m_a.in.size(), nuc, 8 * lde);
      need(L.m2m_b.in.size(), ne, lduc);
      need(L.l2l.in.size(), 8 * lde, lde);
      need(L.dc2de.in.size(), ne, lde);
    }
  }
  /* GEMM columns: inputs read K doubles, outputs write M doubles */
  {
    const long nodes = (long)nn * lde, chk = (long)std::max<size_t>(P.chk_cols, 1) * lduc;
    bool ok = offsets_ok(P.s2m_gemm.in, lduc, chk) && offsets_ok(P.s2m_gemm.out, ne, nodes);
    for (const HostLevel& L : P.lv)
      ok = ok && offsets_ok(L.m2m_a.in, 8L * lde, nodes) && offsets_ok(L.m2m_a.out, nuc, chk) &&
           offsets_ok(L.m2m_b.in, lduc, chk) && offsets_ok(L.m2m_b.out, ne, nodes) &&
           offsets_ok(L.l2l.in, lde, nodes) && offsets_ok(L.l2l.out, 8L * lde, nodes) &&
           offsets_ok(L.dc2de.in, lde, nodes) && offsets_ok(L.dc2de.out, ne, nodes);
    if (!ok) return fail("GEMM column offset out of range");
  }

  /* V-list: child blocks below parents of depth >= 1 and their 27 neighbour slots */
  for (int i = 0; i < nn; i++) {
    if (t->child[i] == -1 || t->depth[i] < 1) continue;
    const int blk = (t->child[i] - 1) / 8;
    P.vblocks.push_back(t->child[i]);
    P.vslot.push_back(blk + 1);
    P.hslot.push_back(blk + 1);
    const int d = t->depth[i], lim = 1 << d;
    for (int o = 0; o < 27; o++) {
      const int off[3] = {o / 9 - 1, (o / 3) % 3 - 1, o % 3 - 1};
      int w[3], slot = 0;
      bool in = true;
      for (int k = 0; k < 3; k++) {
        w[k] = t->path[3 * i + k] + off[k];
        in = in && w[k] >= 0 && w[k] < lim;
      }
      if (in) {
        const int c = find_box(t, d, w);
        if (t->depth[c] == d && t->child[c] != -1) slot = (t->child[c] - 1) / 8 + 1;
      }
      P.hnbr.push_back(slot);
      P.hoct.push_back((unsigned char)(((w[0] & 1) << 2) | ((w[1] & 1) << 1) | (w[2] & 1)));
    }
  }
  for (size_t k = 0; k < P.vblocks.size(); k++)
    if (P.vblocks[k] < 1 || P.vblocks[k] + 8 > nn || P.vslot[k] < 1 || P.vslot[k] > P.nblk || P.hslot[k] < 1 ||
        P.hslot[k] > P.nblk)
      return fail("V-list block out of range");
  for (int v : P.hnbr)
    if (v < 0 || v > P.nblk) return fail("V-list neighbour slot out of range");
  TRY(had_groups(t, P));
  {
    const int np_ = (int)P.hslot.size();
    for (const int4& gq : P.hgroups)
      if (gq.y < 1 || gq.y > 64 || gq.x + gq.y > np_ || gq.w > HAD_CAP || gq.z + gq.w > (int)P.huslots.size())
        return fail("Hadamard group out of range");
  }
  wc.v_entries = t->v_ptr[nn];
  wc.v_cmac_ref = 0.5 * (2.0 * P.F) * wc.v_entries;
  wc.v_cmac = 26.0 * 64.0 * P.F * (double)P.hslot.size();
  wc.fft_bytes = (double)P.vblocks.size() * 8 * (2.0 * 8 * ne + 2.0 * 16 * P.F);
  wc.hadamard_bytes = (double)P.hslot.size() * 8 * 16.0 * P.F * 2 + 343.0 * 16 * P.F;

  /* W, X and L2T work */
  for (int i = 0; i < nn; i++) {
    const bool leaf = t->child[i] == -1;
    const bool trg = (t->tag[i] & KIFMM_TRGNODE) != 0;
    if (trg && leaf && t->w_ptr[i + 1] > t->w_ptr[i]) {
      for (int k = t->w_ptr[i]; k < t->w_ptr[i + 1]; k++) {
        const int s = t->w_idx[k];
        const bool direct = t->child[s] == -1 && t->src_num[s] < ne;
        wc.w_pairs += (double)t->trg_num[i] * (direct ? t->src_num[s] : ne);
      }
    }
    if (trg && t->x_ptr[i + 1] > t->x_ptr[i]) {
      const bool direct = leaf && t->trg_num[i] < ne;
      for (int k = t->x_ptr[i]; k < t->x_ptr[i + 1]; k++)
        wc.x_pairs += (double)t->src_num[t->x_idx[k]] * (direct ? t->trg_num[i] : ne);
    }
    if (trg && leaf && t->trg_num[i] > 0 && t->depth[i] >= 2) {
      P.l2t.push_back(i);
      wc.l2t_pairs += (double)ne * t->trg_num[i];
      for (int c = 0; c < t->trg_num[i]; c += 64)
        P.l2t_items.push_back(make_int4(i, t->trg_beg[i] + c, std::min(64, t->trg_num[i] - c), 0));
    }
  }
  TRY(wx_plan(t, ne, lde, mixed, P));
  for (int i : P.l2t)
    if (t->trg_num[i] < 1) return fail("L2T leaf without targets");
  /* k_l2t reads trg4[it.y .. it.y + it.z - 1] and the leaf's DE densities */
  for (const int4& it : P.l2t_items)
    if (it.x < 0 || it.x >= nn || it.z < 1 || it.z > 64 || it.y < 0 || (long)it.y + it.z > t->n_trg)
      return fail("L2T work item out of range");
  if (nuc > 320) return fail("NP too large for the S2M block");
  return KIFMM_OK;
}

int upload_gemm(kifmm_gpu* g, GemmList& L, const HostGemm& h) {
  L.n = (int)h.in.size();
  TRY(dev_upload(g, &L.in_off, h.in.data(), h.in.size()));
  TRY(dev_upload(g, &L.out_off, h.out.data(), h.out.size()));
  TRY(dev_upload(g, &L.sexp, h.sexp.data(), h.sexp.size()));
  return KIFMM_OK;
}

int build(kifmm_gpu* g, const kifmm_tree_view* t, const kifmm_operators* ops, const Plan& P) {
  const int np = P.np, nn = t->n_nodes, ne = P.n_e, nuc = P.n_uc, lde = P.ld_e, lduc = P.ld_uc;
  g->np = np; g->n_e = ne; g->n_uc = nuc; g->ld_e = lde; g->ld_uc = lduc;
  g->lda_e = P.lda_e; g->lda_uc = P.lda_uc; g->lda_l2l = P.lda_l2l; g->ld_surf = P.ld_surf;
  g->N = P.N; g->H = P.H; g->F = P.F;
  g->n_nodes = nn; g->n_src = t->n_src; g->n_trg = t->n_trg;
  g->coincident = t->coincident;
  g->max_depth = P.max_depth;
  g->counts = P.wc;

  /* points: the caller's coordinate arrays go up as they are and are
   * packed into (x, y, z, w) records on the device (k_pack4) */
  {
    TRY(dev_zero(g, &g->src4, (size_t)t->n_src));
    TRY(dev_zero(g, &g->trg4, (size_t)t->n_trg));
    TRY(dev_zero(g, &g->pot, (size_t)t->n_trg));
    const size_t m = (size_t)std::max(std::max(t->n_src, t->n_trg), 1);
    DeviceArena tmp(g->stream);
    double* const stage = (double*)tmp.get(4 * m * sizeof(double));
    if (!stage) {
      set_error("hipMalloc of the point staging buffer failed");
      return KIFMM_ENOMEM;
    }
    const int blocks = (int)std::min<size_t>(4096, (m + 255) / 256);
    const double* srcs[4] = {t->sx, t->sy, t->sz, t->sden};
    const double* trgs[3] = {t->tx, t->ty, t->tz};
    if (t->n_src > 0) {
      for (int k = 0; k < 4; k++)
        HIP_TRY(hipMemcpyAsync(stage + k * m, srcs[k], sizeof(double) * t->n_src, hipMemcpyHostToDevice, g->stream));
      hipLaunchKernelGGL(k_pack4, dim3(blocks), dim3(256), 0, g->stream, g->src4, stage, stage + m, stage + 2 * m,
                         stage + 3 * m, (size_t)t->n_src);
      HIP_TRY(hipGetLastError());
    }
    if (t->n_trg > 0) {
      HIP_TRY(hipStreamSynchronize(g->stream)); /* the stage is reused */
      for (int k = 0; k < 3; k++)
        HIP_TRY(hipMemcpyAsync(stage + k * m, trgs[k], sizeof(double) * t->n_trg, hipMemcpyHostToDevice, g->stream));
      hipLaunchKernelGGL(k_pack4, dim3(blocks), dim3(256), 0, g->stream, g->trg4, stage, stage + m, stage + 2 * m,
                         nullptr, (size_t)t->n_trg);
      HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipStreamSynchronize(g->stream));
  }
  /* node geometry (fmm/input.cc:113-137) and node arrays */
  {
    std::vector<double4> geo(nn);
    for (int i = 0; i < nn; i++) {
      const double sc = (double)(1 << t->depth[i]);
      geo[i] = make_double4(-1.0 + (2.0 * 1.0) * (t->path[3 * i] + 0.5) / sc,
                            -1.0 + (2.0 * 1.0) * (t->path[3 * i + 1] + 0.5) / sc,
                            -1.0 + (2.0 * 1.0) * (t->path[3 * i + 2] + 0.5) / sc, 1.0 / sc);
    }
    TRY(dev_upload(g, &g->geo, geo.data(), geo.size()));
    TRY(dev_upload(g, &g->snum, t->src_num, nn));
    TRY(dev_upload(g, &g->sbeg, t->src_beg, nn));
    TRY(dev_upload(g, &g->depth, t->depth, nn));
    TRY(dev_upload(g, &g->tag, t->tag, nn));
    TRY(dev_upload(g, &g->u_ptr, t->u_ptr, (size_t)nn + 1));
    TRY(dev_upload(g, &g->u_idx, t->u_idx, t->u_ptr[nn]));
    TRY(dev_zero(g, &g->uden, (size_t)nn * lde));
    TRY(dev_zero(g, &g->dchk, (size_t)nn * lde));
    TRY(dev_zero(g, &g->dden, (size_t)nn * lde));
  }
  /* operators, padded column-major */
  {
    std::vector<double> a((size_t)g->lda_e * lduc, 0.0);
    for (int k = 0; k < nuc; k++)
      for (int i = 0; i < ne; i++) a[(size_t)k * g->lda_e + i] = ops->uc2ue[(size_t)k * ne + i];
    TRY(dev_upload(g, &g->UC2UE, a.data(), a.size()));
    std::vector<double> b((size_t)g->lda_uc * 8 * lde, 0.0);
    for (int o = 0; o < 8; o++)
      for (int k = 0; k < ne; k++)
        for (int i = 0; i < nuc; i++)
          b[(size_t)(o * lde + k) * g->lda_uc + i] = ops->ue2uc[(size_t)o * nuc * ne + (size_t)k * nuc + i];
    TRY(dev_upload(g, &g->UE2UC, b.data(), b.size()));
    std::vector<double> c((size_t)g->lda_e * lde, 0.0);
    for (int k = 0; k < ne; k++)
      for (int i = 0; i < ne; i++) c[(size_t)k * g->lda_e + i] = ops->dc2de[(size_t)k * ne + i];
    TRY(dev_upload(g, &g->DC2DE, c.data(), c.size()));
    std::vector<double> d((size_t)g->lda_l2l * lde, 0.0);
    for (int o = 0; o < 8; o++)
      for (int k = 0; k < ne; k++)
        for (int i = 0; i < ne; i++)
          d[(size_t)k * g->lda_l2l + o * lde + i] = ops->de2dc[(size_t)o * ne * ne + (size_t)k * ne + i];
    TRY(dev_upload(g, &g->DE2DC, d.data(), d.size()));
  }
  /* unit surfaces (fmm/trans.cc:13-26) and DFT tables */
  {
    const int ls = g->ld_surf;
    std::vector<double> s(4 * (size_t)ls, 0.0);
    host_surface(np, 1.0, s, ls); TRY(dev_upload(g, &g->surf_ue, s.data(), s.size()));
    std::fill(s.begin(), s.end(), 0.0);
    host_surface(np + 2, 3.0, s, ls); TRY(dev_upload(g, &g->surf_uc, s.data(), s.size()));
    if (g->precision == KIFMM_PREC_MIXED) {
      std::vector<float> f(s.begin(), s.end());
      TRY(dev_upload(g, &g->surf_uc32, f.data(), f.size()));
    }
    std::fill(s.begin(), s.end(), 0.0);
    host_surface(np, 3.0, s, ls); TRY(dev_upload(g, &g->surf_de, s.data(), s.size()));
    if (g->precision == KIFMM_PREC_MIXED) {
      std::vector<float> f(s.begin(), s.end());
      TRY(dev_upload(g, &g->surf_de32, f.data(), f.size()));
    }
    std::fill(s.begin(), s.end(), 0.0);
    host_surface(np, 1.0, s, ls); TRY(dev_upload(g, &g->surf_dc, s.data(), s.size()));
    {
      std::vector<double4> r(ne);
      for (int j = 0; j < ne; j++)
        r[j] = make_double4(-2.0 * GRAM_SC * s[j], -2.0 * GRAM_SC * s[ls + j], -2.0 * GRAM_SC * s[2 * ls + j],
                            GRAM_SC * GRAM_SC * s[3 * ls + j]);
      TRY(dev_upload(g, &g->dc_gram, r.data(), r.size()));
    }
    const int N = g->N;
    std::vector<double2> w(N);
    for (int m = 0; m < N; m++) {
      const long double a = 2.0L * 3.141592653589793238462643383279502884L * (long double)m / (long double)N;
      w[m] = make_double2((double)cosl(a), (double)(-sinl(a)));
    }
    TRY(dev_upload(g, &g->tw, w.data(), w.size()));
    std::vector<int> c2s(np * np * np, -1), s2c;
    for (int i = 0; i < np; i++)
      for (int j = 0; j < np; j++)
        for (int k = 0; k < np; k++)
          if (i == 0 || i == np - 1 || j == 0 || j == np - 1 || k == 0 || k == np - 1) {
            c2s[(i * np + j) * np + k] = (int)s2c.size();
            s2c.push_back((i * np + j) * np + k);
          }
    TRY(dev_upload(g, &g->cube2surf, c2s.data(), c2s.size()));
    TRY(dev_upload(g, &g->surf2cube, s2c.data(), s2c.size()));
  }
  /* work lists */
  g->n_p2p = (int)P.p2p_items.size();
  TRY(dev_upload(g, &g->p2p_items, P.p2p_items.data(), P.p2p_items.size()));
  g->n_p2p64 = (int)P.p2p_items64.size();
  TRY(dev_upload(g, &g->p2p_items64, P.p2p_items64.data(), P.p2p_items64.size()));
  g->n_p2p5 = (int)P.p2p_items5.size();
  TRY(dev_upload(g, &g->p2p_items5, P.p2p_items5.data(), P.p2p_items5.size()));
  g->u_order_list = P.u_order_list;
  TRY(dev_upload(g, &g->u_order, P.u_order.data(), P.u_order.size()));
  g->n_p2pW = (int)P.p2p_itemsW.size();
  g->wave_g = P.wave_g;
  TRY(dev_upload(g, &g->p2p_itemsW, P.p2p_itemsW.data(), P.p2p_itemsW.size()));
  g->n_p2pP = (int)P.p2p_itemsP.size();
  TRY(dev_upload(g, &g->p2p_itemsP, P.p2p_itemsP.data(), P.p2p_itemsP.size()));
  TRY(dev_zero(g, &g->p2p_counters, 8 * std::max<size_t>(P.cuts.size(), 1)));
  g->cuts = P.cuts;
  g->tiled = P.tiled;
  for (int l = 0; l < 5; l++) {
    g->chunk_beg[l] = P.chunk_beg[l];
    g->u_cost[l] = P.u_cost[l];
  }
  TRY(dev_zero(g, &g->potU, (size_t)t->n_trg));
  TRY(dev_zero(g, &g->den_stage, (size_t)t->n_src));
  {
    int ncu = 0, per_cu = 0;
    HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, g->dev));
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_p2p_ulist_persist<false, P2P_G, false>, 256, 0));
    g->persist_grid[0] = std::max(8, (ncu * std::max(per_cu, 1) + 7) / 8 * 8);
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_p2p_ulist_persist<false, P2P_G5, true>, 256, 0));
    g->persist_grid[1] = std::max(8, (ncu * std::max(per_cu, 1) + 7) / 8 * 8);
  }
  TRY(dev_upload(g, &g->rng_ptr, P.rng_ptr.data(), P.rng_ptr.size()));
  TRY(dev_upload(g, &g->rng, P.rng.data(), P.rng.size()));
  g->n_s2m = (int)P.s2m_items.size();
  TRY(dev_upload(g, &g->s2m_items, P.s2m_items.data(), P.s2m_items.size()));
  TRY(upload_gemm(g, g->s2m_gemm, P.s2m_gemm));
  g->lv.assign(P.max_depth + 1, LevelOps());
  for (int d = 0; d <= P.max_depth; d++) {
    TRY(upload_gemm(g, g->lv[d].m2m_a, P.lv[d].m2m_a));
    TRY(upload_gemm(g, g->lv[d].m2m_b, P.lv[d].m2m_b));
    TRY(upload_gemm(g, g->lv[d].l2l, P.lv[d].l2l));
    TRY(upload_gemm(g, g->lv[d].dc2de, P.lv[d].dc2de));
  }
  g->chk_cols = P.chk_cols;
  TRY(dev_zero(g, &g->chk, std::max<size_t>(P.chk_cols, 1) * lduc));
  g->ws_len = P.ws_len;
  TRY(dev_zero(g, &g->ws, std::max<size_t>(P.ws_len, 1)));
  g->n_vblocks = (int)P.vblocks.size();
  g->n_hpar = (int)P.hslot.size();
  TRY(dev_upload(g, &g->vblocks, P.vblocks.data(), P.vblocks.size()));
  TRY(dev_upload(g, &g->vslot, P.vslot.data(), P.vslot.size()));
  g->n_hgroups = (int)P.hgroups.size();
  TRY(dev_upload(g, &g->hgroups, P.hgroups.data(), P.hgroups.size()));
  TRY(dev_upload(g, &g->huslots, P.huslots.data(), P.huslots.size()));
  TRY(dev_upload(g, &g->hloc, P.hloc.data(), P.hloc.size()));
  TRY(dev_upload(g, &g->hslot, P.hslot.data(), P.hslot.size()));
  const size_t spec = (size_t)(P.nblk + 1) * g->F * 8;
  if (g->precision == KIFMM_PREC_MIXED) {
    TRY(dev_zero(g, &g->Xf, spec));
    TRY(dev_zero(g, &g->Yf, spec));
    TRY(dev_zero(g, &g->Tf, (size_t)g->F * 343));
    TRY(dev_zero(g, &g->src32, (size_t)std::max(g->n_src, 1)));
  } else {
    TRY(dev_zero(g, &g->X, spec));
    TRY(dev_zero(g, &g->Y, spec));
    TRY(dev_zero(g, &g->T, (size_t)g->F * 343));
    TRY(dev_zero(g, &g->That, (size_t)g->F * HAD_FACT));
  }
  g->n_wx = (int)P.wx_items.size() / 2;
  g->n_wxred = (int)P.wx_red.size() / 2;
  g->wx_targets = P.wx_targets;
  for (int xl = 0; xl < 2; xl++) g->wx_cost[xl] = P.wx_cost[xl];
  g->n_xs = (int)P.xs_items.size() / 2;
  g->n_xsred = (int)P.xs_red.size() / 2;
  g->n_l2t = (int)P.l2t_items.size();
  TRY(dev_upload(g, &g->wx_items, P.wx_items.data(), P.wx_items.size()));
  TRY(dev_upload(g, &g->wx_red, P.wx_red.data(), P.wx_red.size()));
  TRY(dev_upload(g, &g->wx_rng, P.wx_rng.data(), P.wx_rng.size()));
  TRY(dev_upload(g, &g->xs_items, P.xs_items.data(), P.xs_items.size()));
  TRY(dev_upload(g, &g->xs_red, P.xs_red.data(), P.xs_red.size()));
  TRY(dev_zero(g, &g->wxpart, std::max((size_t)P.wx_slots * WX_T, (size_t)P.xs_slots * 64)));
  TRY(dev_upload(g, &g->l2t_items, P.l2t_items.data(), P.l2t_items.size()));
  return KIFMM_OK;
}

/* FP32 leaf-local source records of the mixed S2M ((s - c) / h, w): they
 * depend on the positions, fixed for the handle, and the densities, so they
 * are written here at create time and again by kifmm_gpu_set_densities, not
 * in every evaluation. */
int mixed_sources(kifmm_gpu* g) {
  if (g->n_s2m > 0)
    hipLaunchKernelGGL(k_src_local32, dim3(g->n_s2m), dim3(256), 0, g->stream, g->s2m_items, g->geo, g->src4,
                       g->src32);
  HIP_TRY(hipGetLastError());
  return KIFMM_OK;
}

/* Mixed path, once per evaluator: leaves per block for the mixed S2M and
 * L2T, and the FP32 source records. */
int mixed_setup(kifmm_gpu* g) {
  g->mix_lpb = (g->n_s2m > 0 && (double)g->n_src / g->n_s2m < 100.0) ? 4 : 1;
  TRY(mixed_sources(g));
  HIP_TRY(hipStreamSynchronize(g->stream));
  return KIFMM_OK;
}

/* Close pairs of the U-list (k_close_near): a count pass, the exclusive
 * offsets on the device (k_scan_*), then the fill pass.  Only the total
 * comes back to the host, to size the index array.  An input whose list
 * would exceed 16 pairs per target on average is not listed: the mixed path
 * then keeps the in-loop test (k_p2p_ulist_mixed), the FP64 path the
 * difference form. */
int close_list(kifmm_gpu* g) {
  const long long n = g->n_trg;
  const int nb = (int)std::max<long long>(1, (n + SCAN_PER - 1) / SCAN_PER);
  if (nb > SCAN_PER) return KIFMM_OK; /* beyond the scan's reach: not listed */
  DeviceArena tmp(g->stream);
  int* cnt = (int*)tmp.get(sizeof(int) * std::max<long long>(n, 1));
  long long* bsum = (long long*)tmp.get(sizeof(long long) * (nb + 1));
  if (!cnt || !bsum) {
    set_error("hipMalloc failed for the close-pair search");
    return KIFMM_ENOMEM;
  }
  long long* total = bsum + nb;
  const int per5 = (g->n_p2p5 + 7) / 8;
  if (g->n_p2p5 > 0)
    hipLaunchKernelGGL(k_close_near<false>, dim3(8 * per5), dim3(64), 0, g->stream, g->p2p_items5, g->n_p2p5, per5,
                       g->u_ptr, g->u_idx, g->sbeg, g->snum, g->geo, g->src4, g->trg4, cnt, nullptr, nullptr);
  HIP_TRY(hipGetLastError());
  if (n > 0) hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(SCAN_T), 0, g->stream, cnt, n, bsum);
  hipLaunchKernelGGL(k_scan_tops, dim3(1), dim3(SCAN_T), 0, g->stream, bsum, n > 0 ? nb : 0, total);
  HIP_TRY(hipGetLastError());
  long long tot = 0;
  HIP_TRY(hipMemcpyAsync(&tot, total, sizeof tot, hipMemcpyDeviceToHost, g->stream));
  HIP_TRY(hipStreamSynchronize(g->stream));
  const long long cap = std::min<long long>(std::max(16LL * n, 1LL << 20), INT_MAX - 1);
  if (tot > cap) return KIFMM_OK; /* close_listed stays 0 */
  TRY(dev_zero(g, &g->cptr, (size_t)n + 1));
  TRY(dev_zero(g, &g->cidx, (size_t)std::max<long long>(tot, 1)));
  if (n > 0)
    hipLaunchKernelGGL(k_scan_out, dim3(nb), dim3(SCAN_T), 0, g->stream, cnt, n, bsum, total, g->cptr);
  if (g->n_p2p5 > 0)
    hipLaunchKernelGGL(k_close_near<true>, dim3(8 * per5), dim3(64), 0, g->stream, g->p2p_items5, g->n_p2p5, per5,
                       g->u_ptr, g->u_idx, g->sbeg, g->snum, g->geo, g->src4, g->trg4, nullptr, g->cptr, g->cidx);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->n_close = tot;
  g->close_listed = 1;
  return KIFMM_OK;
}

/* The 343 translation spectra (k_trans; compute_fft_trans__gpu_eval,
 * fmm/cuda.cu:874-963, which the reference recomputes every run) and, FP64,
 * their factored form: they depend only on NP, so they are formed once per
 * handle. */
template <int NP>
int trans_setup_np(kifmm_gpu* g) {
  if (g->precision == KIFMM_PREC_MIXED) {
    hipLaunchKernelGGL((k_trans<NP, float2>), dim3(343), dim3(256), 0, g->stream, g->tw, g->Tf);
  } else {
    hipLaunchKernelGGL((k_trans<NP, double2>), dim3(343), dim3(256), 0, g->stream, g->tw, g->T);
    const int n = g->F * HAD_FACT;
    hipLaunchKernelGGL(k_trans_fact, dim3((n + 255) / 256), dim3(256), 0, g->stream, g->T, n, g->That);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(g->stream));
  return KIFMM_OK;
}
int trans_setup(kifmm_gpu* g) {
  switch (g->np) {
    case 3: return trans_setup_np<3>(g);
    case 4: return trans_setup_np<4>(g);
    case 6: return trans_setup_np<6>(g);
    default: set_error("NP must be 3, 4 or 6 on the GPU"); return KIFMM_EUNSUP;
  }
}

/* The per-target records of the Gram form, for the FP64 U-list with listed
 * close pairs (k_p2p_ulist<., ., true>) and the W / X items on targets. */
int gram_setup(kifmm_gpu* g) {
  g->gram_u = g->precision == KIFMM_PREC_FP64 && g->close_listed;
  if (!g->gram_u && !g->wx_targets) return KIFMM_OK;
  TRY(dev_zero(g, &g->trg_gram, (size_t)std::max(g->n_trg, 1)));
  if (g->n_p2p > 0)
    hipLaunchKernelGGL(k_trg_gram, dim3(g->n_p2p), dim3(128), 0, g->stream, g->p2p_items, g->geo, g->trg4,
                       g->trg_gram);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(g->stream));
  return KIFMM_OK;
}

#define LAUNCH_CHECK()                                                           \
  do {                                                                           \
    hipError_t e_ = hipGetLastError();                                           \
    if (e_ != hipSuccess) {                                                      \
      set_error(std::string("kernel launch: ") + hipGetErrorString(e_));         \
      return KIFMM_EDEVICE;                                                      \
    }                                                                            \
  } while (0)

/* Phase events (outside graph capture): E_START before the sequence, then
 * one after each phase in launch order.  A phase's kernels are launched with
 * its event as their stop event, so that the event ends up with the end of
 * the last one: an event recorded between two kernels costs a marker packet
 * and its drain, 2.4 us each, a stop event nothing measurable (ten 15 us kernels: 184
 * us with an event recorded after each, 158 with stop events, 160 without). */
enum { E_START = 0, E_UP, E_FFT, E_TRANS, E_HAD, E_IFFT, E_WX, E_XSURF, E_DOWN, E_U, E_END };
enum { PHASE_EMPTY, PHASE_STAMPED, PHASE_UNSTAMPED }; /* kifmm_gpu::phase_state */

/* one launch on st; start and stop (stop, or both, may be null) take its start and end */
template <typename... P, typename... A>
void launch_on(hipStream_t st, hipEvent_t start, hipEvent_t stop, void (*kernel)(P...), dim3 grid, dim3 block,
               A... args) {
  if (stop) hipExtLaunchKernelGGL(kernel, grid, block, 0, st, start, stop, 0, static_cast<P>(args)...);
  else hipLaunchKernelGGL(kernel, grid, block, 0, st, static_cast<P>(args)...);
}
/* one launch of the current phase on the main stream */
template <typename... P, typename... A>
void launch(kifmm_gpu* g, void (*kernel)(P...), dim3 grid, dim3 block, A... args) {
  launch_on(g->stream, g->start_ev, g->capturing ? nullptr : g->ev[g->phase], kernel, grid, block, args...);
  g->start_ev = nullptr;
  g->phase_state = PHASE_STAMPED;
}
/* boundary e, after the current phase; the launches from here on are phase e + 1's */
int phase_end(kifmm_gpu* g, int e) {
  g->ev_at[e] = g->phase_state == PHASE_EMPTY ? g->ev_at[e - 1] : e;
  if (!g->capturing && g->phase_state == PHASE_UNSTAMPED) HIP_TRY(hipEventRecord(g->ev[e], g->stream));
  g->phase = e + 1;
  g->phase_state = PHASE_EMPTY;
  return KIFMM_OK;
}

int gemm(kifmm_gpu* g, const GemmList& L, int M, int K, const double* A, int lda, const double* in, double* out,
         int accumulate) {
  if (L.n == 0) return KIFMM_OK;
  const GemmShape sh = gemm_shape(L.n, M, K);
  if (sh.nsplit > 1 && (size_t)sh.nsplit * L.n * sh.ldw > g->ws_len) {
    set_error("internal: GEMM workspace too small");
    return KIFMM_EINVAL;
  }
  const hipError_t e = launch_gemm_cols(g->stream, sh, M, K, A, lda, L.n, L.in_off, L.out_off, L.sexp, in, out,
                                        accumulate, g->ws);
  if (e != hipSuccess) {
    set_error(std::string("GEMM launch: ") + hipGetErrorString(e));
    return KIFMM_EDEVICE;
  }
  g->phase_state = PHASE_UNSTAMPED;
  return KIFMM_OK;
}

/* KIFMM_LEVEL_GEMM runs a level's applies as column GEMMs; otherwise (AUTO,
 * FUSED) M2M is two launches of k_level_op, and L2L + DC2DE is the fused
 * kernel, or at NP 6 on levels of up to L2L_SPLIT parents two launches of
 * k_level_op as well (13 us against 25 up to 200 parents, 35 against 39 at 990,
 * 119 against 119 at 4096; at NP 4 the fused kernel's 9 us beat two launches'
 * 11).  The two orders of summation are the same bit for bit. */
bool level_gemm_up(const kifmm_gpu* g) { return g->up_form == KIFMM_LEVEL_GEMM; }
bool level_gemm_down(const kifmm_gpu* g) { return g->down_form == KIFMM_LEVEL_GEMM; }
constexpr int L2L_SPLIT = 2048;

/* L2L of the parents at depth d - 1 and DC2DE of their children, fused */
int l2l_dc2de(kifmm_gpu* g, const GemmList& L, int d) {
  if (L.n == 0) return KIFMM_OK;
  const dim3 grid((L.n + 15) / 16, 8);
  switch ((g->n_e + 15) / 16) {
#define KIFMM_DOWN_CASE(R)                                                                                        \
  case R:                                                                                                         \
    launch(g, k_l2l_dc2de<R>, grid, dim3(256), g->n_e, g->ld_e, g->DE2DC, g->lda_l2l,       \
                       g->DC2DE, g->lda_e, L.n, L.in_off, L.out_off, g->tag, d, g->dchk, g->dden);                 \
    break;
    KIFMM_DOWN_CASE(2)
    KIFMM_DOWN_CASE(4)
    KIFMM_DOWN_CASE(10)
#undef KIFMM_DOWN_CASE
    default:
      set_error("internal: no fused downward kernel for this n_e");
      return KIFMM_EINVAL;
  }
  LAUNCH_CHECK();
  return KIFMM_OK;
}

int level_op(kifmm_gpu* g, const LevelOp& op, int parts, int nin) {
  if (op.ncols == 0) return KIFMM_OK;
  const dim3 grid((op.ncols + 15) / 16, (op.M + 63) / 64, parts);
  if (nin == 1) launch(g, k_level_op<1>, grid, dim3(256), op);
  else launch(g, k_level_op<M2M_PARTS>, grid, dim3(256), op);
  LAUNCH_CHECK();
  return KIFMM_OK;
}

/* UC2UE: check values (lduc apart, in nin slices) to upward densities */
int uc2ue(kifmm_gpu* g, const GemmList& B, int nin) {
  LevelOp op{};
  op.M = g->n_e; op.K = g->ld_uc; op.A = g->UC2UE; op.lda = g->lda_e;
  op.ncols = B.n; op.ldi = g->ld_uc; op.in = g->chk; op.slice = (size_t)B.n * g->ld_uc;
  op.out_off = B.out_off; op.out = g->uden; op.sexp = B.sexp;
  return level_op(g, op, 1, nin);
}

/* M2M of one level in two launches: the UE2UC stack into check values, in
 * m2m_parts slices along K, then UC2UE */
int m2m(kifmm_gpu* g, const GemmList& A, const GemmList& B, int d) {
  const int parts = m2m_parts(A.n, g->precision == KIFMM_PREC_MIXED);
  LevelOp op{};
  op.M = g->n_uc; op.K = 8 * g->ld_e / parts; op.A = g->UE2UC; op.lda = g->lda_uc;
  op.a_z = (size_t)op.K * g->lda_uc; op.in_z = op.K;
  op.ncols = A.n; op.in_off = A.in_off; op.in = g->uden;
  op.ldo = g->ld_uc; op.out_z = (size_t)A.n * g->ld_uc; op.out = g->chk; op.e = d + 1;
  TRY(level_op(g, op, parts, 1));
  return uc2ue(g, B, parts);
}

/* DC2DE of the nodes of depth d */
int dc2de(kifmm_gpu* g, const GemmList& D, int d) {
  LevelOp op{};
  op.M = g->n_e; op.K = g->ld_e; op.A = g->DC2DE; op.lda = g->lda_e;
  op.ncols = D.n; op.in_off = D.in_off; op.in = g->dchk; op.out_off = D.out_off; op.out = g->dden; op.e = -d;
  return level_op(g, op, 1, 1);
}

/* L2L of the parents at depth d - 1, an octant of children per part, then
 * DC2DE of the children */
int l2l_dc2de_split(kifmm_gpu* g, const GemmList& L, const GemmList& D, int d) {
  LevelOp op{};
  op.M = g->n_e; op.K = g->ld_e; op.A = g->DE2DC; op.lda = g->lda_l2l; op.a_z = g->ld_e;
  op.ncols = L.n; op.in_off = L.in_off; op.in = g->dden;
  op.out_off = L.out_off; op.out_z = g->ld_e; op.out = g->dchk; op.e = d - 1; op.accumulate = 1;
  TRY(level_op(g, op, 8, 1));
  return dc2de(g, D, d);
}

/* zeros over p[0 .. n) and q[0 .. m) */
int fill(kifmm_gpu* g, double* p, size_t n, double* q = nullptr, size_t m = 0) {
  const int blocks = (int)std::min<size_t>(4096, (std::max(n, m) + 255) / 256);
  launch(g, k_fill2, dim3(std::max(blocks, 1)), dim3(256), p, n, q, m);
  LAUNCH_CHECK();
  return KIFMM_OK;
}

/* Frequencies per Hadamard block: had_fb as the caller set it; by default
 * (had_auto) it is halved down to 4 while the launch has fewer than two blocks
 * per CU and to 2 below four.  A block runs its
 * frequencies one after another: 4 thousand points NP 3 took 29 us in blocks
 * of 8, 17 of 4 and 12 of 2; 100 thousand NP 4 57 in 800 blocks of 4 and 53 in
 * 1600 of 2, 65 thousand mixed 44 and 41, 16 thousand NP 6 the same.  Above that
 * the prefetch across frequencies pays (465 thousand mixed: 61 us in 680 blocks of
 * 8, 62.5 in 1360 of 4; 4M NP 6: 0.87 ms in blocks of 8, 0.88 of 4).  The sums are
 * the same. */
int had_block_size(const kifmm_gpu* g) {
  int fb = g->had_fb;
  while (g->had_auto && fb > 2 && (long)g->n_hgroups * (g->F / fb) < (fb > 4 ? 512 : 1024)) fb /= 2;
  return fb;
}

/* The V-list's four sub-phases; had launches the Hadamard in 8 per_xcd blocks
 * of fb frequencies in XCD-contiguous order (had_block). */
template <int NP, typename ST, typename HAD>
int vlist_phase(kifmm_gpu* g, ST* X, ST* Y, HAD had) {
  if (g->n_vblocks > 0)
    launch(g, (k_dft_fwd<NP, ST>), dim3(dft_blocks<NP>(g->n_vblocks)), dim3(Grid<NP>::THREADS), g->vblocks, g->n_vblocks, g->vslot,
                       g->depth, g->uden, g->ld_e, g->tw, g->cube2surf, X);
  LAUNCH_CHECK();
  TRY(phase_end(g, E_FFT));
  /* the translation spectra T depend only on NP: computed once at create
   * time (trans_setup), so this sub-phase is empty */
  TRY(phase_end(g, E_TRANS));
  if (g->n_hgroups > 0) {
    const int fb = had_block_size(g);
    TRY(had(fb, (int)(((long)g->n_hgroups * (g->F / fb) + 7) / 8)));
    LAUNCH_CHECK();
  }
  TRY(phase_end(g, E_HAD));
  if (g->n_vblocks > 0)
    launch(g, (k_dft_inv<NP, ST>), dim3(dft_blocks<NP>(g->n_vblocks)), dim3(Grid<NP>::THREADS), g->vblocks, g->n_vblocks, g->vslot, Y,
                       g->tw, g->surf2cube, g->dchk, g->ld_e);
  LAUNCH_CHECK();
  return KIFMM_OK;
}

/* A Hadamard kernel by its block size fb: KERNEL(FB) is the instantiation, T
 * its translation values */
#define KIFMM_HAD_LAUNCH(KERNEL, THREADS, T, X, Y)                                                                 \
  switch (fb) {                                                                                                    \
    case 2: launch(g, KERNEL(2), dim3(8 * per), dim3(THREADS), g->hgroups, g->huslots,       \
                               g->hloc, g->hslot, T, X, Y, g->n_hgroups, per); break;                              \
    case 4: launch(g, KERNEL(4), dim3(8 * per), dim3(THREADS), g->hgroups, g->huslots,       \
                               g->hloc, g->hslot, T, X, Y, g->n_hgroups, per); break;                              \
    case 8: launch(g, KERNEL(8), dim3(8 * per), dim3(THREADS), g->hgroups, g->huslots,       \
                               g->hloc, g->hslot, T, X, Y, g->n_hgroups, per); break;                              \
    case 16: launch(g, KERNEL(16), dim3(8 * per), dim3(THREADS), g->hgroups, g->huslots,     \
                                g->hloc, g->hslot, T, X, Y, g->n_hgroups, per); break;                             \
    default: set_error("internal: unknown Hadamard shape"); return KIFMM_EINVAL;                                   \
  }
#define HAD_V32(FB) (k_hadamard<NP, float2, FB>)
#define HAD_V64(FB) (k_hadamard<NP, double2, FB>)
#define HAD_M32(FB) (k_hadamard_mfma<NP, FB>)
#define HAD_F64(FB) (k_hadamard_fact<NP, FB>)
template <int NP>
int vlist_phase(kifmm_gpu* g) {
  if constexpr (NP <= 4) {
    if (g->precision == KIFMM_PREC_MIXED)
      return vlist_phase<NP>(g, g->Xf, g->Yf, [&](int fb, int per) {
        if (g->had_form == KIFMM_HAD_VALU) KIFMM_HAD_LAUNCH(HAD_V32, 128, g->Tf, g->Xf, g->Yf)
        else KIFMM_HAD_LAUNCH(HAD_M32, 256, g->Tf, g->Xf, g->Yf)
        return KIFMM_OK;
      });
  }
  return vlist_phase<NP>(g, g->X, g->Y, [&](int fb, int per) {
    if (g->had_form == KIFMM_HAD_VALU) KIFMM_HAD_LAUNCH(HAD_V64, 128, g->T, g->X, g->Y)
    else KIFMM_HAD_LAUNCH(HAD_F64, 512, g->That, g->X, g->Y)
    return KIFMM_OK;
  });
}
#undef HAD_V32
#undef HAD_V64
#undef HAD_M32
#undef HAD_F64
#undef KIFMM_HAD_LAUNCH

/* The item list the U-list launch uses: the mixed tau kernel takes sibling
 * pairs and single leaves (list 3), the FP64 Gram-form kernels items of
 * <= P2P_MAXT5 targets (list 2), the STATIC64 shape items of <= 64 (list
 * 1), the difference form, the mixed source-split form and the mixed
 * in-loop test items of <= P2P_MAXT (list 0).  The STATIC Gram form takes
 * a wave per item on small inputs (list 4, u_wave_groups) and the <= 64 list where leaves are small, U_SMALL targets or fewer per
 * item of list 2: its kernel holds 6 waves per SIMD instead of 4, which on
 * short items outweighs the second source walk of the few large leaves.
 * Measured, list 2 -> list 1: 0.503 -> 0.455 ms at 50 targets per item (1M
 * ellipsoid), 0.160 -> 0.137 at 37 (300 thousand, NP 6), 13.16 -> 12.89 at
 * 64 (16M uniform); 5.36 -> 5.59 at 128 (4M uniform).  The sums are the same
 * bit for bit. */
int u_list_index(const kifmm_gpu* g) {
  if (g->precision == KIFMM_PREC_MIXED) return g->close_listed && g->p2p_form != KIFMM_P2P_SPLIT ? 3 : 0;
  if (g->p2p_form == KIFMM_P2P_STATIC64) return 1;
  if (g->p2p_form == KIFMM_P2P_STATIC && g->gram_u && g->wave_g > 0) return 4;
  if (g->p2p_form == KIFMM_P2P_STATIC && g->gram_u && g->n_trg <= U_SMALL * g->n_p2p5) return 1;
  return g->gram_u ? 2 : 0;
}

/* U-list over the items of copy-out chunks [c0, c1) on stream st, writing
 * out[t] = u (accum = 0) or out[t] = u + out[t] (accum = 1), and to host[t]
 * (device address of the pinned buffer) when host is set.  The
 * persistent form's per-XCD counters of the launch are slot c0. */
template <bool MASK>
int launch_u(kifmm_gpu* g, hipStream_t st, int c0, int c1, double* out, double* host, int accum, hipEvent_t stop) {
  const int l = u_list_index(g);
  const int4* list = l == 0 ? g->p2p_items : l == 1 ? g->p2p_items64 : l == 2 ? g->p2p_items5 : l == 3 ? g->p2p_itemsP : g->p2p_itemsW;
  const int beg = g->chunk_beg[l][c0], end = g->chunk_beg[l][c1];
  const int chunk = c0;
  if (end <= beg) return KIFMM_OK;
  const XcdRuns runs = xcd_runs(g->u_cost[l], beg, end);
  int per = 0;
  for (int x = 0; x < 8; x++) per = std::max(per, runs.beg[x + 1] - runs.beg[x]);
  const int4* items = l == g->u_order_list && beg == 0 && end == g->chunk_beg[l].back() ? g->u_order : list;
  if (g->precision == KIFMM_PREC_MIXED) {
    if (g->close_listed && g->p2p_form == KIFMM_P2P_SPLIT)
      launch_on(st, nullptr, stop, k_p2p_ulist_mixed_split<MASK>, dim3(8 * per), dim3(256), items, runs, g->rng_ptr,
                         g->rng, g->geo, g->src4, g->trg4, g->cptr, g->cidx, out, host, accum);
    else if (g->close_listed)
      launch_on(st, nullptr, stop, k_p2p_ulist_mixed_tau<MASK>, dim3(8 * per), dim3(256), items, runs, g->rng_ptr,
                         g->rng, g->geo, g->src4, g->trg4, g->cptr, g->cidx, out, host, accum);
    else
      launch_on(st, nullptr, stop, k_p2p_ulist_mixed<MASK>, dim3(8 * per), dim3(256), items, runs, g->rng_ptr, g->rng,
                         g->geo, g->src4, g->trg4, out, host, accum);
  } else if (l == 4) {
    launch_on(st, nullptr, stop, g->wave_g == 1 ? k_p2p_wave<MASK, 1> : k_p2p_wave<MASK, 2>, dim3(8 * per), dim3(64),
              items, runs, g->rng_ptr, g->rng, g->src4, g->trg4, out, host, g->geo, g->trg_gram, g->cptr, g->cidx, accum);
  } else if (l == 1) {
    if (g->gram_u)
      launch_on(st, nullptr, stop, (k_p2p_ulist64<MASK, true>), dim3(8 * per), dim3(256), items, runs, g->rng_ptr,
                         g->rng, g->src4, g->trg4, out, host, g->geo, g->trg_gram, g->cptr, g->cidx, accum);
    else
      launch_on(st, nullptr, stop, (k_p2p_ulist64<MASK, false>), dim3(8 * per), dim3(256), items, runs, g->rng_ptr,
                         g->rng, g->src4, g->trg4, out, host, g->geo, g->trg_gram, g->cptr, g->cidx, accum);
  } else if (g->p2p_form == KIFMM_P2P_PERSISTENT) {
    int* counters = g->p2p_counters + 8 * std::max(chunk, 0);
    launch_on(st, nullptr, nullptr, k_fill_int, dim3(1), dim3(64), counters, 8, 0);
    if (g->gram_u)
      launch_on(st, nullptr, stop, (k_p2p_ulist_persist<MASK, P2P_G5, true>), dim3(g->persist_grid[1]), dim3(256), items,
                         runs, g->rng_ptr, g->rng, g->src4, g->trg4, out, host, counters, g->geo, g->trg_gram, g->cptr,
                         g->cidx, accum);
    else
      launch_on(st, nullptr, stop, (k_p2p_ulist_persist<MASK, P2P_G, false>), dim3(g->persist_grid[0]), dim3(256), items,
                         runs, g->rng_ptr, g->rng, g->src4, g->trg4, out, host, counters, g->geo, g->trg_gram, g->cptr,
                         g->cidx, accum);
  } else {
    if (g->gram_u)
      launch_on(st, nullptr, stop, (k_p2p_ulist<MASK, P2P_G5, true>), dim3(8 * per), dim3(256), items, runs,
                         g->rng_ptr, g->rng, g->src4, g->trg4, out, host, g->geo, g->trg_gram, g->cptr, g->cidx, accum);
    else
      launch_on(st, nullptr, stop, (k_p2p_ulist<MASK, P2P_G, false>), dim3(8 * per), dim3(256), items, runs,
                         g->rng_ptr, g->rng, g->src4, g->trg4, out, host, g->geo, g->trg_gram, g->cptr, g->cidx, accum);
  }
  LAUNCH_CHECK();
  return KIFMM_OK;
}

int launch_u(kifmm_gpu* g, hipStream_t st, int c0, int c1, double* out, double* host, int accum, hipEvent_t stop) {
  return g->coincident ? launch_u<true>(g, st, c0, c1, out, host, accum, stop)
                       : launch_u<false>(g, st, c0, c1, out, host, accum, stop);
}

/* Copy-out chunks whose U-list runs on the second stream from the start of
 * the evaluation (alongside the far field) rather than after it: none in
 * the default layout (tuning.overlap 0) and the sequential one (4), all of
 * them in the overlap layout (1), the first one or two in the split
 * layouts (2, 3 and their sequential forms 5, 6). */
int early_chunks(const kifmm_gpu* g, unsigned mask) {
  if (!(mask & KIFMM_PHASE_U)) return 0;
  const int nch = (int)g->cuts.size() - 1;
  switch (g->overlap) {
    case 1: return nch;
    case 2: case 5: return std::min(1, nch);
    case 3: case 6: return std::min(2, nch);
    default: return 0;
  }
}

/* W and X in one launch (lists: which of the two) and the sums of their
 * chunks; on the mixed path the X sums onto check surfaces on their own */
int wx_phase(kifmm_gpu* g, unsigned mask) {
  const int lists = (mask & KIFMM_PHASE_W ? WX_W : 0) | (mask & KIFMM_PHASE_X ? WX_X : 0);
  if (lists && g->n_wx > 0) {
    launch(g, k_wx, dim3(g->n_wx), dim3(64), g->wx_items, g->wx_rng, lists, g->geo, g->surf_ue,
                       g->surf_dc, g->ld_surf, g->uden, g->ld_e, g->src4, g->trg4, g->trg_gram, g->dc_gram, g->wxpart);
    LAUNCH_CHECK();
    launch(g, k_wx_reduce, dim3((g->n_wxred + 1) / 2), dim3(64), g->wx_red, g->n_wxred, lists,
                       g->wxpart, g->pot, g->dchk);
    LAUNCH_CHECK();
  }
  TRY(phase_end(g, E_WX));
  if ((lists & WX_X) && g->n_xs > 0) {
    launch(g, k_x_surf, dim3(g->n_xs), dim3(64), g->xs_items, g->wx_rng, g->geo, g->surf_dc,
                       g->ld_surf, g->src4, g->dchk, g->ld_e, g->wxpart);
    LAUNCH_CHECK();
    if (g->n_xsred > 0)
      launch(g, k_x_surf_reduce, dim3(g->n_xsred), dim3(64), g->xs_red, g->ld_e, g->wxpart,
                         g->dchk);
    LAUNCH_CHECK();
  }
  return phase_end(g, E_XSURF);
}

/* One evaluation is three launch sequences on the handle's streams:
 *   enqueue_side  the U-list of the early copy-out chunks (early_chunks) on
 *                 the second stream from the start, into potU, alongside
 *                 the far field;
 *   enqueue_far   the fills, up, V, W, X and down on the main stream (what a
 *                 graph handle captures and replays);
 *   enqueue_near  the join pot = potU + pot of the early chunks, then the
 *                 U-list of the others; both write the finished potentials
 *                 to the host as well (host, the pinned buffer's device
 *                 address, when non-null).  One U-list launch, or with
 *                 chunked (a caller buffer filled by host passes) one per
 *                 chunk, each followed by its event, so that the host copies
 *                 a chunk while the later ones compute.
 * The U-list's accumulating write (u + pot) and the join (potU + pot) add
 * the same two terms, so every layout gives the same bits. */
int enqueue_side(kifmm_gpu* g, unsigned mask) {
  const int e = early_chunks(g, mask);
  if (e == 0) return KIFMM_OK;
  HIP_TRY(hipEventRecord(g->fork_ev, g->stream)); /* after the previous evaluation's join read potU */
  HIP_TRY(hipStreamWaitEvent(g->side, g->fork_ev, 0));
  HIP_TRY(hipEventRecord(g->su0, g->side));
  TRY(launch_u(g, g->side, 0, e, g->potU, nullptr, 0, nullptr));
  HIP_TRY(hipEventRecord(g->su1, g->side));
  HIP_TRY(hipEventRecord(g->join_ev, g->side));
  return KIFMM_OK;
}

int enqueue_far(kifmm_gpu* g, unsigned mask) {
  const int lde = g->ld_e, lduc = g->ld_uc;
  /* zero what this call accumulates into (fill kernels, so the sequence
   * stays capturable): pot (W, X, L2T and the U-list add into it) and dchk
   * (V, X, L2L) always; uden and dden only when their phase, which assigns
   * every entry that is read, is left out */
  TRY(fill(g, g->pot, (size_t)g->n_trg, g->dchk, (size_t)g->n_nodes * lde));
  if (!(mask & KIFMM_PHASE_UP)) TRY(fill(g, g->uden, (size_t)g->n_nodes * lde));
  if (!(mask & KIFMM_PHASE_DOWN)) TRY(fill(g, g->dden, (size_t)g->n_nodes * lde));
  /* up: S2M check potentials, UC2UE, then M2M bottom-up */
  if ((mask & KIFMM_PHASE_UP) && g->n_s2m > 0) {
    /* sources never sit on the check surface: no r = 0 mask */
    if (g->precision == KIFMM_PREC_MIXED) {
      /* the FP32 leaf-local source records (mixed_sources) */
      /* (phases, check points per lane) as in the FP64 S2M; NP <= 4 here (98 or 152 check points) */
      if (g->n_uc > 160) {
        set_error("mixed S2M: more than 160 check points");
        return KIFMM_EUNSUP;
      }
      const bool small = g->n_uc <= 112;
      auto s2m = g->mix_lpb == 4 ? (small ? k_s2m_mixed<4, 4, 7> : k_s2m_mixed<4, 2, 5>)
                                 : (small ? k_s2m_mixed<1, 4, 7> : k_s2m_mixed<1, 2, 5>);
      launch(g, s2m, dim3((g->n_s2m + g->mix_lpb - 1) / g->mix_lpb), dim3(64), g->s2m_items,
                         g->n_s2m, g->geo, g->surf_uc32, g->n_uc, g->ld_surf, g->src32, g->chk, lduc);
    } else {
      /* (phases, check points per lane) by the check surface size: 98, 152, 296 for NP 3, 4, 6 */
      auto s2m = g->n_uc <= 112 ? k_s2m<4, 7> : g->n_uc <= 160 ? k_s2m<2, 5> : k_s2m<1, 5>;
      if (g->n_uc > 320) {
        set_error("S2M: more than 320 check points");
        return KIFMM_EUNSUP;
      }
      launch(g, s2m, dim3(g->n_s2m), dim3(64), g->s2m_items, g->geo, g->surf_uc, g->n_uc,
                         g->ld_surf, g->src4, g->chk, lduc);
    }
    LAUNCH_CHECK();
    /* below LEAF_SPLIT leaves the column GEMM splits K, with a reduction, or
     * has few blocks: 21 -> 6 us at 4096 leaves NP 4, 57 -> 27 at 6592 NP 6
     * (94 us at 32768 NP 6, where this would take about 130).  The mixed path keeps that order: another one flips FP32
     * roundings further on (see k_x_surf) */
    if (g->precision == KIFMM_PREC_FP64 && g->s2m_gemm.n < LEAF_SPLIT)
      TRY(uc2ue(g, g->s2m_gemm, 1));
    else
      TRY(gemm(g, g->s2m_gemm, g->n_e, lduc, g->UC2UE, g->lda_e, g->chk, g->uden, 0));
  }
  for (int d = g->max_depth - 1; d >= 0 && (mask & KIFMM_PHASE_UP); d--) {
    if (g->lv[d].m2m_a.n == 0) continue;
    if (!level_gemm_up(g)) {
      TRY(m2m(g, g->lv[d].m2m_a, g->lv[d].m2m_b, d));
    } else {
      TRY(gemm(g, g->lv[d].m2m_a, g->n_uc, 8 * lde, g->UE2UC, g->lda_uc, g->uden, g->chk, 0));
      TRY(gemm(g, g->lv[d].m2m_b, g->n_e, lduc, g->UC2UE, g->lda_e, g->chk, g->uden, 0));
    }
  }
  TRY(phase_end(g, E_UP));
  /* V-list */
  if (mask & KIFMM_PHASE_V) switch (g->np) {
    case 3: TRY(vlist_phase<3>(g)); break;
    case 4: TRY(vlist_phase<4>(g)); break;
    case 6: TRY(vlist_phase<6>(g)); break;
    default: set_error("NP must be 3, 4 or 6 on the GPU"); return KIFMM_EUNSUP;
  }
  else {
    for (int e : {E_FFT, E_TRANS, E_HAD}) TRY(phase_end(g, e));
  }
  TRY(phase_end(g, E_IFFT));
  /* W and X */
  TRY(wx_phase(g, mask));
  /* down: DC2DE at depth 2, then per level the fused L2L + DC2DE
   * (k_l2l_dc2de over the parents at depth d - 1), then L2T */
  for (int d = 2; d <= g->max_depth && (mask & KIFMM_PHASE_DOWN); d++) {
    if (d >= 3 && !level_gemm_down(g)) {
      if (g->np == 6 && g->lv[d - 1].l2l.n <= L2L_SPLIT) TRY(l2l_dc2de_split(g, g->lv[d - 1].l2l, g->lv[d].dc2de, d));
      else TRY(l2l_dc2de(g, g->lv[d - 1].l2l, d));
      continue;
    }
    if (d == 2 && g->precision == KIFMM_PREC_FP64 && !level_gemm_down(g)) {
      TRY(dc2de(g, g->lv[d].dc2de, d)); /* the mixed path keeps the split column GEMM's order */
      continue;
    }
    if (d >= 3) TRY(gemm(g, g->lv[d - 1].l2l, 8 * lde, lde, g->DE2DC, g->lda_l2l, g->dden, g->dchk, 1));
    TRY(gemm(g, g->lv[d].dc2de, g->n_e, lde, g->DC2DE, g->lda_e, g->dchk, g->dden, 0));
  }
  if ((mask & KIFMM_PHASE_DOWN) && g->n_l2t > 0) {
    if (g->precision == KIFMM_PREC_MIXED)
      launch(g, g->mix_lpb == 4 ? k_l2t_mixed<4> : k_l2t_mixed<1>, dim3((g->n_l2t + g->mix_lpb - 1) / g->mix_lpb),
             dim3(64), g->l2t_items, g->n_l2t, g->geo, g->surf_de32, g->ld_surf, g->n_e, g->dden, lde, g->trg4, g->pot);
    else
      launch(g, k_l2t, dim3(g->n_l2t), dim3(64), g->l2t_items, g->geo, g->surf_de, g->ld_surf,
                         g->n_e, g->dden, lde, g->trg4, g->pot);
  }
  LAUNCH_CHECK();
  TRY(phase_end(g, E_DOWN));
  return KIFMM_OK;
}

int enqueue_near(kifmm_gpu* g, unsigned mask, double* host, bool chunked) {
  const int nch = (int)g->cuts.size() - 1, e = early_chunks(g, mask);
  /* The early chunks' potentials go to the host from the join itself, or from
   * EARLY_COPY targets on, with others to come, by copies on a stream of their
   * own beside those: the join would hold the main stream for as long as PCIe
   * takes.  Two chunks early, join -> copies, into the handle's and a caller's
   * buffer: 2.96 -> 2.63 and 3.15 -> 2.90 ms at 4M points mixed (2.3M targets
   * early), 8.05 -> 7.73 and 8.20 -> 7.89 at 4M NP 6; but 1.55 -> 1.53 and 1.72 ->
   * 1.76 at 1M ellipsoid (0.6M), 1.13 -> 1.16 and 1.20 -> 1.20 at 300 thousand. */
  constexpr int EARLY_COPY = 1 << 20;
  const bool early_copy = e > 0 && e < nch && host && g->cuts[e] >= EARLY_COPY;
  if (e > 0) { /* the early chunks: join */
    g->phase_state = PHASE_UNSTAMPED;
    const int m = g->cuts[e];
    HIP_TRY(hipStreamWaitEvent(g->stream, g->join_ev, 0));
    const int blocks = std::min(4096, (m + 255) / 256);
    if (m > 0)
      hipLaunchKernelGGL(k_join_pot, dim3(std::max(blocks, 1)), dim3(256), 0, g->stream, g->pot,
                         early_copy ? nullptr : host, g->potU, m);
    LAUNCH_CHECK();
    if (early_copy) {
      if (!g->cstream) HIP_TRY(take_stream(g->dev, &g->cstream));
      HIP_TRY(hipEventRecord(g->far_ev, g->stream));
      HIP_TRY(hipStreamWaitEvent(g->cstream, g->far_ev, 0));
    }
    for (int c = 0; c < e && (early_copy || chunked); c++) {
      const int b = g->cuts[c], n = g->cuts[c + 1] - b;
      if (early_copy && n > 0)
        HIP_TRY(hipMemcpyAsync(g->pinned + b, g->pot + b, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost, g->cstream));
      if (chunked) HIP_TRY(hipEventRecord(g->cd_ev[c], early_copy ? g->cstream : g->stream));
    }
    if (early_copy) HIP_TRY(hipEventRecord(g->copied_ev, g->cstream));
  }
  if ((mask & KIFMM_PHASE_U) && e < nch) { /* the other chunks after the far field */
    const int late = chunked ? nch - e : 1;
    const int l = u_list_index(g);
    g->phase_state = late == 1 && g->chunk_beg[l][nch] > g->chunk_beg[l][e] ? PHASE_STAMPED : PHASE_UNSTAMPED;
    /* chunk launches on the two streams in turn (one chunk's last blocks run
     * beside the next chunk's first), or in layouts 4 - 6 one after another
     * on the main stream */
    const bool pairs = late > 1 && g->overlap < 4;
    if (pairs) {
      HIP_TRY(hipEventRecord(g->far_ev, g->stream));
      HIP_TRY(hipStreamWaitEvent(g->side, g->far_ev, 0));
    }
    for (int k = 0; k < late; k++) {
      const int c = e + k;
      hipStream_t st = (pairs && (k & 1)) ? g->side : g->stream;
      TRY(launch_u(g, st, c, chunked ? c + 1 : nch, g->pot, host, 1, late == 1 ? g->ev[E_U] : nullptr));
      if (chunked) HIP_TRY(hipEventRecord(g->cd_ev[c], st));
    }
    if (pairs) {
      HIP_TRY(hipEventRecord(g->sdone_ev, g->side));
      HIP_TRY(hipStreamWaitEvent(g->stream, g->sdone_ev, 0));
    }
  }
  TRY(phase_end(g, E_U));
  if (early_copy) HIP_TRY(hipStreamWaitEvent(g->stream, g->copied_ev, 0));
  return KIFMM_OK;
}

/* pinned potentials -> the caller's buffer, a few host threads */
void host_copy(double* to, const double* from, size_t b, size_t e) {
  const size_t n = e - b;
  const int nt = (int)std::min<size_t>(8, std::max<size_t>(1, n / (1 << 16)));
  if (nt == 1) {
    std::memcpy(to + b, from + b, sizeof(double) * n);
    return;
  }
  std::vector<std::thread> th;
  for (int k = 0; k < nt; k++) {
    const size_t x = b + n * k / nt, y = b + n * (k + 1) / nt;
    th.emplace_back([=] { std::memcpy(to + x, from + x, sizeof(double) * (y - x)); });
  }
  for (auto& t : th) t.join();
}

int evaluate(kifmm_gpu* g, unsigned mask, double* pot_leaf, kifmm_phase_times* times) {
  hipEvent_t* ev = g->ev;
  HIP_TRY(hipSetDevice(g->dev));
  /* a graph handle replays the far-field sequence (fills, up, V, W, X,
   * down) as one graph: HIP runs a graph's nodes in one order on the launch
   * stream, so the U-list chunks and their copies, whose point is to run
   * beside one another, stay outside it */
  const bool graph = g->use_graph && mask == KIFMM_PHASE_ALL;
  /* the potentials land in the handle's pinned buffer (the caller's own
   * buffer when it is that one; otherwise one host pass follows), or without
   * pinned memory straight in the caller's buffer.  The U-list writes them
   * there itself (or the join, in the overlap layouts); without a U-list, or
   * when its items do not cover every target, a copy follows */
  double* const dst = pot_leaf ? (g->pinned ? g->pinned : pot_leaf) : nullptr;
  const bool direct = pot_leaf && g->pinned_dev && g->tiled && (mask & KIFMM_PHASE_U);
  const bool host_pass = pot_leaf && g->pinned && pot_leaf != g->pinned;
  const bool pipelined = direct && host_pass && g->cuts.size() > 2; /* the host pass chunk by chunk */
  if (graph && !g->gexec[0]) {
    HIP_TRY(hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal));
    g->capturing = true;
    const int r = enqueue_far(g, mask);
    hipGraph_t gr = nullptr;
    const hipError_t e = hipStreamEndCapture(g->stream, &gr);
    g->capturing = false;
    if (r != KIFMM_OK) {
      if (gr) (void)hipGraphDestroy(gr);
      return r;
    }
    HIP_TRY(e);
    g->graph[0] = gr;
    HIP_TRY(hipGraphInstantiate(&g->gexec[0], gr, nullptr, nullptr, 0));
  }
  /* E_START: the start of the first fill, unless that is inside the graph or
   * the second stream starts before it */
  g->phase = E_UP;
  g->phase_state = PHASE_EMPTY;
  g->ev_at[E_START] = E_START;
  g->start_ev = nullptr;
  if (graph || early_chunks(g, mask) > 0) HIP_TRY(hipEventRecord(ev[E_START], g->stream));
  else g->start_ev = ev[E_START];
  TRY(enqueue_side(g, mask));
  if (graph) { /* the far field's phases are not told apart */
    HIP_TRY(hipGraphLaunch(g->gexec[0], g->stream));
    for (int i = E_UP; i < E_DOWN; i++) g->ev_at[i] = E_START;
    g->phase_state = PHASE_UNSTAMPED;
    TRY(phase_end(g, E_DOWN));
  } else {
    TRY(enqueue_far(g, mask));
  }
  TRY(enqueue_near(g, mask, direct ? g->pinned_dev : nullptr, pipelined));
  if (dst && !direct && g->n_trg > 0)
    HIP_TRY(hipMemcpyAsync(dst, g->pot, sizeof(double) * (size_t)g->n_trg, hipMemcpyDeviceToHost, g->stream));
  HIP_TRY(hipEventRecord(ev[E_END], g->stream));
  double host_copy_ms = 0.0;
  if (host_pass) {
    const int nch = (int)g->cuts.size() - 1;
    double t0 = 0.0;
    if (pipelined) { /* each chunk as soon as its copy is done */
      for (int c = 0; c < nch; c++) {
        HIP_TRY(hipEventSynchronize(g->cd_ev[c]));
        if (c == nch - 1) t0 = kifmm::wall_seconds();
        host_copy(pot_leaf, g->pinned, (size_t)g->cuts[c], (size_t)g->cuts[c + 1]);
      }
    } else {
      HIP_TRY(hipEventSynchronize(ev[E_END]));
      t0 = kifmm::wall_seconds();
      host_copy(pot_leaf, g->pinned, 0, (size_t)g->n_trg);
    }
    host_copy_ms = (kifmm::wall_seconds() - t0) * 1e3; /* what is left after the device work */
  }
  HIP_TRY(hipEventSynchronize(ev[E_END]));
  g->den_queued = false;
  if (times) {
    float ms[E_END + 1] = {0};
    g->ev_at[E_END] = E_END;
    for (int i = E_UP; i <= E_END; i++)
      if (g->ev_at[i] != g->ev_at[i - 1])
        HIP_TRY(hipEventElapsedTime(&ms[i], ev[g->ev_at[i - 1]], ev[g->ev_at[i]]));
    float tot = 0;
    HIP_TRY(hipEventElapsedTime(&tot, ev[E_START], ev[E_END]));
    std::memset(times, 0, sizeof *times);
    if (!graph) {
      times->up = ms[E_UP];
      times->v_fft_src = ms[E_FFT];
      times->v_trans = ms[E_TRANS];
      times->v_hadamard = ms[E_HAD];
      times->v_ifft = ms[E_IFFT];
      times->vlist = ms[E_FFT] + ms[E_TRANS] + ms[E_HAD] + ms[E_IFFT];
      /* k_wx is one launch, its time split by what the lists' items cost; k_x_surf is X alone */
      const double w = mask & KIFMM_PHASE_W ? g->wx_cost[0] : 0.0, x = mask & KIFMM_PHASE_X ? g->wx_cost[1] : 0.0;
      times->wlist = w > 0.0 ? ms[E_WX] * (w / (w + x)) : 0.0;
      times->xlist = ms[E_WX] - times->wlist + ms[E_XSURF];
      times->down = ms[E_DOWN];
    }
    /* the U-list: its chunks after the far field, plus the span of the
     * early chunks on the second stream (which overlaps the far field) */
    times->ulist = times->p2p_kernel = ms[E_U];
    if (early_chunks(g, mask) > 0) {
      float mu = 0;
      HIP_TRY(hipEventElapsedTime(&mu, g->su0, g->su1));
      times->ulist += mu;
      times->p2p_kernel = early_chunks(g, mask) == (int)g->cuts.size() - 1 ? mu : times->ulist;
    }
    /* the copy left after the last kernel (it overlaps the U-list) */
    times->copy = ms[E_END] + host_copy_ms;
    times->total = tot + host_copy_ms;
  }
  return KIFMM_OK;
}

}  // namespace

extern "C" {

int kifmm_gpu_available(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n > 0 ? 1 : 0;
}

int kifmm_gpu_create(const kifmm_tree_view* tree, const kifmm_operators* ops, const kifmm_gpu_options* opts,
                     kifmm_gpu** out) {
  if (!tree || !ops || !out) {
    set_error("kifmm_gpu_create: null argument");
    return KIFMM_EINVAL;
  }
  *out = nullptr;
  if (tree->np != 3 && tree->np != 4 && tree->np != 6) {
    set_error("kifmm_gpu_create: NP must be 3, 4 or 6 on the GPU (got " + std::to_string(tree->np) + ")");
    return KIFMM_EUNSUP;
  }
  if (ops->np != tree->np || ops->n_e != tree->np * tree->np * tree->np - (tree->np - 2) * (tree->np - 2) * (tree->np - 2)) {
    set_error("kifmm_gpu_create: operators do not match the tree's NP");
    return KIFMM_EINVAL;
  }
  if (tree->n_nodes < 1 || tree->n_src < 0 || tree->n_trg < 0 || (tree->n_nodes - 1) % 8 != 0) {
    set_error("kifmm_gpu_create: malformed tree view");
    return KIFMM_EINVAL;
  }
  /* every index the kernels derive is checked on the host before any device call */
  const double t_plan0 = kifmm::wall_seconds();
  Plan P;
  try {
    const int pr = make_plan(tree, ops, opts && opts->precision == KIFMM_PREC_MIXED, P);
    if (pr != KIFMM_OK) return pr;
  } catch (const std::bad_alloc&) {
    set_error("host allocation failed in kifmm_gpu_create");
    return KIFMM_ENOMEM;
  }
  const double t_plan1 = kifmm::wall_seconds();
  kifmm_gpu* g = new (std::nothrow) kifmm_gpu();
  if (!g) {
    set_error("host allocation failed");
    return KIFMM_ENOMEM;
  }
  g->create_ms[0] = (t_plan1 - t_plan0) * 1e3;
  g->dev = opts ? opts->device : 0;
  g->precision = opts ? opts->precision : KIFMM_PREC_FP64;
  g->use_graph = opts ? (opts->flags & KIFMM_GPU_GRAPH) != 0 : 0;
  if (g->precision != KIFMM_PREC_FP64 && !(g->precision == KIFMM_PREC_MIXED && tree->np <= 4)) {
    set_error("kifmm_gpu_create: precision must be FP64, or MIXED with NP <= 4");
    delete g;
    return KIFMM_EUNSUP;
  }
  int r = KIFMM_OK;
  if (hipSetDevice(g->dev) != hipSuccess) {
    set_error("hipSetDevice failed");
    delete g;
    return KIFMM_EDEVICE;
  }
  if (take_stream(g->dev, &g->stream) != hipSuccess) {
    set_error("hipStreamCreate failed");
    delete g;
    return KIFMM_EDEVICE;
  }
  for (auto& e : g->ev) {
    if (hipEventCreate(&e) != hipSuccess) {
      set_error("hipEventCreate failed");
      kifmm_gpu_destroy(g);
      return KIFMM_EDEVICE;
    }
  }
  g->overlap = opts ? (opts->flags & KIFMM_GPU_OVERLAP) != 0 : 0;
  /* the second stream exists on every handle: the layout is a tuning choice */
  if (take_stream(g->dev, &g->side) != hipSuccess ||
      hipEventCreateWithFlags(&g->fork_ev, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&g->join_ev, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&g->far_ev, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&g->sdone_ev, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&g->copied_ev, hipEventDisableTiming) != hipSuccess ||
      hipEventCreate(&g->su0) != hipSuccess || hipEventCreate(&g->su1) != hipSuccess) {
    set_error("kifmm_gpu_create: second stream or its events could not be created");
    kifmm_gpu_destroy(g);
    return KIFMM_EDEVICE;
  }
  if (scratch_address(g->dev, &g->scratch) != KIFMM_OK) {
    kifmm_gpu_destroy(g);
    return KIFMM_EDEVICE;
  }
  g->cd_ev.assign(P.cuts.size(), nullptr);
  for (size_t c = 0; c < P.cuts.size(); c++)
    if (hipEventCreateWithFlags(&g->cd_ev[c], hipEventDisableTiming) != hipSuccess) {
      set_error("kifmm_gpu_create: copy-out events could not be created");
      kifmm_gpu_destroy(g);
      return KIFMM_EDEVICE;
    }
  if (hipHostMalloc((void**)&g->up_pin, UP_PIN, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    g->up_pin = nullptr;
  }
  try {
    const double t0 = kifmm::wall_seconds();
    r = build(g, tree, ops, P);
    if (r == KIFMM_OK) r = hipStreamSynchronize(g->stream) == hipSuccess ? KIFMM_OK : KIFMM_EDEVICE;
    const double t1 = kifmm::wall_seconds();
    if (r == KIFMM_OK && !(opts && (opts->flags & KIFMM_GPU_NO_CLOSE_LIST))) r = close_list(g);
    const double t2 = kifmm::wall_seconds();
    if (r == KIFMM_OK) r = trans_setup(g);
    if (r == KIFMM_OK && g->precision == KIFMM_PREC_MIXED) r = mixed_setup(g);
    if (r == KIFMM_OK) r = gram_setup(g);
    const double t3 = kifmm::wall_seconds();
    g->create_ms[1] = (t1 - t0) * 1e3;
    g->create_ms[2] = (t2 - t1) * 1e3;
    g->create_ms[3] = (t3 - t2) * 1e3;
  } catch (const std::bad_alloc&) {
    set_error("host allocation failed in kifmm_gpu_create");
    r = KIFMM_ENOMEM;
  }
  (void)hipStreamSynchronize(g->stream); /* staged uploads */
  if (g->up_pin) (void)hipHostFree(g->up_pin);
  g->up_pin = nullptr;
  if (r != KIFMM_OK) {
    kifmm_gpu_destroy(g);
    return r;
  }
  /* pinned buffer of the potentials; without it the copy goes straight to
   * the caller's (pageable) buffer */
  if (hipHostMalloc((void**)&g->pinned, sizeof(double) * std::max(g->n_trg, 1), hipHostMallocDefault) != hipSuccess)
    g->pinned = nullptr;
  if (g->pinned && hipHostGetDevicePointer((void**)&g->pinned_dev, g->pinned, 0) != hipSuccess) g->pinned_dev = nullptr;
  (void)hipGetLastError(); /* of either: done without, and not for the next launch check to find */
  if (hipDeviceSynchronize() != hipSuccess) {
    set_error("device synchronisation failed after upload");
    kifmm_gpu_destroy(g);
    return KIFMM_EDEVICE;
  }
  g->create_ms[4] = (kifmm::wall_seconds() - t_plan0) * 1e3;
  *out = g;
  return KIFMM_OK;
}

int kifmm_gpu_evaluate(kifmm_gpu* g, double* pot_leaf, kifmm_phase_times* times) {
  if (!g) {
    set_error("kifmm_gpu_evaluate: null handle");
    return KIFMM_EINVAL;
  }
  return evaluate(g, KIFMM_PHASE_ALL, pot_leaf, times);
}

int kifmm_gpu_evaluate_phases(kifmm_gpu* g, unsigned phases, double* pot_leaf, kifmm_phase_times* times) {
  if (!g) {
    set_error("kifmm_gpu_evaluate_phases: null handle");
    return KIFMM_EINVAL;
  }
  return evaluate(g, phases & KIFMM_PHASE_ALL, pot_leaf, times);
}

int kifmm_gpu_destroy(kifmm_gpu* g) {
  if (!g) return KIFMM_OK;
  (void)hipSetDevice(g->dev);
  bool ended = true;
  for (hipStream_t s : {g->stream, g->side, g->cstream})
    if (s && hipStreamSynchronize(s) != hipSuccess) ended = false;
  if (g->pinned) (void)hipHostFree(g->pinned);
  if (g->den_pin) (void)hipHostFree(g->den_pin);
  for (int k = 0; k < 2; k++) {
    if (g->gexec[k]) (void)hipGraphExecDestroy(g->gexec[k]);
    if (g->graph[k]) (void)hipGraphDestroy(g->graph[k]);
  }
  g->mem.free(ended);
  for (auto& e : g->ev)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : {g->fork_ev, g->join_ev, g->su0, g->su1, g->far_ev, g->sdone_ev, g->copied_ev})
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : g->cd_ev)
    if (e) (void)hipEventDestroy(e);
  for (hipStream_t s : {g->cstream, g->side, g->stream}) give_stream(g->dev, s);
  delete g;
  return KIFMM_OK;
}

int kifmm_gpu_release_idle(void) {
  drop_idle();
  return KIFMM_OK;
}

/* The split of nt targets over n sources: chunks of the sources until there
 * are DIR_ITEMS work items (four per block slot of the chip at 4 blocks of 4
 * waves per CU, so that the last round is a quarter of the work at most), a
 * chunk being at least one run of every lane.  At 8 chunks or more a multiple
 * of 8: a chunk then stays in one XCD's L2.  groups * n_chunk <= DIR_ITEMS,
 * or one chunk. */
struct DirectPlan {
  int groups, n_chunk, per;
  size_t part() const { return (size_t)groups * n_chunk * DIR_T; }
};
static DirectPlan direct_plan(int nt, int n) {
  constexpr int run = 256 * DIR_RUN;
  DirectPlan p;
  p.groups = (int)(((long)nt + DIR_T - 1) / DIR_T);
  const int most = std::max(1, (int)(((long)n + run - 1) / run));
  int c = std::min(std::max(1, DIR_ITEMS / p.groups), most);
  if (c >= 8) c &= ~7;
  p.n_chunk = c;
  p.per = (int)(((long)n + (long)c * run - 1) / ((long)c * run)) * run;
  return p;
}

/* d: x, y, z, sums [nt] each, then plan.part() double2.  The targets go up
 * in one copy, joined on the host first: three cost 8 us more each */
static int direct_queue(kifmm_gpu* g, const DirectPlan& p, int nt, const double* xyz, double* out, double* d) {
  const size_t b = sizeof(double) * (size_t)nt;
  double* const sums = d + 3 * (size_t)nt;
  double2* const part = reinterpret_cast<double2*>(d + 4 * (size_t)nt);
  HIP_TRY(hipMemcpyAsync(d, xyz, 3 * b, hipMemcpyHostToDevice, g->stream));
  const long items = (long)p.groups * p.n_chunk;
  hipLaunchKernelGGL(k_direct, dim3((unsigned)std::min<long>(items, 1 << 20)), dim3(256), 0, g->stream, nt, d, d + nt,
                     d + 2 * (size_t)nt, g->src4, g->n_src, p.groups, p.n_chunk, p.per, part);
  hipLaunchKernelGGL(k_direct_join, dim3((unsigned)(((long)nt + 63) / 64)), dim3(64), 0, g->stream, nt, p.groups,
                     p.n_chunk, part, sums);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, sums, b, hipMemcpyDeviceToHost, g->stream));
  return KIFMM_OK;
}
static int direct_run(kifmm_gpu* g, const DirectPlan& p, int nt, const double* tx, const double* ty, const double* tz,
                      double* out, double* d) {
  const std::unique_ptr<double[]> xyz(new (std::nothrow) double[3 * (size_t)nt]);
  if (!xyz) {
    set_error("direct sums: out of host memory");
    return KIFMM_ENOMEM;
  }
  std::copy(tx, tx + nt, xyz.get());
  std::copy(ty, ty + nt, xyz.get() + nt);
  std::copy(tz, tz + nt, xyz.get() + 2 * (size_t)nt);
  const int r = direct_queue(g, p, nt, xyz.get(), out, d);
  HIP_TRY(hipStreamSynchronize(g->stream));
  return r;
}

int kifmm_gpu_direct(kifmm_gpu* g, int nt, const double* tx, const double* ty, const double* tz, double* out) {
  if (!g || nt <= 0 || !tx || !ty || !tz || !out) {
    set_error("kifmm_gpu_direct: invalid argument");
    return KIFMM_EINVAL;
  }
  HIP_TRY(hipSetDevice(g->dev));
  const DirectPlan p = direct_plan(nt, g->n_src);
  void* d = nullptr;
  HIP_TRY(device_malloc(&d, sizeof(double) * (4 * (size_t)nt + 2 * p.part())));
  const int r = direct_run(g, p, nt, tx, ty, tz, out, (double*)d);
  (void)hipFree(d);
  return r;
}

int kifmm_gpu_direct_noalloc(kifmm_gpu* g, int nt, const double* tx, const double* ty, const double* tz,
                             double* out) {
  if (!g || nt <= 0 || !tx || !ty || !tz || !out) {
    set_error("kifmm_gpu_direct_noalloc: invalid argument");
    return KIFMM_EINVAL;
  }
  if (nt > KIFMM_DIRECT_NOALLOC_MAX) {
    set_error("kifmm_gpu_direct_noalloc: " + std::to_string(nt) + " points exceed the scratch of " +
              std::to_string(KIFMM_DIRECT_NOALLOC_MAX) + " (use kifmm_gpu_direct)");
    return KIFMM_EINVAL;
  }
  if (!g->scratch) {
    set_error("kifmm_gpu_direct_noalloc: no scratch address for this device");
    return KIFMM_EDEVICE;
  }
  HIP_TRY(hipSetDevice(g->dev));
  /* 4 nt doubles and at most DIR_ITEMS groups of partial sums: MAX / DIR_T
   * groups <= DIR_ITEMS.  The kernels assign every partial and every sum
   * that is read, so nothing needs clearing */
  static_assert(KIFMM_DIRECT_NOALLOC_MAX / DIR_T <= DIR_ITEMS, "one chunk of every group has to fit the scratch");
  return direct_run(g, direct_plan(nt, g->n_src), nt, tx, ty, tz, out, g->scratch);
}

double kifmm_problem_validate_gpu(kifmm_problem* p, kifmm_gpu* g, const double* pot_orig, int nv, int* chk_ids,
                                  double* direct_out) {
  if (!p || !g || !pot_orig || nv <= 0) {
    set_error("kifmm_problem_validate_gpu: invalid argument");
    return -1.0;
  }
  std::vector<int> ids(nv);
  std::vector<double> xyz(3 * (size_t)nv), direct(nv);
  if (kifmm::sample_targets(p, nv, ids.data(), xyz.data()) != KIFMM_OK) return -1.0;
  if (kifmm_gpu_direct(g, nv, xyz.data(), xyz.data() + nv, xyz.data() + 2 * (size_t)nv, direct.data()) != KIFMM_OK)
    return -1.0;
  double vn = 0.0, en = 0.0;
  for (int k = 0; k < nv; k++) {
    const double f = pot_orig[ids[k]];
    vn += f * f;
    en += (direct[k] - f) * (direct[k] - f);
  }
  if (chk_ids) std::memcpy(chk_ids, ids.data(), sizeof(int) * nv);
  if (direct_out) std::memcpy(direct_out, direct.data(), sizeof(double) * nv);
  return std::sqrt(en) / std::sqrt(vn);
}

int kifmm_gpu_plan(const kifmm_tree_view* tree, const kifmm_operators* ops, kifmm_work_counts* out) {
  if (!tree || !ops) {
    set_error("kifmm_gpu_plan: null argument");
    return KIFMM_EINVAL;
  }
  if (tree->np != 3 && tree->np != 4 && tree->np != 6) {
    set_error("kifmm_gpu_plan: NP must be 3, 4 or 6 on the GPU");
    return KIFMM_EUNSUP;
  }
  Plan P;
  int r = KIFMM_OK;
  try {
    r = make_plan(tree, ops, false, P);
  } catch (const std::bad_alloc&) {
    set_error("host allocation failed in kifmm_gpu_plan");
    return KIFMM_ENOMEM;
  }
  if (r == KIFMM_OK && out) *out = P.wc;
  return r;
}

int kifmm_gpu_set_tuning(kifmm_gpu* g, const kifmm_gpu_tuning* t) {
  if (!g || !t) {
    set_error("kifmm_gpu_set_tuning: null argument");
    return KIFMM_EINVAL;
  }
  if (t->p2p_form < KIFMM_P2P_STATIC || t->p2p_form > KIFMM_P2P_SPLIT ||
      (t->hadamard_fb != 2 && t->hadamard_fb != 4 && t->hadamard_fb != 8 && t->hadamard_fb != 16) ||
      t->hadamard_auto < 0 || t->hadamard_auto > 1 ||
      (t->hadamard_form != KIFMM_HAD_VALU && t->hadamard_form != KIFMM_HAD_MFMA) ||
      t->overlap < 0 || t->overlap > 6 || t->up_form < KIFMM_LEVEL_AUTO || t->up_form > KIFMM_LEVEL_FUSED ||
      t->down_form < KIFMM_LEVEL_AUTO || t->down_form > KIFMM_LEVEL_FUSED) {
    set_error("kifmm_gpu_set_tuning: p2p_form must be a KIFMM_P2P_* value, hadamard_fb 2, 4, 8 or 16, "
              "hadamard_auto 0 or 1, hadamard_form a KIFMM_HAD_* value, overlap 0 to 6 and up_form / down_form KIFMM_LEVEL_* "
              "values");
    return KIFMM_EINVAL;
  }
  if (g->precision == KIFMM_PREC_MIXED && t->p2p_form != KIFMM_P2P_STATIC &&
      !(t->p2p_form == KIFMM_P2P_SPLIT && g->close_listed)) {
    set_error("kifmm_gpu_set_tuning: the mixed path has the STATIC and, with a close-pair list, the SPLIT "
              "U-list forms");
    return KIFMM_EUNSUP;
  }
  if (g->precision == KIFMM_PREC_FP64 && t->p2p_form == KIFMM_P2P_SPLIT) {
    set_error("kifmm_gpu_set_tuning: the SPLIT U-list form is the mixed path's");
    return KIFMM_EUNSUP;
  }
  if (t->p2p_form == g->p2p_form && t->hadamard_fb == g->had_fb && t->hadamard_auto == g->had_auto &&
      t->hadamard_form == g->had_form &&
      t->overlap == g->overlap && t->up_form == g->up_form && t->down_form == g->down_form)
    return KIFMM_OK;
  g->p2p_form = t->p2p_form;
  g->had_fb = t->hadamard_fb;
  g->had_auto = t->hadamard_auto;
  g->had_form = t->hadamard_form;
  g->overlap = t->overlap;
  g->up_form = t->up_form;
  g->down_form = t->down_form;
  for (int k = 0; k < 2; k++) {
    if (g->gexec[k]) (void)hipGraphExecDestroy(g->gexec[k]);
    if (g->graph[k]) (void)hipGraphDestroy(g->graph[k]);
    g->gexec[k] = nullptr;
    g->graph[k] = nullptr;
  }
  return KIFMM_OK;
}

int kifmm_gpu_get_tuning(const kifmm_gpu* g, kifmm_gpu_tuning* t) {
  if (!g || !t) {
    set_error("kifmm_gpu_get_tuning: null argument");
    return KIFMM_EINVAL;
  }
  std::memset(t, 0, sizeof *t);
  t->p2p_form = g->p2p_form;
  t->hadamard_fb = g->had_fb;
  t->hadamard_auto = g->had_auto;
  t->hadamard_form = g->had_form;
  t->overlap = g->overlap;
  t->up_form = g->up_form;
  t->down_form = g->down_form;
  return KIFMM_OK;
}

int kifmm_gpu_autotune(kifmm_gpu* g, int reps, kifmm_gpu_tuning* best, double* ms, int n_ms) {
  if (!g || reps < 1 || (ms && n_ms < 0)) {
    set_error("kifmm_gpu_autotune: null handle or reps < 1");
    return KIFMM_EINVAL;
  }
  double t[21];
  std::fill(t, t + 21, -1.0);
  kifmm_gpu_tuning cur{};
  kifmm_gpu_get_tuning(g, &cur);
  /* the fastest of reps timed runs after one warm-up: the U-list, the
   * Hadamard, or the up and the down phase (out[0], out[1]) */
  auto time_phase = [&](unsigned phase, double* out) -> int {
    kifmm_phase_times pt{};
    double m[2] = {0.0, 0.0};
    for (int r = 0; r <= reps; r++) {
      const int rc = evaluate(g, phase, nullptr, &pt);
      if (rc != KIFMM_OK) return rc;
      const double v[2] = {phase == KIFMM_PHASE_U ? pt.ulist : phase == KIFMM_PHASE_V ? pt.v_hadamard : pt.up,
                           pt.down};
      for (int k = 0; k < 2; k++)
        if (r == 1 || (r > 1 && v[k] < m[k])) m[k] = v[k]; /* run 0 warms up */
    }
    out[0] = m[0];
    if (phase == (KIFMM_PHASE_UP | KIFMM_PHASE_DOWN)) out[1] = m[1];
    return KIFMM_OK;
  };
  kifmm_gpu_tuning c = cur;
  /* the U-list forms of the handle's path, with their slot in t */
  std::vector<std::pair<int, int>> forms;
  if (g->precision == KIFMM_PREC_FP64)
    forms = {{KIFMM_P2P_STATIC, 0}, {KIFMM_P2P_PERSISTENT, 1}, {KIFMM_P2P_STATIC64, 2}};
  else if (g->close_listed)
    forms = {{KIFMM_P2P_STATIC, 0}, {KIFMM_P2P_SPLIT, 11}};
  else
    forms = {{KIFMM_P2P_STATIC, 0}};
  int best_form = KIFMM_P2P_STATIC, best_slot = 0;
  for (const auto& f : forms) {
    c.p2p_form = f.first;
    TRY(kifmm_gpu_set_tuning(g, &c));
    TRY(time_phase(KIFMM_PHASE_U, &t[f.second]));
    if (t[f.second] < t[best_slot]) {
      best_form = f.first;
      best_slot = f.second;
    }
  }
  c.p2p_form = best_form;
  c.hadamard_fb = 8;
  c.hadamard_auto = 1;
  TRY(kifmm_gpu_set_tuning(g, &c));
  const int own_fb = had_block_size(g);
  const int fbs[3] = {4, 8, 16};
  int best_v = 0;
  c.hadamard_auto = 0;
  for (int k = 0; k < 6; k++) { /* VALU fb 4, 8, 16, then MFMA fb 4, 8, 16 */
    c.hadamard_form = k / 3;
    c.hadamard_fb = fbs[k % 3];
    TRY(kifmm_gpu_set_tuning(g, &c));
    TRY(time_phase(KIFMM_PHASE_V, &t[3 + k]));
    if (t[3 + k] < t[3 + best_v]) best_v = k;
  }
  double t_v = t[3 + best_v];
  c.hadamard_form = best_v / 3;
  c.hadamard_fb = fbs[best_v % 3];
  if (own_fb < fbs[0] && g->n_hgroups > 0) { /* where the handle picks fewer by itself, they are tried too */
    kifmm_gpu_tuning f = c;
    f.hadamard_fb = own_fb;
    for (f.hadamard_form = 0; f.hadamard_form < 2; f.hadamard_form++) {
      double t_f;
      TRY(kifmm_gpu_set_tuning(g, &f));
      TRY(time_phase(KIFMM_PHASE_V, &t_f));
      if (t_f >= t_v) continue;
      t_v = t_f;
      c = f;
    }
  }
  /* up and down: the column GEMMs against the fused kernels, each phase on
   * its own (slots 14, 15: up; 16, 17: down) */
  for (int k = 0; k < 2; k++) {
    c.up_form = c.down_form = k == 0 ? KIFMM_LEVEL_GEMM : KIFMM_LEVEL_FUSED;
    TRY(kifmm_gpu_set_tuning(g, &c));
    double ud[2];
    TRY(time_phase(KIFMM_PHASE_UP | KIFMM_PHASE_DOWN, ud));
    t[14 + k] = ud[0];
    t[16 + k] = ud[1];
  }
  c.up_form = t[15] < t[14] ? KIFMM_LEVEL_FUSED : KIFMM_LEVEL_GEMM;
  c.down_form = t[17] < t[16] ? KIFMM_LEVEL_FUSED : KIFMM_LEVEL_GEMM;
  /* stream layout, on whole evaluations timed eagerly (a graph handle
   * would otherwise capture here) */
  const int use_graph = g->use_graph;
  g->use_graph = 0;
  /* slots of the layouts 0 .. 6 in t */
  const int lslot[7] = {9, 10, 12, 13, 18, 19, 20};
  int best_l = 0, rc = KIFMM_OK;
  for (int l = 0; l < 7 && rc == KIFMM_OK; l++) {
    c.overlap = l;
    rc = kifmm_gpu_set_tuning(g, &c);
    kifmm_phase_times pt{};
    for (int r = 0; r <= reps && rc == KIFMM_OK; r++) {
      rc = evaluate(g, KIFMM_PHASE_ALL, g->pinned, &pt); /* with the copy-out, as the layouts differ there */
      if (r == 1 || (r > 1 && pt.total < t[lslot[l]])) t[lslot[l]] = pt.total; /* run 0 warms up */
    }
    if (rc == KIFMM_OK && t[lslot[l]] < t[lslot[best_l]]) best_l = l;
  }
  g->use_graph = use_graph;
  TRY(rc);
  c.overlap = best_l;
  TRY(kifmm_gpu_set_tuning(g, &c));
  if (best) *best = c;
  if (ms)
    for (int k = 0; k < std::min(n_ms, 21); k++) ms[k] = t[k];
  return KIFMM_OK;
}

int kifmm_gpu_work_counts(const kifmm_gpu* g, kifmm_work_counts* out) {
  if (!g || !out) return KIFMM_EINVAL;
  *out = g->counts;
  out->close_pairs = g->close_listed ? (double)g->n_close : -1.0;
  out->copy_chunks = (double)std::max<size_t>(g->cuts.size(), 2) - 1.0;
  out->hadamard_block = had_block_size(g);
  return KIFMM_OK;
}

double* kifmm_gpu_output(kifmm_gpu* g) { return g ? g->pinned : nullptr; }

/* Densities of up to DEN_PINNED bytes are copied to pinned memory that the
 * packing kernel reads, and not waited for (the evaluation follows on the same
 * stream); above, the runtime's copy, waited for.  The line is where the two
 * routes meet, by the time of this call and an evaluation (the call alone
 * returns sooner up to 2M points, but one thread fills the pinned memory and
 * the evaluation waits for the kernel to read it): runtime's copy -> pinned at
 * 131 thousand points 530 -> 493 us, 500 thousand 958 -> 940, 700 thousand 1493 ->
 * 1488, 1M 2643 -> 2642, but 1.4M 4770 -> 4915, 2M 8373 -> 8636, 4M 7134 -> 7647. */
constexpr size_t DEN_PINNED = (size_t)8 << 20;

int kifmm_gpu_set_densities(kifmm_gpu* g, const double* den_leaf) {
  if (!g || (!den_leaf && g->n_src > 0)) {
    set_error("kifmm_gpu_set_densities: invalid argument");
    return KIFMM_EINVAL;
  }
  if (g->n_src == 0) return KIFMM_OK;
  HIP_TRY(hipSetDevice(g->dev));
  const size_t bytes = sizeof(double) * (size_t)g->n_src;
  if (bytes <= DEN_PINNED && !g->den_pin) {
    if (hipHostMalloc((void**)&g->den_pin, bytes, hipHostMallocDefault) != hipSuccess) g->den_pin = nullptr;
    else if (hipHostGetDevicePointer((void**)&g->den_pin_dev, g->den_pin, 0) != hipSuccess) g->den_pin_dev = nullptr;
    (void)hipGetLastError();
  }
  const double* den = g->den_stage;
  const bool pinned = bytes <= DEN_PINNED && g->den_pin_dev;
  if (pinned) {
    if (g->den_queued) HIP_TRY(hipStreamSynchronize(g->stream)); /* the previous densities are not read yet */
    g->den_queued = true;
    std::memcpy(g->den_pin, den_leaf, bytes);
    den = g->den_pin_dev;
  } else {
    HIP_TRY(hipMemcpyAsync(g->den_stage, den_leaf, bytes, hipMemcpyHostToDevice, g->stream));
  }
  const int blocks = (int)std::min<size_t>(4096, ((size_t)g->n_src + 255) / 256);
  hipLaunchKernelGGL(k_set_w, dim3(blocks), dim3(256), 0, g->stream, g->src4, den, (size_t)g->n_src);
  HIP_TRY(hipGetLastError());
  if (g->precision == KIFMM_PREC_MIXED) TRY(mixed_sources(g));
  if (!pinned) HIP_TRY(hipStreamSynchronize(g->stream)); /* den_leaf may be released on return */
  return KIFMM_OK;
}

int kifmm_gpu_create_times(const kifmm_gpu* g, double* ms, int n) {
  if (!g || !ms || n < 0) {
    set_error("kifmm_gpu_create_times: invalid argument");
    return KIFMM_EINVAL;
  }
  for (int k = 0; k < std::min(n, 5); k++) ms[k] = g->create_ms[k];
  return KIFMM_OK;
}

long kifmm_gpu_close_list(const kifmm_gpu* g, int* ptr, long n_ptr, int* idx, long n_idx) {
  if (!g || n_ptr < 0 || n_idx < 0 || (n_ptr && !ptr) || (n_idx && !idx)) {
    set_error("kifmm_gpu_close_list: invalid argument");
    return KIFMM_EINVAL;
  }
  if (!g->close_listed) { /* KIFMM_GPU_NO_CLOSE_LIST, or too many pairs */
    set_error("kifmm_gpu_close_list: this handle has no close-pair list");
    return KIFMM_EUNSUP;
  }
  if (n_ptr > (long)g->n_trg + 1 || n_idx > g->n_close) {
    set_error("kifmm_gpu_close_list: count exceeds the list");
    return KIFMM_EINVAL;
  }
  if (hipSetDevice(g->dev) != hipSuccess || hipStreamSynchronize(g->stream) != hipSuccess ||
      (n_ptr && hipMemcpy(ptr, g->cptr, sizeof(int) * n_ptr, hipMemcpyDeviceToHost) != hipSuccess) ||
      (n_idx && hipMemcpy(idx, g->cidx, sizeof(int) * n_idx, hipMemcpyDeviceToHost) != hipSuccess)) {
    set_error("kifmm_gpu_close_list: copy failed");
    return KIFMM_EDEVICE;
  }
  return (long)g->n_close;
}

int kifmm_gpu_copy_intermediate(const kifmm_gpu* g, int which, double* out, long count) {
  if (!g || !out || count < 0) {
    set_error("kifmm_gpu_copy_intermediate: invalid argument");
    return KIFMM_EINVAL;
  }
  const double* src = nullptr;
  long avail = 0;
  switch (which) {
    case 0: src = g->uden; avail = (long)g->n_nodes * g->ld_e; break;
    case 1: src = g->dchk; avail = (long)g->n_nodes * g->ld_e; break;
    case 2: src = g->dden; avail = (long)g->n_nodes * g->ld_e; break;
    case 3: src = g->pot; avail = g->n_trg; break;
    default: set_error("kifmm_gpu_copy_intermediate: which must be 0..3"); return KIFMM_EINVAL;
  }
  if (count > avail) {
    set_error("kifmm_gpu_copy_intermediate: count exceeds the array");
    return KIFMM_EINVAL;
  }
  if (hipSetDevice(g->dev) != hipSuccess || hipStreamSynchronize(g->stream) != hipSuccess ||
      hipMemcpy(out, src, sizeof(double) * count, hipMemcpyDeviceToHost) != hipSuccess) {
    set_error("kifmm_gpu_copy_intermediate: copy failed");
    return KIFMM_EDEVICE;
  }
  return KIFMM_OK;
}

}  // extern "C"
