// Batched (stage-fused) evaluation: many ciphertexts, mixed levels and ring
// dimensions, one launch per pipeline stage per parameter set, the whole
// sequence captured once as a hipGraph and replayed.
//
// A batch is a list of layers; a layer holds independent operations
// (HomMul+relin+rescale, rotate[-and-accumulate], forward/inverse NTT) grouped
// by parameter set.  Layers run in order (each may consume the previous one's
// outputs, as the rotate-and-sum steps of ckks_sumslots do,
// aoa-ntt/src/ckks/ckks.cpp:479-495).  Every stage of a group is one
// descriptor-driven kernel launch covering all its ciphertexts, so a launch
// carries thousands of workgroups even when each ciphertext is small, and
// evaluation keys are shared between them.
#include <algorithm>
#include <cstring>
#include <vector>

#include "internal.hpp"

using namespace aoa;

namespace aoa {

struct BatchGroup {
  const aoa_params* params = nullptr;
  const uint64_t* evk_b = nullptr;
  const uint64_t* evk_a = nullptr;
  std::vector<aoa_mul_item> muls;
  std::vector<aoa_rot_item> rots;
  std::vector<aoa_ntt_item> ntts;
  // descriptor tables (device) and counts, set by batch_fill
  NttDesc* d_pre_fwd = nullptr;
  int n_pre_fwd = 0;
  NttDesc* d_pre_inv = nullptr;
  int n_pre_inv = 0;
  AutoDesc* d_auto = nullptr;
  int n_auto = 0;
  // HomMuls and rotations (fused.hpp): items, HomMuls first, and the limbs of
  // each stage's launches, item << 8 | limb
  FzItem* d_items = nullptr;
  int n_mul = 0, n_rot = 0;
  int max_level = 0;
  uint32_t* d_rows = nullptr;  // d2 = a1 b1 and its inverse rows
  uint32_t* d_keyb = nullptr;  // key products of the special limbs
  uint32_t* d_keyq = nullptr;  // key products of the Q limbs
  int n_rows = 0, n_keyb = 0, n_keyq = 0;
  // leading entries of rows and keyq whose prime is above 2^56 (-1: not split)
  int ns_rows = -1, ns_keyq = -1;
  int field_q = 0, field_b = 0;  // form of the Q primes after q0, of the special primes
};

struct BatchLayer {
  std::vector<BatchGroup> groups;
};

}  // namespace aoa

struct aoa_batch {
  std::vector<BatchLayer> layers;
  aoa_batch_options opt{0, 1, 0, 0};
  bool built = false;
  void* dmem = nullptr;  // descriptors
  void* ws = nullptr;    // workspace
  size_t ws_bytes = 0;
  size_t desc_bytes = 0;
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  BatchLayer* layers_cur = nullptr;  // layer being enqueued
};

namespace aoa {

static BatchGroup& group_for(aoa_batch* b, const aoa_params* p, const uint64_t* kb, const uint64_t* ka) {
  if (b->layers.empty()) b->layers.emplace_back();
  BatchLayer& L = b->layers.back();
  for (auto& g : L.groups)
    if (g.params == p && g.evk_b == kb && g.evk_a == ka) return g;
  L.groups.emplace_back();
  BatchGroup& g = L.groups.back();
  g.params = p;
  g.evk_b = kb;
  g.evk_a = ka;
  return g;
}

// Workspace bytes (max over layers of the layer's sum) and descriptor bytes.
void batch_sizes(const aoa_batch* b, size_t* ws_bytes, size_t* desc_bytes) {
  size_t ws = 0, desc = 0;
  for (auto& L : b->layers) {
    size_t s = 0;
    for (auto& g : L.groups) {
      const size_t N = g.params->host.N, K = g.params->host.K;
      for (auto& it : g.muls) {
        const size_t Lq = it.level + 1;
        s += mul_ws_limbs((int)Lq, (int)K) * N * 8;
        desc += sizeof(FzItem) + (2 * Lq + K) * sizeof(uint32_t);
      }
      for (auto& it : g.rots) {
        const size_t Lq = it.level + 1;
        s += rot_ws_limbs((int)Lq, (int)K) * N * 8;
        desc += sizeof(FzItem) + 2 * Lq * sizeof(AutoDesc) + (Lq + K) * sizeof(uint32_t);
      }
      for (auto& it : g.ntts) desc += 2 * (size_t)(it.level + 1) * sizeof(NttDesc);
      desc += 8 * 256;  // per-table alignment slack
    }
    ws = std::max(ws, s);
  }
  *ws_bytes = ws;
  *desc_bytes = desc;
}

// Fills every descriptor table into `host` (desc_cap bytes) using workspace
// `ws` and device descriptor base `dev`; device table pointers are set to
// dev + offset.  Returns the bytes used, or 0 if desc_cap is too small.
size_t batch_fill(aoa_batch* b, uint64_t* ws, char* host, char* dev, size_t desc_cap) {
  size_t used = 0;
  bool overflow = false;
  auto put = [&](const void* p, size_t bytes) -> char* {
    size_t off = (used + 255) & ~(size_t)255;
    if (off + bytes > desc_cap) {
      overflow = true;
      return nullptr;
    }
    std::memcpy(host + off, p, bytes);
    used = off + bytes;
    return dev + off;
  };
  for (auto& L : b->layers) {
    uint64_t* w = ws;  // layers reuse the workspace
    for (auto& g : L.groups) {
      const DevParams& P = g.params->dev;
      const size_t N = (size_t)P.N;
      const int k = P.k, K = P.K;
      std::vector<NttDesc> prefwd, preinv;
      std::vector<FzItem> items;
      std::vector<uint32_t> rows, keyb, keyq;
      std::vector<AutoDesc> au;
      g.max_level = 0;
      for (auto& it : g.ntts)
        for (int y = 0; y < 2; ++y)
          for (int i = 0; i <= it.level; ++i) {
            uint64_t* l = it.poly[y] + (size_t)i * N;
            (it.dir == AOA_FORWARD ? prefwd : preinv).push_back({l, l, i, 0});
          }
      auto key_entries = [&](uint32_t item, int Lq) {
        for (int m = 0; m < Lq; ++m) keyq.push_back(item << 8 | m);
        for (int m = Lq; m < Lq + K; ++m) keyb.push_back(item << 8 | m);
      };
      for (auto& it : g.muls) {
        const int lv = it.level, Lq = lv + 1;
        const uint32_t item = (uint32_t)items.size();
        g.max_level = std::max(g.max_level, lv);
        FzItem z{};
        z.a0 = it.c1[0];
        z.a1 = it.c1[1];
        z.b0 = it.c2[0];
        z.b1 = it.c2[1];
        z.kb = g.evk_b;
        z.ka = g.evk_a;
        z.D = w;
        z.X = z.D + (size_t)Lq * N;
        z.P0 = z.X + (size_t)K * N;
        z.P1 = z.P0 + (size_t)(Lq + K) * N;
        z.out0 = it.out[0];
        z.out1 = it.out[1];
        z.level = lv;
        z.rescale = 1;
        w += mul_ws_limbs(Lq, K) * N;
        items.push_back(z);
        for (int i = 0; i < Lq; ++i) rows.push_back(item << 8 | i);
        key_entries(item, Lq);
      }
      g.n_mul = (int)items.size();
      for (auto& it : g.rots) {
        const int lv = it.level, Lq = lv + 1;
        const uint32_t item = (uint32_t)items.size();
        g.max_level = std::max(g.max_level, lv);
        uint64_t* R0 = w;
        uint64_t* R1 = R0 + (size_t)Lq * N;
        const uint64_t ginv = galois_inverse(galois_of(it.rot_slots, P.N), P.N);
        for (int i = 0; i < Lq; ++i) {
          const size_t o = (size_t)i * N;
          au.push_back({it.in[0] + o, R0 + o, it.accumulate ? it.in[0] + o : nullptr, ginv, i, 0});
          au.push_back({it.in[1] + o, R1 + o, nullptr, ginv, i, 0});
        }
        FzItem z{};
        z.d = R1;
        z.kb = it.rtk_b;
        z.ka = it.rtk_a;
        z.XQ = R1 + (size_t)Lq * N;
        z.X = z.XQ + (size_t)Lq * N;
        z.P0 = z.X + (size_t)K * N;
        z.P1 = z.P0 + (size_t)(Lq + K) * N;
        z.add0 = R0;
        z.add1 = it.accumulate ? it.in[1] : nullptr;
        z.out0 = it.out[0];
        z.out1 = it.out[1];
        z.level = lv;
        w += rot_ws_limbs(Lq, K) * N;
        items.push_back(z);
        key_entries(item, Lq);
      }
      g.n_rot = (int)items.size() - g.n_mul;
      // Prime-major order: the limbs of one prime from every item run next
      // to each other, so their workgroups (spread over the XCDs by block
      // index) find that prime's twiddles, and in the key stage its key
      // limbs, in the L2 cache.  Entries of a stage are independent.
      // Item order (prime_major = 0) keeps the order of insertion: the limbs of
      // one item after the other.
      const bool pm = b->opt.prime_major != 0;
      auto by_prime = [pm](auto& v) {
        if (pm) std::stable_sort(v.begin(), v.end(), [](const auto& a, const auto& b) { return a.prime < b.prime; });
      };
      by_prime(prefwd);
      by_prime(preinv);
      // Q limbs come first in an item, so in each list the entries of one prime
      // are those of one limb (special limbs: of one place after level + 1)
      auto prime_of = [&](uint32_t e) { return (int)(e & 255) - (items[e >> 8].level + 1); };
      if (pm) {
        auto by_limb = [](uint32_t a, uint32_t b) { return (a & 255) < (b & 255); };
        std::stable_sort(rows.begin(), rows.end(), by_limb);
        std::stable_sort(keyq.begin(), keyq.end(), by_limb);
        std::stable_sort(keyb.begin(), keyb.end(), [&](uint32_t a, uint32_t b) { return prime_of(a) < prime_of(b); });
      }
      // The limbs of primes wider than 2^56 (q0), which sort first, take another
      // form of arithmetic; with them in a launch of their own the others'
      // launch compiles for its form alone and holds fewer registers.  Small
      // stages (a serving step of a few requests) keep one launch by default: 60
      // entries at N = 2^16 0.356 ms in one launch, 0.383 in two; 960 entries
      // 4.32 and 4.31.
      constexpr size_t kSplitMin = 256;
      auto split_at = [&](const std::vector<uint32_t>& v) -> int {
        if (b->opt.strict_split < 0 || !pm) return -1;
        if (b->opt.strict_split == 0 && v.size() < kSplitMin) return -1;
        const auto& dp = g.params->host.dprimes;
        int n = 0;
        while (n < (int)v.size() && dp[v[n] & 255].field == FIELD_STRICT) ++n;
        for (size_t t = n; t < v.size(); ++t)
          if (dp[v[t] & 255].field != dp[v[n] & 255].field) return -1;  // not in order
        return n;
      };
      g.field_q = (int)g.params->host.dprimes[k > 1 ? 1 : 0].field;
      g.field_b = g.params->host.K ? (int)g.params->host.dprimes[k].field : FIELD_LAZY;
      g.ns_rows = split_at(rows);
      g.ns_keyq = split_at(keyq);
      g.n_rows = (int)rows.size();
      g.n_keyb = (int)keyb.size();
      g.n_keyq = (int)keyq.size();
      g.n_pre_fwd = (int)prefwd.size();
      g.n_pre_inv = (int)preinv.size();
      g.n_auto = (int)au.size();
      g.d_pre_fwd = (NttDesc*)(prefwd.empty() ? nullptr : put(prefwd.data(), prefwd.size() * sizeof(NttDesc)));
      g.d_pre_inv = (NttDesc*)(preinv.empty() ? nullptr : put(preinv.data(), preinv.size() * sizeof(NttDesc)));
      g.d_items = (FzItem*)(items.empty() ? nullptr : put(items.data(), items.size() * sizeof(FzItem)));
      auto put_list = [&](const std::vector<uint32_t>& v) {
        return (uint32_t*)(v.empty() ? nullptr : put(v.data(), v.size() * sizeof(uint32_t)));
      };
      g.d_rows = put_list(rows);
      g.d_keyb = put_list(keyb);
      g.d_keyq = put_list(keyq);
      g.d_auto = (AutoDesc*)(au.empty() ? nullptr : put(au.data(), au.size() * sizeof(AutoDesc)));
    }
  }
  return overflow ? 0 : used;
}

// Records a HIP event pair around each stage launch of batch_enqueue (on the
// stream the stage is launched on); used only by aoa_batch_stage_times.
struct StageTimer {
  std::vector<int> stage;
  std::vector<hipEvent_t> ev;  // begin, end pairs
  bool ok = true;
  void begin(int s, hipStream_t st) {
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) { ok = false; return; }
    if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); ok = false; return; }
    stage.push_back(s);
    ev.push_back(e0);
    ev.push_back(e1);
    (void)hipEventRecord(e0, st);
  }
  void end(hipStream_t st) {
    if (ok) (void)hipEventRecord(ev.back(), st);
  }
  ~StageTimer() {
    for (auto e : ev) (void)hipEventDestroy(e);
  }
};

// The batch's NTT split where the group's ring admits it and the group has
// transforms of its own (nothing else uses one), else 0.
static int group_split(const aoa_batch* b, const BatchGroup& g) {
  return !g.ntts.empty() && b->opt.ntt_split && ntt_valid_split(g.params->host.N, b->opt.ntt_split) ? b->opt.ntt_split : 0;
}
// Builds the tables of the batch's split, so that a launch (or a capture) does not.
static int prepare_splits(const aoa_batch* b) {
  for (auto& L : b->layers)
    for (auto& g : L.groups)
      if (const int n1 = group_split(b, g)) {
        DevParams P = g.params->dev;
        if (const int rc = use_split(g.params, n1, &P)) return rc;
      }
  return AOA_OK;
}

// The parameters a group's launches use: its handle's, with the batch's NTT
// split and XCD mapping.
static DevParams launch_params(const aoa_batch* b, const BatchGroup& g) {
  DevParams P = g.params->dev;
  if (const int n1 = group_split(b, g)) (void)use_split(g.params, n1, &P);
  P.xcd_chunks = b->opt.xcd_chunks ? 1 : 0;
  return P;
}

// Issues every stage launch of the batch on stream st (stage order
// AOA_STAGE_*); with a timer, each (layer, stage) launch run is bracketed by
// an event pair.
int batch_enqueue(aoa_batch* b, hipStream_t st, StageTimer* tm) {
  int rc = AOA_OK;
  auto run = [&](int s, auto&& has, auto&& go) {
    bool any = false;
    for (auto& g : b->layers_cur->groups) any = any || has(g);
    if (!any || rc) return;
    if (tm) tm->begin(s, st);
    for (auto& g : b->layers_cur->groups)
      if (has(g) && go(g)) rc = set_error(AOA_ERR_UNSUPPORTED, "no NTT split");
    if (tm) tm->end(st);
  };
  for (auto& L : b->layers) {
    b->layers_cur = &L;
    run(AOA_STAGE_PRE_FWD, [](BatchGroup& g) { return g.n_pre_fwd > 0; },
        [&](BatchGroup& g) { return ntt_forward_desc(launch_params(b, g), g.d_pre_fwd, g.n_pre_fwd, 0, st); });
    run(AOA_STAGE_PRE_INV, [](BatchGroup& g) { return g.n_pre_inv > 0; },
        [&](BatchGroup& g) { return ntt_inverse_desc(launch_params(b, g), g.d_pre_inv, g.n_pre_inv, 0, st); });
    run(AOA_STAGE_AUTOMORPHISM, [](BatchGroup& g) { return g.n_auto > 0; }, [&](BatchGroup& g) {
      launch_automorphism_desc(launch_params(b, g), g.d_auto, g.n_auto, st);
      return 0;
    });
    run(AOA_STAGE_INTT, [](BatchGroup& g) { return g.n_rows > 0; }, [&](BatchGroup& g) {
      return fz_rows_desc(launch_params(b, g), g.d_items, g.d_rows, g.n_rows, g.ns_rows, g.field_q, st);
    });
    auto switches = [](BatchGroup& g) { return g.n_mul + g.n_rot > 0; };
    run(AOA_STAGE_MODUP, switches, [&](BatchGroup& g) {
      const DevParams P = launch_params(b, g);
      if (g.n_mul) fz_up_desc(P, g.d_items, g.n_mul, g.max_level, true, st);
      if (g.n_rot) fz_up_desc(P, g.d_items + g.n_mul, g.n_rot, g.max_level, false, st);
      return 0;
    });
    run(AOA_STAGE_NTT, switches, [&](BatchGroup& g) {
      return fz_key_special_desc(launch_params(b, g), g.d_items, g.d_keyb, g.n_keyb, g.field_b, st);
    });
    run(AOA_STAGE_KEY_INTT, switches, [&](BatchGroup& g) {
      return fz_key_desc(launch_params(b, g), g.d_items, g.d_keyq, g.n_keyq, g.ns_keyq, g.field_q, st);
    });
    run(AOA_STAGE_MODDOWN, switches, [&](BatchGroup& g) {
      fz_down_desc(launch_params(b, g), g.d_items, g.n_mul + g.n_rot, g.max_level, st);
      return 0;
    });
  }
  b->layers_cur = nullptr;
  if (rc) return rc;
  return check_launch("aoa_batch");
}

int batch_add_mul(aoa_batch* b, const aoa_params* p, const uint64_t* evk_b, const uint64_t* evk_a,
                  const aoa_mul_item* items, int n) {
  for (int i = 0; i < n; ++i) {
    const aoa_mul_item& it = items[i];
    if (!it.c1[0] || !it.c1[1] || !it.c2[0] || !it.c2[1] || !it.out[0] || !it.out[1])
      return set_error(AOA_ERR_ARG, "null pointer in item");
    if ((((uintptr_t)it.c1[0] | (uintptr_t)it.c1[1] | (uintptr_t)it.c2[0] | (uintptr_t)it.c2[1]) & 15) != 0)
      return set_error(AOA_ERR_ARG, "device pointers must be 16-byte aligned");
    if (it.level == 0) return set_error(AOA_ERR_LEVEL, "The ciphertext level is 0. No more rescaling is possible.");
    if (it.level < 0 || it.level >= p->host.k) return set_error(AOA_ERR_ARG, "level out of range");
  }
  BatchGroup& g = group_for(b, p, evk_b, evk_a);
  g.muls.insert(g.muls.end(), items, items + n);
  return AOA_OK;
}

int batch_add_rotate(aoa_batch* b, const aoa_params* p, const aoa_rot_item* items, int n) {
  for (int i = 0; i < n; ++i) {
    const aoa_rot_item& it = items[i];
    if (!it.in[0] || !it.in[1] || !it.out[0] || !it.out[1] || !it.rtk_b || !it.rtk_a)
      return set_error(AOA_ERR_ARG, "null pointer in item");
    if (it.level < 0 || it.level >= p->host.k || it.rot_slots < 0) return set_error(AOA_ERR_ARG, "bad item");
  }
  BatchGroup& g = group_for(b, p, nullptr, nullptr);
  g.rots.insert(g.rots.end(), items, items + n);
  return AOA_OK;
}

int batch_add_ntt(aoa_batch* b, const aoa_params* p, const aoa_ntt_item* items, int n) {
  for (int i = 0; i < n; ++i) {
    const aoa_ntt_item& it = items[i];
    if (!it.poly[0] || !it.poly[1]) return set_error(AOA_ERR_ARG, "null pointer in item");
    if (it.level < 0 || it.level >= p->host.k) return set_error(AOA_ERR_ARG, "level out of range");
    if (it.dir != AOA_FORWARD && it.dir != AOA_INVERSE) return set_error(AOA_ERR_ARG, "bad direction");
  }
  BatchGroup& g = group_for(b, p, nullptr, nullptr);
  g.ntts.insert(g.ntts.end(), items, items + n);
  return AOA_OK;
}

void batch_clear(aoa_batch* b) {
  b->layers.clear();
  b->layers.emplace_back();
}

bool batch_empty(const aoa_batch* b) {
  for (auto& L : b->layers)
    for (auto& g : L.groups)
      if (!g.muls.empty() || !g.rots.empty() || !g.ntts.empty()) return false;
  return true;
}

void batch_barrier(aoa_batch* b) {
  if (!b->layers.back().groups.empty()) b->layers.emplace_back();
}

}  // namespace aoa

// ------------------------------------------------------------------ C-ABI --

extern "C" int aoa_batch_create(aoa_batch** out) {
  if (!out) return set_error(AOA_ERR_ARG, "null output handle");
  *out = new aoa_batch();
  (*out)->layers.emplace_back();
  return AOA_OK;
}

extern "C" void aoa_batch_destroy(aoa_batch* b) {
  if (!b) return;
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->cap) (void)hipStreamDestroy(b->cap);
  if (b->dmem) (void)hipFree(b->dmem);
  if (b->ws) (void)hipFree(b->ws);
  delete b;
}

extern "C" int aoa_batch_add_mul(aoa_batch* b, const aoa_params* p, const uint64_t* evk_b, const uint64_t* evk_a,
                                 const aoa_mul_item* items, int n) {
  if (!b || !p || !evk_b || !evk_a || (!items && n > 0)) return set_error(AOA_ERR_ARG, "null argument");
  if (b->built) return set_error(AOA_ERR_ARG, "batch already built");
  return batch_add_mul(b, p, evk_b, evk_a, items, n);
}

extern "C" int aoa_batch_add_rotate(aoa_batch* b, const aoa_params* p, const aoa_rot_item* items, int n) {
  if (!b || !p || (!items && n > 0)) return set_error(AOA_ERR_ARG, "null argument");
  if (b->built) return set_error(AOA_ERR_ARG, "batch already built");
  return batch_add_rotate(b, p, items, n);
}

extern "C" int aoa_batch_add_ntt(aoa_batch* b, const aoa_params* p, const aoa_ntt_item* items, int n) {
  if (!b || !p || (!items && n > 0)) return set_error(AOA_ERR_ARG, "null argument");
  if (b->built) return set_error(AOA_ERR_ARG, "batch already built");
  return batch_add_ntt(b, p, items, n);
}

extern "C" int aoa_batch_barrier(aoa_batch* b) {
  if (!b) return set_error(AOA_ERR_ARG, "null batch");
  if (b->built) return set_error(AOA_ERR_ARG, "batch already built");
  batch_barrier(b);
  return AOA_OK;
}

extern "C" int aoa_batch_build(aoa_batch* b) {
  if (!b) return set_error(AOA_ERR_ARG, "null batch");
  if (b->built) return AOA_OK;
  if (const int rc = prepare_splits(b)) return rc;
  size_t ws = 0, desc = 0;
  batch_sizes(b, &ws, &desc);
  b->ws_bytes = ws;
  if (ws && hipMalloc(&b->ws, ws) != hipSuccess) return set_error(AOA_ERR_HIP, "hipMalloc of batch workspace failed");
  if (desc && hipMalloc(&b->dmem, desc) != hipSuccess) return set_error(AOA_ERR_HIP, "hipMalloc of descriptors failed");
  std::vector<char> host(desc);
  size_t used = batch_fill(b, (uint64_t*)b->ws, host.data(), (char*)b->dmem, desc);
  if (desc && !used) return set_error(AOA_ERR_ARG, "descriptor sizing failed");
  b->desc_bytes = used;
  if (used && hipMemcpy(b->dmem, host.data(), used, hipMemcpyHostToDevice) != hipSuccess)
    return set_error(AOA_ERR_HIP, "hipMemcpy of descriptors failed");
  b->built = true;
  return AOA_OK;
}

extern "C" size_t aoa_batch_workspace_bytes(const aoa_batch* b) { return b ? b->ws_bytes : 0; }

extern "C" void aoa_batch_default_options(aoa_batch_options* o) {
  if (o) *o = aoa_batch_options{0, 1, 0, 0};
}

extern "C" int aoa_batch_get_options(const aoa_batch* b, aoa_batch_options* o) {
  if (!b || !o) return set_error(AOA_ERR_ARG, "null argument");
  *o = b->opt;
  return AOA_OK;
}

static void drop_graph(aoa_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
}

extern "C" int aoa_batch_set_options(aoa_batch* b, const aoa_batch_options* o) {
  if (!b || !o) return set_error(AOA_ERR_ARG, "null argument");
  if (o->strict_split < -1 || o->strict_split > 1) return set_error(AOA_ERR_ARG, "strict_split must be -1, 0 or 1");
  if (o->ntt_split) {
    bool any = false;
    for (auto& L : b->layers)
      for (auto& g : L.groups) any = any || ntt_valid_split(g.params->host.N, o->ntt_split);
    if (!any) return set_error(AOA_ERR_ARG, "the NTT split fits no ring dimension of the batch");
  }
  b->opt = *o;
  b->opt.prime_major = o->prime_major ? 1 : 0;
  b->opt.xcd_chunks = o->xcd_chunks ? 1 : 0;
  if (!b->built) return AOA_OK;
  if (const int rc = prepare_splits(b)) return rc;
  // same descriptors in another order: refill the tables in place
  if (hipDeviceSynchronize() != hipSuccess) return set_error(AOA_ERR_HIP, "hipDeviceSynchronize failed");
  drop_graph(b);
  std::vector<char> host(b->desc_bytes);
  size_t used = batch_fill(b, (uint64_t*)b->ws, host.data(), (char*)b->dmem, b->desc_bytes);
  if (b->desc_bytes && used != b->desc_bytes) return set_error(AOA_ERR_ARG, "descriptor refill failed");
  if (used && hipMemcpy(b->dmem, host.data(), used, hipMemcpyHostToDevice) != hipSuccess)
    return set_error(AOA_ERR_HIP, "hipMemcpy of descriptors failed");
  return AOA_OK;
}

extern "C" int aoa_batch_launch(aoa_batch* b, void* stream, int use_graph) {
  if (!b) return set_error(AOA_ERR_ARG, "null batch");
  int rc = aoa_batch_build(b);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (!use_graph) return batch_enqueue(b, st, nullptr);
  if (!b->exec) {
    if (hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking) != hipSuccess)
      return set_error(AOA_ERR_HIP, "hipStreamCreate failed");
    if (hipStreamBeginCapture(b->cap, hipStreamCaptureModeThreadLocal) != hipSuccess)
      return set_error(AOA_ERR_HIP, "hipStreamBeginCapture failed");
    int erc = batch_enqueue(b, b->cap, nullptr);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->cap, &g);
    if (erc) {
      if (g) (void)hipGraphDestroy(g);
      return erc;
    }
    if (e != hipSuccess || !g) return set_error(AOA_ERR_HIP, "hipStreamEndCapture failed");
    b->graph = g;
    if (hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0) != hipSuccess)
      return set_error(AOA_ERR_HIP, "hipGraphInstantiate failed");
  }
  if (hipGraphLaunch(b->exec, st) != hipSuccess) return set_error(AOA_ERR_HIP, "hipGraphLaunch failed");
  return AOA_OK;
}

extern "C" int aoa_batch_stage_times(aoa_batch* b, void* stream, double* ms, int* launches, int nstages) {
  if (!b || !ms || !launches || nstages < AOA_NSTAGES) return set_error(AOA_ERR_ARG, "bad argument");
  int rc = aoa_batch_build(b);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  StageTimer tm;
  rc = batch_enqueue(b, st, &tm);
  if (!tm.ok) return set_error(AOA_ERR_HIP, "hipEventCreate failed");
  if (rc) return rc;
  if (hipStreamSynchronize(st) != hipSuccess) return set_error(AOA_ERR_HIP, "hipStreamSynchronize failed");
  for (int s = 0; s < nstages; ++s) {
    ms[s] = 0.0;
    launches[s] = 0;
  }
  for (size_t i = 0; i < tm.stage.size(); ++i) {
    float t = 0.f;
    if (hipEventElapsedTime(&t, tm.ev[2 * i], tm.ev[2 * i + 1]) != hipSuccess)
      return set_error(AOA_ERR_HIP, "hipEventElapsedTime failed");
    ms[tm.stage[i]] += t;
    launches[tm.stage[i]] += 1;
  }
  return AOA_OK;
}

// ------------------------------------------------------------ autotuner ----
// The reference fixes its NTT factorisation per ring dimension in a table
// (aoa-ntt/include/newckks/cuda/htrans/ntt.h:13-44).  Here every launch option
// of a batch is timed on the batch itself and the fastest is kept.

// Words of every output of the batch: HomMul outputs after the rescale (level
// limbs), rotation outputs (level + 1 limbs), transformed polynomials.
static void output_ranges(const aoa_batch* b, std::vector<std::pair<const uint64_t*, size_t>>* out) {
  for (auto& L : b->layers)
    for (auto& g : L.groups) {
      const size_t N = g.params->host.N;
      for (auto& it : g.muls)
        for (int y = 0; y < 2; ++y) out->push_back({it.out[y], (size_t)it.level * N});
      for (auto& it : g.rots)
        for (int y = 0; y < 2; ++y) out->push_back({it.out[y], (size_t)(it.level + 1) * N});
      for (auto& it : g.ntts)
        for (int y = 0; y < 2; ++y) out->push_back({it.poly[y], (size_t)(it.level + 1) * N});
    }
}

extern "C" int aoa_batch_autotune(aoa_batch* b, void* stream, int reps, aoa_tune_result* results, int max) {
  if (!b) return -set_error(AOA_ERR_ARG, "null batch");
  if (reps <= 0) reps = 5;
  int rc = aoa_batch_build(b);
  if (rc) return -rc;
  hipStream_t st = (hipStream_t)stream;
  // the handles' own transforms (0) and the splits valid for every ring of the batch
  std::vector<int> splits{0};
  for (int n1 : {64, 128, 256, 2048, 4096}) {
    bool ok = true, any = false;
    for (auto& L : b->layers)
      for (auto& g : L.groups) {
        ok = ok && ntt_valid_split(g.params->host.N, n1);
        any = true;
      }
    if (ok && any) splits.push_back(n1);
  }
  // a split is for the batch's own transforms: without any its candidates are the
  // first one's programs, whose results they get
  bool split_matters = false;
  for (auto& L : b->layers)
    for (auto& g : L.groups) split_matters = split_matters || !g.ntts.empty();
  std::vector<aoa_batch_options> cand;
  for (int n1 : splits)
    for (int xcd = 0; xcd < 2; ++xcd) {
      cand.push_back({n1, 0, xcd, -1});  // item order: no strict split
      for (int ss = -1; ss <= 1; ++ss) cand.push_back({n1, 1, xcd, ss});
    }
  std::vector<std::pair<const uint64_t*, size_t>> outs;
  output_ranges(b, &outs);
  uint64_t* acc = nullptr;
  if (hipMalloc(&acc, sizeof(uint64_t)) != hipSuccess) return -set_error(AOA_ERR_HIP, "hipMalloc failed");
  hipEvent_t e0 = nullptr, e1 = nullptr;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  const aoa_batch_options saved = b->opt;
  auto checksum = [&](uint64_t* v) -> int {
    if (hipMemsetAsync(acc, 0, sizeof(uint64_t), st) != hipSuccess) return set_error(AOA_ERR_HIP, "hipMemsetAsync failed");
    uint64_t off = 0;
    for (auto& r : outs) {
      launch_checksum(r.first, r.second, off, acc, st);
      off += r.second;
    }
    if (hipMemcpyAsync(v, acc, sizeof(uint64_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return set_error(AOA_ERR_HIP, "checksum copy failed");
    return check_launch("aoa_batch_autotune");
  };
  int best = -1, count = 0;
  double best_ms = 1e30;
  uint64_t base_sum = 0;
  bool reproducible = true;
  const size_t distinct = split_matters ? cand.size() : cand.size() / splits.size();
  std::vector<aoa_tune_result> found;
  for (size_t c = 0; c < cand.size() && !rc; ++c) {
    if (c >= distinct) {
      aoa_tune_result r = found[c % distinct];
      r.opt = cand[c];
      if (count < max && results) results[count] = r;
      ++count;
      continue;
    }
    rc = aoa_batch_set_options(b, &cand[c]);
    if (rc) break;
    rc = aoa_batch_launch(b, st, 1);  // warm-up (captures the graph)
    if (rc) break;
    if (hipStreamSynchronize(st) != hipSuccess) {
      rc = set_error(AOA_ERR_HIP, "hipStreamSynchronize failed");
      break;
    }
    (void)hipEventRecord(e0, st);
    for (int r = 0; r < reps && !rc; ++r) rc = aoa_batch_launch(b, st, 1);
    (void)hipEventRecord(e1, st);
    if (rc || hipEventSynchronize(e1) != hipSuccess) {
      if (!rc) rc = set_error(AOA_ERR_HIP, "hipEventSynchronize failed");
      break;
    }
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    uint64_t sum = 0;
    if ((rc = checksum(&sum))) break;
    if (c == 0) {
      // outputs that are a function of unchanged inputs repeat exactly
      base_sum = sum;
      if ((rc = aoa_batch_launch(b, st, 1))) break;
      uint64_t again = 0;
      if ((rc = checksum(&again))) break;
      reproducible = again == base_sum;
    }
    const bool exact = reproducible && sum == base_sum;
    const double t = ms / reps;
    found.push_back(aoa_tune_result{cand[c], t, sum, exact ? 1 : 0});
    if (count < max && results) results[count] = found.back();
    ++count;
    if ((exact || !reproducible) && t < best_ms) {
      best_ms = t;
      best = (int)c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(acc);
  if (rc) {
    (void)aoa_batch_set_options(b, &saved);
    return -rc;
  }
  rc = aoa_batch_set_options(b, best >= 0 ? &cand[best] : &saved);
  return rc ? -rc : count;
}
