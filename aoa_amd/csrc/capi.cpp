// C-ABI entry points (include/aoa.h): argument checks, workspace carving and
// the kernel sequences of the plain (one ciphertext per call) form.
#include <algorithm>
#include <cstring>
#include <exception>
#include <memory>
#include <string>

#include "internal.hpp"

using namespace aoa;

static thread_local std::string g_err;

namespace aoa {

int set_error(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(AOA_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return AOA_OK;
}

uint64_t galois_of(int rot_slots, int N) {
  const uint64_t M = 2 * (uint64_t)N;
  uint64_t r = 1, s = 5 % M, e = (uint64_t)rot_slots;
  while (e) {
    if (e & 1) r = (r * s) % M;
    s = (s * s) % M;
    e >>= 1;
  }
  return r;
}

}  // namespace aoa

// Ciphertext and workspace pointers are moved as 16-byte vectors.
static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

static int fail(int code, const std::string& msg) { return set_error(code, msg); }

extern "C" const char* aoa_last_error(void) { return g_err.c_str(); }

namespace {

// A table on its way to the device: *at becomes its address.
struct Section {
  const void* src;
  size_t bytes;
  const void** at;
};
template <class T, class D>
Section section(const std::vector<T>& v, const D** at) {
  return Section{v.data(), v.size() * sizeof(T), (const void**)at};
}

// One allocation of 256-byte aligned sections.  Those below 1 MiB go up in one
// copy: a copy takes 8 us or more, and small rings have some thirty.
int upload(std::vector<Section>& secs, void** mem) {
  std::stable_partition(secs.begin(), secs.end(), [](const Section& s) { return s.bytes < ((size_t)1 << 20); });
  size_t total = 0, small = 0;
  std::vector<size_t> off;
  for (const Section& s : secs) {
    off.push_back(total);
    total += (s.bytes + 255) & ~(size_t)255;
    if (s.bytes < ((size_t)1 << 20)) small = total;
  }
  std::vector<char> stage(small);
  if (hipMalloc(mem, total) != hipSuccess) return fail(AOA_ERR_HIP, "hipMalloc of parameter tables failed");
  char* b = (char*)*mem;
  bool ok = true;
  for (size_t i = 0; i < secs.size(); ++i) {
    if (off[i] < small)
      std::memcpy(&stage[off[i]], secs[i].src, secs[i].bytes);
    else
      ok = ok && hipMemcpy(b + off[i], secs[i].src, secs[i].bytes, hipMemcpyHostToDevice) == hipSuccess;
    *secs[i].at = b + off[i];
  }
  ok = ok && (!small || hipMemcpy(b, stage.data(), small, hipMemcpyHostToDevice) == hipSuccess);
  return ok ? AOA_OK : fail(AOA_ERR_HIP, "hipMemcpy of parameter tables failed");
}

int create_params(int N, int k, int kl, int prec, aoa_params** out) {
  std::unique_ptr<aoa_params, decltype(&aoa_params_destroy)> h(new aoa_params(), aoa_params_destroy);
  std::string err = build_host_params(N, k, kl, prec, &h->host);
  if (!err.empty()) return fail(AOA_ERR_UNSUPPORTED, err);
  const HostParams& H = h->host;
  FusedTables F;
  build_fused_tables(H, &F);
  if (hipGetDevice(&h->device) != hipSuccess) return fail(AOA_ERR_HIP, "no current device");
  DevParams& D = h->dev;
  FusedDev& Z = D.fz;
  std::vector<Section> secs = {
      section(H.dprimes, &D.primes),
      section(H.inv_qhat, &D.inv_qhat),
      section(H.qhat_mod_b, &D.qhat_mod_b),
      section(H.inv_bhat, &D.inv_bhat),
      section(H.bhat_mod_q, &D.bhat_mod_q),
      section(H.inv_b_mod_q, &D.inv_b_mod_q),
      section(H.b_mod_q, &D.b_mod_q),
      section(H.inv_ql_mod_qi, &D.inv_ql_mod_qi),
      section(H.enc_t[0], &D.enc_t[0]),
      section(H.enc_t[1], &D.enc_t[1]),
      section(H.gauss_cdt, &D.gauss_cdt),
      section(H.md_terms, &D.md_terms),
      section(H.md_thr, &D.md_thr),
      section(H.md_red, &D.md_red),
      section(H.md_fin, &D.md_fin),
      section(H.mu_terms, &D.mu_terms),
      section(F.tw[0], &Z.tw[0]),
      section(F.tw[1], &Z.tw[1]),
      section(F.lc, &Z.lc),
      section(F.lc_b, &Z.lc_b),
      section(F.lc_up, &Z.lc_up),
      section(F.lc_down, &Z.lc_down),
      section(F.bq, &Z.bq),
      section(F.mu_w, &Z.mu_w),
      section(F.md_w, &Z.md_w),
      section(F.mu_out, &Z.mu_out),
      section(F.md_out, &Z.md_out),
      section(F.scr, &Z.scr),
      section(F.scr_thr, &Z.scr_thr),
  };
  const int rc = upload(secs, &h->dmem);
  if (rc) return rc;
  D.N = H.N;
  D.logN = H.logN;
  D.k = H.k;
  D.K = H.K;
  Z.mu_stride = F.mu_stride;
  Z.md_stride = F.md_stride;
  Z.mu_kb = F.mu_kb;
  Z.md_kb = F.md_kb;
  *out = h.release();
  return AOA_OK;
}

}  // namespace

int aoa::use_split(const aoa_params* h, int n1, DevParams* P) try {
  if (n1) {
    std::lock_guard<std::mutex> lock(h->split_mu);
    if (!h->split_mem) {
      const HostParams& H = h->host;
      std::vector<uint64_t> row[3][2];
      parallel_for(6, (size_t)(H.k + H.K) * H.N, [&](int t) {
        row_twiddle_order(t & 1 ? H.tw_inv : H.tw_fwd, H.N, H.k + H.K, 64 << (t >> 1), &row[t >> 1][t & 1]);
      });
      SplitTables t{};
      std::vector<Section> secs = {section(H.tw_fwd, &t.tw_fwd), section(H.tw_inv, &t.tw_inv)};
      for (int i = 0; i < 6; ++i)
        if (!row[i >> 1][i & 1].empty()) secs.push_back(section(row[i >> 1][i & 1], &t.tw_row[i >> 1][i & 1]));
      int prev = 0;
      void* mem = nullptr;
      if (hipGetDevice(&prev) != hipSuccess || hipSetDevice(h->device) != hipSuccess)
        return fail(AOA_ERR_HIP, "the parameter set's device is not usable");
      const int rc = upload(secs, &mem);
      (void)hipSetDevice(prev);
      if (rc) {
        if (mem) (void)hipFree(mem);
        return rc;
      }
      h->split_tables = t;
      h->split_mem = mem;
    }
    P->split = h->split_tables;
  }
  P->ntt_n1 = n1;
  return AOA_OK;
} catch (const std::exception&) {
  return fail(AOA_ERR_HIP, "no memory for a split's tables");
}

extern "C" int aoa_params_create(int N, int k, int kl, int prec, aoa_params** out) {
  if (!out) return fail(AOA_ERR_ARG, "null output handle");
  *out = nullptr;
  try {
    return create_params(N, k, kl, prec, out);
  } catch (const std::exception&) {
    return fail(AOA_ERR_HIP, "no memory for the parameter tables");
  }
}

extern "C" void aoa_params_destroy(aoa_params* h) {
  if (!h) return;
  if (h->dmem) (void)hipFree(h->dmem);
  if (h->split_mem) (void)hipFree(h->split_mem);
  delete h;
}

extern "C" int aoa_params_info(const aoa_params* h, int* N, int* k, int* kl, int* prec) {
  if (!h) return fail(AOA_ERR_ARG, "null params");
  if (N) *N = h->host.N;
  if (k) *k = h->host.k;
  if (kl) *kl = h->host.K;
  if (prec) *prec = h->host.prec;
  return AOA_OK;
}

extern "C" int aoa_params_primes(const aoa_params* h, uint64_t* out, int n) {
  if (!h || !out) return fail(AOA_ERR_ARG, "null argument");
  int R = (int)h->host.primes.size();
  if (n < R) return fail(AOA_ERR_ARG, "output too small");
  std::memcpy(out, h->host.primes.data(), R * sizeof(uint64_t));
  return AOA_OK;
}

extern "C" int64_t aoa_params_table(const aoa_params* h, int which, uint64_t* out, int64_t n) {
  if (!h) return -fail(AOA_ERR_ARG, "null params");
  const HostParams& H = h->host;
  const int R = H.k + H.K;
  std::vector<uint64_t> v;
  auto take = [&](const std::vector<uint64_t>& src, int stride) {
    for (size_t i = 0; i < src.size(); i += stride) v.push_back(src[i]);
  };
  switch (which) {
    case 0: take(H.tw_fwd, 2); break;
    case 1: take(H.tw_inv, 2); break;
    case 2: take(H.inv_qhat, 2); break;
    case 3: take(H.qhat_mod_b, 1); break;
    case 4: take(H.inv_bhat, 2); break;
    case 5: take(H.bhat_mod_q, 2); break;
    case 6: take(H.inv_b_mod_q, 2); break;
    case 7: take(H.b_mod_q, 2); break;
    case 8: take(H.inv_ql_mod_qi, 2); break;
    case 9:
      for (int r = 0; r < R; ++r) v.push_back(H.dprimes[r].mu);
      break;
    case 11:
      v.resize(H.enc_w.size());
      std::memcpy(v.data(), H.enc_w.data(), v.size() * 8);
      break;
    case 12:
      for (uint32_t g : H.rot_group) v.push_back(g);
      break;
    case 13: v = H.gauss_cdt; break;
    case 15: take(H.bscale, 2); break;
    case 14:  // ModDown constants, eight 32-bit words per (i, j) widened to 64 bits
      for (const MdConst& m : H.md_const)
        for (uint32_t x : {m.cl, m.ch, m.cs, m.w0, m.w1, m.w2, m.thr, m.pad}) v.push_back(x);
      break;
    default: return -fail(AOA_ERR_ARG, "unknown table");
  }
  if (!out) return (int64_t)v.size();
  if (n < (int64_t)v.size()) return -fail(AOA_ERR_ARG, "output too small");
  std::memcpy(out, v.data(), v.size() * 8);
  return (int64_t)v.size();
}

static LimbMap limbs_of(uint64_t* base, int res0, int nres, int k) {
  LimbMap m;
  std::memset(&m, 0, sizeof(m));
  m.base[0] = base + 0;
  m.nlimbs = nres;
  m.npolys = 1;
  if (res0 < k) {
    m.prime0 = res0;
    m.qlimbs = std::min(nres, k - res0);
  } else {
    // only special limbs: prime = k + li - qlimbs with qlimbs = k - res0 <= 0
    m.prime0 = 0;
    m.qlimbs = k - res0;
  }
  return m;
}

extern "C" int aoa_ntt(const aoa_params* h, void* stream, uint64_t* d, int res0, int nres, int dir) {
  if (!h || !d) return fail(AOA_ERR_ARG, "null argument");
  const int R = h->host.k + h->host.K;
  if (res0 < 0 || nres <= 0 || res0 + nres > R) return fail(AOA_ERR_ARG, "limb range out of bounds");
  LimbMap m = limbs_of(d + (size_t)res0 * h->host.N, res0, nres, h->host.k);
  hipStream_t st = (hipStream_t)stream;
  int rc = dir == AOA_FORWARD ? ntt_forward(h->dev, m, 0, st) : ntt_inverse(h->dev, m, 0, st);
  if (rc) return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
  return check_launch("aoa_ntt");
}

extern "C" int aoa_eltwise(const aoa_params* h, void* stream, int op, uint64_t* out, const uint64_t* a,
                           const uint64_t* b, const uint64_t* c, int res0, int nres) {
  if (!h || !out || !a) return fail(AOA_ERR_ARG, "null argument");
  if (op != AOA_ADD && op != AOA_SUB && op != AOA_MUL && op != AOA_NEGATE && op != AOA_MULADD)
    return fail(AOA_ERR_ARG, "unknown operation");
  if (op != AOA_NEGATE && !b) return fail(AOA_ERR_ARG, "null operand b");
  if (op == AOA_MULADD && !c) return fail(AOA_ERR_ARG, "null addend c");
  const int R = h->host.k + h->host.K, k = h->host.k;
  if (res0 < 0 || nres <= 0 || res0 + nres > R) return fail(AOA_ERR_ARG, "limb range out of bounds");
  const size_t off = (size_t)res0 * h->host.N;
  int qlimbs = res0 < k ? std::min(nres, k - res0) : k - res0;
  launch_eltwise(h->dev, op, out + off, a + off, b ? b + off : nullptr, c ? c + off : nullptr, nres, qlimbs,
                 res0 < k ? res0 : 0, (hipStream_t)stream);
  return check_launch("aoa_eltwise");
}

extern "C" int aoa_eltwise_scalar(const aoa_params* h, void* stream, int op, uint64_t* out, const uint64_t* a,
                                  uint64_t b, int res0, int nres) {
  if (!h || !out || !a) return fail(AOA_ERR_ARG, "null argument");
  if (op != AOA_ADD && op != AOA_SUB && op != AOA_MUL) return fail(AOA_ERR_ARG, "unknown operation");
  const int R = h->host.k + h->host.K;
  if (res0 < 0 || nres <= 0 || res0 + nres > R) return fail(AOA_ERR_ARG, "limb range out of bounds");
  const size_t off = (size_t)res0 * h->host.N;
  launch_eltwise_scalar(h->dev, op, out + off, a + off, b, nres, res0, (hipStream_t)stream);
  return check_launch("aoa_eltwise_scalar");
}

extern "C" int aoa_conjugate(const aoa_params* h, void* stream, uint64_t* out, const uint64_t* in, int nres) {
  if (!h || !out || !in) return fail(AOA_ERR_ARG, "null argument");
  if (out == in) return fail(AOA_ERR_ARG, "out and in must not overlap");
  if (nres <= 0 || nres > h->host.k + h->host.K) return fail(AOA_ERR_ARG, "limb count out of range");
  launch_conjugate(h->dev, out, in, nres, (hipStream_t)stream);
  return check_launch("aoa_conjugate");
}

static bool slots_ok(const aoa_params* h, int n) { return n >= 1 && n <= h->host.N / 2 && !(n & (n - 1)); }

extern "C" int aoa_special_fft(const aoa_params* h, void* stream, double* vals, int n, int dir) {
  if (!h || !vals) return fail(AOA_ERR_ARG, "null argument");
  if (!slots_ok(h, n)) return fail(AOA_ERR_ARG, "size must be a power of two <= N/2");
  if (dir != AOA_FORWARD && dir != AOA_INVERSE) return fail(AOA_ERR_ARG, "unknown direction");
  if (!aligned16(vals)) return fail(AOA_ERR_ARG, "values must be 16-byte aligned");
  launch_special_fft(h->dev, vals, n, dir == AOA_INVERSE, (hipStream_t)stream);
  return check_launch("aoa_special_fft");
}

extern "C" int aoa_encode(const aoa_params* h, void* stream, uint64_t* out, double* vals, int slots, uint64_t scale,
                          int nres) {
  if (!h || !out || !vals) return fail(AOA_ERR_ARG, "null argument");
  if (!slots_ok(h, slots)) return fail(AOA_ERR_ARG, "slots must be a power of two <= N/2");
  if (scale == 0) return fail(AOA_ERR_ARG, "scale must be positive");
  if (nres <= 0 || nres > h->host.k) return fail(AOA_ERR_ARG, "limb count out of range");
  if (!aligned16(vals)) return fail(AOA_ERR_ARG, "values must be 16-byte aligned");
  launch_encode(h->dev, out, vals, slots, (double)scale, nres, (hipStream_t)stream);
  return check_launch("aoa_encode");
}

extern "C" int aoa_decode(const aoa_params* h, void* stream, double* vals, const uint64_t* in, int slots,
                          uint64_t scale) {
  if (!h || !vals || !in) return fail(AOA_ERR_ARG, "null argument");
  if (!slots_ok(h, slots)) return fail(AOA_ERR_ARG, "slots must be a power of two <= N/2");
  if (scale == 0) return fail(AOA_ERR_ARG, "scale must be positive");
  if (!aligned16(vals)) return fail(AOA_ERR_ARG, "values must be 16-byte aligned");
  launch_decode(h->dev, vals, in, slots, (double)scale, (hipStream_t)stream);
  return check_launch("aoa_decode");
}

extern "C" int aoa_sample(const aoa_params* h, void* stream, uint64_t* out, int res0, int nres, int kind,
                          uint64_t seed, uint64_t nonce) {
  if (!h || !out) return fail(AOA_ERR_ARG, "null argument");
  if (kind < AOA_SAMPLE_UNIFORM || kind > AOA_SAMPLE_NARROW) return fail(AOA_ERR_ARG, "unknown distribution");
  const int R = h->host.k + h->host.K;
  if (res0 < 0 || nres <= 0 || res0 + nres > R) return fail(AOA_ERR_ARG, "limb range out of bounds");
  launch_sample(h->dev, out, res0, nres, kind, seed, nonce, (hipStream_t)stream);
  return check_launch("aoa_sample");
}

extern "C" int aoa_encrypt(const aoa_params* h, void* stream, uint64_t* c0, uint64_t* c1, uint64_t* m,
                           const uint64_t* pk_b, const uint64_t* pk_a, uint64_t seed, uint64_t nonce, void* ws,
                           size_t ws_bytes) {
  if (!h || !c0 || !c1 || !m || !pk_b || !pk_a || !ws) return fail(AOA_ERR_ARG, "null argument");
  const int k = h->host.k;
  const size_t N = (size_t)h->host.N;
  if (ws_bytes < 3 * (size_t)k * N * sizeof(uint64_t)) return fail(AOA_ERR_WORKSPACE, "workspace too small");
  const DevParams& P = h->dev;
  hipStream_t st = (hipStream_t)stream;
  uint64_t* u = (uint64_t*)ws;
  uint64_t* e0 = u + (size_t)k * N;
  uint64_t* e1 = e0 + (size_t)k * N;
  // The fused rows write c0, c1 and m from workgroups of their own, so these
  // must not overlap each other or what they are formed from.
  const size_t kN = (size_t)k * N;
  auto apart = [&](const uint64_t* a, const uint64_t* b, size_t n) { return a + kN <= b || b + n <= a; };
  const bool fused = nt_default(P) && apart(c0, c1, kN) && apart(c0, m, kN) && apart(c1, m, kN) && apart(c0, u, 3 * kN) &&
                     apart(c1, u, 3 * kN) && apart(m, u, 3 * kN) && apart(c0, pk_b, kN) && apart(c0, pk_a, kN) &&
                     apart(c1, pk_b, kN) && apart(c1, pk_a, kN) && apart(m, pk_b, kN) && apart(m, pk_a, kN);
  launch_sample_encrypt(P, u, e0, e1, fused ? m : nullptr, k, seed, nonce, st);
  LimbMap mm;
  std::memset(&mm, 0, sizeof(mm));
  mm.base[0] = m;
  mm.base[1] = u;
  mm.base[2] = e0;
  mm.base[3] = e1;
  mm.nlimbs = k;
  mm.qlimbs = k;
  mm.npolys = 4;
  if (fused) {
    for (int y = 0; y < 4; ++y) mm.src[y] = mm.base[y];
    nt_forward_cols(P, mm, st);
    if (nt_encrypt_rows(P, NtEncrypt{u, e0, e1, pk_b, pk_a, m, c0, c1}, k, st))
      return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
    return check_launch("aoa_encrypt");
  }
  if (ntt_forward(P, mm, 0, st)) return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
  launch_encrypt_combine(P, c0, c1, pk_b, pk_a, u, e0, e1, m, k, st);
  return check_launch("aoa_encrypt");
}

extern "C" int aoa_decrypt(const aoa_params* h, void* stream, uint64_t* m, uint64_t* c0, uint64_t* c1,
                           const uint64_t* s, int level) {
  if (!h || !m || !c0 || !c1 || !s) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  const DevParams& P = h->dev;
  hipStream_t st = (hipStream_t)stream;
  const int L = level + 1;
  // The fused rows read s while other workgroups transform c0 and c1, so it must
  // not overlap them.
  const size_t LN = (size_t)L * P.N;
  auto apart = [&](const uint64_t* c) { return s + LN <= c || c + LN <= s; };
  if (nt_default(P) && apart(c0) && apart(c1)) {
    if (nt_decrypt(P, m, c0, c1, s, L, st)) return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
    return check_launch("aoa_decrypt");
  }
  LimbMap mc;
  std::memset(&mc, 0, sizeof(mc));
  mc.base[0] = c0;
  mc.base[1] = c1;
  mc.nlimbs = L;
  mc.qlimbs = L;
  mc.npolys = 2;
  if (ntt_forward(P, mc, 0, st)) return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
  launch_eltwise(P, ELT_MULADD, m, c1, s, c0, L, L, 0, st);
  LimbMap mo = limbs_of(m, 0, L, h->host.k);
  if (ntt_inverse(P, mo, 0, st)) return fail(AOA_ERR_UNSUPPORTED, "no NTT split for this N");
  return check_launch("aoa_decrypt");
}

extern "C" int aoa_rescale(const aoa_params* h, void* stream, uint64_t* c0, uint64_t* c1, int level) {
  if (!h || !c0 || !c1) return fail(AOA_ERR_ARG, "null argument");
  if (level == 0) return fail(AOA_ERR_LEVEL, "The ciphertext level is 0. No more rescaling is possible.");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  launch_rescale(h->dev, c0, c1, level, (hipStream_t)stream);
  return check_launch("aoa_rescale");
}

extern "C" int aoa_modup(const aoa_params* h, void* stream, uint64_t* d_qb, int level) {
  if (!h || !d_qb) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  launch_modup(h->dev, d_qb, d_qb + (size_t)h->host.k * h->host.N, level, (hipStream_t)stream);
  return check_launch("aoa_modup");
}

extern "C" int aoa_modup_from(const aoa_params* h, void* stream, uint64_t* d_qb, const uint64_t* d_q, int level) {
  if (!h || !d_qb || !d_q) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  const size_t N = (size_t)h->host.N, k = (size_t)h->host.k;
  // the special limbs written must not overlap the Q limbs read (unless they
  // are the same QB polynomial)
  const uint64_t* w0 = d_qb + k * N;
  const uint64_t* w1 = w0 + (size_t)h->host.K * N;
  const uint64_t* r1 = d_q + (size_t)(level + 1) * N;
  if (d_q != d_qb && r1 > w0 && d_q < w1) return fail(AOA_ERR_ARG, "input overlaps the special limbs written");
  launch_modup(h->dev, d_q, d_qb + k * N, level, (hipStream_t)stream);
  return check_launch("aoa_modup_from");
}

extern "C" int aoa_dot(const aoa_params* h, void* stream, uint64_t* c, const uint64_t* const* a,
                       const uint64_t* const* b, int k) {
  if (!h || !c || !a || !b) return fail(AOA_ERR_ARG, "null argument");
  if (k < 0 || k > 1 << 20) return fail(AOA_ERR_ARG, "term count out of range");
  launch_dot(h->dev, c, a, b, k, (hipStream_t)stream);
  return check_launch("aoa_dot");
}

extern "C" int aoa_dr2(const aoa_params* h, void* stream, uint64_t* c21, uint64_t* c22, uint64_t* c23,
                       const uint64_t* a01, const uint64_t* a02, const uint64_t* a11, const uint64_t* a12) {
  if (!h || !c21 || !c22 || !c23 || !a01 || !a02 || !a11 || !a12) return fail(AOA_ERR_ARG, "null argument");
  launch_dr2(h->dev, c21, c22, c23, a01, a02, a11, a12, (hipStream_t)stream);
  return check_launch("aoa_dr2");
}

extern "C" int aoa_rns_primes(int k, int kl, int prec, uint64_t* out, int n) {
  if (kl <= 0) kl = k + 1;
  std::vector<uint64_t> pr;
  const std::string err = select_rns_primes(k, kl, prec, &pr);
  if (!err.empty()) return fail(AOA_ERR_UNSUPPORTED, err);
  if (!out) return fail(AOA_ERR_ARG, "null output");
  if (n < (int)pr.size()) return fail(AOA_ERR_ARG, "output too small");
  std::memcpy(out, pr.data(), pr.size() * sizeof(uint64_t));
  return AOA_OK;
}

extern "C" int aoa_moddown(const aoa_params* h, void* stream, uint64_t* d_q_out, const uint64_t* d_qb_in,
                           int level) {
  if (!h || !d_q_out || !d_qb_in) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  launch_moddown(h->dev, d_qb_in, d_qb_in + (size_t)h->host.k * h->host.N, d_q_out, level, (hipStream_t)stream);
  return check_launch("aoa_moddown");
}

extern "C" int aoa_automorphism(const aoa_params* h, void* stream, uint64_t* out, const uint64_t* in, int nres,
                                int rot_slots) {
  if (!h || !out || !in) return fail(AOA_ERR_ARG, "null argument");
  if (nres <= 0 || nres > h->host.k + h->host.K) return fail(AOA_ERR_ARG, "limb count out of range");
  if (rot_slots < 0) return fail(AOA_ERR_ARG, "negative rotation");
  launch_automorphism(h->dev, out, in, nres, galois_of(rot_slots, h->host.N), (hipStream_t)stream);
  return check_launch("aoa_automorphism");
}

extern "C" size_t aoa_workspace_bytes(const aoa_params* h, int level) {
  if (!h || level < 0 || level >= h->host.k) return 0;
  const size_t L = (size_t)level + 1, K = (size_t)h->host.K;
  return (6 * L + 3 * K) * (size_t)h->host.N * sizeof(uint64_t);
}

// Key switch of d (coefficient domain, L limbs) into (out0 [+ add0], out1).
// Workspace: X (L+K limbs), P0, P1 (L+K limbs each).
static int keyswitch_core(const aoa_params* h, hipStream_t st, uint64_t* out0, uint64_t* out1,
                          const uint64_t* add0, const uint64_t* d, const uint64_t* kb, const uint64_t* ka,
                          int level, uint64_t* ws) {
  const size_t N = (size_t)h->dev.N;
  const int L = level + 1, K = h->dev.K;
  FzItem it{};
  it.d = d;
  it.kb = kb;
  it.ka = ka;
  it.XQ = ws;
  it.X = ws + (size_t)L * N;
  it.P0 = it.XQ + (size_t)(L + K) * N;
  it.P1 = it.P0 + (size_t)(L + K) * N;
  it.add0 = add0;
  it.out0 = out0;
  it.out1 = out1;
  it.level = level;
  return fz_switch(h->dev, it, st) ? fail(AOA_ERR_UNSUPPORTED, "no NTT split") : AOA_OK;
}

extern "C" int aoa_keyswitch(const aoa_params* h, void* stream, uint64_t* out0, uint64_t* out1,
                             const uint64_t* add0, const uint64_t* d_in, const uint64_t* key_b,
                             const uint64_t* key_a, int level, void* ws, size_t ws_bytes) {
  if (!h || !out0 || !out1 || !d_in || !key_b || !key_a || !ws) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  if (ws_bytes < aoa_workspace_bytes(h, level)) return fail(AOA_ERR_WORKSPACE, "workspace too small");
  int rc = keyswitch_core(h, (hipStream_t)stream, out0, out1, add0, d_in, key_b, key_a, level, (uint64_t*)ws);
  if (rc) return rc;
  return check_launch("aoa_keyswitch");
}

int aoa::hommul_core(const aoa_params* h, void* stream, uint64_t* c3_0, uint64_t* c3_1, const uint64_t* a0,
                     const uint64_t* a1, const uint64_t* b0, const uint64_t* b1, const uint64_t* evk_b,
                     const uint64_t* evk_a, int level, void* ws, size_t ws_bytes, int rescale) {
  if (!h || !c3_0 || !c3_1 || !a0 || !a1 || !b0 || !b1 || !evk_b || !evk_a || !ws)
    return fail(AOA_ERR_ARG, "null argument");
  if (!aligned16(c3_0) || !aligned16(c3_1) || !aligned16(a0) || !aligned16(a1) || !aligned16(b0) ||
      !aligned16(b1) || !aligned16(ws))
    return fail(AOA_ERR_ARG, "device pointers must be 16-byte aligned");
  if (level == 0) return fail(AOA_ERR_LEVEL, "The ciphertext level is 0. No more rescaling is possible.");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  if (ws_bytes < aoa_workspace_bytes(h, level)) return fail(AOA_ERR_WORKSPACE, "workspace too small");
  const DevParams& P = h->dev;
  const size_t N = (size_t)P.N;
  const int L = level + 1, K = P.K;
  // d2 after its inverse rows (L limbs), the special limbs (K), the key products (L + K each)
  FzItem it{};
  it.a0 = a0;
  it.a1 = a1;
  it.b0 = b0;
  it.b1 = b1;
  it.kb = evk_b;
  it.ka = evk_a;
  it.D = (uint64_t*)ws;
  it.X = it.D + (size_t)L * N;
  it.P0 = it.X + (size_t)K * N;
  it.P1 = it.P0 + (size_t)(L + K) * N;
  it.out0 = c3_0;
  it.out1 = c3_1;
  it.level = level;
  it.rescale = rescale;
  if (fz_mul(P, it, (hipStream_t)stream)) return fail(AOA_ERR_UNSUPPORTED, "no NTT split");
  return check_launch(rescale ? "aoa_hommul_relin_rescale" : "aoa_hommul_relin");
}

extern "C" int aoa_hommul_relin_rescale(const aoa_params* h, void* stream, uint64_t* c3_0, uint64_t* c3_1,
                                        const uint64_t* a0, const uint64_t* a1, const uint64_t* b0,
                                        const uint64_t* b1, const uint64_t* evk_b, const uint64_t* evk_a,
                                        int level, void* ws, size_t ws_bytes) {
  return aoa::hommul_core(h, stream, c3_0, c3_1, a0, a1, b0, b1, evk_b, evk_a, level, ws, ws_bytes, 1);
}

extern "C" int aoa_hommul_relin(const aoa_params* h, void* stream, uint64_t* c3_0, uint64_t* c3_1,
                                const uint64_t* a0, const uint64_t* a1, const uint64_t* b0, const uint64_t* b1,
                                const uint64_t* evk_b, const uint64_t* evk_a, int level, void* ws,
                                size_t ws_bytes) {
  return aoa::hommul_core(h, stream, c3_0, c3_1, a0, a1, b0, b1, evk_b, evk_a, level, ws, ws_bytes, 0);
}

// rho (aoa-ntt/src/cuda/manager.cu:149-176): Q limbs times B mod q_i, special
// limbs zero.  Any domain (the factor is a scalar per limb).
extern "C" int aoa_rho(const aoa_params* h, void* stream, uint64_t* out, const uint64_t* in) {
  if (!h || !out || !in) return fail(AOA_ERR_ARG, "null argument");
  launch_rho(h->dev, out, in, (hipStream_t)stream);
  return check_launch("aoa_rho");
}

extern "C" int aoa_rotate_left(const aoa_params* h, void* stream, uint64_t* out0, uint64_t* out1,
                               const uint64_t* c0, const uint64_t* c1, const uint64_t* rtk_b,
                               const uint64_t* rtk_a, int rot_slots, int level, void* ws, size_t ws_bytes) {
  if (!h || !out0 || !out1 || !c0 || !c1 || !rtk_b || !rtk_a || !ws) return fail(AOA_ERR_ARG, "null argument");
  if (level < 0 || level >= h->host.k) return fail(AOA_ERR_ARG, "level out of range");
  if (rot_slots < 0) return fail(AOA_ERR_ARG, "negative rotation");
  if (ws_bytes < aoa_workspace_bytes(h, level)) return fail(AOA_ERR_WORKSPACE, "workspace too small");
  const DevParams& P = h->dev;
  hipStream_t st = (hipStream_t)stream;
  const size_t N = (size_t)P.N;
  const int L = level + 1, K = P.K;
  uint64_t* R0 = (uint64_t*)ws;
  uint64_t* R1 = R0 + (size_t)L * N;
  uint64_t* kws = R1 + (size_t)L * N;  // 3(L+K) limbs
  (void)K;
  const uint64_t g = galois_of(rot_slots, P.N);
  launch_automorphism2(P, R0, R1, c0, c1, L, g, st);
  int rc = keyswitch_core(h, st, out0, out1, R0, R1, rtk_b, rtk_a, level, kws);
  if (rc) return rc;
  return check_launch("aoa_rotate_left");
}

// ckks_rotate_right (aoa-ntt/src/ckks/ckks.cpp:953-980): rotate_slots_right is
// rotate_slots_left by N/2 - rotSlots (aoa-ntt/src/ckks/encoder.cu:356-363);
// the key switch is the same, with the right rotation key.
extern "C" int aoa_rotate_right(const aoa_params* h, void* stream, uint64_t* out0, uint64_t* out1,
                                const uint64_t* c0, const uint64_t* c1, const uint64_t* rtk_b,
                                const uint64_t* rtk_a, int rot_slots, int level, void* ws, size_t ws_bytes) {
  if (!h) return fail(AOA_ERR_ARG, "null argument");
  if (rot_slots < 0 || rot_slots > h->host.N / 2) return fail(AOA_ERR_ARG, "rotation out of range [0, N/2]");
  return aoa_rotate_left(h, stream, out0, out1, c0, c1, rtk_b, rtk_a, h->host.N / 2 - rot_slots, level, ws,
                         ws_bytes);
}
