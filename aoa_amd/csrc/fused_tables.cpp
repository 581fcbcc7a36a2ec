// Host tables of the fused kernels (fused.hpp).
#include <cmath>
#include <cstring>

#include "params.hpp"

namespace aoa {

typedef unsigned __int128 u128;

static uint64_t mulm(uint64_t a, uint64_t b, uint64_t p) { return (uint64_t)((u128)a * b % p); }

// c mod p as a double in (-p/2, p/2].
static uint64_t balanced(uint64_t c, uint64_t p) {
  const double d = c > p / 2 ? -(double)(p - c) : (double)c;
  uint64_t b;
  std::memcpy(&b, &d, 8);
  return b;
}

// One last-stage entry: the constants n0 and n1 in the prime's form.
static void put_lc(uint64_t* e, uint64_t n0, uint64_t n1, uint64_t p, uint32_t field) {
  if (field == FIELD_FP64) {
    e[0] = balanced(n0, p);
    e[1] = balanced(n1, p);
    e[2] = e[3] = 0;
  } else {
    e[0] = n0;
    e[1] = shoup_quot(n0, p);
    e[2] = n1;
    e[3] = shoup_quot(n1, p);
  }
}

// The `T` balanced base-256 digits of c mod p (the representative that T
// digits hold: their window is 256^T values wide, so p <= 256^T has one);
// returns it.
static __int128 digits(uint64_t c, uint64_t p, int T, int8_t* d) {
  __int128 top = 0;
  for (int t = 0; t < T; ++t) top = top * 256 + 127;
  __int128 v = c;
  if (v > top) v -= p;
  __int128 x = v;
  for (int t = 0; t < T; ++t) {
    const int g = (int)((x + 128) & 255) - 128;
    d[t] = (int8_t)g;
    x = (x - g) / 256;
  }
  return v;
}

// Accumulates one output's conversion: `n` input slots, each `bytes` bytes
// wide with base constant c; writes the digits to w (block of 16 outputs,
// row m), the layout of FusedDev.
struct ConvRow {
  uint64_t p;
  int T;
  u128 sum_mod = 0;    // 128 sum of constants mod p
  u128 bound = 0;      // 128 sum of |constants|
  void slot(uint8_t* blk, int m, int kbs, int T_blk, int s, int bytes, uint64_t c) {
    uint64_t x = c % p;
    for (int b = 0; b < 8; ++b) {
      int8_t d[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (b < bytes) {
        const __int128 v = digits(x, p, T, d);
        sum_mod = (sum_mod + (u128)128 * x) % p;
        bound += (u128)128 * (u128)(v < 0 ? -v : v);
        x = mulm(x, 256 % p, p);
      }
      // input slot s, byte b: step s / 8, lane group (s % 8) / 2, byte (s % 2) 8 + b of the lane's 16
      const int kb = s / 8, lane = m + 16 * ((s % 8) / 2), at = (s % 2) * 8 + b;
      for (int t = 0; t < T_blk; ++t) blk[(((size_t)t * kbs + kb) * 64 + lane) * 16 + at] = (uint8_t)(t < T ? d[t] : 0);
    }
  }
  // The kernel sums V + off with off = (128 sum) + m p, m p >= |V|, so the
  // total lies in [0, 2^17 p); its quotient estimate is low by 0.02 to 0.2, which
  // leaves a remainder below 1.3 p.
  ConvOut finish() const {
    const uint64_t m = (uint64_t)(bound / p) + 2;
    ConvOut o;
    std::memset(&o, 0, sizeof(o));
    o.p = p;
    o.off = (uint64_t)sum_mod + m * p;
    const double pd = (double)p;
    o.c_48 = (float)(std::ldexp(1.0, 48) / pd);
    o.c_32 = (float)(std::ldexp(1.0, 32) / pd);
    o.c_16 = (float)(std::ldexp(1.0, 16) / pd);
    o.c_b = (float)((double)m + (double)(uint64_t)sum_mod / pd - 0.1);
    return o;
  }
};

void build_fused_tables(const HostParams& h, FusedTables* out) {
  const int N = h.N, k = h.k, K = h.K, R = k + K;
  for (int dir = 0; dir < 2; ++dir) {
    const std::vector<uint64_t>& tw = dir ? h.tw_inv : h.tw_fwd;
    std::vector<uint64_t>& o = out->tw[dir];
    o.assign((size_t)R * N * 2, 0);
    parallel_for(R, (size_t)N, [&](int r) {
      const uint64_t p = h.primes[r];
      const uint64_t* src = &tw[(size_t)r * N * 2];
      uint64_t* dst = &o[(size_t)r * N * 2];
      if (h.dprimes[r].field == FIELD_FP64) {
        for (int i = 0; i < N; ++i) dst[i] = balanced(src[2 * (size_t)i], p);
      } else {
        std::memcpy(dst, src, (size_t)N * 16);
      }
    });
  }
  out->lc.assign((size_t)R * 4, 0);
  out->lc_b.assign((size_t)K * 4, 0);
  out->lc_down.assign((size_t)(k + 1) * k * 4, 0);
  for (int r = 0; r < R; ++r) {
    const DevPrime& d = h.dprimes[r];
    put_lc(&out->lc[4 * r], d.ninv, d.w1ninv, d.p, d.field);
    if (r < k) continue;
    const uint64_t s = h.inv_bhat[2 * (r - k)];
    put_lc(&out->lc_b[4 * (r - k)], mulm(d.ninv, s, d.p), mulm(d.w1ninv, s, d.p), d.p, d.field);
  }
  // ModDown's factor of limb i: B^-1, with a rescale from level l > i also q_l^-1
  auto down_factor = [&](int l, int i) {
    return l < k && i < l ? h.md_fin[((size_t)l * k + i) * 2] : h.inv_b_mod_q[2 * i];
  };
  for (int l = 0; l <= k; ++l)
    for (int i = 0; i < k; ++i) {
      const DevPrime& d = h.dprimes[i];
      const uint64_t s = down_factor(l, i);
      put_lc(&out->lc_down[((size_t)l * k + i) * 4], mulm(d.ninv, s, d.p), mulm(d.w1ninv, s, d.p), d.p, d.field);
    }
  out->lc_up.assign((size_t)k * k * 4, 0);
  for (int l = 0; l < k; ++l)
    for (int i = 0; i <= l; ++i) {
      const DevPrime& d = h.dprimes[i];
      const uint64_t s = h.inv_qhat[((size_t)l * k + i) * 2];
      put_lc(&out->lc_up[((size_t)l * k + i) * 4], mulm(d.ninv, s, d.p), mulm(d.w1ninv, s, d.p), d.p, d.field);
    }
  out->bq.assign((size_t)k * 2, 0);
  for (int i = 0; i < k; ++i) {
    const DevPrime& d = h.dprimes[i];
    const uint64_t b = h.b_mod_q[2 * i];
    out->bq[2 * i] = d.field == FIELD_FP64 ? balanced(b, d.p) : b;
    out->bq[2 * i + 1] = d.field == FIELD_FP64 ? 0 : shoup_quot(b, d.p);
  }
  // ModUp at level l: inputs v_i (i <= l), outputs j.
  const int jb_n = (K + 15) / 16;
  const int Tb = K ? conv_digits((int)h.dprimes[k].nb) : 0;  // special primes share their bit length
  out->mu_kb = (k + 7) / 8;
  out->mu_stride = (uint32_t)(jb_n * Tb * out->mu_kb * 1024);
  out->mu_w.assign((size_t)k * out->mu_stride, 0);
  out->mu_out.assign((size_t)k * K, ConvOut{});
  parallel_for(k, (size_t)k * K * 64, [&](int l) {
    for (int j = 0; j < K; ++j) {
      ConvRow row;
      row.p = h.primes[k + j];
      row.T = Tb;
      uint8_t* blk = &out->mu_w[(size_t)l * out->mu_stride + (size_t)(j / 16) * Tb * out->mu_kb * 1024];
      for (int i = 0; i <= l; ++i)
        row.slot(blk, j % 16, out->mu_kb, Tb, i, ((int)h.dprimes[i].nb + 7) / 8,
                 h.qhat_mod_b[((size_t)l * K + j) * k + i]);
      out->mu_out[(size_t)l * K + j] = row.finish();
    }
  });
  // ModDown's result of limb i is f_i x_i - sum_j f_i c_ij a_j - q_l^-1 top (the
  // last with a rescale from level l, top in slot K); one table per l, and
  // index k without a rescale.
  const int ib_n = (k + 15) / 16;
  out->md_kb = (K + 8) / 8;
  out->md_stride = (uint32_t)(ib_n * 8 * out->md_kb * 1024);
  out->md_w.assign((size_t)(k + 1) * out->md_stride, 0);
  out->md_out.assign((size_t)(k + 1) * k, ConvOut{});
  parallel_for(k + 1, (size_t)k * K * 64, [&](int l) {
    for (int i = 0; i < k; ++i) {
      if (l < k && i >= l) continue;
      const uint64_t q = h.primes[i], f = down_factor(l, i);
      // digits of the widest prime of the block (the first)
      const int T_blk = conv_digits((int)h.dprimes[i / 16 * 16].nb);
      ConvRow row;
      row.p = q;
      row.T = conv_digits((int)h.dprimes[i].nb);
      uint8_t* blk = &out->md_w[(size_t)l * out->md_stride + (size_t)(i / 16) * 8 * out->md_kb * 1024];
      for (int j = 0; j < K; ++j)
        row.slot(blk, i % 16, out->md_kb, T_blk, j, 7, q - mulm(h.bhat_mod_q[((size_t)i * K + j) * 2], f, q));
      if (l < k) row.slot(blk, i % 16, out->md_kb, T_blk, K, 7, q - h.inv_ql_mod_qi[((size_t)l * k + i) * 2]);
      out->md_out[(size_t)l * k + i] = row.finish();
    }
  });
  // Screen of the ModDown products: frac(a c/q) = frac(al c/q + ah frac(2^28 c/q)), a = al + ah 2^28.
  out->scr.assign((size_t)K * 64 * 2, 0.0);
  out->scr_thr.assign(64, 0.0);
  for (int i = 0; i < k; ++i) {
    const uint64_t q = h.primes[i];
    for (int j = 0; j < K; ++j) {
      const uint64_t c = h.bhat_mod_q[((size_t)i * K + j) * 2];
      const uint64_t c28 = (uint64_t)(((u128)c << 28) % q);
      double* e = &out->scr[((size_t)j * 64 + i) * 2];
      e[0] = (double)((long double)c / (long double)q);
      e[1] = (double)((long double)c28 / (long double)q);
    }
    const DevPrime& d = h.dprimes[i];
    const uint64_t thr = d.quirk_thr < q ? d.quirk_thr : q;
    out->scr_thr[i] = (double)((long double)thr / (long double)q) + std::ldexp(1.0, -20);
  }
}

}  // namespace aoa
