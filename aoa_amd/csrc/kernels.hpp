// Host-side launchers of the gfx950 kernels (all stream-ordered, no sync).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.hpp"
#include "params.hpp"

namespace aoa {

enum EltOp { ELT_ADD = 0, ELT_SUB = 1, ELT_MUL = 2, ELT_NEG = 3, ELT_MULADD = 5 };
// Sampler distributions (same values as the C-ABI's AOA_SAMPLE_*).
enum SampleKind { SAMPLE_UNIFORM = 0, SAMPLE_GAUSSIAN = 1, SAMPLE_ZO = 2, SAMPLE_HW = 3, SAMPLE_NARROW = 4 };
constexpr int kHwMaxAttempts = 4096;

bool ntt_valid_split(int N, int N1);
// Forward / inverse NTT of every limb in `m`.  N1 = 0: the set's split, or
// without one nt_forward / nt_inverse.
int ntt_forward(const DevParams& P, LimbMap m, int N1, hipStream_t st);
int ntt_inverse(const DevParams& P, LimbMap m, int N1, hipStream_t st);

// Fused key switching (fused.hpp).  fz_mul: HomMul + relinearisation (+ rescale)
// of one item; fz_switch: key switching of one item.  Workspace in the item.
int fz_mul(const DevParams& P, const FzItem& it, hipStream_t st);
int fz_switch(const DevParams& P, const FzItem& it, hipStream_t st);
int fz_rows_item(const DevParams& P, const FzItem& it, hipStream_t st);
void fz_up_item(const DevParams& P, const FzItem& it, bool mul, hipStream_t st);
int fz_key_item(const DevParams& P, const FzItem& it, hipStream_t st);
void fz_down_item(const DevParams& P, const FzItem& it, hipStream_t st);
// The same stage by stage over device tables: `list` entries are item << 8 | limb.
// nstrict >= 0: the first nstrict entries are of primes wider than 2^56 and the
// others of form `field`; the special limbs' key products have a list of their own.
int fz_rows_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int nstrict, int field,
                 hipStream_t st);
void fz_up_desc(const DevParams& P, const FzItem* items, int n, int max_level, bool mul, hipStream_t st);
int fz_key_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int nstrict, int field,
                hipStream_t st);
int fz_key_special_desc(const DevParams& P, const FzItem* items, const uint32_t* list, int n, int field, hipStream_t st);
void fz_down_desc(const DevParams& P, const FzItem* items, int n, int max_level, hipStream_t st);

// Plain transforms on the fused kernels' split (fused_ntt.hip), the default
// where no split was asked for.
bool nt_default(const DevParams& P);
int nt_forward(const DevParams& P, const LimbMap& m, hipStream_t st);
int nt_inverse(const DevParams& P, const LimbMap& m, hipStream_t st);
int nt_forward_desc(const DevParams& P, const NttDesc* d, int n, hipStream_t st);
int nt_inverse_desc(const DevParams& P, const NttDesc* d, int n, hipStream_t st);
// Encryption after the forward columns of m, u, e0 + m and e1 (limbs of N words).
struct NtEncrypt {
  const uint64_t *u, *e0, *e1, *pkb, *pka;
  uint64_t *m, *c0, *c1;
};
int nt_encrypt_rows(const DevParams& P, const NtEncrypt& a, int nlimbs, hipStream_t st);
void nt_forward_cols(const DevParams& P, const LimbMap& m, hipStream_t st);
// c0, c1 -> NTT domain, m = c0 + c1 s in the coefficient domain.
int nt_decrypt(const DevParams& P, uint64_t* m, uint64_t* c0, uint64_t* c1, const uint64_t* s, int nlimbs, hipStream_t st);

// out = a op b (out = a*b + c for MULADD) over nlimbs limbs mapped to primes
// as in LimbMap (qlimbs Q limbs from prime0, then special limbs).
void launch_encrypt_combine(const DevParams& P, uint64_t* c0, uint64_t* c1, const uint64_t* pkb,
                            const uint64_t* pka, const uint64_t* u, const uint64_t* e0, const uint64_t* e1,
                            const uint64_t* m, int nlimbs, hipStream_t st);
void launch_eltwise(const DevParams& P, int op, uint64_t* out, const uint64_t* a, const uint64_t* b,
                    const uint64_t* c, int nlimbs, int qlimbs, int prime0, hipStream_t st);

void launch_eltwise_scalar(const DevParams& P, int op, uint64_t* out, const uint64_t* a, uint64_t b, int nlimbs,
                           int prime0, hipStream_t st);
void launch_conjugate(const DevParams& P, uint64_t* out, const uint64_t* in, int nlimbs, hipStream_t st);

// Sampler: limbs res0..res0+nres-1 of out (poly base pointer, limb r at
// out + r*N) from distribution `kind`, keyed by (seed, nonce).
void launch_sample(const DevParams& P, uint64_t* out, int res0, int nres, int kind, uint64_t seed, uint64_t nonce,
                   hipStream_t st);
// u (ZO) at nonce, e0 and e1 (Gaussian) at nonce + 1 and nonce + 2, limbs
// 0..nres-1, in one launch; with m, e0 + m.
void launch_sample_encrypt(const DevParams& P, uint64_t* u, uint64_t* e0, uint64_t* e1, const uint64_t* m, int nres,
                           uint64_t seed, uint64_t nonce, hipStream_t st);

// CKKS encoder (FP64).  vals holds n complex values (re, im interleaved); the
// special FFT runs in place (inverse: encoding direction, with the division by
// n).  encode: the inverse FFT of vals in place and k limbs of N residues of its
// values; decode: the FFT of limb 0's (coefficient domain) slot values.
void launch_special_fft(const DevParams& P, double* vals, int n, int inverse, hipStream_t st);
void launch_encode(const DevParams& P, uint64_t* out, double* vals, int slots, double scale, int k, hipStream_t st);
void launch_decode(const DevParams& P, double* vals, const uint64_t* in, int slots, double scale, hipStream_t st);
// ModUp: x holds Q limbs 0..level (coefficient domain, stride N); writes K
// special limbs to outB (stride N).
void launch_modup(const DevParams& P, const uint64_t* x, uint64_t* outB, int level, hipStream_t st);

// ModDown: inQ holds Q limbs 0..level, inB the K special limbs (coefficient
// domain).  out limb i = (inQ_i - conv_i(inB)) B^-1 mod q_i.
void launch_moddown(const DevParams& P, const uint64_t* inQ, const uint64_t* inB, uint64_t* out, int level,
                    hipStream_t st);

// Rescale c0 and c1 in place (coefficient domain) from `level`.
void launch_rescale(const DevParams& P, uint64_t* c0, uint64_t* c1, int level, hipStream_t st);
// acc += sum_i x[i] (2 (i + off) + 1) mod 2^64 over n words (acc on the device).
void launch_checksum(const uint64_t* x, size_t n, uint64_t off, uint64_t* acc, hipStream_t st);

// Galois automorphism X -> X^g (g odd) in the coefficient domain, gather form.
void launch_automorphism(const DevParams& P, uint64_t* out, const uint64_t* in, int nlimbs,
                         uint64_t galois, hipStream_t st);
// Both polynomials of a rotation in one launch.
void launch_automorphism2(const DevParams& P, uint64_t* out0, uint64_t* out1, const uint64_t* in0, const uint64_t* in1,
                          int nlimbs, uint64_t galois, hipStream_t st);
uint64_t galois_inverse(uint64_t galois, int N);

// rho of a QB polynomial: Q limbs times (B mod q_i), special limbs zero.
void launch_rho(const DevParams& P, uint64_t* out, const uint64_t* in, hipStream_t st);
void launch_dot(const DevParams& P, uint64_t* c, const uint64_t* const* a, const uint64_t* const* b, int k,
                hipStream_t st);
void launch_dr2(const DevParams& P, uint64_t* c21, uint64_t* c22, uint64_t* c23, const uint64_t* a01,
                const uint64_t* a02, const uint64_t* a11, const uint64_t* a12, hipStream_t st);

// Descriptor-driven (stage-fused) forms used by batches: one launch covers
// every descriptor of the table (device memory).
int ntt_forward_desc(const DevParams& P, const NttDesc* d, int ndesc, int N1, hipStream_t st);
int ntt_inverse_desc(const DevParams& P, const NttDesc* d, int ndesc, int N1, hipStream_t st);
void launch_automorphism_desc(const DevParams& P, const AutoDesc* d, int ndesc, hipStream_t st);

}  // namespace aoa
