// Exact negacyclic products a*s mod (X^N + 1, 2^32) for encrypt and decrypt.
//
// The reference computes b = a*s + e (tLweSymEncryptZero, eval/idash.cpp:625)
// and phase = b - a*s (tLwePhase, :714) through TFHE's floating-point FFT.
// Here the key s is binary, and a*s is computed exactly two ways:
//  - k_ring_mfma (the default for both directions): a product of the a-rows
//    with the key's negacyclic Toeplitz matrix on int8 MFMA, described there;
//    encryption first runs k_encrypt_ae for a and b = e + messages.
//  - k_encrypt / k_decrypt<J> (IHE_ENCRYPT_KERNEL / IHE_DECRYPT_KERNEL =
//    valu): (a*s)[j] = sum_{k : s_k = 1} A2[j - k + N], A2 = [-a[0..N), a[0..N)],
//    a sum of signed coefficients. One wavefront owns one ciphertext: a is
//    staged in LDS as A2 (padded one word per J so lanes reading J-strided
//    words hit distinct banks), lane l owns the J consecutive outputs
//    j = l*J + u and slides a J-register window down A2 as k advances, so each
//    key bit costs one LDS read per lane plus, when the bit is set, J adds. The
//    key bits are kernel arguments, hence wave-uniform branches.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>

#include "ihe_internal.h"
#include "ihe_rules.h"

// Work counters of ihe_decrypt_noalloc: the ring kernel's per-XCD item
// counters and its count of finished workgroups, in a file-scope device array
// instead of a context's allocation. Each GPU holds its own copy for the life
// of the process; host code uses the address hipGetSymbolAddress gives on
// that device, never this name.
static __device__ __align__(256) uint32_t scratch[ihe::kRingQueueWords];

namespace ihe {

constexpr int kWavesPerBlock = 4;

template <int J>
__device__ __forceinline__ uint32_t lds_pad(uint32_t t) {
  if constexpr (J == 1) return t;
  else return t + t / J;
}

template <int J>
constexpr uint32_t lds_words() {
  return J == 1 ? 2 * kN : 2 * kN + 2 * kN / J;
}

// acc[u] = (a*s)[jb + u] for u < J, A2 staged (padded) in lds.
template <int J>
__device__ __forceinline__ void negacyclic_window(const int32_t *lds, const KeyBits &key,
                                                  uint32_t jb, uint32_t acc[J]) {
  uint32_t win[J];
#pragma unroll
  for (int u = 0; u < J; ++u) {
    acc[u] = 0;
    win[u] = (uint32_t)lds[lds_pad<J>(jb + kN + u)];
  }
  // At step k the logical element u (= A2[jb + N + u - k]) sits in
  // win[(u - k) mod J]; after the step the slot of u = J-1 receives the new
  // logical u = 0 of step k+1.
  for (uint32_t kb = 0; kb < kN; kb += J) {
    const uint32_t bits = (key.w[kb / 32] >> (kb % 32)) & (J == 32 ? 0xFFFFFFFFu : ((1u << J) - 1u));
#pragma unroll
    for (int d = 0; d < J; ++d) {
      if ((bits >> d) & 1u) {
#pragma unroll
        for (int u = 0; u < J; ++u) acc[u] += win[(u - d) & (J - 1)];
      }
      const uint32_t t = jb + kN - (kb + (uint32_t)d) - 1u;
      win[(J - 1 - d) & (J - 1)] = (uint32_t)lds[lds_pad<J>(t)];
    }
  }
}

template <int J>
__global__ __launch_bounds__(64 * kWavesPerBlock) void k_decrypt(const int32_t *__restrict__ in,
                                                                 uint32_t num_cts, uint32_t ns,
                                                                 KeyBits key,
                                                                 float *__restrict__ out) {
  __shared__ int32_t lds_all[kWavesPerBlock][lds_words<J>()];
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t ct = blockIdx.x * kWavesPerBlock + wave;
  const bool active = ct < num_cts;
  int32_t *lds = lds_all[wave];
  if (active) {
    const int32_t *a = in + (size_t)ct * kCtWords;
    for (uint32_t t = lane; t < kN; t += 64) {
      const int32_t x = a[t];
      lds[lds_pad<J>(t)] = (int32_t)(0u - (uint32_t)x);
      lds[lds_pad<J>(t + kN)] = x;
    }
  }
  __syncthreads();
  if (!active) return;
  const uint32_t jb = lane * J;
  if (jb >= ns) return;
  uint32_t acc[J];
  negacyclic_window<J>(lds, key, jb, acc);
  const int32_t *b = in + (size_t)ct * kCtWords + kN;
#pragma unroll
  for (int u = 0; u < J; ++u) {
    const uint32_t j = jb + u;
    if (j < ns) {
      const int32_t phase = (int32_t)((uint32_t)b[j] - acc[u]);
      // t32tod then float: the int32 -> float conversion rounds to nearest
      // even; scaling by 2^-32 is exact.
      out[(size_t)ct * ns + j] = (float)phase * 0x1p-32f;
    }
  }
}

// a ^ b ^ c in one instruction (truth table 0x96)
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
  return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0x96);
}

// Philox4x32-10 (Salmon et al., SC'11).
__device__ __forceinline__ void philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                       uint32_t k0, uint32_t k1, uint32_t r[4]) {
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    // one 32 x 32 -> 64-bit product per multiplier
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t lo0 = (uint32_t)p0, hi0 = (uint32_t)(p0 >> 32);
    const uint32_t lo1 = (uint32_t)p1, hi1 = (uint32_t)(p1 >> 32);
    c0 = xor3(hi1, c1, k0);
    c1 = lo1;
    c2 = xor3(hi0, c3, k1);
    c3 = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  r[0] = c0;
  r[1] = c1;
  r[2] = c2;
  r[3] = c3;
}

// |e| = smallest k with (u >> 1) < table[k]; sign from bit 0. The table is
// non-decreasing and table[LEN - 1] = 2^63 exceeds every m, so k is the count
// of entries <= m among the first LEN - 1, found in a fixed 11 steps (no
// data-dependent loop, so the samples of a lane interleave).
__device__ __forceinline__ int32_t noise_sample(uint64_t u, const uint64_t *__restrict__ table) {
  static_assert(IHE_NOISE_TABLE_LEN - 1 <= 2047, "11 steps cover the table");
  const uint64_t m = u >> 1;
  uint32_t k = 0;
#pragma unroll
  for (uint32_t step = 1024; step > 0; step >>= 1) {
    const uint32_t nk = k + step;
    const uint64_t tv = table[min(nk, IHE_NOISE_TABLE_LEN - 1) - 1];
    k = nk <= IHE_NOISE_TABLE_LEN - 1 && tv <= m ? nk : k;
  }
  return (u & 1) ? -(int32_t)k : (int32_t)k;
}

// The same samples of four words at once, each search started from its bucket
// (lut: low end, and entries in the bucket up to kNoiseLutMany, from
// build_noise_lut). Three steps do where every bucket of the wave spans at most
// 7 entries; two more are taken where one spans up to 30 (beyond about 3.2
// sigma, one wave in four), the remaining six beyond 3.6 sigma (one in sixteen).
// The four words take them together, so that their LDS reads overlap, and
// kNoisePad entries above every m follow the table in place of a bound.
constexpr uint32_t kNoiseLutMany = 31;
constexpr uint32_t kNoisePad = 32;
__device__ __forceinline__ void noise_sample4(const uint64_t u[4], const uint64_t *table,
                                              const uint16_t *lut, uint32_t e[4]) {
  static_assert(IHE_NOISE_TABLE_LEN < 2048, "the low end takes 11 bits");
  uint32_t k[4], many = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t l = lut[(uint32_t)(u[i] >> (64 - kNoiseLutBits))];
    k[i] = l & 2047u;
    many = max(many, l >> 11);
  }
  auto step4 = [&](uint32_t step, bool pad) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t at = pad ? k[i] + step : min(k[i] + step, IHE_NOISE_TABLE_LEN);
      k[i] += table[at - 1] <= (u[i] >> 1) ? step : 0;
    }
  };
  if (__builtin_expect(__any(many > 7), 0)) {
    if (__any(many >= kNoiseLutMany))
      for (uint32_t step = 1024; step > 16; step >>= 1) step4(step, false);
    step4(16, true);
    step4(8, true);
  }
  step4(4, true);
  step4(2, true);
  step4(1, true);
#pragma unroll
  for (int i = 0; i < 4; ++i) e[i] = (u[i] & 1) ? 0u - k[i] : k[i];
}

// ---------------------------------------------------------------------------
// Decryption and encryption on int8 MFMA. For every ciphertext c and word j,
//   (a_c * s)[j] = sum_i a_c[i] T[i][j],  T[i][j] = S[j - i],
// with S[m] = s[m] for m >= 0 and -s[m + N] for m < 0 (the negacyclic wrap),
// so decryption is the product of the ciphertexts' a-rows with one Toeplitz
// matrix of entries in {-1, 0, 1}. Each a word is recoded into balanced
// signed bytes (x = sum_p 2^(8p) d_p, d_p = byte_p(x + 0x80808080) - 128), one
// v_mfma_i32_32x32x32_i8 per byte plane and K-block of 32 coefficients, all into
// one int32 accumulator that wraps mod 2^32.
//
// Work items are 32 ciphertexts x 8 TPW column tiles of 32 words (TPW = 1 .. 4
// tiles a wave; all 1,024 words at TPW = 4). One workgroup of 8 waves per CU
// holds an item's a-words as byte planes in LDS (128 KB) and stays for further
// items, taken from its XCD's counter.
//  - Planes outermost: a wave multiplies all 32 K-blocks of the highest plane
//    into its tiles' accumulators, shifts them by 8 and goes on with the next
//    plane (Horner mod 2^32; the MFMA's int32 sums wrap). So a tile costs 16
//    accumulator registers instead of 64, a wave owns four tiles, and an A
//    operand read feeds TPW MFMAs. The b words enter with the last shift.
//  - The B operand of word tile nt and K-block ks depends on nt - ks only: a
//    wave with adjacent tiles keeps them in a register window that moves by one
//    block per K-block, one LDS read for TPW MFMAs. Lane (h, c) reads the 16
//    bytes of u[N + x] = S[-x] from N - 32 (nt - ks) - c + 16 h on; LDS holds
//    every such 16-byte run (32 KB), consecutive lanes on consecutive runs,
//    which leaves no bank conflicts (shifted copies of u conflict once per 16
//    lanes wherever they lie).
//  - A: each thread loads 16 pieces of four words (16 lanes x 16 bytes of a
//    row), recodes them to digits and writes each plane's four bytes. The rows
//    of the planes' 16-byte cells are XORed with the K half and the K-block's
//    parity, which spreads the writes over the banks.
//  - Everything that touches memory is spread over the K-block steps of some
//    pass: results of the item before in plane 3's pass, b words in plane 2's,
//    the next item's a-words in plane 1's and 0's (from plane 3's on where the
//    registers allow, TPW < 4), their recoding in plane 0's. A wave that issues
//    64 loads or stores in a row stalls on the memory pipe and keeps the matrix
//    pipe idle. Two barriers an item: planes 3 and 2 are rewritten between the
//    passes 1 and 0, planes 1 and 0 in the next item's pass 3.
// Decryption (words j < NS) ends with phase = b - a*s as a float (u negated);
// encryption (all N words; k_encrypt_ae has written a and b = e + messages)
// adds a*s to b in place.
//
// What bounds it: at 242,646 ciphertexts x 1,024 words 0.75 ms (0.92 ms with 64
// accumulators a tile, two tiles a wave and 256-word items). The matrix pipe is
// busy 82 % of the cycles (58 % before), and the chip then lowers its clock to
// 1.7 GHz for power; with the MFMAs left out the same kernel takes 0.52 ms
// (5.7 TB/s). At 45,011 x 203 words: 0.064 ms (0.083 ms before), HBM and the last,
// half-filled round of workgroups.
struct RingParams {
  const int32_t *in;
  float *out;     // decryption: phases [num_cts][ns]
  int32_t *bout;  // encryption: the ciphertexts of `in` (same buffer), b halves updated
  uint32_t num_cts, ns, col_groups, num_items;
  // kRingQueueWords zero words: a workgroup's first item is fixed, the others
  // are taken from its XCD's counter; null: every gridDim / 8-th of its range
  uint32_t *queue;
};


// u[y] = S[N - y]: s[N - y] for 1 <= y <= N, -s[2N - y] for N < y < 2N, else 0
// (key words in LDS); NEG: its negative.
template <bool NEG>
__device__ __forceinline__ uint32_t u_byte(uint32_t y, const uint32_t *kw) {
  const uint32_t m = (0u - y) & (kN - 1);
  const uint32_t bit = y ? (kw[m / 32] >> (m % 32)) & 1u : 0u;
  return bit * ((y > kN) != NEG ? 0xFFu : 1u);
}

static_assert(kRuns == 2 * kN - 16, "16-byte runs of u that B operands are made of");
constexpr uint32_t kRingThreads = 512, kRingWaves = kRingThreads / 64;

struct RingLds {
  uint32_t planes[4][kN / 32][256];  // [plane][K-block][k half][row, swizzled][4 dwords]
  uint32_t u[kRuns][4];  // run e: bytes u[e + 1 .. e + 16]
  uint32_t next;                 // the item after the next one
};
static_assert(sizeof(RingLds) <= 160 * 1024, "one workgroup's LDS");

// NT: a-words by streaming (nt) loads, for decryptions of kRingStreamCts
// ciphertexts and more. Their a-words (4 KB each) pass through the 256 MB
// infinity cache without being found there again, and loads that leave lines
// behind made 242,646 x 256 take 298 us and x 160 271 us; streaming they take 280
// and 248 us (three inputs in turn: 294 and 266; the kernel of 256-word items: 290
// and 260). Below it they find part of an input that was decrypted before:
// 45,011 x 256 takes 55.6 us plain and 61.7 us streaming, 100,000 x 256 128 and
// 122 us. At four tiles a wave the MFMAs hide either (242,646 x 1,024: 742, 743 us).
constexpr uint32_t kRingStreamCts = 3u << 15;

template <bool ENC, int TPW, bool NT = false>
__global__ __launch_bounds__(kRingThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_ring_mfma(RingParams P, KeyBits key) {
  typedef int int4v __attribute__((ext_vector_type(4)));
  typedef int int16v __attribute__((ext_vector_type(16)));
  typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
  constexpr int kRsrc3 = 0x00020000;  // raw buffer descriptor, dword 3
  constexpr uint32_t kDrop = 0x80000000u;  // an offset past every buffer: loads 0, stores nothing
  constexpr uint32_t kCtBytes = kCtWords * 4;
  constexpr bool kEarly = TPW < 4;  // registers left to load the next item from pass 3 on
  __shared__ __attribute__((aligned(16))) RingLds S;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const uint32_t h = lane / 32, c = lane % 32;
  const uint32_t lim = ENC ? kN : P.ns;
  const uint32_t xcd = blockIdx.x % 8, per_xcd = gridDim.x / 8;
  const uint32_t chunk = (P.num_items + 7) / 8;
  const uint32_t it_beg = min(xcd * chunk, P.num_items);
  const uint32_t it_end = min((xcd + 1) * chunk, P.num_items);
  // this item, the next (loaded meanwhile) and, in S.next, the one after it
  uint32_t item = it_beg + blockIdx.x / 8, next = item + per_xcd;

  // loader role: words 64 i + 4 lc .. + 3 of row lr, i < 16
  const uint32_t lr = threadIdx.x / 16, lc = threadIdx.x % 16;
  const uint32_t wpar = lc / 8, whalf = (lc % 8) / 4;
  uint32_t *const wp =
      &S.planes[0][wpar][whalf * 128 + ((lr ^ (4 * whalf) ^ (2 * wpar)) * 4) + lc % 4];
  u32x4v q[16];
  auto rows_of = [&](uint32_t it) { return min(32u, P.num_cts - (it / P.col_groups) * 32); };
  auto in_rsrc = [&](uint32_t it, bool on) {
    return __builtin_amdgcn_make_buffer_rsrc(
        (void *)(P.in + (size_t)(it / P.col_groups) * 32 * kCtWords), (short)0,
        on ? (int)(32 * kCtBytes) : 0, kRsrc3);
  };
  auto a_off = [&](uint32_t it) { return min(lr, rows_of(it) - 1) * kCtBytes + lc * 16; };
  auto load_a = [&](const __amdgpu_buffer_rsrc_t &R, uint32_t vo, int i) {
    q[i] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(R, vo + 256 * i, 0,
                                                                          NT ? 2 : 0));
  };
  auto put = [&](int p, int i) { wp[p * 8192 + i * 512] = q[i][p]; };
  // piece i: four words -> their digits by plane; planes 3 and 2 written
  auto recode = [&](int i) {
    u32x4v y;
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = (q[i][k] + 0x80808080u) ^ 0x80808080u;
    const uint32_t t0 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
    q[i][0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    q[i][1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    q[i][2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    q[i][3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
    put(3, i);
    put(2, i);
  };

  {
    const __amdgpu_buffer_rsrc_t R = in_rsrc(item < it_end ? item : 0, item < it_end);
    const uint32_t vo = a_off(item < it_end ? item : 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) load_a(R, vo, i);
  }
  uint32_t taken = 0;
  if (P.queue && threadIdx.x == 0) taken = atomicAdd(&P.queue[xcd], 1u);
  // u itself, in the space of the planes, then its runs
  uint32_t *const kw = &S.planes[0][0][0], *const u0 = &S.planes[1][0][0];
  if (threadIdx.x < kN / 32) kw[threadIdx.x] = key.w[threadIdx.x];
  __syncthreads();
  {
    uint32_t v = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) v |= u_byte<!ENC>(4 * threadIdx.x + i, kw) << (8 * i);
    u0[threadIdx.x] = v;
  }
  if (P.queue && threadIdx.x == 0) S.next = it_beg + per_xcd + taken;
  __syncthreads();
  if (threadIdx.x < kRuns / 4) {  // runs 4 t .. 4 t + 3: dwords t .. t + 4 of u
    uint32_t x[5];
#pragma unroll
    for (uint32_t i = 0; i < 5; ++i) x[i] = u0[threadIdx.x + i];
#pragma unroll
    for (int s = 1; s <= 4; ++s) {
      u32x4v v;
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = s < 4 ? __builtin_amdgcn_alignbyte(x[k + 1], x[k], s) : x[k + 1];
      *(u32x4v *)S.u[4 * threadIdx.x + s - 1] = v;
    }
  }
  if (P.queue) next = __builtin_amdgcn_readfirstlane(S.next);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) recode(i);
  __syncthreads();

  // A operand addresses of this lane in even and odd K-blocks
  const uint8_t *const ra0 = (const uint8_t *)&S.planes[0][0][h * 128 + ((c ^ (4 * h)) * 4)];
  const uint8_t *const ra1 = (const uint8_t *)&S.planes[0][0][h * 128 + ((c ^ (4 * h) ^ 2) * 4)];
  const uint32_t ostride = ENC ? kCtBytes : P.ns * 4;
  int16v br[TPW];  // an item's b words, then its results
  uint32_t vo[TPW];
  uint32_t p_item = 0, p_rows = 0;  // the item of the results in br; 0 rows: none
  auto out_rsrc = [&](uint32_t it, bool on) {
    const size_t ct0 = (size_t)(it / P.col_groups) * 32;
    return __builtin_amdgcn_make_buffer_rsrc(
        ENC ? (void *)(P.bout + ct0 * kCtWords) : (void *)(P.out + ct0 * P.ns), (short)0,
        on ? (int)(32 * ostride) : 0, kRsrc3);
  };
  // a value that what depends on it is computed from where it is used, not earlier
  auto late = [](uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  // value v of a tile: row m + 4 h of the item, m = 8 (v / 4) + v % 4
  auto row_of = [](int v) -> uint32_t { return 8 * (v / 4) + v % 4; };
  auto store = [&](const __amdgpu_buffer_rsrc_t &R, int i) {
    const int v = i / TPW, t = i % TPW;
    __builtin_amdgcn_raw_buffer_store_b32(br[t][v], R, vo[t], row_of(v) * ostride, 2);
  };
  auto store_part = [&]() {
    const __amdgpu_buffer_rsrc_t R = out_rsrc(p_item, true);
    const uint32_t r0 = late(4 * h);
#pragma unroll
    for (int i = 0; i < 16 * TPW; ++i) {
      const int v = i / TPW, t = i % TPW;
      __builtin_amdgcn_raw_buffer_store_b32(
          br[t][v], R, row_of(v) + r0 < p_rows ? vo[t] : kDrop, row_of(v) * ostride, 2);
    }
  };
#pragma unroll
  for (int t = 0; t < TPW; ++t) br[t] = int16v{}, vo[t] = kDrop;

  while (item < it_end) {
    const uint32_t rows = rows_of(item);
    const uint32_t nt0 = (item % P.col_groups) * (kRingWaves * TPW) + wave * TPW;
    const bool active = nt0 * 32 < lim, full = rows == 32, more = next < it_end;
    const __amdgpu_buffer_rsrc_t nr = in_rsrc(more ? next : item, more);
    const uint32_t nvo = a_off(more ? next : item);
    const int4v *const bl = (const int4v *)S.u + ring_run(nt0, h, c);
    int16v acc[TPW];
    // plane p's K-blocks; hook(ks) issues the step's share of other work, and a
    // scheduling barrier keeps it there
    auto pass = [&](int p, auto hook) {
      constexpr int kSlots = TPW + 2;  // the block of tile t at K-block ks: slot (t - ks) mod kSlots
      auto slot = [](int d) { return (d + 32 * kSlots) % kSlots; };
      int4v w[kSlots], a[3];
#pragma unroll
      for (int t = 0; t < TPW; ++t)
        w[t] = bl[kRingWordTiles % TPW ? 32 * ((int)nt0 - (int)ring_operand_tile(nt0 + t)) : -32 * t];
      w[slot(-1)] = bl[32];
      a[0] = *(const int4v *)(ra0 + p * 32768);
      a[1] = *(const int4v *)(ra1 + p * 32768 + 1024);
      if (p < 3) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) acc[t] = p == 0 ? (acc[t] << 8) + br[t] : acc[t] << 8;
      }
#pragma unroll
      for (int ks = 0; ks < 32; ++ks) {
        if (ks + 2 < 32) {
          w[slot(-(ks + 2))] = bl[32 * (ks + 2)];
          a[(ks + 2) % 3] = *(const int4v *)((ks & 1 ? ra1 : ra0) + p * 32768 + (ks + 2) * 1024);
        }
        hook(ks);
#pragma unroll
        for (int t = 0; t < TPW; ++t)
          acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
              a[ks % 3], w[slot(t - ks)], p == 3 && ks == 0 ? int16v{} : acc[t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (P.queue && threadIdx.x == 0) taken = atomicAdd(&P.queue[xcd], 1u);
    // whole results go out in pass 3, a partial group's (or an idle wave's) at once
    const bool whole = active && p_rows == 32;
    if (!whole && p_rows) store_part();
    const __amdgpu_buffer_rsrc_t orr = out_rsrc(p_item, whole);
    const __amdgpu_buffer_rsrc_t ir = in_rsrc(item, full);
    uint32_t vb[TPW];
    if (active) {
      pass(3, [&](int ks) {
        if (ks < 16) {
          put(1, ks);
          put(0, ks);
          if constexpr (kEarly) load_a(nr, nvo, ks);
        }
#pragma unroll
        for (int i = ks * TPW / 2; i < (ks + 1) * TPW / 2; ++i) store(orr, i);
      });
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const uint32_t j = (nt0 + t) * 32 + c;
        vb[t] = j < lim ? 4 * h * kCtBytes + (kN + j) * 4 : kDrop;
        vo[t] = j < lim ? 4 * h * ostride + ((ENC ? kN : 0) + j) * 4 : kDrop;
      }
      pass(2, [&](int ks) {
#pragma unroll
        for (int i = ks * TPW / 2; i < (ks + 1) * TPW / 2; ++i) {
          const int v = i / TPW, t = i % TPW;
          br[t][v] = __builtin_amdgcn_raw_buffer_load_b32(ir, vb[t], row_of(v) * kCtBytes, 0);
        }
      });
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        put(1, i);
        put(0, i);
        if constexpr (kEarly) load_a(nr, nvo, i);
      }
    }
    __syncthreads();
    if (P.queue && threadIdx.x == 0) S.next = it_beg + per_xcd + taken;
    if (active) {
      pass(1, [&](int ks) {
        if (!kEarly && ks >= 16 && ks % 2 == 0) load_a(nr, nvo, (ks - 16) / 2);
      });
      if (!full) {
        const __amdgpu_buffer_rsrc_t pr = in_rsrc(item, true);
        const uint32_t r0 = late(4 * h);
#pragma unroll
        for (int i = 0; i < 16 * TPW; ++i) {
          const int v = i / TPW, t = i % TPW;
          br[t][v] = __builtin_amdgcn_raw_buffer_load_b32(
              pr, row_of(v) + r0 < rows ? vb[t] : kDrop, row_of(v) * kCtBytes, 0);
        }
      }
      pass(0, [&](int ks) {
        if (!kEarly && ks < 16 && ks % 2 == 0) load_a(nr, nvo, 8 + ks / 2);
        if (ks >= 16) recode(ks - 16);
      });
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          br[t][v] = ENC ? acc[t][v] : __builtin_bit_cast(int, (float)acc[t][v] * 0x1p-32f);
    } else {
      if constexpr (!kEarly) {
#pragma unroll
        for (int i = 0; i < 16; ++i) load_a(nr, nvo, i);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) recode(i);
    }
    p_item = item;
    p_rows = active ? rows : 0;
    __syncthreads();
    item = next;
    next = P.queue ? (uint32_t)__builtin_amdgcn_readfirstlane(S.next) : next + per_xcd;
  }
  if (p_rows) store_part();
  // the last workgroup to finish clears the counters for the next launch
  if (P.queue && threadIdx.x == 0) {
    if (atomicAdd(&P.queue[8], 1u) == gridDim.x - 1)
      for (uint32_t i = 0; i <= 8; ++i) atomicExch(&P.queue[i], 0u);
  }
}

struct EncryptParams {
  const int8_t *__restrict__ geno;
  const uint64_t *__restrict__ table;
  const uint32_t *__restrict__ lut;
  int32_t *__restrict__ out;
  double *__restrict__ out_var;
  uint32_t num_cts, num_cols, ns, R, rs;
  uint32_t seed_lo, seed_hi;
  uint64_t rs_recip;  // ceil(2^32 / rs): j / rs = (j * rs_recip) >> 32 for every word j < N
};

// One wavefront per ciphertext c (FeatIndex):
//   a = Philox stream 0, b = a*s + e + one-hot messages (setScore); without
//   genotypes (geno == nullptr) the ciphertexts encrypt zero (tLweSymEncryptZero).
__global__ __launch_bounds__(64 * kWavesPerBlock) void k_encrypt(EncryptParams P, KeyBits key) {
  constexpr int J = 16;
  __shared__ int32_t lds_all[kWavesPerBlock][lds_words<J>()];
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t ct = blockIdx.x * kWavesPerBlock + wave;
  const bool active = ct < P.num_cts;
  int32_t *lds = lds_all[wave];
  const uint32_t jb = lane * J;
  if (active) {
    int32_t *a = P.out + (size_t)ct * kCtWords;
#pragma unroll
    for (int q = 0; q < J / 4; ++q) {
      uint32_t r[4];
      const uint32_t w0 = jb + 4 * q;
      philox(w0 / 4, ct, 0, 0, P.seed_lo, P.seed_hi, r);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        a[w0 + t] = (int32_t)r[t];
        lds[lds_pad<J>(w0 + t)] = (int32_t)(0u - r[t]);
        lds[lds_pad<J>(w0 + t + kN)] = (int32_t)r[t];
      }
    }
  }
  __syncthreads();
  if (!active) return;
  uint32_t acc[J];
  negacyclic_window<J>(lds, key, jb, acc);
  int32_t *b = P.out + (size_t)ct * kCtWords + kN;
#pragma unroll
  for (int q = 0; q < J / 2; ++q) {
    uint32_t r[4];
    const uint32_t j0 = jb + 2 * q;
    philox(j0 / 2, ct, 1, 0, P.seed_lo, P.seed_hi, r);
    const uint64_t u0 = (uint64_t)r[0] | ((uint64_t)r[1] << 32);
    const uint64_t u1 = (uint64_t)r[2] | ((uint64_t)r[3] << 32);
    acc[2 * q] += (uint32_t)noise_sample(u0, P.table);
    acc[2 * q + 1] += (uint32_t)noise_sample(u1, P.table);
  }
#pragma unroll
  for (int u = 0; u < J; ++u) {
    const uint32_t j = jb + u;
    const uint32_t r = (uint32_t)(((uint64_t)j * P.rs_recip) >> 32), s = j - r * P.rs;
    uint32_t v = acc[u];
    if (P.geno && r < P.R && s < P.ns) {
      const uint32_t bidx = ct * P.R + r;
      if (bidx < P.num_cols) {
        const uint32_t tag = bidx / 3, val = bidx - 3 * tag;
        const int8_t g = P.geno[(size_t)tag * P.ns + s];
        if (g == 0 || g == 1 || g == 2) {
          if ((uint32_t)g == val) v += kOne;
        } else {
          v += val == 0 ? kNan[0] : (val == 1 ? kNan[1] : kNan[2]);
        }
      }
    }
    b[j] = (int32_t)v;
  }
  if (lane == 0) P.out_var[ct] = 0x1p-50;
}

// Everything of encryption but a*s, with k_encrypt's streams and counters: a
// (Philox stream 0, one counter per four words), b = e + messages (stream 1,
// one counter per two words, e sampled from the CDF table), and the variance.
// k_ring_mfma<true> then adds a*s to b. Persistent workgroups copy the CDF
// table to LDS (its searches are scattered reads) and take ciphertexts in
// turn, a thread four words j..j+3 of each. VALU-bound (54 multiply-adds of
// Philox, four searches and four messages a thread), so searches and messages
// are selects instead of branches. As many workgroups share a CU as registers
// and LDS (bucket index in 16 bits) allow, and the grid is that many: the grid
// of eight before left its last quarter to a second, half-empty wave of
// workgroups (48,552 ciphertexts, encryption: 314 us with branches and a grid of
// eight; 268 us at 5 and 6 a CU, 299 at 7 and 341 at 8, where registers spill).
//
// ONE is for one region (NS > 512): a ciphertext is one column, its tag and
// value are scalars and a word's genotype byte lies at the word's own offset,
// which saves 40 of some 300 vector instructions and leaves registers for seven
// workgroups: 261.3 -> 252.4 us (253.9 at six).
template <bool ONE>
constexpr uint32_t kAeBlocks = ONE ? 7 : 6;
template <bool ONE>
__global__ __launch_bounds__(256, kAeBlocks<ONE>) void k_encrypt_ae(EncryptParams P) {
  typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
  constexpr int kRsrc3 = 0x00020000;  // raw buffer descriptor, dword 3
  __shared__ uint64_t s_table[IHE_NOISE_TABLE_LEN + kNoisePad];
  __shared__ uint16_t s_lut[1u << kNoiseLutBits];
  for (uint32_t t = threadIdx.x; t < IHE_NOISE_TABLE_LEN + kNoisePad; t += 256)
    s_table[t] = t < IHE_NOISE_TABLE_LEN ? P.table[t] : ~0ull;
  for (uint32_t t = threadIdx.x; t < (1u << kNoiseLutBits); t += 256) {
    const uint32_t l = P.lut[t];
    s_lut[t] = (uint16_t)((l & 0xFFFFu) | min(l >> 16, kNoiseLutMany) << 11);
  }
  __syncthreads();
  const uint32_t q = threadIdx.x;
  // word 4 q's region and sample; the next words follow in the same region or
  // at the start of the next one
  const uint32_t rr0 = (uint32_t)(((uint64_t)(4 * q) * P.rs_recip) >> 32), sj0 = 4 * q - rr0 * P.rs;
  for (uint32_t ct = blockIdx.x; ct < P.num_cts; ct += gridDim.x) {
    int32_t *a = P.out + (size_t)ct * kCtWords;
    // The genotype bytes of this thread's four b words (setScore) are loaded
    // first, so that their latency runs under the Philox rounds below. Words
    // without a message load nothing and match no genotype.
    int32_t g[4] = {0, 0, 0, 0};
    uint32_t val[4] = {3, 3, 3, 3};
    if (ONE && P.geno) {
      const uint32_t tag = ct / 3;
      const __amdgpu_buffer_rsrc_t row = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<int8_t *>(P.geno + (size_t)tag * P.ns), 0, P.ns, kRsrc3);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        val[u] = 4 * q + u < P.ns ? ct - 3 * tag : 3u;
        g[u] = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(row, 4 * q + u, 0, 0);
      }
    } else if (P.geno) {
      const uint32_t col0 = ct * P.R, tag0 = col0 / 3;
      const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<int8_t *>(P.geno + (size_t)tag0 * P.ns), 0, 0x7FFFFFFF, kRsrc3);
      uint32_t rr = rr0, sj = sj0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t col = col0 - 3 * tag0 + rr, tag = col * 683 >> 11;  // col / 3, col < 2,048
        const bool has = rr < P.R && sj < P.ns && col0 + rr < P.num_cols;
        const uint32_t off = has ? tag * P.ns + sj : ~0u;
        val[u] = has ? col - 3 * tag : 3u;
        g[u] = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rows, off, 0, 0);
        ++sj;
        rr += sj == P.rs;
        sj = sj == P.rs ? 0 : sj;
      }
    }
    uint32_t r[4];
    philox(q, ct, 0, 0, P.seed_lo, P.seed_hi, r);
    *(u32x4v *)(a + 4 * q) = u32x4v{r[0], r[1], r[2], r[3]};
    uint64_t w[4];
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      philox(2 * q + pr, ct, 1, 0, P.seed_lo, P.seed_hi, r);
      w[2 * pr] = (uint64_t)r[0] | ((uint64_t)r[1] << 32);
      w[2 * pr + 1] = (uint64_t)r[2] | ((uint64_t)r[3] << 32);
    }
    uint32_t b[4];
    noise_sample4(w, s_table, s_lut, b);
#pragma unroll
    for (int u = 0; u < 4; ++u) b[u] += (uint32_t)g[u] == val[u] ? kOne : 0u;
    if (max(max((uint32_t)g[0], (uint32_t)g[1]), max((uint32_t)g[2], (uint32_t)g[3])) > 2) {
      // missing genotypes (a word without a message has g = 0)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t t = val[u] == 0 ? kNan[0] : (val[u] == 1 ? kNan[1] : kNan[2]);
        b[u] += (uint32_t)g[u] > 2 ? t : 0u;
      }
    }
    *(u32x4v *)(a + kN + 4 * q) = u32x4v{b[0], b[1], b[2], b[3]};
    if (q == 0) P.out_var[ct] = 0x1p-50;
  }
}

// Largest decrypt of ihe_decrypt_noalloc: its item count (32-ciphertext groups
// x column groups of 1024 words) stays far inside the 32-bit counters.
constexpr uint32_t kNoallocMaxCts = 1u << 26;

// Column tiles per wave (TPW). A round of workgroups, one per CU, takes about
// 5 us for an item's a-words and 2.5 us for each tile that a SIMD's waves own
// (waves w and w + 4 share a SIMD); fewer tiles a wave make more items, which
// pays where the ciphertexts alone leave CUs idle (33 ciphertexts x 1,024
// words: 13.4 us at TPW = 1, 24.7 us at 4; 242,646: 1,024 and 742 us), and
// three or four tiles keep NS = 300 or 512 to one wave per SIMD (242,646 x 300:
// 372 us at TPW = 3, 384 us at 2). Ties go to more tiles, which read less LDS
// (45,011 x 512: 82.6 us at 4, 87.4 us at 2). IHE_RING_TILES = 1 .. 4 sets it;
// IHE_RING_QUEUE=0 gives the workgroups fixed items instead of the counters.
uint32_t ring_tiles_per_wave(uint32_t groups, uint32_t tiles, uint32_t num_cus) {
  const char *e = std::getenv("IHE_RING_TILES");
  if (e && e[0] >= '1' && e[0] <= '4' && !e[1]) return (uint32_t)(e[0] - '0');
  uint64_t best = ~0ull;
  uint32_t tpw = 1;
  for (uint32_t t = 1; t <= 4; ++t) {
    const uint32_t per_item = kRingWaves * t, cg = (tiles + per_item - 1) / per_item;
    const uint64_t rounds = ((uint64_t)groups * cg + num_cus - 1) / num_cus;
    const bool one_wave = cg == 1 && tiles <= kRingWaves / 2 * t;  // per SIMD
    const uint64_t cost = rounds * (2 + (one_wave ? t : 2 * t));
    if (cost <= best) {
      best = cost;
      tpw = t;
    }
  }
  return tpw;
}

// Launch shape: one persistent workgroup per CU, a multiple of the 8 XCDs.
template <bool ENC>
void launch_ring(hipStream_t stream, RingParams P, const KeyBits &key, uint32_t num_cus,
                 uint32_t *queue) {
  static_assert(kRingQueueWords >= 9, "eight XCD counters and a finished count");
  const char *q = std::getenv("IHE_RING_QUEUE");
  P.queue = (q && std::strcmp(q, "0") == 0) ? nullptr : queue;
  const uint32_t tiles = ((ENC ? kN : P.ns) + 31) / 32, groups = (P.num_cts + 31) / 32;
  const uint32_t tpw = ring_tiles_per_wave(groups, tiles, num_cus);
  P.col_groups = (tiles + kRingWaves * tpw - 1) / (kRingWaves * tpw);
  P.num_items = groups * P.col_groups;
  const dim3 grid(std::min<uint32_t>((num_cus + 7) / 8 * 8, (P.num_items + 7) / 8 * 8));
  const dim3 block(kRingThreads);
  // encryption reads back the a-words that it has just written
  const bool nt = !ENC && P.num_cts >= kRingStreamCts;
  const auto launch = [&](void (*plain)(RingParams, KeyBits), void (*stream_a)(RingParams, KeyBits)) {
    hipLaunchKernelGGL(nt ? stream_a : plain, grid, block, 0, stream, P, key);
  };
  switch (tpw) {
    case 1: launch(k_ring_mfma<ENC, 1>, k_ring_mfma<ENC, 1, !ENC>); break;
    case 2: launch(k_ring_mfma<ENC, 2>, k_ring_mfma<ENC, 2, !ENC>); break;
    case 3: launch(k_ring_mfma<ENC, 3>, k_ring_mfma<ENC, 3, !ENC>); break;
    default: launch(k_ring_mfma<ENC, 4>, k_ring_mfma<ENC, 4>); break;
  }
}

__global__ void k_clear_words(uint32_t *p, uint32_t n) {
  if (threadIdx.x < n) p[threadIdx.x] = 0;
}

// Per device: the address of `scratch` and the CU count, looked up on the
// first ihe_decrypt_noalloc call on that device (with that device current).
constexpr int kMaxDevices = 64;
struct NoallocDevice {
  uint32_t *scratch = nullptr;
  uint32_t num_cus = 0;
};
std::mutex g_noalloc_mu;
NoallocDevice g_noalloc[kMaxDevices];

int noalloc_device(int dev, NoallocDevice &out) {
  if (dev < 0 || dev >= kMaxDevices) return fail(IHE_ERR_UNSUPPORTED, "device index beyond 63");
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  NoallocDevice &d = g_noalloc[dev];
  if (!d.scratch) {
    hipDeviceProp_t prop;
    IHE_HIP(hipGetDeviceProperties(&prop, dev));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
      return fail(IHE_ERR_UNSUPPORTED, std::string("kernels are built for gfx950, device is ") +
                                           prop.gcnArchName);
    void *p = nullptr;
    IHE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(IHE_ERR_HIP, "hipGetSymbolAddress gave no address for the work counters");
    d.num_cus = (uint32_t)prop.multiProcessorCount;
    d.scratch = static_cast<uint32_t *>(p);
  }
  out = d;
  return IHE_OK;
}

int noalloc_setup(int device) {
  NoallocDevice d;
  return noalloc_device(device, d);
}

}  // namespace ihe

using namespace ihe;

extern "C" {

int ihe_key_create(ihe_ctx *ctx, const int32_t *key, ihe_key **out) {
  if (int rc = check_ctx(ctx)) return rc;
  if (!key || !out) return fail(IHE_ERR_ARG, "null argument");
  *out = nullptr;
  ihe_key *k = new ihe_key();
  k->ctx = ctx;
  std::memset(&k->bits, 0, sizeof(k->bits));
  for (uint32_t i = 0; i < kN; ++i) {
    if (key[i] != 0 && key[i] != 1) {
      delete k;
      return fail(IHE_ERR_ARG, "TLWE key must be binary");
    }
    if (key[i]) k->bits.w[i / 32] |= 1u << (i % 32);
  }
  *out = k;
  return IHE_OK;
}

int ihe_key_destroy(ihe_key *key) {
  delete key;
  return IHE_OK;
}

int ihe_encrypt(ihe_ctx *ctx, const ihe_key *key, const ihe_layout *layout, uint32_t num_tags,
                const int8_t *d_geno, uint64_t seed, int32_t *d_out, double *d_out_var) {
  if (int rc = check_ctx(ctx)) return rc;
  if (!key || key->ctx->device != ctx->device)
    return fail(IHE_ERR_ARG, "key is not on this context's device");
  if (!layout) return fail(IHE_ERR_ARG, "null layout");
  const uint32_t NS = layout->num_samples;
  if (NS == 0 || NS > kN || layout->num_regions != kN / NS ||
      layout->region_size != kN / layout->num_regions)
    return fail(IHE_ERR_ARG, "layout must satisfy R = N / NS and RS = N / R (eval/idash.cpp:409-410)");
  if (num_tags == 0) return IHE_OK;
  if (!d_out || !d_out_var) return fail(IHE_ERR_ARG, "null buffer");
  if (num_tags > 0x55555555u) return fail(IHE_ERR_ARG, "too many tags");
  if (int rc = make_current(ctx)) return rc;
  EncryptParams P;
  P.geno = d_geno;
  P.table = ctx->d_noise_table;
  P.lut = ctx->d_noise_lut;
  P.out = d_out;
  P.out_var = d_out_var;
  P.num_cols = 3 * num_tags;
  P.R = layout->num_regions;
  P.rs = layout->region_size;
  P.rs_recip = ((1ull << 32) + P.rs - 1) / P.rs;
  P.ns = NS;
  P.num_cts = (P.num_cols + P.R - 1) / P.R;
  P.seed_lo = (uint32_t)seed;
  P.seed_hi = (uint32_t)(seed >> 32);
  const char *force = std::getenv("IHE_ENCRYPT_KERNEL");
  if (!(force && std::strcmp(force, "valu") == 0)) {
    // a and b = e + messages, then b += a*s on the MFMA kernel
    const RingParams D{d_out, nullptr, d_out, P.num_cts, NS, 0, 0, nullptr};
    ScopedTimer t(ctx, IHE_TIMER_ENCRYPT);
    static_assert(kN / 4 == 256, "a thread per four words of a ciphertext");
    const auto launch_ae = [&](void (*ae)(EncryptParams), uint32_t blocks) {
      hipLaunchKernelGGL(ae, dim3(std::min<uint32_t>(P.num_cts, (uint32_t)ctx->num_cus * blocks)),
                         dim3(256), 0, ctx->stream, P);
    };
    if (P.R == 1) launch_ae(k_encrypt_ae<true>, kAeBlocks<true>);
    else launch_ae(k_encrypt_ae<false>, kAeBlocks<false>);
    launch_ring<true>(ctx->stream, D, key->bits, (uint32_t)ctx->num_cus, ctx->d_ring_queue);
    IHE_HIP(hipGetLastError());
    return IHE_OK;
  }
  const dim3 grid((P.num_cts + kWavesPerBlock - 1) / kWavesPerBlock), block(64 * kWavesPerBlock);
  {
    ScopedTimer t(ctx, IHE_TIMER_ENCRYPT);
    hipLaunchKernelGGL(k_encrypt, grid, block, 0, ctx->stream, P, key->bits);
  }
  IHE_HIP(hipGetLastError());
  return IHE_OK;
}

int ihe_decrypt(ihe_ctx *ctx, const ihe_key *key, uint32_t num_samples, const int32_t *d_in,
                uint32_t num_cts, float *d_out) {
  if (int rc = check_ctx(ctx)) return rc;
  if (!key || key->ctx->device != ctx->device)
    return fail(IHE_ERR_ARG, "key is not on this context's device");
  if (num_samples == 0 || num_samples > kN) return fail(IHE_ERR_ARG, "NUM_SAMPLES must be in [1, 1024]");
  if (num_cts == 0) return IHE_OK;
  if (!d_in || !d_out) return fail(IHE_ERR_ARG, "null buffer");
  if (int rc = make_current(ctx)) return rc;
  ScopedTimer t(ctx, IHE_TIMER_DECRYPT);
  const char *force = std::getenv("IHE_DECRYPT_KERNEL");
  if (!(force && std::strcmp(force, "valu") == 0)) {
    const RingParams P{d_in, d_out, nullptr, num_cts, num_samples, 0, 0, nullptr};
    launch_ring<false>(ctx->stream, P, key->bits, (uint32_t)ctx->num_cus, ctx->d_ring_queue);
    IHE_HIP(hipGetLastError());
    return IHE_OK;
  }
  const dim3 grid((num_cts + kWavesPerBlock - 1) / kWavesPerBlock), block(64 * kWavesPerBlock);
  // J = outputs per lane, the smallest power of two with 64 * J >= NS.
  if (num_samples <= 64) hipLaunchKernelGGL(k_decrypt<1>, grid, block, 0, ctx->stream, d_in, num_cts, num_samples, key->bits, d_out);
  else if (num_samples <= 128) hipLaunchKernelGGL(k_decrypt<2>, grid, block, 0, ctx->stream, d_in, num_cts, num_samples, key->bits, d_out);
  else if (num_samples <= 256) hipLaunchKernelGGL(k_decrypt<4>, grid, block, 0, ctx->stream, d_in, num_cts, num_samples, key->bits, d_out);
  else if (num_samples <= 512) hipLaunchKernelGGL(k_decrypt<8>, grid, block, 0, ctx->stream, d_in, num_cts, num_samples, key->bits, d_out);
  else hipLaunchKernelGGL(k_decrypt<16>, grid, block, 0, ctx->stream, d_in, num_cts, num_samples, key->bits, d_out);
  IHE_HIP(hipGetLastError());
  return IHE_OK;
}

int ihe_decrypt_noalloc(const int32_t *key, uint32_t num_samples, const int32_t *d_in,
                        uint32_t num_cts, float *d_out, void *hip_stream) {
  if (!key) return fail(IHE_ERR_ARG, "null key");
  if (num_samples == 0 || num_samples > kN) return fail(IHE_ERR_ARG, "NUM_SAMPLES must be in [1, 1024]");
  if (num_cts > kNoallocMaxCts)
    return fail(IHE_ERR_ARG, "ihe_decrypt_noalloc takes at most 2^26 ciphertexts per call, got " +
                                 std::to_string(num_cts));
  KeyBits bits;
  std::memset(&bits, 0, sizeof(bits));
  for (uint32_t i = 0; i < kN; ++i) {
    if (key[i] != 0 && key[i] != 1) return fail(IHE_ERR_ARG, "TLWE key must be binary");
    if (key[i]) bits.w[i / 32] |= 1u << (i % 32);
  }
  if (num_cts == 0) return IHE_OK;
  if (!d_in || !d_out) return fail(IHE_ERR_ARG, "null buffer");
  int dev = 0;
  IHE_HIP(hipGetDevice(&dev));
  NoallocDevice D;
  if (int rc = noalloc_device(dev, D)) return rc;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const RingParams P{d_in, d_out, nullptr, num_cts, num_samples, 0, 0, nullptr};
  // the counters start at zero (a fill kernel: no memset node under capture)
  hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(64), 0, stream, D.scratch, kRingQueueWords);
  launch_ring<false>(stream, P, bits, D.num_cus, D.scratch);
  IHE_HIP(hipGetLastError());
  return IHE_OK;
}

}  // extern "C"
