// CKKS slot encode and decode on gfx950 (binary64).
//
// Slot order as fhelium_amd/codec.py and the reference's generator-3
// convention (fhelium/engine/slot_embedding.py, galois.py:10-26): slot j is
// the evaluation at zeta^{e_j}, zeta = e^{i pi / N}, e_j = 3^{-j} mod 2N, and
// pos_j = (e_j - 1) / 2 is its index among the N odd exponents.
//
//   encode:  z[pos_j] = m_j, z[N-1-pos_j] = conj(m_j)      (every index once)
//            a = FFT_N(z) / N * conj(twist), twist_k = zeta^k
//            coefficient_k = rint(Re(a_k) * scale), residues mod each prime
//   decode:  x_k = centered CRT of the residues over two primes (Garner)
//            z = sum_k x_k twist_k e^{+2 pi i j k / N}    (an FFT with + sign)
//            m_j = z[pos_j] / scale
//
// The FFT is iterative radix-2 on bit-reversed input (butterflies of half
// size h = 2^s, twiddle e^{i pi k / h}), executed in one of two ways:
//   * 2^12 <= N <= 2^16, with the caller's tables (fh_codec_tables): two
//     passes over the elements, one on 256-element tiles (8 stages) and one
//     on columns of stride 256 (the other logN - 8).  Each thread holds 16
//     elements, four stages per LDS exchange, and twiddles come from a table
//     instead of a sincospi per butterfly.  Encode gathers its slots, runs
//     the butterflies below in the same order (its rounded coefficients are
//     the same bits) and ends in them; decode reads its residues in natural
//     order, runs the stages in the opposite order and ends in the slots.
//   * any other N (fh_ckks_encode, fh_ckks_decode): one launch per stage.
// One launch per stage spends its time on 16 passes over the 16-byte
// elements and a sincospi per butterfly: at N = 2^16 the stages took 85 us
// for 12 encoded entries and 87 us for 9 decoded ones, besides 59 us of
// 64-bit remainders onto 27 rows and 28 us of 128-bit ones in the CRT; the
// two passes take 25 us and 28 us, everything included (the remainders onto the
// rows moved into the transform that reads them).
#include "fh_common.h"
#include "fh_views.h"
#include "ntt_core.h"

namespace fh {
namespace {

constexpr int kCodecBlock = 256;

__device__ __forceinline__ uint32_t bitrev(uint32_t x, int bits) { return __brev(x) >> (32 - bits); }

// z: [B, N] complex as (re, im) pairs.
__global__ __launch_bounds__(kCodecBlock) void k_encode_scatter(const double* slots, int64_t s, const int32_t* pos,
                                                               int log_n, double2* z) {
  const int64_t b = blockIdx.y;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  if (j >= s) return;
  const int64_t n = int64_t{1} << log_n;
  const double re = slots[(b * s + j) * 2], im = slots[(b * s + j) * 2 + 1];
  const uint32_t p = static_cast<uint32_t>(pos[j]);
  z[b * n + bitrev(p, log_n)] = make_double2(re, im);
  z[b * n + bitrev(static_cast<uint32_t>(n - 1) - p, log_n)] = make_double2(re, -im);
}

// One radix-2 stage of half size h on bit-reversed-input data; sign -1 is
// the forward DFT (e^{-2 pi i jk/N}), +1 the positive-exponent sum.
__global__ __launch_bounds__(kCodecBlock) void k_fft_stage(double2* z, int log_n, int64_t h, double sign) {
  const int64_t b = blockIdx.y;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  const int64_t n = int64_t{1} << log_n;
  if (t >= n / 2) return;
  const int64_t k = t & (h - 1);
  const int64_t i0 = ((t - k) << 1) + k;
  const int64_t i1 = i0 + h;
  double sn, cs;
  sincospi(sign * static_cast<double>(k) / static_cast<double>(h), &sn, &cs);
  double2* row = z + b * n;
  const double2 u = row[i0], v = row[i1];
  const double vr = v.x * cs - v.y * sn, vi = v.x * sn + v.y * cs;
  row[i0] = make_double2(u.x + vr, u.y + vi);
  row[i1] = make_double2(u.x - vr, u.y - vi);
}

// coefficient_k = rint(Re(z_k conj(twist_k)) / N * scale), then its residue
// for each prime: out [B, L, N] canonical standard.
__global__ __launch_bounds__(kCodecBlock) void k_encode_finish(const double2* z, int log_n, double scale,
                                                              const int64_t* moduli, int64_t limbs, int64_t* out) {
  const int64_t b = blockIdx.y;
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  const int64_t n = int64_t{1} << log_n;
  if (k >= n) return;
  const double2 v = z[b * n + k];
  double sn, cs;
  sincospi(static_cast<double>(k) / static_cast<double>(n), &sn, &cs);
  const double re = (v.x * cs + v.y * sn) / static_cast<double>(n);  // Re(v * conj(twist))
  const int64_t c = static_cast<int64_t>(rint(re * scale));
  for (int64_t l = 0; l < limbs; ++l) {
    const int64_t q = moduli[l];
    int64_t r = c % q;
    if (r < 0) r += q;
    out[(b * limbs + l) * n + k] = r;
  }
}

// x_k centered over q_a q_b by Garner, times twist_k, written bit-reversed.
__global__ __launch_bounds__(kCodecBlock) void k_decode_crt(const int64_t* ra, const int64_t* rb, int64_t batch_stride,
                                                           int64_t qa, int64_t qb, int64_t qa_inv_b, int log_n,
                                                           double2* z) {
  const int64_t b = blockIdx.y;
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  const int64_t n = int64_t{1} << log_n;
  if (k >= n) return;
  const uint64_t a = static_cast<uint64_t>(ra[b * batch_stride + k]);
  const uint64_t bb = static_cast<uint64_t>(rb[b * batch_stride + k]);
  // t = (b - a) qa^{-1} mod qb; x = a + qa t in [0, qa qb)
  const uint64_t qbu = static_cast<uint64_t>(qb);
  const uint64_t diff = (bb + qbu - a % qbu) % qbu;
  const unsigned __int128 prod = static_cast<unsigned __int128>(diff) * static_cast<uint64_t>(qa_inv_b);
  int64_t t = static_cast<int64_t>(static_cast<uint64_t>(prod % qbu));
  // centre: x > (qa qb - 1) / 2 = (qb - 1) / 2 qa + (qa - 1) / 2
  const int64_t half = (qb - 1) / 2;
  if (t > half || (t == half && a > static_cast<uint64_t>(qa - 1) / 2)) t -= qb;
  // |x| < 2^62: one rounding from the exact int64 value; larger: binary64.
  const double x = (t >= -3 && t <= 3)
                       ? static_cast<double>(static_cast<int64_t>(a) + qa * t)
                       : static_cast<double>(static_cast<int64_t>(a)) + static_cast<double>(qa) * static_cast<double>(t);
  double sn, cs;
  sincospi(static_cast<double>(k) / static_cast<double>(n), &sn, &cs);
  z[b * n + bitrev(static_cast<uint32_t>(k), log_n)] = make_double2(x * cs, x * sn);
}

__global__ __launch_bounds__(kCodecBlock) void k_decode_gather(const double2* z, const int32_t* pos, int64_t s,
                                                              int log_n, double inv_scale, double* slots) {
  const int64_t b = blockIdx.y;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  if (j >= s) return;
  const int64_t n = int64_t{1} << log_n;
  const double2 v = z[b * n + pos[j]];
  slots[(b * s + j) * 2] = v.x * inv_scale;
  slots[(b * s + j) * 2 + 1] = v.y * inv_scale;
}

int fft_stages(double2* z, int64_t batch, int log_n, double sign, hipStream_t st) {
  const int64_t n = int64_t{1} << log_n;
  const dim3 grid(static_cast<uint32_t>(ceil_div(n / 2, kCodecBlock)), static_cast<uint32_t>(batch));
  for (int s = 0; s < log_n; ++s) {
    hipLaunchKernelGGL(k_fft_stage, grid, dim3(kCodecBlock), 0, st, z, log_n, int64_t{1} << s, sign);
    FH_CHECK_LAUNCH("codec fft stage");
  }
  return kOk;
}

// ---------------------------------------------------------------------------
// Two-pass execution, 12 <= logN <= 16.
// ---------------------------------------------------------------------------
constexpr int kFftTile = 256;       // elements of a tile (first eight stages)
constexpr int kTileThreads = 64;    // four tiles of 16 threads per block, one wave
constexpr int kColThreads = 128;    // encode's column pass: T threads x C columns
constexpr int kCrtThreads = 256;    // decode's: 128-byte runs of residues

// twiddles[h + k] = e^{i pi k / h}, h a power of two up to N, k < h;
// slot_map[p] = j where pos_j = p, ~j where N - 1 - pos_j = p.
__global__ __launch_bounds__(kCodecBlock) void k_codec_tables(const int32_t* pos, int log_n, double2* twiddles,
                                                             int32_t* slot_map) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  const int64_t n = int64_t{1} << log_n;
  if (i >= 2 * n) return;
  if (i == 0) {
    twiddles[0] = make_double2(0.0, 0.0);
  } else {
    const int64_t h = int64_t{1} << (63 - __builtin_clzll(static_cast<uint64_t>(i)));
    double sn, cs;
    sincospi(static_cast<double>(i - h) / static_cast<double>(h), &sn, &cs);
    twiddles[i] = make_double2(cs, sn);
  }
  if (i < n / 2) {
    const int32_t p = pos[i];
    slot_map[p] = static_cast<int32_t>(i);
    slot_map[static_cast<int32_t>(n - 1) - p] = ~static_cast<int32_t>(i);
  }
}

// k_fft_stage's butterfly with sign -1 (the table holds the conjugate).
__device__ __forceinline__ void fft_butterfly(double2& a, double2& b, double2 w) {
  const double cs = w.x, sn = -w.y;
  const double2 u = a, v = b;
  const double vr = v.x * cs - v.y * sn, vi = v.x * sn + v.y * cs;
  a = make_double2(u.x + vr, u.y + vi);
  b = make_double2(u.x - vr, u.y - vi);
}

// First eight stages of one tile's 256 elements by 16 threads: thread t
// starts with elements 16t + k and ends with t + 16k.
__device__ __forceinline__ void fft_tile(double2 (&v)[16], int t, const double2* tw, double2* sh) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int h = 1 << s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & h) continue;
      fft_butterfly(v[k], v[k + h], tw[h + (k & (h - 1))]);
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) sh[17 * t + k] = v[k];
  ntt::tile_sync();
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = sh[ntt::tile_pad(t + 16 * k)];
#pragma unroll
  for (int s = 4; s < 8; ++s) {
    const int h = 1 << s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & (h >> 4)) continue;
      fft_butterfly(v[k], v[k + (h >> 4)], tw[h + ((t + 16 * k) & (h - 1))]);
    }
  }
}

struct FftArgs {
  double2* z;               // [B, N]
  const double2* twiddles;  // [2N]
  const int32_t* slot_map;  // [N]
  int log_n;
};

// Grid (N / 1024, B).  Slots [B, S] at their bit-reversed positions.
__global__ __launch_bounds__(kTileThreads) void k_encode_tiles(FftArgs a, const double2* slots) {
  __shared__ double2 lds[4 * (kFftTile + kFftTile / 16)];
  const int64_t n = int64_t{1} << a.log_n;
  const int m = threadIdx.x / 16, t = threadIdx.x % 16;
  const uint32_t r = blockIdx.x * 4 + m;
  const double2* row = slots + static_cast<int64_t>(blockIdx.y) * (n / 2);
  double2 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int32_t j = a.slot_map[bitrev(r * kFftTile + 16 * t + k, a.log_n)];
    const double2 x = row[j < 0 ? ~j : j];
    v[k] = make_double2(x.x, j < 0 ? -x.y : x.y);
  }
  fft_tile(v, t, a.twiddles, lds + m * (kFftTile + kFftTile / 16));
  double2* out = a.z + static_cast<int64_t>(blockIdx.y) * n + r * kFftTile;
#pragma unroll
  for (int k = 0; k < 16; ++k) out[t + 16 * k] = v[k];
}

// The second pass: stages of half size 256 .. N/2 on the 2^S1 rows of C
// columns.  Ends with each thread's elements handed to
// finish(element, value).
template <int S1, class Finish>
__device__ __forceinline__ void fft_columns(const FftArgs& a, double2* lds, Finish finish) {
  constexpr int R1 = 1 << S1;
  constexpr int T = R1 / 16;
  constexpr int C = kColThreads / T;
  const int64_t n = int64_t{1} << a.log_n;
  const int c = threadIdx.x % C;
  const int t = threadIdx.x / C;
  const int col = blockIdx.x * C + c;
  const double2* z = a.z + static_cast<int64_t>(blockIdx.y) * n;
  const double2* tw = a.twiddles;
  double2 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = z[(16 * t + k) * kFftTile + col];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int h = 1 << s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & h) continue;
      fft_butterfly(v[k], v[k + h], tw[(h + (k & (h - 1))) * kFftTile + col]);
    }
  }
  if constexpr (S1 > 4) {
#pragma unroll
    for (int k = 0; k < 16; ++k) lds[(16 * t + k) * C + c] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = lds[(t + T * k) * C + c];
#pragma unroll
    for (int s = 4; s < S1; ++s) {
      const int h = 1 << s;
      const int half = 1 << (s - (S1 - 4));  // the row bit as a bit of k
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (k & half) continue;
        fft_butterfly(v[k], v[k + half], tw[(h + ((t + T * k) & (h - 1))) * kFftTile + col]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) finish((S1 > 4 ? t + T * k : 16 * t + k) * kFftTile + col, v[k]);
}

template <int S1>
constexpr int fft_lds_elements() {
  return S1 > 4 ? (1 << S1) * (kColThreads / ((1 << S1) / 16)) : 1;
}

// Grid (256 / C, B).  coefficient_k = rint(Re(z_k conj(twist_k)) / N scale).
template <int S1>
__global__ __launch_bounds__(kColThreads) void k_encode_columns(FftArgs a, double scale, int64_t* out) {
  __shared__ double2 lds[fft_lds_elements<S1>()];
  const int64_t n = int64_t{1} << a.log_n;
  const double inv_n = 1.0 / static_cast<double>(n);
  int64_t* row = out + static_cast<int64_t>(blockIdx.y) * n;
  fft_columns<S1>(a, lds, [&](int i, double2 v) {
    const double2 w = a.twiddles[n + i];
    const double re = (v.x * w.x + v.y * w.y) * inv_n;  // Re(v * conj(twist)); 1/N is exact
    row[i] = static_cast<int64_t>(rint(re * scale));
  });
}

// Two residues of each coefficient, over q_a and q_b, with an optional
// addend (canonical or any representative within 2^51 of zero times q).
struct CrtArgs {
  const int64_t* ra;
  const int64_t* rb;
  int64_t batch_stride;
  const int64_t* add_a;  // null: none
  const int64_t* add_b;
  int64_t add_batch_stride;
  int64_t add_coef_stride;
  int64_t qa, qb;
  double qa_inv, qb_inv;        // 1 / q
  uint64_t inv, inv_shoup;      // qa^{-1} mod qb and floor(inv 2^64 / qb)
};

// Decode runs the stages from the largest half size down (natural input,
// bit-reversed output), so that the residues are read as whole cache lines;
// its slots are scattered in any case.  At bit-reversed positions the reads
// touch a line per residue.
__device__ __forceinline__ void dif_butterfly(double2& a, double2& b, double2 w) {
  const double dx = a.x - b.x, dy = a.y - b.y;
  a = make_double2(a.x + b.x, a.y + b.y);
  b = make_double2(dx * w.x - dy * w.y, dx * w.y + dy * w.x);
}

// Grid (256 / C, B): the centered CRT of k_decode_crt (its 64- and 128-bit
// divisions replaced by reciprocals and a Shoup product), times the twist,
// and the stages of half size N/2 .. 256 on C columns.
template <int S1>
__global__ __launch_bounds__(kCrtThreads) void k_decode_columns(FftArgs a, CrtArgs q) {
  constexpr int R1 = 1 << S1;
  constexpr int T = R1 / 16;
  constexpr int C = kCrtThreads / T;
  __shared__ double2 lds[S1 > 4 ? R1 * C : 1];
  const int64_t n = int64_t{1} << a.log_n;
  const int c = threadIdx.x % C;
  const int t = threadIdx.x / C;
  const int col = blockIdx.x * C + c;
  const int64_t b = blockIdx.y;
  const uint64_t qa = static_cast<uint64_t>(q.qa), qb = static_cast<uint64_t>(q.qb);
  auto plus = [](int64_t x, int64_t y, uint64_t mod, double inv) -> int64_t {
    const uint64_t s = static_cast<uint64_t>(x) + static_cast<uint64_t>(canonical_operand(y, mod, inv));
    return static_cast<int64_t>(s >= mod ? s - mod : s);
  };
  int64_t xa[16], xb[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int64_t i = b * q.batch_stride + (t + T * k) * kFftTile + col;
    xa[k] = q.ra[i];
    xb[k] = q.rb[i];
  }
  if (q.add_a != nullptr) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int64_t i = b * q.add_batch_stride + ((t + T * k) * kFftTile + col) * q.add_coef_stride;
      xa[k] = plus(xa[k], q.add_a[i], qa, q.qa_inv);
      xb[k] = plus(xb[k], q.add_b[i], qb, q.qb_inv);
    }
  }
  double2 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    // t = (b - a) qa^{-1} mod qb; x = a + qa t in [0, qa qb)
    uint64_t diff = static_cast<uint64_t>(xb[k]) + qb - static_cast<uint64_t>(canonical_operand(xa[k], qb, q.qb_inv));
    diff = diff >= qb ? diff - qb : diff;
    int64_t td = static_cast<int64_t>(shoup_mulmod(q.inv, q.inv_shoup, diff, qb));
    // centre: x > (qa qb - 1) / 2 = (qb - 1) / 2 qa + (qa - 1) / 2
    const int64_t half = (q.qb - 1) / 2;
    if (td > half || (td == half && xa[k] > (q.qa - 1) / 2)) td -= q.qb;
    // |x| < 2^62: one rounding from the exact int64 value; larger: binary64.
    const double x = (td >= -3 && td <= 3)
                         ? static_cast<double>(xa[k] + q.qa * td)
                         : static_cast<double>(xa[k]) + static_cast<double>(q.qa) * static_cast<double>(td);
    const double2 w = a.twiddles[n + (t + T * k) * kFftTile + col];
    v[k] = make_double2(x * w.x, x * w.y);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int half = 8 >> s;
    const int h = (R1 / 2) >> s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & half) continue;
      dif_butterfly(v[k], v[k + half], a.twiddles[(h + ((t + T * k) & (h - 1))) * kFftTile + col]);
    }
  }
  double2* z = a.z + b * n;
  if constexpr (S1 > 4) {
#pragma unroll
    for (int k = 0; k < 16; ++k) lds[(t + T * k) * C + c] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = lds[(16 * t + k) * C + c];
#pragma unroll
    for (int s = 4; s < S1; ++s) {
      const int h = (R1 / 2) >> s;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (k & h) continue;
        dif_butterfly(v[k], v[k + h], a.twiddles[(h + (k & (h - 1))) * kFftTile + col]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) z[(S1 > 4 ? 16 * t + k : t + T * k) * kFftTile + col] = v[k];
}

// Grid (N / 1024, B): the stages of half size 128 .. 1 inside the tiles; the
// element at position p is coefficient bitrev(p) of the embedding.
__global__ __launch_bounds__(kTileThreads) void k_decode_tiles(FftArgs a, double inv_scale, double2* slots) {
  __shared__ double2 lds[4 * (kFftTile + kFftTile / 16)];
  const int64_t n = int64_t{1} << a.log_n;
  const int m = threadIdx.x / 16, t = threadIdx.x % 16;
  const uint32_t r = blockIdx.x * 4 + m;
  const double2* z = a.z + static_cast<int64_t>(blockIdx.y) * n + r * kFftTile;
  double2* sh = lds + m * (kFftTile + kFftTile / 16);
  double2 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = z[t + 16 * k];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int half = 8 >> s;
    const int h = 128 >> s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & half) continue;
      dif_butterfly(v[k], v[k + half], a.twiddles[h + ((t + 16 * k) & (h - 1))]);
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) sh[ntt::tile_pad(t + 16 * k)] = v[k];
  ntt::tile_sync();
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = sh[17 * t + k];
#pragma unroll
  for (int s = 4; s < 8; ++s) {
    const int h = 128 >> s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k & h) continue;
      dif_butterfly(v[k], v[k + h], a.twiddles[h + (k & (h - 1))]);
    }
  }
  double2* row = slots + static_cast<int64_t>(blockIdx.y) * (n / 2);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int32_t j = a.slot_map[bitrev(r * kFftTile + 16 * t + k, a.log_n)];
    if (j >= 0) row[j] = make_double2(v[k].x * inv_scale, v[k].y * inv_scale);
  }
}

#define FH_CODEC_COLUMNS(K, THREADS, LOG_N, ...)                                                               \
  switch (static_cast<int>(LOG_N) - 8) {                                                                      \
    case 4: hipLaunchKernelGGL(K<4>, dim3(256 * 1 / THREADS, batch32), dim3(THREADS), 0, st, __VA_ARGS__); break;  \
    case 5: hipLaunchKernelGGL(K<5>, dim3(256 * 2 / THREADS, batch32), dim3(THREADS), 0, st, __VA_ARGS__); break;  \
    case 6: hipLaunchKernelGGL(K<6>, dim3(256 * 4 / THREADS, batch32), dim3(THREADS), 0, st, __VA_ARGS__); break;  \
    case 7: hipLaunchKernelGGL(K<7>, dim3(256 * 8 / THREADS, batch32), dim3(THREADS), 0, st, __VA_ARGS__); break;  \
    default: hipLaunchKernelGGL(K<8>, dim3(256 * 16 / THREADS, batch32), dim3(THREADS), 0, st, __VA_ARGS__); break; \
  }

// The CRT of both residue rows and the embedding (two launches).
int decode_two_pass(CrtArgs q, int64_t batch, int64_t log_n, const int32_t* slot_map, const double* twiddles,
                    double scale, double* workspace, double* slots, hipStream_t st) {
  FH_CHECK_ARG(q.qa > 2 && q.qb > 4096 && (q.qb & 1) && q.inv > 0 && q.inv < static_cast<uint64_t>(q.qb),
               "decode moduli must be odd primes with a^{-1} mod b given");
  FH_CHECK_ARG(scale > 0.0, "decode scale must be positive");
  q.qa_inv = 1.0 / static_cast<double>(q.qa);
  q.qb_inv = 1.0 / static_cast<double>(q.qb);
  q.inv_shoup = static_cast<uint64_t>((static_cast<unsigned __int128>(q.inv) << 64) / static_cast<uint64_t>(q.qb));
  FftArgs a{reinterpret_cast<double2*>(workspace), reinterpret_cast<const double2*>(twiddles), slot_map,
            static_cast<int>(log_n)};
  const uint32_t batch32 = static_cast<uint32_t>(batch);
  FH_CODEC_COLUMNS(k_decode_columns, kCrtThreads, log_n, a, q)
  FH_CHECK_LAUNCH("decode crt + column stages");
  hipLaunchKernelGGL(k_decode_tiles, dim3(static_cast<uint32_t>((int64_t{1} << log_n) / (4 * kFftTile)), batch32),
                     dim3(kTileThreads), 0, st, a, 1.0 / scale, reinterpret_cast<double2*>(slots));
  FH_CHECK_LAUNCH("decode tile stages");
  return kOk;
}

// out[b, l, i] = (c[b, i] mod q_l) R mod q_l, canonical.
__global__ __launch_bounds__(kCodecBlock) void k_lift_montgomery(const int64_t* coefficients, int64_t n,
                                                                const NttRow* rows, ParamView params,
                                                                int64_t limbs, int64_t* out) {
  const int64_t l = blockIdx.y;
  const int64_t b = blockIdx.z;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kCodecBlock + threadIdx.x;
  if (i >= n) return;
  const Mont m = load_mont(params, l);
  const int64_t c = canonical_operand(coefficients[b * n + i], m.q, rows[l].qinv);
  out[(b * limbs + l) * n + i] = mont_mul(c, m.r2, m);
}

}  // namespace
}  // namespace fh

using namespace fh;

FH_API int fh_ckks_encode(const double* slots, int64_t batch, int64_t log_n, const int32_t* slot_positions,
                          double scale, const int64_t* moduli, int64_t limbs, double* workspace, int64_t* out,
                          void* stream) {
  FH_CHECK_ARG(log_n >= 2 && log_n <= 17, "encode supports logN 2..17");
  FH_CHECK_ARG(batch >= 1 && batch <= 65535 && limbs >= 1, "bad encode batch or limb count");
  FH_CHECK_ARG(scale > 0.0 && scale < 0x1.0p62, "encode scale must be positive and below 2^62");
  FH_CHECK_ARG(slots && slot_positions && moduli && workspace && out, "encode: null operand");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t n = int64_t{1} << log_n;
  const int64_t s = n / 2;
  double2* z = reinterpret_cast<double2*>(workspace);
  hipLaunchKernelGGL(k_encode_scatter, dim3(static_cast<uint32_t>(ceil_div(s, kCodecBlock)), static_cast<uint32_t>(batch)),
                     dim3(kCodecBlock), 0, st, slots, s, slot_positions, static_cast<int>(log_n), z);
  FH_CHECK_LAUNCH("encode scatter");
  int rc = fft_stages(z, batch, static_cast<int>(log_n), -1.0, st);
  if (rc != kOk) return rc;
  hipLaunchKernelGGL(k_encode_finish, dim3(static_cast<uint32_t>(ceil_div(n, kCodecBlock)), static_cast<uint32_t>(batch)),
                     dim3(kCodecBlock), 0, st, z, static_cast<int>(log_n), scale, moduli, limbs, out);
  FH_CHECK_LAUNCH("encode finish");
  return kOk;
}

FH_API int fh_ckks_decode(const int64_t* residues_a, const int64_t* residues_b, int64_t batch_stride, int64_t batch,
                          int64_t log_n, int64_t modulus_a, int64_t modulus_b, int64_t modulus_a_inverse_mod_b,
                          const int32_t* slot_positions, double scale, double* workspace, double* slots,
                          void* stream) {
  FH_CHECK_ARG(log_n >= 2 && log_n <= 17, "decode supports logN 2..17");
  FH_CHECK_ARG(batch >= 1 && batch <= 65535, "bad decode batch");
  FH_CHECK_ARG(modulus_a > 2 && modulus_b > 2 && (modulus_b & 1) && modulus_a_inverse_mod_b > 0 &&
                   modulus_a_inverse_mod_b < modulus_b,
               "decode moduli must be odd primes with a^{-1} mod b given");
  FH_CHECK_ARG(scale > 0.0, "decode scale must be positive");
  FH_CHECK_ARG(residues_a && residues_b && slot_positions && workspace && slots, "decode: null operand");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t n = int64_t{1} << log_n;
  const int64_t s = n / 2;
  double2* z = reinterpret_cast<double2*>(workspace);
  hipLaunchKernelGGL(k_decode_crt, dim3(static_cast<uint32_t>(ceil_div(n, kCodecBlock)), static_cast<uint32_t>(batch)),
                     dim3(kCodecBlock), 0, st, residues_a, residues_b, batch_stride, modulus_a, modulus_b,
                     modulus_a_inverse_mod_b, static_cast<int>(log_n), z);
  FH_CHECK_LAUNCH("decode crt");
  int rc = fft_stages(z, batch, static_cast<int>(log_n), 1.0, st);
  if (rc != kOk) return rc;
  hipLaunchKernelGGL(k_decode_gather, dim3(static_cast<uint32_t>(ceil_div(s, kCodecBlock)), static_cast<uint32_t>(batch)),
                     dim3(kCodecBlock), 0, st, z, slot_positions, s, static_cast<int>(log_n), 1.0 / scale, slots);
  FH_CHECK_LAUNCH("decode gather");
  return kOk;
}

FH_API int fh_codec_tables(int64_t log_n, const int32_t* slot_positions, double* twiddles, int32_t* slot_map,
                           void* stream) {
  FH_CHECK_ARG(log_n >= 12 && log_n <= 16, "codec tables are for logN 12..16");
  FH_CHECK_ARG(slot_positions && twiddles && slot_map, "codec tables: null operand");
  hipLaunchKernelGGL(k_codec_tables, dim3(static_cast<uint32_t>((int64_t{2} << log_n) / kCodecBlock)),
                     dim3(kCodecBlock), 0, static_cast<hipStream_t>(stream), slot_positions, static_cast<int>(log_n),
                     reinterpret_cast<double2*>(twiddles), slot_map);
  FH_CHECK_LAUNCH("codec tables");
  return kOk;
}

FH_API int fh_ckks_encode_coefficients(const double* slots, int64_t batch, int64_t log_n, const int32_t* slot_map,
                                       const double* twiddles, double scale, double* workspace, int64_t* out,
                                       void* stream) {
  FH_CHECK_ARG(log_n >= 12 && log_n <= 16, "two-pass encode supports logN 12..16");
  FH_CHECK_ARG(batch >= 1 && batch <= 65535, "bad encode batch");
  FH_CHECK_ARG(scale > 0.0 && scale < 0x1.0p62, "encode scale must be positive and below 2^62");
  FH_CHECK_ARG(slots && slot_map && twiddles && workspace && out, "encode: null operand");
  hipStream_t st = static_cast<hipStream_t>(stream);
  FftArgs a{reinterpret_cast<double2*>(workspace), reinterpret_cast<const double2*>(twiddles), slot_map,
            static_cast<int>(log_n)};
  const uint32_t batch32 = static_cast<uint32_t>(batch);
  hipLaunchKernelGGL(k_encode_tiles, dim3(static_cast<uint32_t>((int64_t{1} << log_n) / (4 * kFftTile)), batch32),
                     dim3(kTileThreads), 0, st, a, reinterpret_cast<const double2*>(slots));
  FH_CHECK_LAUNCH("encode tile stages");
  FH_CODEC_COLUMNS(k_encode_columns, kColThreads, log_n, a, scale, out)
  FH_CHECK_LAUNCH("encode column stages");
  return kOk;
}

FH_API int fh_ckks_lift_montgomery(const int64_t* coefficients, int64_t batch, int64_t limbs, int64_t n,
                                   const void* ntt_rows, int64_t row_start, fh_table2 rns_params, int64_t* out,
                                   void* stream) {
  FH_CHECK_ARG(batch >= 0 && limbs >= 0 && n >= 0 && batch <= 65535 && limbs <= 65535, "bad lift extent");
  if (batch == 0 || limbs == 0 || n == 0) return kOk;
  FH_CHECK_ARG(coefficients && ntt_rows && rns_params.data && out && row_start >= 0, "lift: null operand");
  hipLaunchKernelGGL(k_lift_montgomery,
                     dim3(static_cast<uint32_t>(ceil_div(n, kCodecBlock)), static_cast<uint32_t>(limbs),
                          static_cast<uint32_t>(batch)),
                     dim3(kCodecBlock), 0, static_cast<hipStream_t>(stream), coefficients, n,
                     static_cast<const NttRow*>(ntt_rows) + row_start,
                     ParamView{rns_params.data, rns_params.stride_row, rns_params.stride_col}, limbs, out);
  FH_CHECK_LAUNCH("lift to Montgomery");
  return kOk;
}

FH_API int fh_ckks_decode_rows(const int64_t* residues_a, const int64_t* residues_b, int64_t batch_stride,
                               int64_t batch, int64_t log_n, int64_t modulus_a, int64_t modulus_b,
                               int64_t modulus_a_inverse_mod_b, const int32_t* slot_map, const double* twiddles,
                               double scale, double* workspace, double* slots, void* stream) {
  FH_CHECK_ARG(log_n >= 12 && log_n <= 16, "two-pass decode supports logN 12..16");
  FH_CHECK_ARG(batch >= 1 && batch <= 65535, "bad decode batch");
  FH_CHECK_ARG(residues_a && residues_b && slot_map && twiddles && workspace && slots, "decode: null operand");
  CrtArgs q{residues_a, residues_b, batch_stride, nullptr, nullptr, 0, 0, modulus_a, modulus_b, 0.0, 0.0,
            static_cast<uint64_t>(modulus_a_inverse_mod_b), 0};
  return decode_two_pass(q, batch, log_n, slot_map, twiddles, scale, workspace, slots,
                         static_cast<hipStream_t>(stream));
}

FH_API int fh_ckks_decrypt_decode(fh_view3 c0, fh_view3 c1, int64_t batch, int64_t log_n, int64_t row_start,
                                  const void* ntt_rows, const int64_t* forward_twiddles,
                                  const int64_t* forward_twiddles_shoup, const int64_t* inverse_twiddles,
                                  const int64_t* inverse_twiddles_shoup, const int64_t* secret,
                                  int64_t secret_row_stride, int64_t modulus_a, int64_t modulus_b,
                                  int64_t modulus_a_inverse_mod_b, const int32_t* slot_map, const double* twiddles,
                                  double scale, int64_t* product, double* workspace, double* slots, void* stream) {
  FH_CHECK_ARG(log_n >= 12 && log_n <= 16, "fused decryption supports logN 12..16");
  FH_CHECK_ARG(batch >= 1 && batch <= 32767 && row_start >= 0, "bad decryption batch or row start");
  FH_CHECK_ARG(c0.data && c1.data && ntt_rows && forward_twiddles && forward_twiddles_shoup && inverse_twiddles &&
                   inverse_twiddles_shoup && secret && slot_map && twiddles && product && workspace && slots,
               "decrypt: null operand");
  FH_CHECK_ARG(c1.stride_coef == 1, "decrypt: c1 needs a unit coefficient stride");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t n = int64_t{1} << log_n;
  int rc = ntt::product_internal(product, c1.data, batch, 2, static_cast<int>(log_n), c1.stride_batch, c1.stride_limb,
                                 static_cast<const NttRow*>(ntt_rows), forward_twiddles, forward_twiddles_shoup,
                                 inverse_twiddles, inverse_twiddles_shoup, row_start, secret, secret_row_stride, st);
  if (rc != kOk) return rc;
  CrtArgs q{product + n, product, 2 * n, c0.data + c0.stride_limb, c0.data, c0.stride_batch, c0.stride_coef,
            modulus_a, modulus_b, 0.0, 0.0, static_cast<uint64_t>(modulus_a_inverse_mod_b), 0};
  return decode_two_pass(q, batch, log_n, slot_map, twiddles, scale, workspace, slots, st);
}
