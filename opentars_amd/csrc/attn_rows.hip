// Attention of prompt rows: the per-head triple FDOT_NT (scores) -> causal ROW_SOFTMAX -> FDOT_NN
// (P V) of the reference's lowering (tars_mini/llm.py:736-746) for many query rows, bit for bit.
//
// The contract rounds every product and every sum on its own and fixes the order of the sums, so
// neither an FMA nor a matrix instruction can form the dots. What a matrix instruction can do is
// the products alone: v_mfma_f32_16x16x1_4b_f32 (four 16 x 16 outer products, one k each) on a C of
// -0 returns RN(a * b) of every pair with its sign, subnormals kept (x + -0 = x for every x), while
// the vector ALU adds the products of the step before. The contract's flushes then cost nothing: the
// products are formed with fp32 subnormals kept (MODE denorm = keep, captured when the MFMA
// issues) and added with them flushed (MODE denorm = flush), and a flushing v_add_f32 is exactly
// fadd: it takes ftz(product) and ftz(acc), and flushes the sum (a sum of two fp32 values in the
// subnormal range is exact, so flushing after rounding or before is the same). A flushing multiply
// would not be: a product in [2^-126 - 2^-150, 2^-126) rounds up to a normal value in the contract
// and to zero there. Both facts were checked against numpy on products at the edge of the subnormal
// range, and by the attention tests' planted values. q, K and V elements are flushed on arrival.
// NaN payloads are canonicalized where a value is stored; they reach nothing else.
//
// A workgroup owns 16 query rows of one head, its scores in LDS. Per (query, key) pair the contract
// leaves 2 hd adds (4 cycles of a SIMD per 64 of them): 8208 vector instructions per SIMD for 512 causal
// rows of 16 heads over 512 keys, 14 us, of the 17915 (30 us) that the kernel issues there in 55 us, next to
// 16896 busy cycles of the matrix cores (7 us). The rest is the uneven load of the causal tiles, whose
// workgroups are all resident at once, and a wave left alone on its SIMD at the end.
//  1. scores, 16 keys per tile, tiles dealt to the waves. Block b of the MFMA takes the chains
//     4 b + e of sum16 (element 16 u + 4 b + e in step u), e one after another: lane l holds the 16
//     bytes 64 u + 16 (l / 16) of query row and key row l % 16, so q stays in registers for the
//     whole kernel and a tile's K arrives in hd / 16 loads of 16 rows x 64 bytes. The fold's first two
//     levels join the four e of a block, the last two the blocks: registers only, no lane exchange.
//  2. softmax, 16 lanes per row: the maximum, then exp and the 16-lane sum in one pass, then the
//     products with the reciprocal.
//  3. P V: a wave takes RW rows x 64 columns, keys in order, on v_mfma_f32_4x4x1_16b_f32 (4 rows x 64
//     columns of products; lane = column). V rows come by buffer loads two 16-key blocks ahead, the first
//     before the softmax. Keys past the last one any row of the tile may see are left out of both
//     products: their probabilities are +0, and acc + (+-0) = acc unless acc is -0 or the V element is
//     infinite or NaN; a scan of those V elements and of the sums decides, and the keys run if need be.
//
// Measured on MI355X. f32 MFMA and vector adds do not overlap there: per 64 products and sums 4.5 - 4.8
// cycles of a SIMD with two or more waves (a product by v_mul costs the same 2.4 cycles as its share of
// an MFMA, but needs its operands spread over the lanes), 7.5 - 8 with one wave, which issues a vector
// instruction every 4.9 cycles at best. So the split aims at two waves per SIMD: 8 rows per P V wave (4
// waves at head size 128) when the grid gives more than a workgroup per CU, else 4 rows (8 waves):
// 128 rows of 8 heads over 512 keys 50 -> 45 us with 4; 512 rows of 16 heads, causal, 55 us with 8 and
// 68 us with 4. Steps from the first form (64 columns x 16 rows per P V wave on the 16 x 16 x 1 MFMA,
// 110 us there): 8 rows per wave 75, straight-line softmax 68, buffer loads with scalar row offsets 61
// (64-bit lane addresses cost a quarter-rate add per load), probabilities always from LDS 55.
// One workgroup per head, row by row, took 11.7 ms.
#include <mutex>
#include <type_traits>

#include "kernels.h"
#include "row_sums.h"

namespace tars {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kTile = 16;  // query rows per workgroup, keys per scores tile
constexpr int kKeys = 16;  // keys per block of P V
constexpr int kAhead = 2;  // blocks of V rows in flight
constexpr size_t kLds = 163840;  // LDS of a CU

__device__ __forceinline__ v16f splat(float x) {
  v16f v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = x;
  return v;
}

// the products of one step, in a keep region of their own (b's tie holds the MFMA there)
__device__ __forceinline__ v16f products(float a, float b, const v16f& neg0) {
  keep_denorms();
  tie(b);
  v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, neg0, 0, 0, 0);
  tie(d);
  flush_denorms();
  return d;
}

// RW: query rows per P V wave (4 or 8); the workgroup has 16 / RW * HD / 64 waves
template <int HD, bool VHALF, int RW>
__global__ __launch_bounds__(64 * (16 / RW) * (HD / 64), 2) void attn_rows_kernel(AttnArgs a, int tr, int lds_row,
                                                                                   int tiles) {
  constexpr int U = HD / 16, nw = 16 / RW * (HD / 64);
  extern __shared__ __align__(16) float sp[];  // [tr][lds_row]
  const int t = threadIdx.x, lane = t & 63, l = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // Workgroups are dealt round-robin over the 8 XCDs: with the heads a multiple of 8 each XCD gets
  // heads / 8 consecutive ones, so a K / V head is read through one L2. The last rows first: they see
  // the most keys.
  const int nh = a.heads, b = blockIdx.x, hb = b % nh;
  const int h = nh % 8 == 0 ? (hb % 8) * (nh / 8) + hb / 8 : hb;
  const int m0 = (tiles - 1 - b / nh) * tr;
  const int rows = min(tr, a.M - m0), nk = a.nk;
  const int limit = causal_valid(nk, a.causal_k, m0 + rows - 1);  // keys some row sees
  const bool last = h == nh - 1;
  const int score_keys = last && a.sc ? nk : limit;
  const v16f neg0 = splat(-0.0f);

  // ---- 1. scores
  {
    const float* qrow = frow_f32(a.q[h], a.ldq, m0 + min(l, rows - 1)) + 4 * lg;
    const float* kbase = a.k[h] + 4 * lg;
    float4 q4[U];
#pragma unroll
    for (int u = 0; u < U; ++u) q4[u] = *reinterpret_cast<const float4*>(qrow + 16 * u);
    float q[4][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      q[0][u] = ftz(q4[u].x);
      q[1][u] = ftz(q4[u].y);
      q[2][u] = ftz(q4[u].z);
      q[3][u] = ftz(q4[u].w);
    }
    float4 kn[U];
    auto load = [&](int kt) {
      const float* kr = frow_f32(kbase, a.ldk, min(16 * kt + l, nk - 1));  // past the end: computed and unused
#pragma unroll
      for (int u = 0; u < U; ++u) kn[u] = *reinterpret_cast<const float4*>(kr + 16 * u);
    };
    const int nt = (score_keys + kTile - 1) / kTile;
    // the next tile's K rows arrive during a tile's chains, but at head size 256, whose registers two tiles
    // would not fit
    constexpr bool kPrefetch = HD <= 128;
    if (kPrefetch && wave < nt) load(wave);
    for (int kt = wave; kt < nt; kt += nw) {
      if (!kPrefetch) load(kt);
      float k[4][U];
      flush_denorms();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        k[0][u] = kn[u].x;
        k[1][u] = kn[u].y;
        k[2][u] = kn[u].z;
        k[3][u] = kn[u].w;
#pragma unroll
        for (int e = 0; e < 4; ++e) flush_in_place(k[e][u]);
      }
      if (kPrefetch && kt + nw < nt) load(kt + nw);
      v16f acc, even, part;
      v16f d = products(q[0][0], k[0][0], neg0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          v16f dn;
          if (u + 1 < U) dn = products(q[e][u + 1], k[e][u + 1], neg0);
          else if (e < 3) dn = products(q[e + 1][0], k[e + 1][0], neg0);
          tie(d);
          acc = (u == 0 ? splat(0.0f) : acc) + d;
          tie(acc);
          if (u + 1 < U || e < 3) d = dn;
        }
        // chain end: (c0 + c1) + (c2 + c3)
        if (e == 0) even = acc;
        else if (e == 1) part = even + acc;
        else if (e == 2) even = acc;
        else part = part + (even + acc);
        if (e & 1) tie(part);
      }
      float sv[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {  // the blocks: (B0 + B1) + (B2 + B3)
        sv[v] = (part[v] + part[4 + v]) + (part[8 + v] + part[12 + v]);
        tie(sv[v]);
      }
      keep_denorms();
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 4 * lg + v, j = 16 * kt + l;
        if (r < tr) sp[r * lds_row + j] = sv[v];
        if (last && a.sc && r < rows && j < nk)
          *reinterpret_cast<float*>(reinterpret_cast<char*>(a.sc) + (m0 + r) * a.ldsc + 4 * j) = canon(sv[v]);
      }
    }
  }
  // ---- P V operands: RW rows x 64 columns per wave
  constexpr int NC = HD / 64, ES = VHALF ? 2 : 4, H4 = RW / 4;
  const int cg = wave % NC, r0 = wave / NC * RW;
  const int pad = (limit + 15) / 16 * 16;  // P V runs over whole blocks of 16 keys
  const char* vcol = static_cast<const char*>(a.v[h]) + 64 * ES * cg;
  // V elements (as stored) of keys j0 .. j0 + kKeys - 1 (j0 < nk); past the matrix the last row's again
  struct Keys {
    uint32_t v[kKeys];
  };
  const int ldv = static_cast<int>(a.ldv);
  auto load = [&](Keys& o, int j0) __attribute__((always_inline)) {
    // buffer loads: the block's base in the resource, the row's offset scalar, the lane's column in a VGPR
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vcol) + static_cast<int64_t>(j0) * a.ldv, 0,
                                                        -1, 0x00027000);
    const int left = nk - 1 - j0;
#pragma unroll
    for (int i = 0; i < kKeys; ++i) {
      const int row = min(i, left) * ldv;
      if constexpr (VHALF) o.v[i] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, ES * lane, row, 0);
      else o.v[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, ES * lane, row, 0);
    }
  };
  // the first blocks' V rows, in flight while the softmax runs
  Keys vq[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) load(vq[i], min(i * kKeys, nk - 1));
  __syncthreads();

  // ---- 2. softmax: 16 lanes per row
  for (int r = t >> 4; r < tr; r += 4 * nw) {
    float* s = sp + r * lds_row;
    const int m = m0 + min(r, rows - 1);
    const int V = causal_valid(nk, a.causal_k, m);
    // the lane's n elements l, l + 16, ... of the row, eight at a time (their chains of steps side by side)
    const int n = pad >> 4;
    auto each = [&](auto&& f) {
      int i = 0;
      for (; i + 8 <= n; i += 8) f(i, std::integral_constant<int, 8>{});
      for (; i < n; ++i) f(i, std::integral_constant<int, 1>{});
    };
    uint32_t key = 0;
    each([&](int i0, auto size) {
      constexpr int B = decltype(size)::value;
      float x[B];
#pragma unroll
      for (int i = 0; i < B; ++i) x[i] = s[l + 16 * (i0 + i)];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const uint32_t k = is_nan(x[i]) ? 0xFFFFFFFFu : fmax_key(x[i]);
        key = l + 16 * (i0 + i) < V ? max(key, k) : key;
      }
    });
    key = static_cast<uint32_t>(group_reduce<16>(static_cast<int>(key), OpMaxU{}));
    const float nmx = fneg(key == 0xFFFFFFFFu ? ffrom(kCanonNaN) : fmax_from_key(key));
    // exp values are 0, normal, infinite or NaN, so their plain sums are the contract's
    float acc = 0.0f;
    each([&](int i0, auto size) {
      constexpr int B = decltype(size)::value;
      float x[B];
#pragma unroll
      for (int i = 0; i < B; ++i) x[i] = s[l + 16 * (i0 + i)];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const float e = exp_f(fadd(x[i], nmx));
        x[i] = l + 16 * (i0 + i) < V ? e : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < B; ++i) acc = __fadd_rn(acc, x[i]);
#pragma unroll
      for (int i = 0; i < B; ++i) s[l + 16 * (i0 + i)] = x[i];
    });
    const float inv = recip_f(fold16(acc));
    const float zero = fmul(0.0f, inv);  // a masked probability: +0 (NaN when the row's sum is)
    float* prow = last && a.pr && r < rows
                      ? reinterpret_cast<float*>(reinterpret_cast<char*>(a.pr) + (m0 + r) * a.ldpr) : nullptr;
    each([&](int i0, auto size) {
      constexpr int B = decltype(size)::value;
      float x[B];
#pragma unroll
      for (int i = 0; i < B; ++i) x[i] = s[l + 16 * (i0 + i)];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int j = l + 16 * (i0 + i);
        const float p = fmul(x[i], inv);
        // past the matrix: -0, whose product with the +0 standing in for V leaves every sum as it is
        s[j] = j < nk ? p : -0.0f;
        if (prow && j < nk) prow[j] = p;
      }
    });
    if (prow)
      for (int j = pad + l; j < nk; j += 16) prow[j] = zero;
  }
  __syncthreads();

  // ---- 3. P V
  if (r0 >= rows) return;
  // MFMA h (h < H4) takes rows r0 + 4 h .. + 3; its lane's operand row (a row past tr is clamped, unstored)
  const float* prow[H4];
#pragma unroll
  for (int i = 0; i < H4; ++i) prow[i] = sp + min(r0 + 4 * i + (lane & 3), tr - 1) * lds_row;
  v4f acc[H4];
#pragma unroll
  for (int i = 0; i < H4; ++i) acc[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const v4f n0 = {-0.0f, -0.0f, -0.0f, -0.0f};
  // kKeys keys from j on: their V rows in o (refilled with the block kAhead on when that is before j1), their
  // probabilities from LDS. Four keys' products are formed while the four before are added.
  auto block = [&](Keys& o, int j, int j1) __attribute__((always_inline)) {
      float v[kKeys];
      float4 p[H4][kKeys / 4];
#pragma unroll
      for (int i = 0; i < H4; ++i)
#pragma unroll
        for (int c = 0; c < kKeys / 4; ++c)
          p[i][c] = *reinterpret_cast<const float4*>(prow[i] + j + 4 * c);
      flush_denorms();
#pragma unroll
      for (int i = 0; i < kKeys; ++i) {
        v[i] = VHALF ? fp16_to_f32_keep_nan(o.v[i]) : ffrom(o.v[i]);
        if constexpr (!VHALF) flush_in_place(v[i]);
      }
      if (j + kKeys > nk) {
#pragma unroll
        for (int i = 0; i < kKeys; ++i) v[i] = j + i < nk ? v[i] : 0.0f;
      }
      if (j + kAhead * kKeys < j1) load(o, j + kAhead * kKeys);
      auto quad = [&](v4f (&d)[4][H4], int c) __attribute__((always_inline)) {
        keep_denorms();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          tie(v[4 * c + k]);
#pragma unroll
          for (int i = 0; i < H4; ++i) {
            const float4 q = p[i][c];
            d[k][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w, v[4 * c + k], n0,
                                                         0, 0, 0);
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int i = 0; i < H4; ++i) tie(d[k][i]);
        flush_denorms();
      };
      v4f d[2][4][H4];
      quad(d[0], 0);
#pragma unroll
      for (int c = 0; c < kKeys / 4; ++c) {
        if (c + 1 < kKeys / 4) quad(d[(c + 1) & 1], c + 1);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
          for (int i = 0; i < H4; ++i) {
            tie(d[c & 1][k][i]);
            acc[i] = acc[i] + d[c & 1][k][i];
          }
        }
#pragma unroll
        for (int i = 0; i < H4; ++i) tie(acc[i]);
      }
  };
  // the keys some row sees; then, if they can change a sum (see the file notes), the masked ones
  for (int j0 = 0, j1 = pad;; j0 = pad, j1 = (nk + kKeys - 1) / kKeys * kKeys) {
    for (int j = j0; j < j1; j += kAhead * kKeys) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
        if (j + i * kKeys < j1) block(vq[i], j + i * kKeys, j1);
    }
    keep_denorms();
    if (j1 >= nk) break;
    bool need = false;
#pragma unroll
    for (int i = 0; i < H4; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float x = acc[i][v];
        need |= fbits(x) == kSign;
      }
    constexpr int LPR = 64 * ES / 16;  // lanes per 64-column row piece
    for (int js = pad + lane / LPR; js < nk; js += 4 * (64 / LPR)) {
      uint4 w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = *reinterpret_cast<const uint4*>(vcol + static_cast<int64_t>(min(js + i * (64 / LPR), nk - 1)) * a.ldv +
                                               16 * (lane % LPR));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t x[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if constexpr (VHALF) need |= (x[c] & 0x7C00u) == 0x7C00u || (x[c] & 0x7C000000u) == 0x7C000000u;
          else need |= (x[c] & kExpo) == kExpo;
        }
      }
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(need) == 0, 1)) break;
    // their probabilities into this wave's rows (the waves of a row write the same values): +0, -0 past the matrix
    for (int r = r0; r < min(r0 + RW, tr); ++r)
      for (int j = pad + lane; j < (nk + kKeys - 1) / kKeys * kKeys; j += 64) sp[r * lds_row + j] = j < nk ? 0.0f : -0.0f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load(vq[i], min(pad + i * kKeys, nk - 1));
  }
#pragma unroll
  for (int i = 0; i < H4; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = r0 + 4 * i + v;
      const float y = acc[i][v];
      if (r < rows) store_out(a.att[h], (m0 + r) * a.ldatt, 64 * cg + lane, a.out, chain_end(y), a.out_scale);
    }
}

// More than 64 KiB of dynamic LDS is asked for once per device and instance.
template <int HD, bool VHALF, int RW>
hipError_t go(const AttnArgs& a, int tr, int lds_row, hipStream_t s) {
  static std::mutex mu;
  static bool ready[64] = {};
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!ready[dev]) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_rows_kernel<HD, VHALF, RW>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
      if (e != hipSuccess) return e;
      ready[dev] = true;
    }
  }
  const int tiles = (a.M + tr - 1) / tr;
  hipLaunchKernelGGL((attn_rows_kernel<HD, VHALF, RW>), dim3(static_cast<unsigned>(tiles) * a.heads),
                     dim3(64 * (16 / RW) * (HD / 64)), static_cast<size_t>(4) * tr * lds_row, s, a, tr, lds_row, tiles);
  return hipGetLastError();
}

template <bool VHALF>
hipError_t rows(const AttnArgs& a, hipStream_t s) {
  // row pitch 4 * odd: an MFMA operand read (16-byte pieces of several rows) and a scores store touch
  // every bank once; 16 rows per workgroup while they fit, else 8
  const int lds_row = (a.nk + 15) / 16 * 16 + 4;
  const int tr = static_cast<size_t>(64) * lds_row <= kLds ? 16 : 8;
  if (a.hd == 64) return go<64, VHALF, 4>(a, tr, lds_row, s);
  if (a.hd == 256) return go<256, VHALF, 8>(a, tr, lds_row, s);
  const bool few = static_cast<int64_t>((a.M + tr - 1) / tr) * a.heads <= 256;
  return few ? go<128, VHALF, 4>(a, tr, lds_row, s) : go<128, VHALF, 8>(a, tr, lds_row, s);
}

}  // namespace

hipError_t launch_attention_rows(const AttnArgs& a, hipStream_t s) {
  return a.v_fp16 ? rows<true>(a, s) : rows<false>(a, s);
}

}  // namespace tars
