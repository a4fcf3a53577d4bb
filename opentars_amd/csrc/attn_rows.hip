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
// A workgroup owns 16 query rows of one head, its scores in LDS. Per (query, key) pair that is 2 hd
// adds (4 cycles per 64 of them), which bounds the kernel; the MFMAs run beside them.
//  1. scores, 16 keys per tile, tiles dealt to the waves. Block b of the MFMA takes the chains
//     4 b + e of sum16 (element 16 u + 4 b + e in step u), e one after another: lane l holds the 16
//     bytes 64 u + 16 (l / 16) of query row and key row l % 16, so q stays in registers for the
//     whole kernel and a tile's K arrives in hd / 16 loads of 16 rows x 64 bytes. The fold's first two
//     levels join the four e of a block, the last two the blocks: registers only, no lane exchange.
//  2. softmax, 16 lanes per row: the maximum, then exp and the 16-lane sum in one pass, then the
//     products with the reciprocal.
//  3. P V: wave w takes output columns 64 w .. + 63 (block b columns 16 b .. + 15), keys in order.
//     Keys past the last one any row of the tile may see are left out of both products: their
//     probabilities are +0, and acc + (+-0) = acc unless acc is -0 or the V element is infinite or
//     NaN; a scan of those V elements and of the sums decides, and the keys run if need be.
#include <mutex>

#include "kernels.h"
#include "row_sums.h"

namespace tars {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kTile = 16;  // query rows per workgroup, keys per scores tile

// fp32 subnormals kept / flushed (MODE bits 4-5) from here on. The values an instruction of a region
// takes or gives pass through tie() inside it: the compiler keeps volatile statements in order, so
// it cannot move the instruction out of its region. Between kernels' phases the mode is "keep", the
// one the rest of the library is compiled for.
__device__ __forceinline__ void keep_denorms() { __builtin_amdgcn_s_setreg(1 | (4 << 6) | (1 << 11), 3); }
__device__ __forceinline__ void flush_denorms() { __builtin_amdgcn_s_setreg(1 | (4 << 6) | (1 << 11), 0); }
template <class T>
__device__ __forceinline__ void tie(T& x) {
  asm volatile("" : "+v"(x));
}
// ftz in a flush region (a maximum flushes its operands)
__device__ __forceinline__ void flush_in_place(float& x) { asm volatile("v_max_f32 %0, %0, %0" : "+v"(x)); }

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

template <int HD, bool VHALF>
__global__ __launch_bounds__(256, HD == 256 ? 1 : 2) void attn_rows_kernel(AttnArgs a, int tr, int lds_row, int tiles) {
  constexpr int U = HD / 16, NWV = HD / 64;
  extern __shared__ __align__(16) float sp[];  // [tr][lds_row]
  const int t = threadIdx.x, lane = t & 63, l = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), nw = blockDim.x >> 6;
  // Workgroups are dealt round-robin over the 8 XCDs: with the heads a multiple of 8 each XCD gets
  // heads / 8 consecutive ones, so a K / V head is read through one L2. The last rows first: they see
  // the most keys.
  const int nh = a.heads, b = blockIdx.x, hb = b % nh;
  const int h = nh % 8 == 0 ? (hb % 8) * (nh / 8) + hb / 8 : hb;
  const int m0 = (tiles - 1 - b / nh) * tr;
  const int rows = min(tr, a.M - m0), nk = a.nk;
  const int limit = a.causal_k > 0 ? min(nk, a.causal_k + m0 + rows - 1) : nk;  // keys some row sees
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
    if (wave < nt) load(wave);
    for (int kt = wave; kt < nt; kt += nw) {
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
      if (kt + nw < nt) load(kt + nw);  // in flight during this tile's chains
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
  __syncthreads();

  // ---- 2. softmax: 16 lanes per row
  const int pad = (limit + 15) / 16 * 16;  // P V runs over whole blocks of 16 keys
  for (int r = t >> 4; r < tr; r += blockDim.x >> 4) {
    float* s = sp + r * lds_row;
    const int m = m0 + min(r, rows - 1);
    const int V = a.causal_k > 0 ? min(nk, a.causal_k + m) : nk;
    uint32_t key = 0;
    for (int j0 = l; j0 < V; j0 += 128) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = s[min(j0 + 16 * i, V - 1)];  // a repeat changes no maximum
#pragma unroll
      for (int i = 0; i < 8; ++i) key = max(key, is_nan(x[i]) ? 0xFFFFFFFFu : fmax_key(x[i]));
    }
    key = static_cast<uint32_t>(group_reduce<16>(static_cast<int>(key), OpMaxU{}));
    const float nmx = fneg(key == 0xFFFFFFFFu ? ffrom(kCanonNaN) : fmax_from_key(key));
    // exp values are 0, normal, infinite or NaN, so their plain sums are the contract's
    float acc = 0.0f;
    for (int j0 = l; j0 < pad; j0 += 64) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = s[min(j0 + 16 * i, pad - 1)];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + 16 * i;
        x[i] = j < V ? exp_f(fadd(x[i], nmx)) : 0.0f;
        acc = __fadd_rn(acc, x[i]);
        if (j < pad) s[j] = x[i];
      }
    }
    const float inv = recip_f(fold16(acc));
    const float zero = fmul(0.0f, inv);  // a masked probability: +0 (NaN when the row's sum is)
    float* prow = last && a.pr && r < rows
                      ? reinterpret_cast<float*>(reinterpret_cast<char*>(a.pr) + (m0 + r) * a.ldpr) : nullptr;
    for (int j0 = l; j0 < pad; j0 += 64) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = s[min(j0 + 16 * i, pad - 1)];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + 16 * i;
        const float p = fmul(x[i], inv);
        // past the matrix: -0, whose product with the +0 standing in for V leaves every sum as it is
        if (j < pad) s[j] = j < nk ? p : -0.0f;
        if (prow && j < min(pad, nk)) prow[j] = p;
      }
    }
    if (prow)
      for (int j = pad + l; j < nk; j += 16) prow[j] = zero;
  }
  __syncthreads();

  // ---- 3. P V: 64 columns per wave
  if (wave >= NWV) return;
  constexpr int ES = VHALF ? 2 : 4;
  const char* vcol = static_cast<const char*>(a.v[h]) + 64 * ES * wave;
  const float* prow = sp + min(l, tr - 1) * lds_row;
  struct Block {
    uint32_t v[16];  // V elements as stored
    float4 p[4];
  };
  auto load = [&](Block& o, int j0, bool probs) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const char* p = vcol + static_cast<int64_t>(min(j0 + i, nk - 1)) * a.ldv + ES * lane;
      if constexpr (VHALF) o.v[i] = *reinterpret_cast<const uint16_t*>(p);
      else o.v[i] = *reinterpret_cast<const uint32_t*>(p);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (probs) o.p[i] = *reinterpret_cast<const float4*>(prow + j0 + 4 * i);
      else  // masked keys: probability +0 (-0 past the matrix)
        o.p[i] = make_float4(j0 + 4 * i < nk ? 0.0f : -0.0f, j0 + 4 * i + 1 < nk ? 0.0f : -0.0f,
                             j0 + 4 * i + 2 < nk ? 0.0f : -0.0f, j0 + 4 * i + 3 < nk ? 0.0f : -0.0f);
    }
  };
  v16f acc = splat(0.0f);
  // keys [j0, j1) (multiples of 16), the next block's V rows and probabilities loaded during a block's steps
  auto chains = [&](int j0, int j1, bool probs) {
    Block nxt;
    load(nxt, j0, probs);
    for (int j = j0; j < j1; j += 16) {
      float v[16], p[16];
      flush_denorms();
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        v[i] = VHALF ? fp16_to_f32_keep_nan(nxt.v[i]) : ffrom(nxt.v[i]);
        if constexpr (!VHALF) flush_in_place(v[i]);
      }
      if (j + 16 > nk) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = j + i < nk ? v[i] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) p[4 * i] = nxt.p[i].x, p[4 * i + 1] = nxt.p[i].y, p[4 * i + 2] = nxt.p[i].z, p[4 * i + 3] = nxt.p[i].w;
      if (j + 16 < j1) load(nxt, j + 16, probs);
      v16f d = products(p[0], v[0], neg0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        v16f dn;
        if (i + 1 < 16) dn = products(p[i + 1], v[i + 1], neg0);
        tie(d);
        acc = acc + d;
        tie(acc);
        if (i + 1 < 16) d = dn;
      }
    }
    keep_denorms();
  };
  chains(0, pad, true);
  if (pad < nk) {  // masked keys of every row (see the file notes)
    bool need = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float x = acc[i];
      need |= fbits(x) == kSign;
    }
    constexpr int LPR = 64 * ES / 16;  // lanes per 64-column row piece
    for (int j0 = pad + lane / LPR; j0 < nk; j0 += 4 * (64 / LPR)) {
      uint4 w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = *reinterpret_cast<const uint4*>(vcol + static_cast<int64_t>(min(j0 + i * (64 / LPR), nk - 1)) * a.ldv +
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
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(need) != 0, 0)) chains(pad, (nk + 15) / 16 * 16, false);
  }
#pragma unroll
  for (int blk = 0; blk < 4; ++blk)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 4 * lg + v;
      const float y = acc[4 * blk + v];
      if (r < rows) store_out(a.att[h], (m0 + r) * a.ldatt, 64 * wave + 16 * blk + l, a.out, chain_end(y), a.out_scale);
    }
}

// More than 64 KiB of dynamic LDS is asked for once per device and instance.
template <int HD, bool VHALF>
hipError_t go(const AttnArgs& a, hipStream_t s) {
  constexpr size_t kLds = 163840;
  static std::mutex mu;
  static bool ready[64] = {};
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!ready[dev]) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_rows_kernel<HD, VHALF>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
      if (e != hipSuccess) return e;
      ready[dev] = true;
    }
  }
  // row pitch 4 * odd: an MFMA operand read (16 rows x 16 bytes) and a scores store touch every
  // bank once; 16 rows per workgroup while they fit, else 8
  const int lds_row = (a.nk + 15) / 16 * 16 + 4;
  const int tr = static_cast<size_t>(64) * lds_row <= kLds ? 16 : 8;
  const size_t lds = static_cast<size_t>(4) * tr * lds_row;
  const int tiles = (a.M + tr - 1) / tr;
  // 4 waves (a wave per SIMD) where LDS leaves at most two workgroups per CU, else the P V waves alone
  const int nw = kLds / lds <= 2 ? 4 : (HD / 64 > 2 ? HD / 64 : 2);
  hipLaunchKernelGGL((attn_rows_kernel<HD, VHALF>), dim3(static_cast<unsigned>(tiles) * a.heads), dim3(64 * nw), lds, s, a, tr,
                     lds_row, tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_attention_rows(const AttnArgs& a, hipStream_t s) {
  if (a.hd == 64) return a.v_fp16 ? go<64, true>(a, s) : go<64, false>(a, s);
  if (a.hd == 128) return a.v_fp16 ? go<128, true>(a, s) : go<128, false>(a, s);
  return a.v_fp16 ? go<256, true>(a, s) : go<256, false>(a, s);
}

}  // namespace tars
