// Float32 prefill on the matrix cores (attn_f32.hpp has the decode side).
//
// fp32 MFMA (v_mfma_f32_32x32x2_f32, 256 FLOP per cycle per CU) computes both
// products in fp32 end to end.  On the vector ALUs every key row cost a
// column D/4 lanes' products plus log2(D/4) cross-lane sums: one sequence of
// 512 tokens, 32/8 heads, head_dim 64 (1.08 GFLOP) took 113.8 us at 9.5
// TFLOP/s; here 19.1 us.
//
// A work-group covers 32 columns, (query row, query head) pairs of one KV
// head in row-major order, so a causal group of G = 4 spans 8 rows.  Its 4
// waves take every fourth 32-key tile and merge their softmax states through
// LDS: 512 tokens at 8 KV heads are then 512 groups and the longest chain is
// 4 tiles, where one wave per 32 columns would leave half of the SIMDs idle
// behind a chain of 16.  Per tile a wave computes S^T = K Q^T (keys as rows,
// columns as columns) and O^T += V^T P^T, whose B operand is S^T's output
// register by register, so P never moves; K, V and q come straight from
// memory in operand order (the contraction index and the dimension order of
// an MFMA tile are free, so every load is 16 bytes or a whole row).  K of the
// next tile and V of this one are in flight under S^T's MFMAs; at head_dim 128
// and 256 the registers hold a quarter or an eighth of each twice, loaded that
// much ahead (two waves per SIMD up to 128).
#include "attn_f32.hpp"
#include "host_util.hpp"

namespace sia {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// x of lanes l and l ^ 32
__device__ __forceinline__ void halves(float x, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                 false, false);
  lo = __builtin_bit_cast(float, (uint32_t)r[0]);
  hi = __builtin_bit_cast(float, (uint32_t)r[1]);
}

// Dimension held by element e of row r (0..31) of the O^T tiles, and the V
// elements lane r loads per key: [ET r, + ET) up to head_dim 128, pieces of 4
// at [4 r] and [128 + 4 r] at 256.  (head_dim 16: rows past 15 are zero.)
template <int D>
__device__ __forceinline__ int f32_dim(int r, int e) {
  constexpr int ET = D < 32 ? 1 : D / 32;
  return ET <= 4 ? ET * r + e : 128 * (e >> 2) + 4 * r + (e & 3);
}

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1)))
void attn_f32_prefill(const F32Args a) {
  constexpr int ET = D < 32 ? 1 : D / 32;       // 32-dimension tiles of O^T
  constexpr int KQ = D / 8;                      // 16-byte pieces of a row per half wave
  constexpr bool kAhead = D <= 32;               // whole tiles of K and V in flight (else parts of them)
  __shared__ float sm_o[2][16 * ET][64];
  __shared__ float sm_m[4][32], sm_l[4][32];
  __shared__ f32x4 sm_q[kAhead ? 1 : KQ][64];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  // heaviest (last) columns first; the groups of one (b, KV head) are a
  // multiple of B Hkv apart, so with 8 KV heads each XCD's L2 serves its own.
  // A grid of one to two groups per CU is resident at once: its second half
  // runs lightest first, so that every CU holds a heavy and a light group.
  const int bhn = a.B * a.Hkv;
  const int lin = a.fold && (int)blockIdx.x >= a.fold ? a.fold + (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
  const int ck = lin / bhn;
  const int bh = lin - ck * bhn;
  const int chunk = a.nchunk - 1 - ck;
  const int b = bh / a.Hkv, hkv = bh - b * a.Hkv;
  const int col = chunk * kF32TileCols + l32;
  const bool live = col < a.ncol;
  const int i = live ? col / a.G : 0, g = live ? col - i * a.G : 0;
  const int off = a.Tk - a.Tq + 1;               // keys visible to row 0 under the causal mask
  const int lim = !live ? 0 : a.causal ? max(0, min(a.Tk, off + i)) : a.Tk;
  const int i_last = uniform(min(chunk * kF32TileCols + kF32TileCols - 1, a.ncol - 1) / a.G);
  const int hi = a.causal ? max(0, min(a.Tk, off + i_last)) : a.Tk;   // keys of the group's last column
  const int lim0 = a.causal ? min(a.Tk, off + uniform(chunk * kF32TileCols / a.G)) : a.Tk;   // of its first one

  const char* qp = a.q + b * a.q_sb + (int64_t)(hkv * a.G + g) * a.q_sh + (int64_t)i * a.q_sm + 16 * h;
  // q operand: column l32, dims 8 j + 4 h + [0, 4) of piece j (dead columns
  // read column 0; never stored).  The 4 waves share it: from head_dim 64 on
  // it sits in LDS, read piece by piece (16 bytes per 4 MFMAs), which leaves
  // the registers to the accumulators.
  f32x4 q[kAhead ? KQ : 1];
  if constexpr (kAhead) {
#pragma unroll
    for (int j = 0; j < KQ; ++j) q[j] = *(const f32x4*)(qp + 32 * j);
  } else {
#pragma unroll
    for (int j = 0; j < KQ / 4; ++j) sm_q[wave * (KQ / 4) + j][lane] = *(const f32x4*)(qp + 32 * (wave * (KQ / 4) + j));
    __syncthreads();
  }
  const char* kb = a.k + b * a.k_s0 + (int64_t)hkv * a.k_sh + 16 * h;
  const char* vb = a.v + b * a.v_s0 + (int64_t)hkv * a.v_sh;

  // K operand of tile t: key row l32, dims 8 j + 4 h + [0, 4) (rows past the
  // last key read it again: their scores are masked); pieces [j0, j0 + n)
  auto load_k = [&](int t, f32x4* k, int j0, int n) {
    const char* kp = kb + (int64_t)min(t * 32 + l32, hi - 1) * a.k_sn;
#pragma unroll
    for (int j = 0; j < n; ++j) k[j] = *(const f32x4*)(kp + 32 * (j0 + j));
  };
  // V operand of tile t: for S^T register j, key 8 (j / 4) + 4 h + j % 4 of
  // the tile, EP of the ET dimensions of row l32; registers [j0, j0 + n), dimensions from e0 on
  // (past the last key: that row of the tile again, with zero weights)
  constexpr int EP = ET < 4 ? ET : 4;            // 32-dimension tiles per V load
  auto load_v1 = [&](int key, float* x, int e0) {
    const char* vp = vb + (int64_t)key * a.v_sn + 4 * f32_dim<D>(D < 32 ? l32 & (D - 1) : l32, e0);
    if constexpr (EP == 1) {
      x[0] = *(const float*)vp;
    } else if constexpr (EP == 2) {
      const f32x2 y = *(const f32x2*)vp;
      x[0] = y[0]; x[1] = y[1];
    } else {
      const f32x4 y = *(const f32x4*)vp;
      x[0] = y[0]; x[1] = y[1]; x[2] = y[2]; x[3] = y[3];
    }
  };
  auto load_v = [&](int t, float (*v)[EP], int j0, int n, int e0) {
#pragma unroll
    for (int j = 0; j < n; ++j)
      load_v1(min(t * 32 + 8 * ((j0 + j) >> 2) + 4 * h + ((j0 + j) & 3), hi - 1), v[j], e0);
  };

  f32x16 o[ET];
#pragma unroll
  for (int e = 0; e < ET; ++e) o[e] = f32x16{};
  float m = -INFINITY, l = 0.f;
  // scores of tile t to weights, (m, l, o) brought to the new max
  auto softmax = [&](int t, f32x16& s) {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int key = t * 32 + 8 * (j >> 2) + 4 * h + (j & 3);
      s[j] = key < lim ? s[j] : -INFINITY;
      mx = fmaxf(mx, s[j]);
    }
    float lo, up;
    halves(mx, lo, up);
    const float M = fmaxf(m, fmaxf(lo, up) * a.qk_scale);
    const float mu = M == -INFINITY ? 0.f : M;     // nothing visible yet
    const float alpha = fast_exp2(m - mu);
    float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      s[j] = fast_exp2(__builtin_fmaf(s[j], a.qk_scale, -mu));
      ps[j & 3] += s[j];
    }
    l = l * alpha + ((ps[0] + ps[1]) + (ps[2] + ps[3]));
    m = M;
#pragma unroll
    for (int e = 0; e < ET; ++e) o[e] *= alpha;
  };
  // S^T over pieces [j0, j0 + N) of the rows: 4 dimensions (2 MFMAs) at a time
  // from zero, added up in a tree
  auto qk = [&](const f32x4* k, int j0, auto nn) {
    constexpr int N = 2 * decltype(nn)::value;
    f32x16 part[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const f32x4 qj = kAhead ? q[kAhead ? j0 + j / 2 : 0] : sm_q[kAhead ? 0 : j0 + j / 2][lane];
      const int e = 2 * (j & 1);
      part[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[j / 2][e], qj[e], f32x16{}, 0, 0, 0);
      part[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[j / 2][e + 1], qj[e + 1], part[j], 0, 0, 0);
      // (finished pairs are added at once: few parts are live)
#pragma unroll
      for (int w = 1; w < N; w *= 2) {
        if ((j + 1) % (2 * w) != 0) break;
        part[j + 1 - 2 * w] += part[j + 1 - w];
      }
    }
    return part[0];
  };
  // O^T over registers [j0, j0 + n) of the weights, one key at a time, each
  // column taking only the keys that it sees
  auto pv_each = [&](int t, int j0, int n, int e0, const f32x16& s) {
    for (int q = 0; q < 2 * n; ++q) {
      const int jr = j0 + (q >> 1), key = t * 32 + 8 * (jr >> 2) + 4 * (q & 1) + (jr & 3);
      if (key >= hi) continue;
      float p = 0.f, x[EP], lo, up;
#pragma unroll
      for (int j = 0; j < 16; ++j) p = j == jr ? s[j] : p;
      halves(p, lo, up);
      p = q & 1 ? up : lo;
      load_v1(key, x, e0);
#pragma unroll
      for (int e = 0; e < EP; ++e) {
        const f32x16 part = __builtin_amdgcn_mfma_f32_32x32x2f32(h == 0 ? x[e] : 0.f, h == 0 ? p : 0.f, f32x16{}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 16; ++j) o[e0 + e][j] += key < lim ? part[j] : 0.f;
      }
    }
  };
  // The same: 8 keys (4 MFMAs) from zero, two such sums (one from head_dim 128
  // on) added to O together.  (One by one, the error of 37 rows over 1500 keys
  // was 2.0-2.1e-7 of the result up to head_dim 64, now 1.9e-7.)  In a tile
  // with keys that not every column sees (they weigh 0), values that are not
  // finite go one key at a time, as 0 times those is NaN: so a hidden key's
  // never reach a column, whichever columns share the group.
  auto pv = [&](const float (*v)[EP], int t, int j0, int n, int e0, const f32x16& s, auto check) {
    if (decltype(check)::value && t * 32 + 31 >= lim0) {
      float z[4] = {0.f, 0.f, 0.f, 0.f};               // (0 x Inf and 0 x NaN are NaN, and stay)
#pragma unroll
      for (int j = 0; j < n; ++j)
#pragma unroll
        for (int e = 0; e < EP; ++e) z[(j * EP + e) & 3] = __builtin_fmaf(v[j][e], 0.f, z[(j * EP + e) & 3]);
      const float any = (z[0] + z[1]) + (z[2] + z[3]);
      if (__any(any != any)) {
        pv_each(t, j0, n, e0, s);
        return;
      }
    }
#pragma unroll
    for (int j = 0; j < n; j += 8)
#pragma unroll
      for (int e = 0; e < EP; ++e) {
        f32x16 part[2] = {f32x16{}, f32x16{}};
#pragma unroll
        for (int i2 = 0; i2 < min(8, n); ++i2)
          part[i2 >> 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[j + i2][e], s[j0 + j + i2], part[i2 >> 2], 0, 0, 0);
        o[e0 + e] += n > 4 ? part[0] + part[1] : part[0];
      }
  };
  if constexpr (kAhead) {
    auto tile = [&](int t, const f32x4* k, f32x4* knext) {
      float v[16][EP];
      load_v(t, v, 0, 16, 0);
      if ((t + 4) * 32 < hi) load_k(t + 4, knext, 0, KQ);
      f32x16 s = qk(k, 0, std::integral_constant<int, KQ>{});
      softmax(t, s);
      pv(v, t, 0, 16, 0, s, std::true_type{});
    };
    f32x4 ka[KQ], kn[KQ];
    int t = wave;
    if (t * 32 < hi) load_k(t, ka, 0, KQ);
    for (; t * 32 < hi; t += 8) {
      tile(t, ka, kn);
      if ((t + 4) * 32 < hi) tile(t + 4, kn, ka);
    }
  } else {
    constexpr int NC = D <= 128 ? D / 32 : 4;      // K and V in NC parts
    constexpr int KC = KQ / NC, VC = 16 / NC;      // K pieces and V registers per part
    constexpr int NH = ET / EP, NV = NC * NH;      // V parts: VC registers, EP tiles of dimensions
    f32x4 k[2][KC];
    float v[2][VC][EP];
    if (wave * 32 < hi) load_k(wave, k[0], 0, KC);
    auto tile = [&](int t, auto check) {
      f32x16 s;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (c < NC - 1) load_k(t, k[(c + 1) & 1], (c + 1) * KC, KC);
        else load_v(t, v[0], 0, VC, 0);
        __builtin_amdgcn_sched_barrier(0);
        {
          const f32x16 part = qk(k[c & 1], c * KC, std::integral_constant<int, KC>{});
          if (c == 0) s = part;
          else s += part;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      softmax(t, s);
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        if (c < NV - 1) load_v(t, v[(c + 1) & 1], VC * ((c + 1) / NH), VC, EP * ((c + 1) % NH));
        else load_k(t + 4, k[0], 0, KC);           // (past the last tile: the last key again, unused)
        __builtin_amdgcn_sched_barrier(0);
        pv(v[c & 1], t, VC * (c / NH), VC, EP * (c % NH), s, check);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int t = wave;
    for (; t * 32 + 31 < lim0; t += 4) tile(t, std::false_type{});   // (with the check 2-4% slower from 512 tokens on)
    for (; t * 32 < hi; t += 4) tile(t, std::true_type{});
  }

  // merge the 4 waves: every state scaled to the common max, then added
  float lo, up;
  halves(l, lo, up);
  l = lo + up;
  if (h == 0) {
    sm_m[wave][l32] = m;
    sm_l[wave][l32] = l;
  }
  __syncthreads();
  float M = sm_m[0][l32];
#pragma unroll
  for (int w = 1; w < 4; ++w) M = fmaxf(M, sm_m[w][l32]);
  const float mu = M == -INFINITY ? 0.f : M;
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) L += sm_l[w][l32] * fast_exp2(sm_m[w][l32] - mu);
  const float wt = fast_exp2(m - mu);
#pragma unroll
  for (int e = 0; e < ET; ++e) o[e] *= wt;
  auto put = [&](float (*dst)[64]) {
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int e = 0; e < ET; ++e) dst[j * ET + e][lane] = o[e][j];
  };
  auto add = [&](float (*src)[64]) {
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int e = 0; e < ET; ++e) o[e][j] += src[j * ET + e][lane];
  };
  if (wave >= 2) put(sm_o[wave - 2]);
  __syncthreads();
  if (wave < 2) add(sm_o[wave]);
  if (wave == 1) put(sm_o[1]);
  __syncthreads();
  if (wave != 0 || chunk * kF32TileCols + l32 >= a.ncol) return;
  add(sm_o[1]);
  const float inv = L == 0.f ? 0.f : 1.0f / L;     // no visible key: zeros (the reference's l_safe guard)
  int c2 = (int)threadIdx.x & 31;
  asm volatile("" : "+v"(c2));                     // (computed again: held through the loop, they were spilled)
  c2 += chunk * kF32TileCols;
  const int i2 = c2 / a.G;
  char* op = a.out + b * a.o_sb + (int64_t)(hkv * a.G + c2 - i2 * a.G) * a.o_sh + (int64_t)i2 * a.o_sm;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int r = 8 * (j >> 2) + 4 * h + (j & 3);
    if (D < 32 && r >= D) continue;
    if constexpr (ET == 1) {
      *(float*)(op + 4 * r) = o[0][j] * inv;
    } else if constexpr (ET == 2) {
      *(f32x2*)(op + 8 * r) = f32x2{o[0][j] * inv, o[1][j] * inv};
    } else {
#pragma unroll
      for (int p = 0; p < ET / 4; ++p)
        *(f32x4*)(op + 512 * p + 16 * r) = f32x4{o[4 * p][j] * inv, o[4 * p + 1][j] * inv, o[4 * p + 2][j] * inv,
                                                 o[4 * p + 3][j] * inv};
    }
  }
}

template <int D>
static int launch_d(F32Launch& L) {
  const int64_t items = (int64_t)L.a.B * L.a.Hkv * L.a.nchunk;
  if (items > 0x7fffffff) return fail(SIA_ERR_UNSUPPORTED, "fp32 attention: too many work items");
  if (items == 0) return SIA_OK;
  const int cus = device_info().cus;
  L.a.fold = L.a.causal && items > cus && items <= 2 * (int64_t)cus && D <= 128 ? cus : 0;
  hipLaunchKernelGGL((attn_f32_prefill<D>), dim3((unsigned)items), dim3(256), 0, L.stream, L.a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SIA_OK : fail(SIA_ERR_LAUNCH, "fp32 prefill launch: %s", hipGetErrorString(e));
}

int launch_attn_f32_prefill(F32Launch& L) {
  switch (L.D) {
    case 16: return launch_d<16>(L);
    case 32: return launch_d<32>(L);
    case 64: return launch_d<64>(L);
    case 128: return launch_d<128>(L);
    case 256: return launch_d<256>(L);
    default: return fail(SIA_ERR_UNSUPPORTED, "head_dim %d not supported (16, 32, 64, 128, 256)", L.D);
  }
}

}  // namespace sia
