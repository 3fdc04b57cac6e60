// Clip factors (fixed / AUTO-S, global or per group) and the clipped batch
// sum of stored per-segment gradients.
//
// The scale arithmetic follows clip_pytree / auto_scale_pytree
// (opaque-engine/.../clipping/_pytree.py:106-142, 345-431, 475-564): fp64
// norms, ratio C/||g|| (or R/(||g||+gamma)), the storage guard
// ratio*rel - abs evaluated as two separately rounded fp64 operations,
// min(1, .) for fixed clipping with NaN propagating as in torch.minimum,
// non-finite -> 0, clamp at 0, then rounded to the leaf dtype the way
// torch casts a float64 tensor (to float32, then to bfloat16).
#include <mutex>
#include <type_traits>

#include "odp_internal.h"

namespace {

constexpr int CL_THREADS = 1024;  // one workgroup per example
constexpr int CL_DEPTH = 8;      // loads in flight per thread (a power of two)
constexpr int CL_LONG = 16 * 64 * CL_DEPTH * 2;  // partials a wave sums in 16 rounds of loads
constexpr int CL_MAX_GROUPS = 1024;
static_assert(CL_MAX_GROUPS <= CL_THREADS, "thread g finishes group g");
constexpr int SS_THREADS = 256;
constexpr int SS_ELEMS = 4;  // elements per thread of the element-wise form
#define ODP_CONST __attribute__((address_space(4)))  // uniform values through the scalar path

// The scale as the leaf dtype holds it (float64 leaves keep every bit).
__device__ __forceinline__ double finalize_scale(double ratio, double rel, double abs_, int clamp_one,
                                                 int dtype) {
  double s = __dsub_rn(__dmul_rn(ratio, rel), abs_);
  if (clamp_one && !(s < 1.0) && !isnan(s)) s = 1.0;
  if (!isfinite(s)) s = 0.0;
  if (s < 0.0) s = 0.0;
  if (dtype == ODP_DTYPE_F64) return s;
  return (double)odp_round_to((float)s, dtype);
}

// Waves per group: 16 for one group, halved until the groups fit side by side
// (one wave each beyond 8 groups, in rounds of 16 groups).
__host__ __device__ inline int clip_waves(int n_groups) {
  int wpg = CL_THREADS / 64;
  while (wpg > 1 && wpg * n_groups > CL_THREADS / 64) wpg >>= 1;
  return wpg;
}
// Whether a call may have a group too long for its waves.  Four waves come
// close to what the CU can have in flight, so a group on four or more needs no
// help.
inline bool clip_long(int64_t n_slots, int n_groups) {
  const int wpg = clip_waves(n_groups);
  return wpg < 4 && n_slots > (int64_t)CL_LONG * wpg;
}

// One workgroup per example.  Group g owns slots [gstart[g], gstart[g+1]).
// The sum of an example's partials (a few hundred KB on Llama-shaped
// models) is bound by what one CU can have in flight, so each thread issues
// CL_DEPTH 16-byte loads at once; the order of additions is fixed (it does
// not depend on which loads are masked: a fixed tree within each wave by DPP
// and lane reads, then the group's waves in order), so runs are bitwise
// reproducible.  Several groups are summed side by side, the 16 waves split
// evenly among them: one after the other, each by the whole workgroup, they
// are a chain of load latencies and barriers (14 groups of 584 partials: 16
// us, 5 us side by side; one group: 6 us either way).  A group far longer than
// the others, left on one or two waves, would be summed by them alone (about
// 0.3 us a wave for 1024 partials), so it takes the whole workgroup after the
// rest: past CL_LONG partials a wave (below, a round of all the waves costs
// what it saves) and four times its waves' even share (one of 40960 among
// 16: 17 -> 9 us, of 200000: 67 -> 18; 16 of 8192 each stay side by side, 11 us
// against 23).  LONG: the call has slots enough for such a group on waves few
// enough (clip_long); looking for one costs a call 0.4 us.
// `status` (optional): a word that k_sqnorm sets when it dropped a write
// outside the partials; every example then gets a NaN norm, zero scales and
// clear masks, since the partials are incomplete.
template <bool LONG>
__global__ __launch_bounds__(CL_THREADS) void k_clip_factors(
    const double* __restrict__ part, int64_t n_slots, int n_ex, const int64_t* __restrict__ gstart, int n_groups,
    const double* __restrict__ thr, double eff_thr, int mode, double gamma, int n_cls,
    const double* __restrict__ guard, const int32_t* __restrict__ cls_dtype,
    double* __restrict__ scale_out, float* __restrict__ norm_out, float* __restrict__ gnorm_out,
    uint8_t* __restrict__ clip_out, uint8_t* __restrict__ clip_total_out, const uint32_t* __restrict__ status) {
  const int ex = blockIdx.x;
  const int t = threadIdx.x;
  if (status != nullptr && *status != 0u) {
    if (t == 0) {
      norm_out[ex] = __builtin_nanf("");
      if (clip_total_out) clip_total_out[ex] = 0;
    }
    if (t < n_groups) {
      if (gnorm_out) gnorm_out[(int64_t)t * n_ex + ex] = __builtin_nanf("");
      if (clip_out) clip_out[(int64_t)t * n_ex + ex] = 0;
      for (int k = 0; k < n_cls; ++k) scale_out[((int64_t)k * n_groups + t) * n_ex + ex] = 0.0;
    }
    return;
  }
  __shared__ double red[CL_THREADS / 64];
  __shared__ double gsq[CL_MAX_GROUPS];
  __shared__ double sguard[16];
  __shared__ int scls[8], slong[CL_THREADS / 64];
  const double* row = part + (int64_t)ex * n_slots;
  // The inputs of the scale arithmetic are read now, so that their load
  // latency overlaps the partials' instead of following the reduction
  // (n_groups <= CL_THREADS: thread g finishes group g; the barriers of the
  // reduction publish sguard and scls).
  const double thr_t = t < n_groups ? thr[t] : 0.0;
  if (t < 2 * n_cls) sguard[t] = guard[t];
  if (t < n_cls) scls[t] = cls_dtype[t];

  // This thread's part of the sum of slots [lo, hi), taken by nth threads of
  // which it is the tg-th.
  auto sum_slots = [&](int64_t lo, int64_t hi, int tg, int nth) __attribute__((always_inline)) {
    double a[CL_DEPTH];
#pragma unroll
    for (int q = 0; q < CL_DEPTH; ++q) a[q] = 0.0;
    // Slots are read in 16-byte pairs from the first 16-byte aligned one (by
    // address, so any 8-byte aligned partials buffer works; a leading and a
    // trailing odd slot go to the group's first thread), and every load of a
    // round is issued before the first add (masked past the group's end).
    int64_t la = lo + (int64_t)((((uintptr_t)(row + lo)) >> 3) & 1u);
    la = la < hi ? la : hi;
    const int64_t npair = (hi - la) >> 1;
    if (tg == 0) {
      if (lo < la) a[0] += row[lo];
      if (la + 2 * npair < hi) a[1] += row[hi - 1];
    }
    const double2* pr = (const double2*)(row + la);
    for (int64_t q0 = tg; q0 < npair; q0 += CL_DEPTH * nth) {
      double2 v[CL_DEPTH];
#pragma unroll
      for (int q = 0; q < CL_DEPTH; ++q)
        v[q] = q0 + q * nth < npair ? pr[q0 + q * nth] : double2{0.0, 0.0};
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < CL_DEPTH; ++q) a[q] = (a[q] + v[q].x) + v[q].y;
    }
    // Pairwise over the accumulators, in a fixed order.
#pragma unroll
    for (int w = CL_DEPTH / 2; w > 0; w >>= 1)
#pragma unroll
      for (int q = 0; q < w; ++q) a[q] = a[2 * q] + a[2 * q + 1];
    return a[0];
  };
  constexpr int NWAVE = CL_THREADS / 64;
  const int wpg = clip_waves(n_groups);
  const int64_t all = LONG ? gstart[n_groups] - gstart[0] : 0;
  auto is_long = [&](int64_t n) { return LONG && n > (int64_t)CL_LONG * wpg && 4 * n > wpg * all; };
  const int wave = t >> 6, nth = 64 * wpg, tg = t & (nth - 1);
  if (LONG && t < NWAVE) slong[t] = 0;
  for (int g0 = 0; g0 < n_groups; g0 += NWAVE / wpg) {
    const int g = g0 + wave / wpg;
    double part_sum = 0.0;
    bool longer = false;
    if (g < n_groups) {
      const int64_t lo = gstart[g], hi = gstart[g + 1];
      longer = is_long(hi - lo);
      if (!longer) part_sum = sum_slots(lo, hi, tg, nth);
    }
    const double ws = rows_sum4(row_sum16(part_sum));
    if ((t & 63) == 0) red[wave] = ws;
    __syncthreads();
    if (g < n_groups && tg == 0) {
      double tot = 0.0;
      for (int w = 0; w < wpg; ++w) tot += red[wave + w];
      gsq[g] = tot;
      if (longer) slong[wave] = 1;
    }
    __syncthreads();
  }
  if (LONG && __builtin_amdgcn_ballot_w64(slong[t & (NWAVE - 1)] != 0) != 0) {
    for (int g = 0; g < n_groups; ++g) {
      const int64_t lo = gstart[g], hi = gstart[g + 1];
      if (!is_long(hi - lo)) continue;  // the same for every thread
      const double ws = rows_sum4(row_sum16(sum_slots(lo, hi, t, CL_THREADS)));
      if ((t & 63) == 0) red[wave] = ws;
      __syncthreads();
      if (t == 0) {
        double tot = 0.0;
        for (int w = 0; w < NWAVE; ++w) tot += red[w];
        gsq[g] = tot;
      }
      __syncthreads();
    }
  }

  if (t == 0) {
    double total = 0.0;
    for (int g = 0; g < n_groups; ++g) total += gsq[g];
    const double norm = sqrt(total);
    const float normf = (float)norm;
    norm_out[ex] = normf;
    if (clip_total_out) clip_total_out[ex] = normf > (float)eff_thr ? 1 : 0;
  }
  if (t < n_groups) {
    const int g = t;
    const double gn = sqrt(gsq[g]);
    if (gnorm_out) gnorm_out[(int64_t)g * n_ex + ex] = (float)gn;
    if (clip_out) clip_out[(int64_t)g * n_ex + ex] = (float)gn > (float)thr_t ? 1 : 0;
    const double c = thr_t > 0.0 ? thr_t : 0.0;
    const double ratio = mode == ODP_CLIP_AUTOS ? c / (gn + gamma) : c / gn;
    for (int k = 0; k < n_cls; ++k)
      scale_out[((int64_t)k * n_groups + g) * n_ex + ex] =
          finalize_scale(ratio, sguard[2 * k], sguard[2 * k + 1], mode == ODP_CLIP_FIXED, scls[k]);
  }
}

auto clip_kernel(int64_t n_slots, int n_groups) {
  return clip_long(n_slots, n_groups) ? k_clip_factors<true> : k_clip_factors<false>;
}

// Clipped sum of one leaf per problem, element by element: SS_ELEMS
// consecutive elements per thread, summed over the leaf's segments in
// segment order.  Each term is scale * value rounded to the value's dtype
// (clip_pytree's `scale.to(dtype) * leaf`), accumulated in float32, or in
// float64 (Acc = double) for float64 values or a float64 compute dtype.
// This form serves float64, the float64 sums, raw sums and transposed leaves
// that the form below does not take (rows off the 16-byte grid, rank above
// SS_THREADS); that one has float32, bfloat16 and float16.  `raw`: the values
// are already scaled (a caller's scale function): each is summed as it is,
// with scale 1 and no nan_to_num, as the reference sums a scale function's
// output (_clipped_fun.py:673-700, 777-782).
template <typename Acc>
__device__ __forceinline__ void scale_sum_generic(const void* pe, int pdt, int64_t E, int64_t e0, int n_seg,
                                                  int seg_first, const int32_t* __restrict__ sex,
                                                  const double* __restrict__ sc, float normalize_by, void* out,
                                                  void* out2, int odt, int transpose, int64_t M, int rank,
                                                  bool raw) {
  Acc acc[SS_ELEMS], acc2[SS_ELEMS];
#pragma unroll
  for (int i = 0; i < SS_ELEMS; ++i) acc[i] = acc2[i] = (Acc)0;
  for (int s = 0; s < n_seg; ++s) {
    const double c = raw ? 1.0 : sc[sex[seg_first + s]];
#pragma unroll
    for (int i = 0; i < SS_ELEMS; ++i) {
      if (e0 + i >= E) break;
      const double v = odp_load_as_double(pe, (int64_t)s * E + e0 + i, pdt);
      double y = 0.0, yy = 0.0;
      if (raw || isfinite(v)) {  // nan_to_num of the per-example value
        if (pdt == ODP_DTYPE_F64) {
          y = c * v;
          yy = y * y;
        } else {
          y = (double)odp_round_to(__fmul_rn((float)c, (float)v), pdt);
          yy = (double)odp_round_to(__fmul_rn((float)y, (float)y), pdt);
        }
      }
      acc[i] += (Acc)y;
      acc2[i] += (Acc)yy;
    }
  }
#pragma unroll
  for (int i = 0; i < SS_ELEMS; ++i) {
    const int64_t e = e0 + i;
    if (e >= E) break;
    const int64_t k = e / M, m = e - k * M;
    const int64_t o = transpose ? m * rank + k : e;
    // Cast to the output dtype, then divide in it (the reference's order).
    if (odt == ODP_DTYPE_F64) {
      const double x = (double)acc[i], x2 = (double)acc2[i];
      odp_store_from_double(out, o, odt, normalize_by != 1.0f ? x / (double)normalize_by : x);
      if (out2) odp_store_from_double(out2, o, odt, normalize_by != 1.0f ? x2 / (double)normalize_by : x2);
    } else {
      float x = odp_round_to((float)acc[i], odt), x2 = odp_round_to((float)acc2[i], odt);
      if (normalize_by != 1.0f) {
        x = odp_round_to(__fdiv_rn(x, normalize_by), odt);
        x2 = odp_round_to(__fdiv_rn(x2, normalize_by), odt);
      }
      odp_store_from_float(out, o, odt, x);
      if (out2) odp_store_from_float(out2, o, odt, x2);
    }
  }
}

// One clipped-sum term: the per-example value with non-finite entries zeroed
// (nan_to_num), times the scale, rounded to the values' dtype when it is a
// 16-bit one (scale.to(dtype) * leaf); accumulated in float32.  For float32
// values the compiler contracts product and sum into one fused multiply-add
// (__fmul_rn and __fadd_rn do not keep it from that), so the product is not
// rounded by itself as torch and the element-wise form round it: the sums
// differ from theirs by at most half a unit in the last place a term (1.1e-7
// of a sum over 64 examples) and lie no further from the float64 sum.
template <int PDT>
__device__ __forceinline__ float ss_round(float v) {
  if (PDT == ODP_DTYPE_BF16) return odp_round_bf16(v);
  if (PDT == ODP_DTYPE_F16) return (float)(_Float16)v;
  return v;
}
template <bool SECOND, int PDT>
__device__ __forceinline__ void ss_term(float v, float c, float& acc, float& acc2) {
  if (!isfinite(v)) v = 0.f;
  const float y = ss_round<PDT>(__fmul_rn(c, v));
  acc = __fadd_rn(acc, y);
  if (SECOND) acc2 = __fadd_rn(acc2, ss_round<PDT>(__fmul_rn(y, y)));
}

// The sum cast to the output dtype, then divided in it (the reference's order).
__device__ __forceinline__ float ss_finish(float acc, float normalize_by, int odt) {
  float x = odp_round_to(acc, odt);
  if (normalize_by != 1.0f) x = odp_round_to(__fdiv_rn(x, normalize_by), odt);
  return x;
}

typedef uint32_t ss_u32x4 __attribute__((ext_vector_type(4)));

// Values per 16-byte piece.
template <int PDT>
__host__ __device__ constexpr int ss_vec() { return PDT == ODP_DTYPE_F32 ? 4 : 8; }

template <int PDT>
__device__ __forceinline__ void ss_unpack(const ss_u32x4& w, float (&v)[ss_vec<PDT>()]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (PDT == ODP_DTYPE_F32) {
      v[i] = __uint_as_float(w[i]);
    } else if (PDT == ODP_DTYPE_BF16) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    } else {
      v[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)w[i]);
      v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16));
    }
  }
}

// V consecutive outputs (finished values): 16-byte stores where `vec`.
template <int V>
__device__ __forceinline__ void ss_put(void* dst, int64_t o, int odt, bool vec, const float (&y)[V]) {
  if (!vec) {
#pragma unroll
    for (int i = 0; i < V; ++i) odp_store_from_float(dst, o + i, odt, y[i]);
  } else if (odt == ODP_DTYPE_F32) {
#pragma unroll
    for (int i = 0; i < V; i += 4)
      odp_gstore((f32x4_t*)((float*)dst + o + i), f32x4_t{y[i], y[i + 1], y[i + 2], y[i + 3]});
  } else {
    uint32_t w[V / 2];
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
      if (odt == ODP_DTYPE_BF16)
        w[i] = (uint32_t)odp_f2bf(y[2 * i]) | ((uint32_t)odp_f2bf(y[2 * i + 1]) << 16);
      else
        w[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)y[2 * i]) |
               ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)y[2 * i + 1]) << 16);
    }
    if (V == 8)
      odp_gstore((ss_u32x4*)((uint16_t*)dst + o), ss_u32x4{w[0], w[1], w[V / 2 - 2], w[V / 2 - 1]});
    else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      odp_gstore((u32x2*)((uint16_t*)dst + o), u32x2{w[0], w[1]});
    }
  }
}

// The sums of float32, bfloat16 and float16 values into float32, bfloat16
// or float16 outputs, a few segments at a time: the values of a group are
// all loaded before the first of them is accumulated, and the accumulation
// order (and so every sum) is that of one segment at a time.  The clip
// factors come by scalar loads issued behind the values'.  Stored
// per-example values are read once, non-temporally.  A workgroup takes
// tiles b, b + nblk, ... of the leaf, each SS_THREADS pieces of V values:
//   rows: consecutive elements, one 16-byte load per piece and segment
//         (VEC false, a row length or an address off the 16-byte grid: one
//         element per thread, so pieces of one value);
//   transposed ([rank][M] values, [M][rank] outputs): `rank` rows of a run
//         of columns, turned around through LDS so that the outputs leave as
//         one contiguous run.
template <int PDT>
__host__ __device__ constexpr int ss_sg() { return PDT == ODP_DTYPE_F32 ? 8 : 4; }  // 8 KB a wave and group
constexpr int SS_FEW = 4, SS_FEW_VALUES = 16;  // scale_sum_few's segments and values a thread
constexpr int SS_TILE = SS_THREADS * 8 + SS_THREADS / 4;  // words
// A transposed tile's element in LDS: one word of skew every 32, so that the
// column writes (strides of V * rank words) spread over the banks and aligned
// runs of 8 stay contiguous.
__device__ __forceinline__ int ss_at(int i) { return i + (i >> 5); }

template <bool SECOND, int PDT, bool VEC>
__device__ __forceinline__ void scale_sum_fast(const void* pe, int64_t M, int rank, bool transpose, int b, int nblk,
                                               int n_seg, int seg_first, const int32_t* __restrict__ sex,
                                               const double* __restrict__ sc, float normalize_by, void* out,
                                               void* out2, int odt, float* tile) {
  constexpr int V = VEC ? ss_vec<PDT>() : 1, ES = PDT == ODP_DTYPE_F32 ? 4 : 2;
  const int tid = threadIdx.x;
  const int64_t E = M * rank;
  // Transposed: pieces per thread, columns per tile (a multiple of V; a run of
  // 128 bytes of a row up to rank 64 in float32, 64 bytes in 16 bits), pieces
  // per row.
  constexpr int SUB = PDT == ODP_DTYPE_F32 ? 2 : 1;
  const int cols = transpose ? SS_THREADS * V * SUB / rank / V * V : 0, ppr = transpose ? cols / V : 1;
  const int64_t ntile = transpose ? (M + cols - 1) / cols : (E + SS_THREADS * V - 1) / (SS_THREADS * V);
  const ODP_CONST int32_t* ex = (const ODP_CONST int32_t*)(sex + seg_first);
  const ODP_CONST double* csc = (const ODP_CONST double*)sc;
  // The finished sums of the piece at element e0 of segment 0, if `on`.
  auto piece = [&](int64_t e0, bool on, float (&x)[V], float (&x2)[V]) __attribute__((always_inline)) {
    float acc[V], acc2[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = acc2[i] = 0.f;
    // Segments [s, s + n), n <= SG, all loaded before the first is added.
    // The barriers keep the compiler from widening every piece at once.
    constexpr int SG = VEC ? ss_sg<PDT>() : 8;
    auto group = [&](int s, int n) __attribute__((always_inline)) {
      float c[SG], v[VEC ? V : SG];
      ss_u32x4 w[VEC ? SG : 1];
      const char* src = (const char*)pe + ((int64_t)s * E + e0) * ES;
#pragma unroll
      for (int q = 0; q < SG; ++q, src += E * ES)
        if (q < n) {
          if constexpr (VEC)
            w[q] = __builtin_nontemporal_load((const ODP_GMEM ss_u32x4*)(const ODP_GMEM void*)src);
          else
            v[q] = odp_load_as_float(src, 0, PDT);
        }
#pragma unroll
      for (int q = 0; q < SG; ++q)
        if (q < n) c[q] = (float)csc[ex[s + q]];
#pragma unroll
      for (int q = 0; q < SG; ++q) {
        __builtin_amdgcn_sched_barrier(0);
        if (q < n) {
          if constexpr (VEC) {
            ss_unpack<PDT>(w[q], v);
#pragma unroll
            for (int i = 0; i < V; ++i) ss_term<SECOND, PDT>(v[i], c[q], acc[i], acc2[i]);
          } else {
            ss_term<SECOND, PDT>(v[q], c[q], acc[0], acc2[0]);
          }
        }
      }
    };
    if (on) {
      int s = 0;
      for (; s + SG <= n_seg; s += SG) group(s, SG);
      if (s < n_seg) group(s, n_seg - s);
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
      x[i] = ss_finish(acc[i], normalize_by, odt);
      if (SECOND) x2[i] = ss_finish(acc2[i], normalize_by, odt);
    }
  };
  for (int64_t t = b; t < ntile; t += nblk) {
    float x[V], x2[V];
    if constexpr (VEC) if (transpose) {
      // Tile as [column][rank]: the run out[t * cols * rank ...).
      const int64_t m0 = t * cols;
#pragma unroll 1
      for (int h = 0; h < SUB; ++h) {
        const int idx = tid + h * SS_THREADS, k = idx / ppr, c0 = (idx - k * ppr) * V;
        const bool on = k < rank && m0 + c0 < M;
        piece((int64_t)k * M + m0 + c0, on, x, x2);
        if (h == 0) __syncthreads();  // the previous tile has been stored
        if (on) {
#pragma unroll
          for (int i = 0; i < V; ++i) {
            tile[ss_at((c0 + i) * rank + k)] = x[i];
            if (SECOND) tile[SS_TILE + ss_at((c0 + i) * rank + k)] = x2[i];
          }
        }
      }
      __syncthreads();
      const int run = (int)((M - m0 < cols ? M - m0 : cols) * rank);
      const int oes = odp_dtype_size(odt);
#pragma unroll 1
      for (int h = 0; h < (SECOND ? 2 : 1); ++h) {
        void* dst = h ? out2 : out;
        const float* src = tile + h * SS_TILE;
        for (int i = tid * V; i < run; i += SS_THREADS * V) {
          const int64_t o = m0 * rank + i;
          if (i + V <= run) {
#pragma unroll
            for (int q = 0; q < V; ++q) x[q] = src[ss_at(i) + q];
            ss_put<V>(dst, o, odt, (((uintptr_t)dst + o * oes) & (V * oes - 1) & 15) == 0, x);
          } else {
            for (int q = i; q < run; ++q) odp_store_from_float(dst, m0 * rank + q, odt, src[ss_at(q)]);
          }
        }
      }
      continue;
    }
    const int64_t e0 = t * (SS_THREADS * V) + tid * V;
    const bool on = e0 < E;
    piece(e0, on, x, x2);
    if constexpr (!VEC) {
      if (!on) continue;
      odp_store_from_float(out, e0, odt, x[0]);
      if (SECOND) odp_store_from_float(out2, e0, odt, x2[0]);
    } else {
      const int oes = odp_dtype_size(odt);
      if (on) {
        ss_put<V>(out, e0, odt, (((uintptr_t)out + e0 * oes) & (V * oes - 1) & 15) == 0, x);
        if (SECOND) ss_put<V>(out2, e0, odt, (((uintptr_t)out2 + e0 * oes) & (V * oes - 1) & 15) == 0, x2);
      }
    }
  }
}

// Row leaves of at most SS_FEW segments with fewer workgroups than tiles: one
// piece a thread would leave one to
// four loads in flight, so a thread takes SS_FEW_VALUES values, a piece in each
// of as many consecutive tiles, two segments at a time.  The sums are
// scale_sum_fast's, bit for bit (the same terms in the same order).  2^26
// values in float32, one example: 157 -> 83 us (6.4 TB/s), two: 176 -> 124;
// bfloat16: 100 -> 75 and 104 -> 80.
template <bool SECOND, int PDT>
__device__ __forceinline__ void scale_sum_few(const void* pe, int64_t E, int b, int nblk, int n_seg, int seg_first,
                                              const int32_t* __restrict__ sex, const double* __restrict__ sc,
                                              float normalize_by, void* out, void* out2, int odt) {
  constexpr int V = ss_vec<PDT>(), ES = PDT == ODP_DTYPE_F32 ? 4 : 2, NT = SS_FEW_VALUES / V;
  constexpr int64_t TILE = SS_THREADS * V;
  const ODP_CONST int32_t* ex = (const ODP_CONST int32_t*)(sex + seg_first);
  const ODP_CONST double* csc = (const ODP_CONST double*)sc;
  const int oes = odp_dtype_size(odt);
  for (int64_t e0 = (int64_t)b * NT * TILE + threadIdx.x * V; e0 < E; e0 += (int64_t)nblk * NT * TILE) {
    float acc[NT][V], acc2[NT][V];
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int i = 0; i < V; ++i) acc[k][i] = acc2[k][i] = 0.f;
    // Pieces past the end read the last one: no branch between the loads.
    int64_t at[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) at[k] = (e0 + k * TILE < E ? e0 + k * TILE : E - V) * ES;
    auto group = [&](int s, auto N) __attribute__((always_inline)) {
      constexpr int n = decltype(N)::value;
      ss_u32x4 w[n][NT];
#pragma unroll
      for (int q = 0; q < n; ++q)
#pragma unroll
        for (int k = 0; k < NT; ++k)
          w[q][k] = __builtin_nontemporal_load(
              (const ODP_GMEM ss_u32x4*)(const ODP_GMEM void*)((const char*)pe + (int64_t)(s + q) * E * ES + at[k]));
#pragma unroll
      for (int q = 0; q < n; ++q) {
        const float c = (float)csc[ex[s + q]];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
          float v[V];
          __builtin_amdgcn_sched_barrier(0);
          ss_unpack<PDT>(w[q][k], v);
#pragma unroll
          for (int i = 0; i < V; ++i) ss_term<SECOND, PDT>(v[i], c, acc[k][i], acc2[k][i]);
        }
      }
    };
    int s = 0;
    for (; s + 2 <= n_seg; s += 2) group(s, std::integral_constant<int, 2>{});
    if (s < n_seg) group(s, std::integral_constant<int, 1>{});
    // One piece's finish in a loop, the pieces moved down: unrolled, the six
    // forms' finishes were half of the kernel's code.
#pragma unroll 1
    for (int64_t e = e0; e < E && e < e0 + NT * TILE; e += TILE) {
      float x[V];
#pragma unroll
      for (int i = 0; i < V; ++i) x[i] = ss_finish(acc[0][i], normalize_by, odt);
      ss_put<V>(out, e, odt, (((uintptr_t)out + e * oes) & (V * oes - 1) & 15) == 0, x);
      if (SECOND) {
#pragma unroll
        for (int i = 0; i < V; ++i) x[i] = ss_finish(acc2[0][i], normalize_by, odt);
        ss_put<V>(out2, e, odt, (((uintptr_t)out2 + e * oes) & (V * oes - 1) & 15) == 0, x);
      }
#pragma unroll
      for (int k = 0; k + 1 < NT; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) {
          acc[k][i] = acc[k + 1][i];
          if (SECOND) acc2[k][i] = acc2[k + 1][i];
        }
    }
  }
}

__global__ __launch_bounds__(SS_THREADS) void k_scale_sum(
    const int64_t* __restrict__ probs, const int32_t* __restrict__ ws, int n_prob,
    const int32_t* __restrict__ sex, const double* __restrict__ scales, int n_ex, int n_groups,
    float normalize_by) {
  __shared__ float tile[2 * SS_TILE];  // sums and second moments of a transposed tile
  const int bid = blockIdx.x;
  const int p = odp_find_problem(ws, n_prob, bid);
  const int64_t* f = probs + (int64_t)p * ODP_SS_FIELDS;
  const void* pe = (const void*)f[ODP_SS_PE];
  const int64_t M = f[ODP_SS_M];
  const int rank = (int)f[ODP_SS_RANK];
  const int seg_first = (int)f[ODP_SS_SEG_FIRST], n_seg = (int)f[ODP_SS_NSEG];
  void* out = (void*)f[ODP_SS_OUT];
  void* out2 = (void*)f[ODP_SS_OUT2];
  const int64_t flags = f[ODP_SS_FLAGS];
  const int odt = (int)(flags & 0xff);
  const int transpose = (int)((flags >> 8) & 0xff);
  const int grp = (int)((flags >> 16) & 0xffffff);
  const int cls = (int)((flags >> 40) & 0xff);
  const int wide = (int)((flags >> 48) & 1);
  const bool raw = ((flags >> 52) & 1) != 0;
  const int pdt = (int)((flags >> 56) & 0xff);
  const int64_t E = M * rank;
  const double* sc = scales + ((int64_t)cls * n_groups + grp) * n_ex;
  const int b = bid - ws[p], nblk = ws[p + 1] - ws[p];
  const int vec = pdt == ODP_DTYPE_F32 ? 4 : 8;
  const bool aligned = ((uintptr_t)pe & 15) == 0;
  // Transposed leaves need whole 16-byte pieces of a row and a tile of at
  // least one piece per rank; row leaves take any length.
  const bool fast_t = transpose && aligned && M % vec == 0 && rank <= SS_THREADS;
  const bool generic = wide || raw || pdt == ODP_DTYPE_F64 || odt == ODP_DTYPE_F64 || (transpose && !fast_t);
  if (generic) {
    for (int64_t e0 = ((int64_t)b * SS_THREADS + threadIdx.x) * SS_ELEMS; e0 < E;
         e0 += (int64_t)nblk * SS_THREADS * SS_ELEMS) {
      if (wide || pdt == ODP_DTYPE_F64)
        scale_sum_generic<double>(pe, pdt, E, e0, n_seg, seg_first, sex, sc, normalize_by, out, out2, odt, transpose,
                                  M, rank, raw);
      else
        scale_sum_generic<float>(pe, pdt, E, e0, n_seg, seg_first, sex, sc, normalize_by, out, out2, odt, transpose,
                                 M, rank, raw);
    }
    return;
  }
  const bool rows16 = aligned && E % vec == 0;
  const bool few = n_seg <= SS_FEW && rows16 && !transpose && (int64_t)nblk * SS_THREADS * vec < E;
#define ODP_SS_RUN(SECOND, PDT)                                                                                  \
  do {                                                                                                           \
    if (__builtin_expect(few, 0))                                                                                \
      scale_sum_few<SECOND, PDT>(pe, E, b, nblk, n_seg, seg_first, sex, sc, normalize_by, out, out2, odt);       \
    else if (transpose || rows16)                                                                                \
      scale_sum_fast<SECOND, PDT, true>(pe, M, rank, transpose != 0, b, nblk, n_seg, seg_first, sex, sc,         \
                                        normalize_by, out, out2, odt, tile);                               \
    else                                                                                                         \
      scale_sum_fast<SECOND, PDT, false>(pe, M, rank, false, b, nblk, n_seg, seg_first, sex, sc, normalize_by,   \
                                         out, out2, odt, tile);                                            \
  } while (0)
  if (out2 != nullptr) {
    if (pdt == ODP_DTYPE_F32) ODP_SS_RUN(true, ODP_DTYPE_F32);
    else if (pdt == ODP_DTYPE_BF16) ODP_SS_RUN(true, ODP_DTYPE_BF16);
    else ODP_SS_RUN(true, ODP_DTYPE_F16);
  } else {
    if (pdt == ODP_DTYPE_F32) ODP_SS_RUN(false, ODP_DTYPE_F32);
    else if (pdt == ODP_DTYPE_BF16) ODP_SS_RUN(false, ODP_DTYPE_BF16);
    else ODP_SS_RUN(false, ODP_DTYPE_F16);
  }
#undef ODP_SS_RUN
}

// Per-segment sums of squares of materialised per-example tensors: x^2 in
// clip_pytree's accumulation dtype (float32, or float64 with the flag bit 8
// of ODP_SQ_DTYPE, as for float64 leaves), summed in fp64.  Each workgroup
// reduces SQ_CHUNK elements of one segment and writes one slot.  HBM-bound:
// 16-byte loads, SQ_DEPTH of them in flight per thread, of the aligned middle
// of the chunk (a segment's row of n elements may start anywhere), the few
// elements before and after it one by one.
constexpr int SQ_THREADS = 256;
constexpr int64_t SQ_CHUNK = 8192;
constexpr int SQ_DEPTH = 4;

// One element's square in fp64; non-finite values count as 0 unless `raw`.
__device__ __forceinline__ double sq_term(float x, bool raw) {
  if (!raw && !isfinite(x)) x = 0.f;
  return (double)__fmul_rn(x, x);
}

template <int PDT>
__device__ __forceinline__ double sq_chunk(const void* X, int64_t at, int n, bool raw) {
  constexpr int V = ss_vec<PDT>(), ES = PDT == ODP_DTYPE_F32 ? 4 : 2;
  const char* p = (const char*)X + at * ES;
  int head = (int)((16 - ((uintptr_t)p & 15)) & 15) / ES;
  head = head < n ? head : n;
  const int pieces = (n - head) / V, tail = head + pieces * V;
  const ODP_GMEM ss_u32x4* v = (const ODP_GMEM ss_u32x4*)(const ODP_GMEM void*)(p + head * ES);
  double a = 0.0, b = 0.0;
  if ((int)threadIdx.x < head) a = sq_term(odp_load_as_float(X, at + threadIdx.x, PDT), raw);
  if (tail + (int)threadIdx.x < n) b = sq_term(odp_load_as_float(X, at + tail + threadIdx.x, PDT), raw);
  for (int i0 = threadIdx.x; i0 < pieces; i0 += SQ_DEPTH * SQ_THREADS) {
    ss_u32x4 w[SQ_DEPTH];
#pragma unroll
    for (int q = 0; q < SQ_DEPTH; ++q) w[q] = i0 + q * SQ_THREADS < pieces ? v[i0 + q * SQ_THREADS] : ss_u32x4{0u, 0u, 0u, 0u};
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < SQ_DEPTH; ++q) {
      float x[V];
      ss_unpack<PDT>(w[q], x);
#pragma unroll
      for (int i = 0; i < V; i += 2) {
        a += sq_term(x[i], raw);
        b += sq_term(x[i + 1], raw);
      }
    }
  }
  return a + b;
}

// Writes outside the partials ([0, n_ex) x [0, part_stride)) are dropped;
// `status` (optional) is then set to 1.
__global__ __launch_bounds__(SQ_THREADS) void k_sqnorm(const int64_t* __restrict__ probs,
                                                       const int32_t* __restrict__ ws, int n_prob,
                                                       const int32_t* __restrict__ sex,
                                                       double* __restrict__ part,
                                                       int64_t part_stride, int n_ex, uint32_t* status) {
  const int bid = blockIdx.x;
  const int p = odp_find_problem(ws, n_prob, bid);
  const int64_t* f = probs + (int64_t)p * ODP_SQ_FIELDS;
  const void* X = (const void*)f[ODP_SQ_X];
  const int64_t n = f[ODP_SQ_N];
  const int seg_first = (int)f[ODP_SQ_SEG_FIRST];
  const int64_t slot = f[ODP_SQ_SLOT];
  const int dt = (int)(f[ODP_SQ_DTYPE] & 0xff);
  const bool sq64 = ((f[ODP_SQ_DTYPE] >> 8) & 1) != 0;
  const bool raw = ((f[ODP_SQ_DTYPE] >> 9) & 1) != 0;  // no nan_to_num
  const int nchunk = (int)((n + SQ_CHUNK - 1) / SQ_CHUNK);
  const int local = bid - ws[p];
  const int seg = local / nchunk, chunk = local - seg * nchunk;
  const int64_t lo = chunk * SQ_CHUNK, hi = lo + SQ_CHUNK < n ? lo + SQ_CHUNK : n;
  double acc = 0.0;
  if (sq64) {
    for (int64_t i = lo + threadIdx.x; i < hi; i += SQ_THREADS) {
      double x = odp_load_as_double(X, seg * n + i, dt);
      if (!raw && !isfinite(x)) x = 0.0;  // nan_to_num before the norm
      acc += x * x;
    }
  } else if (dt == ODP_DTYPE_F32) {
    acc = sq_chunk<ODP_DTYPE_F32>(X, seg * n + lo, (int)(hi - lo), raw);
  } else if (dt == ODP_DTYPE_BF16) {
    acc = sq_chunk<ODP_DTYPE_BF16>(X, seg * n + lo, (int)(hi - lo), raw);
  } else if (dt == ODP_DTYPE_F16) {
    acc = sq_chunk<ODP_DTYPE_F16>(X, seg * n + lo, (int)(hi - lo), raw);
  } else {
    for (int64_t i = lo + threadIdx.x; i < hi; i += SQ_THREADS)
      acc += sq_term(odp_load_as_float(X, seg * n + i, dt), raw);
  }
  __shared__ double red[SQ_THREADS / 64];
  acc = rows_sum4(row_sum16(acc));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double tot = (red[0] + red[1]) + (red[2] + red[3]);
    const int ex = sex[seg_first + seg];
    if (ex >= 0 && ex < n_ex && slot >= 0 && slot + chunk < part_stride)
      part[(int64_t)ex * part_stride + slot + chunk] = tot;
    else if (status != nullptr)
      odp_gstore(status, 1u);  // every such writer stores the same value
  }
}

}  // namespace

extern "C" int64_t odp_sqnorm_blocks(int64_t n) {
  return n <= 0 ? 0 : (n + SQ_CHUNK - 1) / SQ_CHUNK;
}

extern "C" int odp_sqnorm(odp_stream_t stream, const int64_t* problems, const int32_t* work_start,
                          int32_t n_prob, int32_t total_blocks, const int32_t* seg_example,
                          double* part, int64_t part_stride) {
  int rc = odp_check_table("odp_sqnorm", problems, work_start, n_prob, total_blocks);
  if (rc != ODP_OK) return rc;
  if (total_blocks == 0) return ODP_OK;
  if (seg_example == nullptr || part == nullptr || part_stride <= 0) {
    odp_set_error("odp_sqnorm: null seg_example/part or part_stride <= 0");
    return ODP_ERR_INVALID_ARGUMENT;
  }
  hipLaunchKernelGGL(k_sqnorm, dim3(total_blocks), dim3(SQ_THREADS), 0, odp_hip_stream(stream),
                     problems, work_start, n_prob, seg_example, part, part_stride, INT32_MAX, nullptr);
  return odp_check_launch("odp_sqnorm");
}

// Argument checks shared by odp_clip_factors and its allocation-free
// variant (everything but the partials pointer).
static int check_clip_args(const char* what, int64_t n_slots, int32_t n_ex, const int64_t* group_slot_start,
                           int32_t n_groups, const double* thresholds, int32_t mode, double gamma, int32_t n_cls,
                           const double* guard, const int32_t* cls_dtype, const double* scale_out,
                           const float* norm_out) {
  if (n_ex < 0 || n_slots < 0) {
    odp_set_error("%s: negative n_ex or n_slots", what);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  if (n_groups < 1 || n_groups > CL_MAX_GROUPS) {
    odp_set_error("%s: n_groups=%d outside [1, %d]", what, n_groups, CL_MAX_GROUPS);
    return ODP_ERR_UNSUPPORTED;
  }
  if (n_cls < 1 || n_cls > 8) {
    odp_set_error("%s: n_cls=%d outside [1, 8]", what, n_cls);
    return ODP_ERR_UNSUPPORTED;
  }
  if (mode != ODP_CLIP_FIXED && mode != ODP_CLIP_AUTOS) {
    odp_set_error("%s: unknown mode %d", what, mode);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  if (mode == ODP_CLIP_AUTOS && !(gamma > 0.0)) {
    odp_set_error("%s: gamma must be positive, got %g", what, gamma);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  if (n_ex > 0 && (group_slot_start == nullptr || thresholds == nullptr || guard == nullptr ||
                   cls_dtype == nullptr || scale_out == nullptr || norm_out == nullptr)) {
    odp_set_error("%s: null required pointer", what);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  return ODP_OK;
}

extern "C" int odp_clip_factors(odp_stream_t stream, const double* part, int64_t n_slots,
                                int32_t n_ex, const int64_t* group_slot_start, int32_t n_groups,
                                const double* thresholds, double effective_threshold, int32_t mode,
                                double gamma, int32_t n_cls, const double* guard,
                                const int32_t* cls_dtype, double* scale_out, float* norm_out,
                                float* group_norm_out, uint8_t* clipped_out,
                                uint8_t* clipped_total_out) {
  int rc = check_clip_args("odp_clip_factors", n_slots, n_ex, group_slot_start, n_groups, thresholds, mode,
                           gamma, n_cls, guard, cls_dtype, scale_out, norm_out);
  if (rc != ODP_OK) return rc;
  if (n_ex == 0) return ODP_OK;
  if (n_slots > 0 && part == nullptr) {
    odp_set_error("odp_clip_factors: null required pointer");
    return ODP_ERR_INVALID_ARGUMENT;
  }
  hipLaunchKernelGGL(clip_kernel(n_slots, n_groups), dim3(n_ex), dim3(CL_THREADS), 0, odp_hip_stream(stream), part,
                     n_slots, n_ex, group_slot_start, n_groups, thresholds, effective_threshold, mode,
                     gamma, n_cls, guard, cls_dtype, scale_out, norm_out, group_norm_out,
                     clipped_out, clipped_total_out, nullptr);
  return odp_check_launch("odp_clip_factors");
}

extern "C" int64_t odp_scale_sum_blocks(int64_t n_elems) {
  const int64_t per = (int64_t)SS_THREADS * 8;  // a tile of 16-bit values
  return n_elems <= 0 ? 0 : (n_elems + per - 1) / per;
}

extern "C" int odp_scale_sum(odp_stream_t stream, const int64_t* problems, const int32_t* work_start,
                             int32_t n_prob, int32_t total_blocks, const int32_t* seg_example,
                             const double* scales, int32_t n_ex, int32_t n_groups,
                             float normalize_by) {
  int rc = odp_check_table("odp_scale_sum", problems, work_start, n_prob, total_blocks);
  if (rc != ODP_OK) return rc;
  if (!(normalize_by > 0.0f)) {
    odp_set_error("odp_scale_sum: normalize_by must be > 0, got %g", (double)normalize_by);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  if (total_blocks == 0) return ODP_OK;
  if (seg_example == nullptr || scales == nullptr || n_ex <= 0 || n_groups <= 0) {
    odp_set_error("odp_scale_sum: null seg_example/scales or non-positive n_ex/n_groups");
    return ODP_ERR_INVALID_ARGUMENT;
  }
  hipLaunchKernelGGL(k_scale_sum, dim3(total_blocks), dim3(SS_THREADS), 0, odp_hip_stream(stream),
                     problems, work_start, n_prob, seg_example, scales, n_ex, n_groups,
                     normalize_by);
  return odp_check_launch("odp_scale_sum");
}

// ---------------------------------------------------------------------------
// Allocation-free clipping of materialised per-example gradients.
//
// odp_sqnorm fills caller-provided fp64 partials that odp_clip_factors then
// reads.  Callers that cannot allocate device memory (code under HIP graph
// capture, serving loops, harnesses that forbid hipMalloc) call
// odp_clip_materialized_noalloc instead: the partials live in `scratch`, a
// file-scope device array each GPU holds until the process ends.  The array
// is found by its address per device (hipGetSymbolAddress on the first call
// made with that device current); host code never passes the array's name
// itself to a kernel.  Every call on a GPU shares that GPU's array, so calls
// that overlap on one GPU race.
// ---------------------------------------------------------------------------
// The partials, then one status word (k_sqnorm's dropped writes).
static __device__ __align__(256) double scratch[ODP_NOALLOC_MAX_PARTIALS + 32];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

// The address of this device's `scratch`, looked up once per device.
int scratch_on_current_device(double** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    odp_set_error("odp_clip_materialized_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
    return ODP_ERR_HIP;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    odp_set_error("odp_clip_materialized_noalloc: device %d outside [0, %d)", dev, kMaxDevices);
    return ODP_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      odp_set_error("odp_clip_materialized_noalloc: hipGetSymbolAddress(scratch) failed: %s",
                    hipGetErrorString(e));
      return ODP_ERR_HIP;
    }
    g_scratch_ptr[dev] = (double*)ptr;
  }
  *out = g_scratch_ptr[dev];
  return ODP_OK;
}

// Clears n partials and the status word (a kernel, not a memset: the call
// may be captured into a graph).
__global__ __launch_bounds__(256) void k_zero_partials(double* __restrict__ p, int64_t n, uint32_t* status) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0.0;
  if (i == 0) *status = 0u;
}

}  // namespace

extern "C" int64_t odp_noalloc_max_partials(void) { return ODP_NOALLOC_MAX_PARTIALS; }

extern "C" int odp_clip_materialized_noalloc(
    odp_stream_t stream, const int64_t* sq_problems, const int32_t* sq_work_start, int32_t sq_n_prob,
    int32_t sq_total_blocks, const int32_t* seg_example, int64_t n_slots, int32_t n_ex,
    const int64_t* group_slot_start, int32_t n_groups, const double* thresholds, double effective_threshold,
    int32_t mode, double gamma, int32_t n_cls, const double* guard, const int32_t* cls_dtype, double* scale_out,
    float* norm_out, float* group_norm_out, uint8_t* clipped_out, uint8_t* clipped_total_out) {
  const char* what = "odp_clip_materialized_noalloc";
  int rc = odp_check_table(what, sq_problems, sq_work_start, sq_n_prob, sq_total_blocks);
  if (rc != ODP_OK) return rc;
  rc = check_clip_args(what, n_slots, n_ex, group_slot_start, n_groups, thresholds, mode, gamma, n_cls, guard,
                       cls_dtype, scale_out, norm_out);
  if (rc != ODP_OK) return rc;
  if (n_ex == 0) return ODP_OK;
  if (n_slots > ODP_NOALLOC_MAX_PARTIALS / n_ex) {
    odp_set_error("%s: %d examples x %lld slots exceed the %lld partials of the static scratch", what, n_ex,
                  (long long)n_slots, (long long)ODP_NOALLOC_MAX_PARTIALS);
    return ODP_ERR_UNSUPPORTED;
  }
  if (sq_total_blocks > 0 && seg_example == nullptr) {
    odp_set_error("%s: null seg_example", what);
    return ODP_ERR_INVALID_ARGUMENT;
  }
  double* part = nullptr;
  rc = scratch_on_current_device(&part);
  if (rc != ODP_OK) return rc;
  uint32_t* status = (uint32_t*)(part + ODP_NOALLOC_MAX_PARTIALS);
  hipStream_t s = odp_hip_stream(stream);
  const int64_t n = (int64_t)n_ex * n_slots;
  hipLaunchKernelGGL(k_zero_partials, dim3((unsigned)((n + 255) / 256 > 0 ? (n + 255) / 256 : 1)), dim3(256), 0, s,
                     part, n, status);
  rc = odp_check_launch(what);
  if (rc != ODP_OK) return rc;
  if (sq_total_blocks > 0) {
    // The kernel's bounds checks keep every write inside the n_ex x n_slots
    // partials (a malformed table cannot write past the static array).
    hipLaunchKernelGGL(k_sqnorm, dim3(sq_total_blocks), dim3(SQ_THREADS), 0, s, sq_problems, sq_work_start,
                       sq_n_prob, seg_example, part, n_slots, n_ex, status);
    rc = odp_check_launch(what);
    if (rc != ODP_OK) return rc;
  }
  hipLaunchKernelGGL(clip_kernel(n_slots, n_groups), dim3(n_ex), dim3(CL_THREADS), 0, s, part, n_slots, n_ex, group_slot_start,
                     n_groups, thresholds, effective_threshold, mode, gamma, n_cls, guard, cls_dtype, scale_out,
                     norm_out, group_norm_out, clipped_out, clipped_total_out, status);
  return odp_check_launch(what);
}
