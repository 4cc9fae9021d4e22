// Top-k prox columns by selection: the top-k simplex, the top-k cone and
// their biased forms for the columns the register kernel does not take
// (topk_in_registers) and for those it defers (the U/M searches).
//
// One group of BT threads per column: a wave up to kRegMaxM rows (four
// independent waves per workgroup), the whole workgroup beyond.  The column
// is read once into registers.  A cut that certainly lies below every value
// the thresholds depend on comes from the 64 maxima of 64 disjoint parts of
// the column (the k + 1 largest of them are k + 1 of its values, so the
// (k + 1)-th of the maxima is at most its (k + 1)-th largest); the values
// above the cut, a few more than k + 1 of them, are compacted into LDS,
// sorted by one wave in its registers and given prefix sums.  The
// reference's special cases (topk_cone.h:18-55), the knapsack's partition
// (knapsack_eq.h:25-109) and the U/M searches (topk_cone.h:58-133,
// topk_cone_biased.h:9-106) are then found on that short sorted list, one
// rank or one candidate partition per lane.  Sorting the whole column
// instead (a bitonic network over m values in LDS, then one lane per |U|
// walking M) took 45 network stages at m = 1000 and 105 at 10,000 for a
// list of a dozen values that matter.
//
// What bounds it: HBM from about 1000 rows on (one read, one write), below
// that the fixed work per column (two sorts of 64 values, the searches).
// Measured on MI355X, 40e6 fp32 entries, us per launch, sorting the whole
// column -> selection:
//   top-k simplex k = 10:  m = 700 2568 -> 92, 1000 1875 -> 68, 1500 2261 -> 63
//   top-k simplex k = 5, 4096 columns of 10,000:  7364 -> 201
//   top-k cone k = 5 on margins (U/M searches):  m = 100 12812 -> 653,
//                          1000 15076 -> 443, 3000 7918 -> 105
// (one read and one write of them take 52 us at the rate of a large copy
// kernel).  A column that the list cannot decide (more than kSelectMax values
// above the cut and no plain knapsack, +inf or NaN, ties with zero, a
// partition that may reach past the list) is sorted whole by the group that
// holds it (prox_sorted.hpp).  Classes masked by -inf are left out.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "prox_impl.hpp"
#include "prox_launch.hpp"
#include "prox_select.hpp"
#include "prox_sorted.hpp"

namespace sdca_gpu {

namespace {

// Waves per workgroup of the wave-per-column form.
constexpr int kSelectWaves = 4;

// Group-wide synchronisation of a column's LDS.
template <int BT>
__device__ inline void select_sync() {
  if constexpr (BT > 64) __syncthreads();
  else wave_lds_sync();
}
template <int BT>
__device__ inline int select_lane() {
  return static_cast<int>(threadIdx.x) & (BT > 64 ? BT - 1 : 63);
}

// (One wave per column, up to 16 slots, fp32: four waves per SIMD, one
// register fewer than the compiler takes by itself; at three waves k = 10,
// m = 1000 took 105 us per 50,000 columns instead of 94.  In fp64 the bound
// spills: m = 1000 124 -> 188 us.)
template <class D, class R, int BT, int C>
__global__ void __launch_bounds__(BT > 64 ? BT : 64 * kSelectWaves,
                                  (BT == 64 && C <= 16 && sizeof(D) + sizeof(R) == 8) ? 4 : 1)
prox_select_kernel(const D* __restrict__ in, D* __restrict__ out, int64_t m64, int64_t n,
                   ProxParamsT<R> pp, sdca_thresholds* __restrict__ thr, int* __restrict__ slow,
                   int all_columns, int pow2, int group_bytes, int vec,
                   sdca_prox_sets* __restrict__ sets) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ SelectRecord<R> sh_rec[BT > 64 ? 1 : kSelectWaves];
  __shared__ D sh_cut[BT > 64 ? 1 : kSelectWaves];
  __shared__ int sh_cnt[2];  // the workgroup's compaction counter, two in turn
  constexpr int NG = BT > 64 ? 1 : kSelectWaves;  // groups per workgroup
  // A float workgroup's column (of more than 2048 values) whose sets rounding
  // decides takes the sorted column's steps: with the numerator at sums of
  // thousands, a dozen values free, they place t a hundred ulps off, and a
  // result should not depend on the path its column takes.
  constexpr bool kClose = BT > 64 && sizeof(R) == 4;
  // The sums over the column are rounded to R once, as the sorted column's.
  typedef typename WideSum<R>::type S;
  // (their loops unrolled further would set the kernel's register peak)
  constexpr int UF = (sizeof(R) == 4 && BT > 64) ? 4 : 1;
  __shared__ R sh_mag[kClose ? BT / 64 : 1];
  const int grp = BT > 64 ? 0 : static_cast<int>(threadIdx.x) >> 6;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const bool lead = BT == 64 || threadIdx.x < 64;  // the wave that solves
  // The group's LDS: the sorted list and its prefix sums (and the waves'
  // part maxima), or the whole column where it is sorted.
  unsigned char* const base = smem_raw + static_cast<size_t>(grp) * group_bytes;
  double* const ps = reinterpret_cast<double*>(base);
  D* const list = reinterpret_cast<D*>(base + 8 * (kSelectMax + 2));
  D* const parts = list + kSelectMax;
  D* const whole = reinterpret_cast<D*>(base);
  SelectRecord<R>& rec_lds = sh_rec[grp];
  const int m = static_cast<int>(m64);
  const int k = pp.k;
  const bool cone = pp.op == OP_TOPK_CONE || pp.op == OP_TOPK_CONE_BIASED;
  const int64_t count = all_columns ? n : static_cast<int64_t>(slow[0]);
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * NG + grp; w < count;
       w += static_cast<int64_t>(gridDim.x) * NG) {
    const int64_t j = all_columns ? w : static_cast<int64_t>(slow[2 + w]);
    const D* const col = in + j * m64;
    // (opaque per column: the slots' indices and addresses, hoisted out of
    // this loop, would hold three registers per slot)
    int tid = select_lane<BT>();
    asm("" : "+v"(tid));
    D v[C];
    // Neither +inf nor NaN.  A value of -inf is a masked class: it ends at 0
    // and is left out like the padding.
    bool finite = true;
    // sum |a_i|, for the test of a close call (kClose; infinite with a masked
    // class, which makes every call a close one)
    R mag = 0;
    if (vec) {
      constexpr int E = 16 / static_cast<int>(sizeof(D));
      typedef D word __attribute__((ext_vector_type(E)));
#pragma unroll
      for (int q = 0; q < C / E; ++q) {
        const int i = (q * BT + tid) * E;
        const bool ok = i < m;
        const word x = *reinterpret_cast<const word*>(col + (ok ? i : 0));
#pragma unroll
        for (int l = 0; l < E; ++l) {
          finite = finite && x[l] < num<D>::inf();
          if constexpr (kClose) mag += ok ? static_cast<R>(fabs(x[l])) : R(0);
          v[q * E + l] = ok ? x[l] : -num<D>::inf();
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = c * BT + tid;
        const D x = col[i < m ? i : 0];
        finite = finite && x < num<D>::inf();
        if constexpr (kClose) mag += i < m ? static_cast<R>(fabs(x)) : R(0);
        v[c] = i < m ? x : -num<D>::inf();
      }
    }
    // The maxima of the column's 64 parts (part l: lane l of every wave),
    // descending over the solving wave's lanes.
    D part = v[0];
#pragma unroll
    for (int c = 1; c < C; ++c) part = (v[c] > part) ? v[c] : part;
    if (!finite) part = num<D>::inf();  // seen below: the column goes to the sort
    if constexpr (BT > 64) {
      parts[threadIdx.x] = part;
      if constexpr (kClose) {
        mag = wave_total(mag);
        if (lane == 0) sh_mag[threadIdx.x >> 6] = mag;
      }
      if (threadIdx.x == 0) sh_cnt[0] = sh_cnt[1] = 0;
      __syncthreads();
      if (lead) {
#pragma unroll
        for (int i = 1; i < BT / 64; ++i) {
          const D y = parts[64 * i + lane];
          part = (y > part) ? y : part;
        }
        if constexpr (kClose) {
          mag = R(0);
#pragma unroll
          for (int i = 0; i < BT / 64; ++i) mag += sh_mag[i];
        }
      }
    }
    if (lead) {
      D one[1] = {part};
      wave_sort_desc<1>(one);
      part = one[0];
    }
    SelectRecord<R> rec;
    rec.state = SEL_WIDER;
    rec.t = rec.hi = R(0);
    rec.branch = rec.n_hi = rec.n_mid = 0;
    D cut = -num<D>::inf();
    // At most three lists: the cut for the operator's usual case, a higher
    // one if that list is too long, a lower one if a search needs more.
    for (int attempt = 0; attempt < 3; ++attempt) {
      if (lead) {
        const D top = read_lane(part, 0);
        // (a short column is its own list: -inf is the padding)
        D c = -num<D>::max_finite();
        if (m > kSelectMax) {
          // the k + 1 largest, and for the knapsack every value above
          // a_(k) - hi; a search's list from further down
          c = read_lane(part, (cone && attempt == 0 && k < kSearchRank) ? kSearchRank : k);
          if (!cone && attempt != 1) {
            const R b = static_cast<R>(c);
            const D lower = static_cast<D>(b - pp.rhs_k -
                                           (fabs(b) + pp.rhs_k) * (R(16) * num<R>::eps()));
            c = lower < c ? lower : c;
          }
          if (attempt == 2) {
            const D last = read_lane(part, kSearchRankLast);
            c = last < c ? last : c;
          }
        }
        // (fewer than k + 1 parts hold an unmasked class: all of those)
        if (c < -num<D>::max_finite()) c = -num<D>::max_finite();
        if (!(top < num<D>::inf())) c = num<D>::quiet_nan();
        cut = c;
        if constexpr (BT > 64) {
          if (threadIdx.x == 0) sh_cut[0] = c;
        }
      }
      if constexpr (BT > 64) {
        __syncthreads();
        cut = sh_cut[0];
      }
      if (!(cut == cut)) {
        rec.state = SEL_SLOW;
        break;
      }
      // The values at or above the cut, in any order.
      int cnt = 0;
      if constexpr (BT == 64) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const bool pr = v[c] >= cut;
          const unsigned long long mask = __ballot(pr);
          if (mask) {
            const int at = cnt + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                static_cast<unsigned>(mask >> 32),
                __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0)));
            if (pr && at < kSelectMax) list[at] = v[c];
            cnt += __popcll(mask);
          }
        }
        wave_lds_sync();
      } else {
        int mine = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) mine += __popcll(__ballot(v[c] >= cut));
        int at0 = 0;
        if (mine > 0) {
          if (lane == 0) at0 = atomicAdd(&sh_cnt[attempt & 1], mine);
          at0 = __builtin_amdgcn_readfirstlane(at0);
#pragma unroll
          for (int c = 0; c < C; ++c) {
            const bool pr = v[c] >= cut;
            const unsigned long long mask = __ballot(pr);
            if (mask) {
              const int at = at0 + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                  static_cast<unsigned>(mask >> 32),
                  __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0)));
              if (pr && at < kSelectMax) list[at] = v[c];
              at0 += __popcll(mask);
            }
          }
        }
        __syncthreads();
        cnt = sh_cnt[attempt & 1];
        if (threadIdx.x == 0) sh_cnt[(attempt & 1) ^ 1] = 0;
      }
      if (cnt > kSelectMax) {
        if (attempt == 0) continue;  // the higher cut of attempt 1
        rec.state = SEL_SLOW;
        break;
      }
      if (lead) {
        if (cnt <= 64) list_sort<1>(list, ps, cnt);
        else if (cnt <= 128) list_sort<2>(list, ps, cnt);
        else list_sort<4>(list, ps, cnt);
        rec = list_record<D, R>(list, ps, cnt, m, cut, pp, cone || attempt != 1);
        if constexpr (kClose) {
          // The fixing's numerator sums up to sum |a_i| in R, so its
          // threshold strays by a few ulps of that over the free values; a
          // value so near to t or t + hi may fall on either side there.
          if (rec.state == SEL_DONE && rec.branch == SDCA_BRANCH_KNAPSACK) {
            const R stray = num<R>::eps() * mag / static_cast<R>(rec.n_mid);
            const int u = rec.n_hi, e = rec.n_hi + rec.n_mid;
            const R low = static_cast<R>(e < cnt ? list[e] : list_rest(cut));
            // (none free: the fixing keeps its t)
            if (e == u || (u > 0 && static_cast<R>(list[u - 1]) - rec.t - rec.hi < stray) ||
                rec.t + rec.hi - static_cast<R>(list[u]) < stray ||
                static_cast<R>(list[e - 1]) - rec.t < stray || rec.t - low < stray)
              rec.state = SEL_FIX;
          }
        }
      }
      if constexpr (BT > 64) {
        if (threadIdx.x == 0) rec_lds = rec;
        __syncthreads();
        rec = rec_lds;
      }
      if (rec.state == SEL_U0) {
        // topk_cone_search with U empty: t = 0, M = {x > 16 eps}, then the
        // n_z values within 16 eps of zero one by one.  (This pass
        // and the fixing below read the column again, from the L2: unrolled
        // over the slots they set the kernel's register peak.)
        const R eps16 = R(16) * num<R>::eps();
        S sum_p = 0;
        int n_p = 0, n_z = 0;
#pragma unroll UF
        for (int i = tid; i < m; i += BT) {
          const R x = static_cast<R>(col[i]);
          const bool pos = x > eps16;
          add_if(sum_p, pos, x);
          n_p += pos ? 1 : 0;
          n_z += (!pos && x >= -eps16) ? 1 : 0;
        }
        group_sums<BT>(sum_p, n_p, n_z);
        const R s_p = static_cast<R>(sum_p);
        const R K = static_cast<R>(k);
        const R hi = (K * s_p) / (K * K);
        const R largest = n_p > 0 ? static_cast<R>(list[0]) : -num<R>::inf();
        rec.state = SEL_DONE;
        rec.t = R(0);
        rec.hi = hi;
        rec.branch = SDCA_BRANCH_SCAN;
        rec.n_hi = 0;
        rec.n_mid = n_p;
        if (largest - eps16 <= hi) {
          // accepted at the first end the reference tries
        } else if (largest - eps16 <= hi + static_cast<R>(n_z) * eps16) {
          rec.state = SEL_SLOW;  // the values near zero may decide
        } else {
          if (lead) rec = list_cone<D, R>(list, ps, cnt, m, cut, k, R(0), 1);
          if constexpr (BT > 64) {
            __syncthreads();
            if (threadIdx.x == 0) rec_lds = rec;
            __syncthreads();
            rec = rec_lds;
          }
        }
      }
      if (rec.state == SEL_FIX) {
        // Variable fixing over the slots, the free set as the value interval
        // (lc, hc]: more candidates than the list holds, or a workgroup's
        // column too close to call (below).  A wave's column starts from the
        // bound of the k-th value; a workgroup's takes the sorted column's
        // steps (knapsack_sorted: the same start, the numerator carried on
        // in R, the sums rounded to R once), so that it ends with the same
        // sets.
        const R hi = pp.rhs_k, rhs = pp.rhs;
        const R eps = num<R>::eps() * dmax(R(1), fabs(rhs));
        R lc = -num<R>::inf(), hc = num<R>::inf();
        if constexpr (BT == 64) {
          const R kth = static_cast<R>(list[k - 1]);
          const R slack = (fabs(kth) + hi) * (R(16) * num<R>::eps());
          lc = kth - hi - slack;
          hc = kth + hi + slack;
        }
        S s_f = 0, s_u = 0;
        int n_f = 0, n_u = 0;
#pragma unroll UF
        for (int i = tid; i < m; i += BT) {
          const R x = static_cast<R>(col[i]);
          const bool f = x > lc && x <= hc;
          add_if(s_f, f, x);
          n_f += f ? 1 : 0;
          add_if(s_u, x > hc, x);
          n_u += x > hc ? 1 : 0;
        }
        group_sums<BT>(s_f, s_u, n_f, n_u);
        R t, t_fix;
        if constexpr (BT > 64) t = (static_cast<R>(s_f) - rhs) / static_cast<R>(n_f);
        else t = (static_cast<R>(s_f) + static_cast<R>(n_u) * hi - rhs) / static_cast<R>(n_f);
        for (int iter = 0; iter <= m; ++iter) {
          const R c_hi = hi + t;
          S s_lo = 0, s_hi = 0;
          int n_lo = 0, n_hi = 0;
#pragma unroll UF
          for (int i = tid; i < m; i += BT) {
            const R x = static_cast<R>(col[i]);
            const bool f = x > lc && x <= hc;
            add_if(s_lo, f && x <= t, x);
            n_lo += (f && x <= t) ? 1 : 0;
            add_if(s_hi, f && x > c_hi, x);
            n_hi += (f && x > c_hi) ? 1 : 0;
          }
          group_sums<BT>(s_lo, s_hi, n_lo, n_hi);
          const R r_lo = static_cast<R>(s_lo), r_hi = static_cast<R>(s_hi);
          const R sh = static_cast<R>(n_hi) * hi;
          const R infeas = r_hi + r_lo - sh - static_cast<R>(n_hi + n_lo) * t;
          const bool fix_hi = n_hi > 0 && infeas > eps;
          const bool fix_lo = !fix_hi && n_lo > 0 && infeas < -eps;
          const R mc = static_cast<R>(n_f);
          t_fix = t;
          if (fix_hi || (!fix_lo && n_hi > 0)) {
            hc = c_hi;
            n_u += n_hi;
            s_u += s_hi;
            n_f -= n_hi;
          }
          if (fix_lo || (!fix_hi && n_lo > 0)) {
            lc = t;
            n_f -= n_lo;
          }
          if (n_f <= 0) break;
          if constexpr (BT > 64) {
            if (fix_hi) t = (mc * t - r_hi + sh) / static_cast<R>(n_f);
            else if (fix_lo) t = (mc * t - r_lo) / static_cast<R>(n_f);
          }
          if (BT > 64 && (fix_hi || fix_lo)) continue;
          s_f = 0;
#pragma unroll UF
          for (int i = tid; i < m; i += BT) {
            const R x = static_cast<R>(col[i]);
            add_if(s_f, x > lc && x <= hc, x);
          }
          s_f = group_sum<BT>(s_f);
          if constexpr (BT > 64)
            t = (static_cast<R>(s_f) + static_cast<R>(n_u) * hi - rhs) / static_cast<R>(n_f);
          else
            t = t_fix = (static_cast<R>(s_f) + static_cast<R>(n_u) * hi - rhs) / static_cast<R>(n_f);
          if (!fix_hi && !fix_lo) break;
        }
        bool lt;
        const R K = static_cast<R>(k), num_u = static_cast<R>(n_u);
        if (n_u == 0) lt = t_fix < pp.rho * rhs - eps;
        else
          lt = K * (static_cast<R>(s_u) + (K - num_u) * t_fix) < rhs * (num_u + pp.rho * K * K) - eps;
        const R sum_k = list_sum<R>(list, ps, 0, k);
        const bool constant =
            static_cast<R>(list[k - 1]) - sum_k / (K + pp.rho * K * K) >=
            static_cast<R>(k < cnt ? list[k] : list_rest(cut)) - R(16) * num<R>::eps();
        rec.state = (lt && !constant) ? SEL_SLOW : SEL_DONE;
        rec.t = t;
        rec.hi = hi;
        rec.branch = SDCA_BRANCH_KNAPSACK;
        rec.n_hi = n_u;
        rec.n_mid = n_f;
        break;
      }
      if (rec.state != SEL_WIDER) break;
      // One wider list, where this was the usual one.
      if (m <= kSelectMax || attempt != 0) {
        rec.state = SEL_SLOW;
        break;
      }
      if constexpr (BT > 64) __syncthreads();
      else wave_lds_sync();
      attempt = 1;  // the lower cut next
      if constexpr (BT > 64) {
        if (threadIdx.x == 0) sh_cnt[0] = 0;
        __syncthreads();
      }
    }
    R lo = R(0);
    if (rec.state != SEL_DONE) {
      // The whole column sorted in the group's LDS.
      select_sync<BT>();
      for (int i = tid; i < pow2; i += BT) whole[i] = (i < m) ? col[i] : -num<D>::inf();
      select_sync<BT>();
      for (int size = 2; size <= pow2; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
          for (int i = tid; i < pow2; i += BT) {
            const int partner = i ^ stride;
            if (partner > i) {
              const bool desc = (i & size) == 0;
              const D a = whole[i], b = whole[partner];
              if (desc ? (a < b) : (b < a)) {
                whole[i] = b;
                whole[partner] = a;
              }
            }
          }
          select_sync<BT>();
        }
      }
      // (without the masked classes at the end, unless a value is not finite)
      const int kept = cut == cut ? prefix_end<R>(whole, 0, m, -num<R>::inf()) : m;
      if (lead)
        thresholds_sorted<D, R, true>(whole, kept, pp.op, pp.lo, pp.hi, pp.rhs, pp.rho, k, rec.t, lo,
                                      rec.hi, rec.branch, rec.n_hi, rec.n_mid);
      if constexpr (BT > 64) {
        if (threadIdx.x == 0) rec_lds = rec;
        __syncthreads();
        rec = rec_lds;
      }
      lo = R(0);
    }
    if (tid == 0) {
      if (thr)
        thr[j] = sdca_thresholds{static_cast<double>(rec.t), static_cast<double>(lo),
                                 static_cast<double>(rec.hi)};
      if (sets) sets[j] = sdca_prox_sets{rec.n_hi, rec.n_mid, rec.branch, 0};
    }
    const D t = static_cast<D>(rec.t), dlo = D(0), dhi = static_cast<D>(rec.hi);
    asm("" : "+v"(tid));
    D* const dst = out + j * m64;
    if (vec) {
      constexpr int E = 16 / static_cast<int>(sizeof(D));
      typedef D word __attribute__((ext_vector_type(E)));
#pragma unroll
      for (int q = 0; q < C / E; ++q) {
        const int i = (q * BT + tid) * E;
        word y;
#pragma unroll
        for (int l = 0; l < E; ++l) y[l] = clamp_ref(v[q * E + l] - t, dlo, dhi);
        if (i < m) __builtin_nontemporal_store(y, reinterpret_cast<word*>(dst + i));
      }
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = c * BT + tid;
        if (i < m) dst[i] = clamp_ref(v[c] - t, dlo, dhi);
      }
    }
    select_sync<BT>();  // the column's LDS before the next one's
  }
  // List mode: the list's counters [count, done] must be zero for the next
  // call on the stream.  With an empty list they already are; otherwise the
  // workgroups that took columns count themselves out and the last of them
  // zeroes both (each has read the count before it increments done).
  if (!all_columns) {
    const int64_t groups = (count + NG - 1) / NG;
    const int64_t workers = groups < static_cast<int64_t>(gridDim.x) ? groups : gridDim.x;
    if (NG > 1) __syncthreads();
    if (static_cast<int64_t>(blockIdx.x) < workers && threadIdx.x == 0) {
      __threadfence();
      if (atomicAdd(slow + 1, 1) == static_cast<int>(workers) - 1) {
        atomicExch(slow, 0);
        atomicExch(slow + 1, 0);
      }
    }
  }
}

template <class D, class R, int BT, int C>
hipError_t select_one(const ProxLaunch& a, bool all_columns) {
  ProxParamsT<R> pp;
  pp.lo = static_cast<R>(a.lo);
  pp.hi = static_cast<R>(a.hi);
  pp.rhs = static_cast<R>(a.rhs);
  const bool biased = a.op == OP_TOPK_SIMPLEX_BIASED || a.op == OP_TOPK_CONE_BIASED;
  pp.rho = biased ? static_cast<R>(a.rho) : R(0);
  pp.k = static_cast<int>(a.k);
  pp.rhs_k = pp.rhs / static_cast<R>(a.k);
  pp.op = a.op;
  pp.p = static_cast<int>(a.p);
  if (a.m > static_cast<int64_t>(BT) * C) return hipErrorInvalidValue;
  int pow2 = 1;
  while (pow2 < a.m) pow2 <<= 1;
  constexpr int NG = BT > 64 ? 1 : kSelectWaves;
  constexpr int E = 16 / static_cast<int>(sizeof(D));
  const int64_t list_bytes = 8 * (kSelectMax + 2) +
                             (kSelectMax + (BT > 64 ? BT : 0)) * static_cast<int64_t>(sizeof(D));
  const int64_t sort_bytes = static_cast<int64_t>(pow2) * static_cast<int64_t>(sizeof(D));
  const int64_t group_bytes = (std::max(list_bytes, sort_bytes) + 15) / 16 * 16;
  const int vec = a.m % E == 0 &&
                  ((reinterpret_cast<uintptr_t>(a.in) | reinterpret_cast<uintptr_t>(a.out)) & 15) == 0;
  // List mode: the list is usually empty or a small fraction of the n
  // columns; the grid grows with the batch (256 to 1024 workgroups), so that
  // a long list finds four waves on every SIMD while an empty one costs
  // little to launch.
  const int64_t groups = (a.n + NG - 1) / NG;
  const int64_t work = a.n * a.m / 16384;
  const int64_t cap = all_columns ? max_blocks(BT > 64 ? BT : 64 * NG)
                                  : std::min<int64_t>(1024, std::max<int64_t>(256, work));
  const int64_t grid = std::max<int64_t>(1, std::min(groups, cap));
  hipLaunchKernelGGL((prox_select_kernel<D, R, BT, C>), dim3(static_cast<unsigned>(grid)),
                     dim3(BT > 64 ? BT : 64 * NG), static_cast<size_t>(group_bytes * NG), a.stream,
                     static_cast<const D*>(a.in), static_cast<D*>(a.out), a.m, a.n, pp, a.thr,
                     a.slow, all_columns ? 1 : 0, pow2, static_cast<int>(group_bytes), vec, a.sets);
  return hipGetLastError();
}

template <class D, class R>
hipError_t select_by_m(const ProxLaunch& a, bool all_columns) {
  if (a.m <= 256) return select_one<D, R, 64, 4>(a, all_columns);
  if (a.m <= 512) return select_one<D, R, 64, 8>(a, all_columns);
  if (a.m <= 1024) return select_one<D, R, 64, 16>(a, all_columns);
  if (a.m <= 2048) return select_one<D, R, 64, 32>(a, all_columns);
  if (a.m <= 4096) return select_one<D, R, 256, 16>(a, all_columns);
  if (a.m <= 8192) return select_one<D, R, 512, 16>(a, all_columns);
  // (1024 threads of 16 slots spill: 128 registers.  m = 10,000: 4096 fp32
  // columns 265 us so, 201 with 512 threads; 2000 fp64 columns 547, 88.)
  if (a.m <= 16384) return select_one<D, R, 512, 32>(a, all_columns);
  if constexpr (sizeof(D) == 4) return select_one<D, R, 1024, 32>(a, all_columns);
  return hipErrorInvalidValue;
}

}  // namespace

// k + 1 part maxima give the cut, and the last search's rank must lie past
// them; a column of at most kSelectMax rows is its own list.
bool select_supported(const ProxLaunch& a) {
  const bool topk = a.op == OP_TOPK_SIMPLEX || a.op == OP_TOPK_CONE ||
                    a.op == OP_TOPK_SIMPLEX_BIASED || a.op == OP_TOPK_CONE_BIASED;
  return topk && a.m <= max_rows(a.data) && (a.m <= kSelectMax || a.k < kSearchRankLast);
}

hipError_t launch_select(const ProxLaunch& a, bool all_columns) {
  if (a.data == SDCA_F32 && a.result == SDCA_F32) return select_by_m<float, float>(a, all_columns);
  if (a.data == SDCA_F32 && a.result == SDCA_F64) return select_by_m<float, double>(a, all_columns);
  if (a.data == SDCA_F64 && a.result == SDCA_F64) return select_by_m<double, double>(a, all_columns);
  if (a.data == SDCA_F64 && a.result == SDCA_F32) return select_by_m<double, float>(a, all_columns);
  return hipErrorInvalidValue;
}

}  // namespace sdca_gpu
