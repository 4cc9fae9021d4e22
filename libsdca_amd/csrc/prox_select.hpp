// Thresholds from a short sorted list of a column's largest values, by one
// wave: the list's sort and prefix sums, the knapsack's partition
// (knapsack_eq.h:25-109) with one rank per lane, the U/M searches of the top-k
// cones (topk_cone.h:58-133, topk_cone_biased.h:9-106) with one candidate end
// per lane.
#ifndef SDCA_HIP_PROX_SELECT_HPP
#define SDCA_HIP_PROX_SELECT_HPP

#include <climits>

#include "common.hpp"
#include "prox_impl.hpp"
#include "prox_launch.hpp"
#include "prox_sorted.hpp"

namespace sdca_gpu {

// Most values of the sorted list (four per lane of a wave).
constexpr int kSelectMax = 256;
// Part maxima whose rank gives the cut for a search that may need more than
// the k + 1 largest: about 64 log(64 / (64 - r)) values lie above the r-th.
constexpr int kSearchRank = 24;
constexpr int kSearchRankLast = 56;

// Descending bitonic sort of a wave's 64 * CC values, element l * CC + c in
// slot c of lane l; each compare-exchange is one median with a bound of +inf
// (keep the larger) or -inf (keep the smaller), as in group_sort_desc.
template <int SIZE, int STRIDE, int CC, class D>
__device__ inline void wave_sort_stage(D (&x)[CC], int lane, D pinf) {
  constexpr int N = 64 * CC;
  if constexpr (STRIDE < CC) {
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if ((c & STRIDE) == 0) {
        const bool desc = SIZE >= N || (SIZE < CC ? (c & SIZE) == 0 : (lane & (SIZE / CC)) == 0);
        const D a = x[c], b = x[c + STRIDE];
        const D bound = desc ? pinf : -pinf;
        x[c] = max_or_min(a, b, bound);
        x[c + STRIDE] = max_or_min(a, b, -bound);
      }
    }
  } else {
    constexpr int L = STRIDE / CC;
    const bool desc = SIZE >= N || (lane & (SIZE / CC)) == 0;
    const D bound = (desc == ((lane & L) == 0)) ? pinf : -pinf;
#pragma unroll
    for (int c = 0; c < CC; ++c) x[c] = max_or_min(x[c], xor_lane<L, true>(x[c]), bound);
  }
  if constexpr (STRIDE > 1) wave_sort_stage<SIZE, STRIDE / 2, CC>(x, lane, pinf);
}
template <int SIZE, int CC, class D>
__device__ inline void wave_sort_from(D (&x)[CC], int lane, D pinf) {
  wave_sort_stage<SIZE, SIZE / 2, CC>(x, lane, pinf);
  if constexpr (SIZE < 64 * CC) wave_sort_from<2 * SIZE, CC>(x, lane, pinf);
}
template <int CC, class D>
__device__ inline void wave_sort_desc(D (&x)[CC]) {
  wave_sort_from<2, CC>(x, static_cast<int>(threadIdx.x) & 63, net_inf(D(0)));
}

// Exclusive prefix sum over the wave: the inclusive one (as
// wave_exclusive_scan_dpp) of the lane before.  (Not the inclusive sum less
// the lane's own value: next to a value far below the others, a masked
// class at -1e9 say, that would round the sum of the others away.)
__device__ inline double wave_exclusive_scan(double x) {
  double incl = x;
  incl = dpp_add<0x111, 0xF, true>(incl);   // row_shr:1
  incl = dpp_add<0x112, 0xF, true>(incl);   // row_shr:2
  incl = dpp_add<0x114, 0xF, true>(incl);   // row_shr:4
  incl = dpp_add<0x118, 0xF, true>(incl);   // row_shr:8
  incl = dpp_add<0x142, 0xA, false>(incl);  // row_bcast:15
  incl = dpp_add<0x143, 0xC, false>(incl);  // row_bcast:31
  const long long u = __double_as_longlong(incl);
  const int lo = dpp_bits<0x138, 0xF, true>(static_cast<int>(u & 0xffffffffll));  // wave_shr:1
  const int hi = dpp_bits<0x138, 0xF, true>(static_cast<int>(u >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              static_cast<long long>(static_cast<unsigned>(lo)));
}

// A wave's sorted values x (value l CC + c in slot c of lane l, -inf from
// cnt on) with their prefix sums in double: ex[c] = the sum of the values
// before slot c's.
template <int CC, class D>
__device__ inline void list_prefix(const D (&x)[CC], double (&ex)[CC], int cnt) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  double tot = 0;
#pragma unroll
  for (int c = 0; c < CC; ++c) tot += (lane * CC + c < cnt) ? static_cast<double>(x[c]) : 0.0;
  double run = wave_exclusive_scan(tot);
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    ex[c] = run;
    run += (lane * CC + c < cnt) ? static_cast<double>(x[c]) : 0.0;
  }
}
// The same list in LDS: list[i], and ps[i] = the sum of its first i values,
// i <= cnt.
template <int CC, class D>
__device__ inline void list_store(const D (&x)[CC], const double (&ex)[CC], D* list, double* ps,
                                  int cnt) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  wave_lds_sync();
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int i = lane * CC + c;
    if (i < cnt) {
      list[i] = x[c];
      ps[i] = ex[c];
      if (i == cnt - 1) ps[cnt] = ex[c] + static_cast<double>(x[c]);
    }
  }
  wave_lds_sync();
}
// The list's cnt <= 64 CC values sorted in place, with the prefix sums.
template <int CC, class D>
__device__ inline void list_sort(D* list, double* ps, int cnt) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  D x[CC];
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int i = lane * CC + c;
    x[c] = (i < cnt) ? list[i] : -num<D>::inf();
  }
  wave_sort_desc<CC>(x);
  double ex[CC];
  list_prefix<CC>(x, ex, cnt);
  list_store<CC>(x, ex, list, ps, cnt);
}

// The record of a column, or why there is none yet.
enum { SEL_DONE = 0, SEL_FIX = 1, SEL_U0 = 2, SEL_WIDER = 3, SEL_SLOW = 4 };
template <class R>
struct SelectRecord {
  R t, hi;
  int state, branch, n_hi, n_mid;
};

// A bound of the values past a list of every value at or above the cut: the
// cut, or -inf where that is the type's lowest value (masked classes alone
// are left then).
template <class D>
__device__ inline D list_rest(D cut) {
  return cut > -num<D>::max_finite() ? cut : -num<D>::inf();
}

// The sum of the list's values [b, e) rounded to R once, in every lane: from
// the prefix sums in double for float; for double compensated, a few values
// one after the other (the lanes' six exchanges of pairs are a longer chain).
template <class R, class D>
__device__ inline SumPair list_sum_pair(const D* list, int b, int e) {
  SumPair s = 0.0;
  if (e - b <= 12) {
    for (int i = b; i < e; ++i) s += static_cast<R>(list[i]);
    return s;
  }
  for (int i = b + (static_cast<int>(threadIdx.x) & 63); i < e; i += 64)
    s += static_cast<R>(list[i]);
  return wave_total(s);
}
template <class R, class D>
__device__ inline R list_sum(const D* list, const double* ps, int b, int e) {
  if constexpr (sizeof(R) == 4) return static_cast<R>(ps[e] - ps[b]);
  else return static_cast<R>(list_sum_pair<R>(list, b, e));
}

// The partition of the knapsack sum_i clamp(a_i - t, 0, hi) = rhs on the
// sorted list (every value above t is in it): rank r is above t where
// f(a_r) < rhs and at hi where f(a_r - hi) <= rhs, one rank per lane, f from
// the prefix sums and a binary search for the ranks at hi (or inside) at
// that point.  The same eps as the fixing's (topk_sorted_root).  No rank at
// or below a_(k) - hi is above t (there the k largest alone give k hi); far
// below, the rounding of the test's large terms could say otherwise.  The
// threshold is formed from the direct sum over the free ranks; with none
// free any t of [a_u, a_(u-1) - hi] is the same projection and the record
// takes the middle.
template <class D, class R>
__device__ inline void list_knapsack(const D* list, const double* ps, int cnt, int m, D cut, int k,
                                     R hi_r, R rhs_r, R& t_out, int& u_out, int& e_out) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const double hi = static_cast<double>(hi_r), rhs = static_cast<double>(rhs_r);
  const double eps = static_cast<double>(num<R>::eps() * dmax(R(1), fabs(rhs_r)));
  const double kth = static_cast<double>(list[k - 1]);
  const double least = kth - hi - 16.0 * static_cast<double>(num<R>::eps()) * (fabs(kth) + hi);
  int e = 0, u = 0;
  for (int base = 0; base < cnt; base += 64) {
    const int r = base + lane;
    bool above = false, at_hi = false;
    const double a = r < cnt ? static_cast<double>(list[r]) : -num<double>::inf();
    if (a > least) {
      int b = 0, w = r;
      while (b < w) {  // ranks above a + hi
        const int mid = (b + w) >> 1;
        if (static_cast<double>(list[mid]) > a + hi) b = mid + 1;
        else w = mid;
      }
      above = ps[r] - ps[w] - static_cast<double>(r - w) * a + static_cast<double>(w) * hi <
              rhs - eps;
      int z = cnt;
      b = r + 1;
      while (b < z) {  // ranks above a - hi
        const int mid = (b + z) >> 1;
        if (static_cast<double>(list[mid]) > a - hi) b = mid + 1;
        else z = mid;
      }
      at_hi = static_cast<double>(r + 1) * hi + (ps[z] - ps[r + 1]) -
                  static_cast<double>(z - r - 1) * (a - hi) <= rhs + eps;
    }
    e += __popcll(__ballot(above));
    u += __popcll(__ballot(at_hi));
    if (base + 64 > e && base + 64 > u) break;  // no later rank is above t
  }
  if (u > e) u = e;
  if (e > u) {
    double s = 0;
    if constexpr (sizeof(R) == 4) {
      for (int i = u + lane; i < e; i += 64) s += static_cast<double>(list[i]);
      s = wave_total(s);
    } else {
      s = list_sum<R>(list, ps, u, e);
    }
    t_out = static_cast<R>((s + static_cast<double>(u) * hi - rhs) / static_cast<double>(e - u));
  } else {
    const double top = (u > 0 ? static_cast<double>(list[u - 1]) : static_cast<double>(list[0])) - hi;
    double low = top;
    if (u < cnt) low = static_cast<double>(list[u]);
    else if (u < m && list_rest(cut) > -num<D>::inf()) low = static_cast<double>(cut);
    t_out = static_cast<R>(0.5 * (low + top));
  }
  u_out = u;
  e_out = e;
}

// t = (nu sum_M - k_u sum_U) / den and hi = (|M| sum_U + k_u sum_M) / den of
// the partition U = [0, u), M = [u, e), whose terms may cancel: in double for
// float; for double from compensated sums, the products' rounding kept (fma).
template <class D>
__device__ inline void list_cone_values(const D*, const double* ps, int u, int e, float k_u,
                                        float nu, float& t, float& hi) {
  const double su = ps[u], sm = ps[e] - su;
  const double ku = k_u, n = nu, n_m = e - u, den = ku * ku + n_m * n;
  t = static_cast<float>(div_near(n * sm - ku * su, den));
  hi = static_cast<float>(div_near(n_m * su + ku * sm, den));
}
__device__ inline double two_products(double a, const SumPair& x, double b, const SumPair& y) {
  const double p = a * x.s, q = b * y.s;
  SumPair r(p);
  r += q;
  return r.s + (r.c + ((fma(a, x.s, -p) + fma(b, y.s, -q)) + (a * x.c + b * y.c)));
}
template <class D>
__device__ inline void list_cone_values(const D* list, const double*, int u, int e, double k_u,
                                        double nu, double& t, double& hi) {
  const SumPair su = list_sum_pair<double>(list, 0, u), sm = list_sum_pair<double>(list, u, e);
  const double n_m = e - u, den = k_u * k_u + n_m * nu;
  t = two_products(nu, sm, -k_u, su) / den;
  hi = two_products(n_m, su, k_u, sm) / den;
}

// topk_cone_search (topk_cone.h:58-133) and its biased form
// (topk_cone_biased.h:9-106) on the sorted list, from |U| = u_first on: for
// each |U| = u the candidate ends e of M = ranks [u, e) are tried by the
// lanes, the smallest accepted e of the smallest u wins, as in the
// reference's order.  The list holds the column's cnt largest values, the
// others are at most list_rest(cut).  Where a search for some u may continue past
// the list (no end accepted, and t not certainly above every M that would;
// the bound of cone_biased_regs) the result is SEL_WIDER.
template <class D, class R>
__device__ inline SelectRecord<R> list_cone(const D* list, const double* ps, int cnt, int m, D cut,
                                            int k, R rho, int u_first) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const R eps = R(16) * num<R>::eps();
  const R K = static_cast<R>(k);
  const R rest = static_cast<R>(list_rest(cut));
  SelectRecord<R> rec;
  rec.state = SEL_DONE;
  rec.branch = SDCA_BRANCH_SCAN;
  for (int u = u_first; u <= k; ++u) {
    const R k_u = static_cast<R>(k - u);
    const R nu = rho * K * K + static_cast<R>(u);
    const double pu = ps[u];
    const R sum_u = static_cast<R>(pu);
    const R min_u = u > 0 ? static_cast<R>(list[u - 1]) : num<R>::inf();
    const R first = u < cnt ? static_cast<R>(list[u]) : -num<R>::inf();
    for (int e0 = u;; e0 += 64) {
      const int e = e0 + lane;
      const bool in = e <= cnt;
      const int ei = in ? e : cnt;
      const R n_m = static_cast<R>(ei - u);
      const R sum_m = static_cast<R>(ps[ei] - pu);
      const R den = k_u * k_u + n_m * nu;
      const R t = (nu * sum_m - k_u * sum_u) / den;
      const R hi = (n_m * sum_u + k_u * sum_m) / den;
      const R max_m = ei > u ? first : -num<R>::inf();
      const R min_m = ei > u ? static_cast<R>(list[ei - 1]) : num<R>::inf();
      const R tt = hi + t;
      const bool pass = in && max_m - eps <= tt && tt <= min_u + eps && t <= min_m + eps;
      const R next = ei < cnt ? static_cast<R>(list[ei]) : rest;
      const bool take = pass && (ei == m || next - eps <= t);
      const unsigned long long taken = __ballot(take);
      if (taken) {
        rec.n_hi = u;
        rec.n_mid = e0 + __ffsll(taken) - 1 - u;
        list_cone_values(list, ps, u, u + rec.n_mid, k_u, nu, rec.t, rec.hi);
        return rec;
      }
      // Nothing accepted up to e: where t is certainly above every later
      // min(M) (the bound above, next the largest value still to come), the
      // search for this u is over.
      const R tol = R(2) * eps + R(8) * num<R>::eps() * dmax(fabs(t), fabs(next));
      const bool ends = !(next > -num<R>::inf()) ||
                        den * (t - next) > tol * (den + static_cast<R>(m - ei) * nu);
      if (e0 + 64 > cnt) {
        if (cnt < m && __ballot(in && e == cnt && (pass || !ends))) {
          rec.state = SEL_WIDER;
          return rec;
        }
        break;
      }
      if (__ballot(in && ends)) break;
    }
  }
  rec.t = rec.hi = R(0);
  rec.branch = SDCA_BRANCH_DEFAULT;
  rec.n_hi = rec.n_mid = 0;
  return rec;
}

// The record from the sorted list (list_sort): thresholds_topk_cone,
// thresholds_topk_simplex and the biased forms (topk_cone.h:18-157,
// topk_simplex.h:39-68, topk_simplex_biased.h:40-71,
// topk_cone_biased.h:98-113).  complete: every value above the knapsack's
// threshold is in the list (otherwise the special cases only, and SEL_FIX).
template <class D, class R>
__device__ inline SelectRecord<R> list_record(const D* list, const double* ps, int cnt, int m, D cut,
                                              const ProxParamsT<R>& pp, bool complete) {
  const int k = pp.k;
  const R K = static_cast<R>(k);
  const R rho = pp.rho, rhs = pp.rhs;
  const R eps16 = R(16) * num<R>::eps();
  const bool cone = pp.op == OP_TOPK_CONE || pp.op == OP_TOPK_CONE_BIASED;
  SelectRecord<R> rec;
  rec.state = SEL_DONE;
  rec.t = rec.hi = R(0);
  rec.branch = SDCA_BRANCH_ZERO;
  rec.n_hi = rec.n_mid = 0;
  if (cnt < k) return rec;  // masked classes among the k largest: no sum above 0
  const R sum_k = list_sum<R>(list, ps, 0, k);
  if (sum_k <= eps16) return rec;
  const R hi_c = sum_k / (K + rho * K * K);
  const R t_c = static_cast<R>(list[k - 1]) - hi_c;
  const bool constant =
      k == m || t_c >= static_cast<R>(k < cnt ? list[k] : list_rest(cut)) - eps16;
  const R eps = num<R>::eps() * dmax(R(1), fabs(rhs));
  if (constant && (cone || !(K * hi_c > rhs + eps))) {
    rec.t = t_c;
    rec.hi = hi_c;
    rec.branch = SDCA_BRANCH_CONSTANT;
    rec.n_hi = k;
    return rec;
  }
  if (!cone) {
    if (!complete) {
      rec.state = SEL_FIX;
      return rec;
    }
    int u, e;
    list_knapsack<D, R>(list, ps, cnt, m, cut, k, pp.rhs_k, rhs, rec.t, u, e);
    bool lt = false;
    if (!constant) {
      if (u == 0) {
        lt = rec.t < rho * rhs - eps;
      } else {
        const R num_u = static_cast<R>(u);
        lt = K * (list_sum<R>(list, ps, 0, u) + (K - num_u) * rec.t) < rhs * (num_u + rho * K * K) - eps;
      }
    }
    if (!lt) {
      rec.hi = pp.rhs_k;
      rec.branch = SDCA_BRANCH_KNAPSACK;
      rec.n_hi = u;
      rec.n_mid = e - u;
      return rec;
    }
  }
  // Without the bias the search's U = 0 partition is every value above 16
  // eps: its sum needs the whole column.
  if (rho == R(0)) {
    rec.state = SEL_U0;
    return rec;
  }
  return list_cone<D, R>(list, ps, cnt, m, cut, k, rho, 0);
}

}  // namespace sdca_gpu

#endif
