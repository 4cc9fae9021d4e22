// Thresholds from a short sorted list of a column's largest values, by one
// wave: the list's sort and prefix sums, the knapsack's partition
// (knapsack_eq.h:25-109) with one rank per lane, the U/M searches of the top-k
// cones (topk_cone.h:58-133, topk_cone_biased.h:9-106) with one candidate end
// per lane.  Used by the selection kernel of the top-k operators and by the
// SDCA epoch.
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

// Exclusive prefix sum over the wave (as wave_exclusive_scan_dpp).
__device__ inline double wave_exclusive_scan(double x) {
  double incl = x;
  incl = dpp_add<0x111, 0xF, true>(incl);   // row_shr:1
  incl = dpp_add<0x112, 0xF, true>(incl);   // row_shr:2
  incl = dpp_add<0x114, 0xF, true>(incl);   // row_shr:4
  incl = dpp_add<0x118, 0xF, true>(incl);   // row_shr:8
  incl = dpp_add<0x142, 0xA, false>(incl);  // row_bcast:15
  incl = dpp_add<0x143, 0xC, false>(incl);  // row_bcast:31
  return incl - x;
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

// The partition of the knapsack sum_i clamp(a_i - t, 0, hi) = rhs on the
// sorted list (every value above t is in it): rank r is above t where
// f(a_r) < rhs and at hi where f(a_r - hi) <= rhs, one rank per lane, f from
// the prefix sums and a binary search for the ranks at hi (or inside) at
// that point.  The same eps as the fixing's (topk_sorted_root).  The
// threshold is formed from the direct sum over the free ranks; with none
// free any t of [a_u, a_(u-1) - hi] is the same projection and the record
// takes the middle.  With inv_rho > 0 the right side is t inv_rho instead
// (the biased knapsack with its sum constraint inactive,
// knapsack_le_biased.h:10-92; f(t) - t inv_rho is decreasing as f is).
template <class D, class R>
__device__ inline void list_knapsack(const D* list, const double* ps, int cnt, int m, D cut, R hi_r,
                                     R rhs_r, R& t_out, int& u_out, int& e_out,
                                     R inv_rho_r = R(0)) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const double hi = static_cast<double>(hi_r), rhs = static_cast<double>(rhs_r);
  const double eps = static_cast<double>(num<R>::eps() * dmax(R(1), fabs(rhs_r)));
  const double inv_rho = static_cast<double>(inv_rho_r);
  auto target = [&](double v) { return inv_rho > 0 ? v * inv_rho : rhs; };
  int e = 0, u = 0;
  for (int base = 0; base < cnt; base += 64) {
    const int r = base + lane;
    bool above = false, at_hi = false;
    if (r < cnt) {
      const double a = static_cast<double>(list[r]);
      int b = 0, w = r;
      while (b < w) {  // ranks above a + hi
        const int mid = (b + w) >> 1;
        if (static_cast<double>(list[mid]) > a + hi) b = mid + 1;
        else w = mid;
      }
      above = ps[r] - ps[w] - static_cast<double>(r - w) * a + static_cast<double>(w) * hi <
              target(a) - eps;
      int z = cnt;
      b = r + 1;
      while (b < z) {  // ranks above a - hi
        const int mid = (b + z) >> 1;
        if (static_cast<double>(list[mid]) > a - hi) b = mid + 1;
        else z = mid;
      }
      at_hi = static_cast<double>(r + 1) * hi + (ps[z] - ps[r + 1]) -
                  static_cast<double>(z - r - 1) * (a - hi) <= target(a - hi) + eps;
    }
    e += __popcll(__ballot(above));
    u += __popcll(__ballot(at_hi));
    if (base + 64 > e && base + 64 > u) break;  // no later rank is above t
  }
  if (u > e) u = e;
  if (e > u) {
    double s = 0;
    for (int i = u + lane; i < e; i += 64) s += static_cast<double>(list[i]);
    s = wave_total(s);
    t_out = inv_rho > 0 ? static_cast<R>((s + static_cast<double>(u) * hi) /
                                         (inv_rho + static_cast<double>(e - u)))
                        : static_cast<R>((s + static_cast<double>(u) * hi - rhs) /
                                         static_cast<double>(e - u));
  } else if (inv_rho > 0) {
    t_out = static_cast<R>(static_cast<double>(u) * hi / inv_rho);
  } else {
    const double top = (u > 0 ? static_cast<double>(list[u - 1]) : static_cast<double>(list[0])) - hi;
    double low = top;
    if (u < cnt) low = static_cast<double>(list[u]);
    else if (u < m) low = static_cast<double>(cut);
    t_out = static_cast<R>(0.5 * (low + top));
  }
  u_out = u;
  e_out = e;
}

// topk_cone_search (topk_cone.h:58-133) and its biased form
// (topk_cone_biased.h:9-106) on the sorted list, from |U| = u_first on: for
// each |U| = u the candidate ends e of M = ranks [u, e) are tried by the
// lanes, the smallest accepted e of the smallest u wins, as in the
// reference's order.  The list holds the column's cnt largest values, the
// others are at most `cut`.  Where a search for some u may continue past
// the list (no end accepted, and t not certainly above every M that would;
// the bound of cone_biased_regs) the result is SEL_WIDER.
template <class D, class R>
__device__ inline SelectRecord<R> list_cone(const D* list, const double* ps, int cnt, int m, D cut,
                                            int k, R rho, int u_first) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const R eps = R(16) * num<R>::eps();
  const R K = static_cast<R>(k);
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
      const R next = ei < cnt ? static_cast<R>(list[ei]) : static_cast<R>(cut);
      const bool take = pass && (ei == m || next - eps <= t);
      const unsigned long long taken = __ballot(take);
      if (taken) {
        const int l = __ffsll(taken) - 1;
        rec.t = read_lane(t, __builtin_amdgcn_readfirstlane(l));
        rec.hi = read_lane(hi, __builtin_amdgcn_readfirstlane(l));
        rec.n_hi = u;
        rec.n_mid = e0 + l - u;
        return rec;
      }
      // Nothing accepted up to e: where t is certainly above every later
      // min(M) (the bound above, next the largest value still to come), the
      // search for this u is over.
      const R tol = R(2) * eps + R(8) * num<R>::eps() * dmax(fabs(t), fabs(next));
      const bool ends = den * (t - next) > tol * (den + static_cast<R>(m - ei) * nu);
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
// CHAIN: the cone search by the sorted column's own chain of sums.
template <class D, class R, bool CHAIN = false>
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
  const R sum_k = static_cast<R>(ps[k]);
  if (sum_k <= eps16) return rec;
  const R hi_c = sum_k / (K + rho * K * K);
  const R t_c = static_cast<R>(list[k - 1]) - hi_c;
  const bool constant = k == m || t_c >= static_cast<R>(list[k < cnt ? k : k - 1]) - eps16;
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
    list_knapsack<D, R>(list, ps, cnt, m, cut, pp.rhs_k, rhs, rec.t, u, e);
    bool lt = false;
    if (!constant) {
      if (u == 0) {
        lt = rec.t < rho * rhs - eps;
      } else {
        const R num_u = static_cast<R>(u);
        lt = K * (static_cast<R>(ps[u]) + (K - num_u) * rec.t) < rhs * (num_u + rho * K * K) - eps;
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
  if constexpr (CHAIN) {
    if (!cone_search_sorted<D, R>(list, cnt, m, static_cast<R>(cut), k, rho, rec.t, rec.hi,
                                  rec.branch, rec.n_hi, rec.n_mid))
      rec.state = SEL_WIDER;
    return rec;
  }
  return list_cone<D, R>(list, ps, cnt, m, cut, k, rho, 0);
}

// Value i (uniform) of a wave's list, or of its prefix sums.
template <int CC, class T>
__device__ inline T list_at(const T (&x)[CC], int i) {
  T r = read_lane(x[0], i / CC);
#pragma unroll
  for (int c = 1; c < CC; ++c) r = (i % CC == c) ? read_lane(x[c], i / CC) : r;
  return r;
}

// The prefix sums of list_prefix in R (the register solves below decide the
// partition with them; the threshold comes from a direct sum).
__device__ inline float wave_exclusive_scan(float x) {
  float incl = x;
  incl = dpp_add<0x111, 0xF, true>(incl);   // row_shr:1
  incl = dpp_add<0x112, 0xF, true>(incl);   // row_shr:2
  incl = dpp_add<0x114, 0xF, true>(incl);   // row_shr:4
  incl = dpp_add<0x118, 0xF, true>(incl);   // row_shr:8
  incl = dpp_add<0x142, 0xA, false>(incl);  // row_bcast:15
  incl = dpp_add<0x143, 0xC, false>(incl);  // row_bcast:31
  return incl - x;
}
template <int CC, class D, class R>
__device__ inline void regs_prefix(const D (&x)[CC], R (&ex)[CC], int cnt) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  R tot = 0;
#pragma unroll
  for (int c = 0; c < CC; ++c) tot += (lane * CC + c < cnt) ? static_cast<R>(x[c]) : R(0);
  R run = wave_exclusive_scan(tot);
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    ex[c] = run;
    run += (lane * CC + c < cnt) ? static_cast<R>(x[c]) : R(0);
  }
}

// sum_{i < r} min(a_i - a_r, hi) for each value a_r of the sorted list, its
// prefix sums less what lies above a_r + hi, which only the `most` largest
// can: the knapsack's sum at t = a_r where hi most >= the sums of interest.
template <int CC, class D, class R>
__device__ inline void regs_sums(const D (&x)[CC], const R (&ex)[CC], int most, R hi, R (&f)[CC]) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  R over[CC];
#pragma unroll
  for (int c = 0; c < CC; ++c) over[c] = R(0);
  for (int j = 0; j < most; ++j) {
    const R top = static_cast<R>(list_at<CC>(x, j)) - hi;
#pragma unroll
    for (int c = 0; c < CC; ++c) over[c] += dmax(top - static_cast<R>(x[c]), R(0));
  }
#pragma unroll
  for (int c = 0; c < CC; ++c)
    f[c] = ex[c] - static_cast<R>(lane * CC + c) * static_cast<R>(x[c]) - over[c];
}

// list_knapsack on the list in the wave's registers, for hi k >= rhs with at
// most k values at hi: the end e of the values above t from regs_sums, and
// the |U| = u whose t_u = (sum_M a + u hi - rhs) / (e - u) puts a_(u-1) at or
// above t_u + hi and a_u below it, one u per lane (topk_sorted_root's tests).
// False where no u fits (M empty, ties at rounding level): list_knapsack
// decides.
template <int CC, class D, class R>
__device__ inline bool regs_knapsack(const D (&x)[CC], const R (&ex)[CC], int cnt, int k, R hi, R rhs,
                                     R inv_rho, R& t_out, int& u_out, int& e_out, R& sum_u) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const R eps = num<R>::eps() * dmax(R(1), fabs(rhs));
  const int most = k < cnt ? k : cnt;
  R f[CC];
  regs_sums<CC, D, R>(x, ex, most, hi, f);
  int e = 0;
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const R goal = inv_rho > 0 ? static_cast<R>(x[c]) * inv_rho : rhs;
    e += __popcll(__ballot(lane * CC + c < cnt && f[c] < goal - eps));
  }
  if (e == 0) return false;
  // the sum of the first e values
  const R pe = list_at<CC>(ex, e - 1) + static_cast<R>(list_at<CC>(x, e - 1));
  // a_(r - 1): the slot before, or the last slot of the lane before (wave_shr:1)
  int u = INT_MAX;
  D before;
  if constexpr (sizeof(D) == 4) {
    before = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x[CC - 1]), 0x138, 0xF, 0xF,
                                                        true));
  } else {
    const long long b = __double_as_longlong(x[CC - 1]);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b & 0xffffffffll), 0x138, 0xF, 0xF,
                                               true);
    const int up = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), 0x138, 0xF, 0xF, true);
    before = __longlong_as_double((static_cast<long long>(up) << 32) |
                                  static_cast<long long>(static_cast<unsigned>(lo)));
  }
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int r = lane * CC + c;
    const D prev = c == 0 ? before : x[c > 0 ? c - 1 : 0];
    const R left = static_cast<R>(e - r);
    const R den = inv_rho > 0 ? inv_rho + left : left;
    const R num_r = (pe - ex[c]) + static_cast<R>(r) * hi - (inv_rho > 0 ? R(0) : rhs);
    const bool fits = r < most && r < e && (r == 0 || (static_cast<R>(prev) - hi) * den >= num_r) &&
                      (static_cast<R>(x[c]) - hi) * den < num_r;
    const unsigned long long mask = __ballot(fits);
    if (mask) {
      const int first = (__ffsll(mask) - 1) * CC + c;
      u = first < u ? first : u;
    }
  }
  if (u == INT_MAX) return false;
  sum_u = list_at<CC>(ex, u);
  double s = 0;
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int r = lane * CC + c;
    s += (r >= u && r < e) ? static_cast<double>(x[c]) : 0.0;
  }
  s = wave_total(s) + static_cast<double>(u) * static_cast<double>(hi);
  const double left = static_cast<double>(e - u);
  t_out = inv_rho > 0 ? static_cast<R>(div_near(s, static_cast<double>(inv_rho) + left))
                      : static_cast<R>(div_near(s - static_cast<double>(rhs), left));
  u_out = u;
  e_out = e;
  return true;
}

// list_record on the list in the wave's registers where it is decided there
// (the special cases and the knapsack); false leaves it to list_record.
template <int CC, class D, class R>
__device__ inline bool regs_record(const D (&x)[CC], const R (&ex)[CC], int cnt, int m,
                                   const ProxParamsT<R>& pp, SelectRecord<R>& rec) {
  const int k = pp.k;
  if (pp.op == OP_TOPK_CONE || pp.op == OP_TOPK_CONE_BIASED || k >= 64 * CC || k > cnt) return false;
  const R K = static_cast<R>(k);
  const R rho = pp.rho, rhs = pp.rhs;
  const R eps16 = R(16) * num<R>::eps();
  rec.state = SEL_DONE;
  rec.t = rec.hi = R(0);
  rec.branch = SDCA_BRANCH_ZERO;
  rec.n_hi = rec.n_mid = 0;
  const R kth = static_cast<R>(list_at<CC>(x, k - 1));
  const R sum_k = list_at<CC>(ex, k - 1) + kth;
  if (sum_k <= eps16) return true;
  const R hi_c = sum_k / (K + rho * K * K);
  const R t_c = kth - hi_c;
  // (past the list: -inf, only where the column ends there)
  const bool constant = k == m || t_c >= static_cast<R>(list_at<CC>(x, k)) - eps16;
  const R eps = num<R>::eps() * dmax(R(1), fabs(rhs));
  if (constant && !(K * hi_c > rhs + eps)) {
    rec.t = t_c;
    rec.hi = hi_c;
    rec.branch = SDCA_BRANCH_CONSTANT;
    rec.n_hi = k;
    return true;
  }
  int u, e;
  R sum_u;
  if (!regs_knapsack<CC, D, R>(x, ex, cnt, k, pp.rhs_k, rhs, R(0), rec.t, u, e, sum_u)) return false;
  if (!constant) {
    bool lt;
    const R num_u = static_cast<R>(u);
    if (u == 0) lt = rec.t < rho * rhs - eps;
    else lt = K * (sum_u + (K - num_u) * rec.t) < rhs * (num_u + rho * K * K) - eps;
    if (lt) return false;
  }
  rec.hi = pp.rhs_k;
  rec.branch = SDCA_BRANCH_KNAPSACK;
  rec.n_hi = u;
  rec.n_mid = e - u;
  return true;
}

// A lower bound of the threshold of sum_i clamp(a_i - t, 0, hi) = rhs over a
// column from its 64 sorted part maxima, rank r in lane r (hi k >= rhs):
// f over the maxima alone is at most f over the column, so their first rank
// with f >= rhs is at most t, and so is a_(k) - hi (maximum k bounds a_(k)).
// Less rounding (f's own, relative to its terms, through its slope of at
// least one).
template <class D, class R>
__device__ inline D parts_lower(const D (&part)[1], int k, R hi, R rhs) {
  R ex[1], f[1];
  regs_prefix<1, D, R>(part, ex, 64);
  regs_sums<1, D, R>(part, ex, k, hi, f);
  const unsigned long long mask = __ballot(f[0] >= rhs);
  R b = static_cast<R>(read_lane(part[0], k)) - hi;
  const R top = static_cast<R>(read_lane(part[0], 0));
  if (mask) {
    const R p = static_cast<R>(read_lane(part[0], __ffsll(mask) - 1)) -
                (fabs(top) + rhs) * (R(256) * num<R>::eps());
    b = p > b ? p : b;
  }
  return static_cast<D>(b - (fabs(b) + hi) * (R(16) * num<R>::eps()));
}

}  // namespace sdca_gpu

#endif
