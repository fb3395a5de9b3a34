// Refine, coarsen and swap passes, the independent set, the adapt driver
// and warp_to_limit, on a device-resident mesh.  Every per-entity loop is
// a gfx950 kernel; the host only sequences passes and reads counts.
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>

#include "ohx_adapt.hpp"
#include "ohx_geom.hpp"
#include "ohx_prims.hpp"
#include "ohx_scan.hpp"
#include "ohx_tables.hpp"

namespace ohx {

int g_verbose = 0;
// indset.cpp:33 stops after 100 rounds; raising it is an extension
u32 g_indset_max_rounds = 100;
// the most rounds a set that went to the checked loop needed (a set that
// settles in the first unchecked batch needs at most 8)
std::atomic<u32> g_indset_rounds_seen{0};
// FP32 screening with FP64 re-evaluation near every decision (extension)
bool g_mixed = false;

static double now_s() {
  using namespace std::chrono;
  return duration<double>(steady_clock::now().time_since_epoch()).count();
}

// scratch word slots (zeroed by a fill kernel before each use)
enum { W_ANY = 0, W_CACHED = 1, W_FLAGS = 8, W_STATS = 40 };
// FP32-mixed statistics: two slotted u64 counters (decisions settled in
// FP32, FP64 re-evaluations) in a buffer of their own, float bits of the
// max |q32 - q64| at scratch word 40
struct ScreenStats {
  unsigned long long* screened;
  unsigned long long* reeval;
  u32* max_err;
};
constexpr size_t STAT_WORDS = (size_t) STAT_SLOTS * STAT_STRIDE;
static unsigned long long* stat_counters() {
  // one buffer per thread, for the life of the thread, zeroed once
  static thread_local unsigned long long* c = nullptr;
  if (!c) {
    c = static_cast<unsigned long long*>(dev_alloc(2 * STAT_WORDS * sizeof(unsigned long long)));
    OHX_CHECK(hipMemsetAsync(c, 0, 2 * STAT_WORDS * sizeof(unsigned long long), stream()));
  }
  return c;
}
static ScreenStats screen_stats() {
  unsigned long long* c = stat_counters();
  return ScreenStats{c, c + STAT_WORDS, scratch_words() + W_STATS};
}

void mixed_stats(double* max_err, unsigned long long* screened, unsigned long long* reeval) {
  std::vector<unsigned long long> c(2 * STAT_WORDS);
  to_host(c.data(), stat_counters(), c.size());
  unsigned long long a = 0, b = 0;
  for (u32 k = 0; k < STAT_SLOTS; ++k) {
    a += c[(size_t) k * STAT_STRIDE];
    b += c[STAT_WORDS + (size_t) k * STAT_STRIDE];
  }
  u32 h = read_at(scratch_words(), W_STATS);
  float e;
  std::memcpy(&e, &h, 4);
  if (max_err) *max_err = e;
  if (screened) *screened = a;
  if (reeval) *reeval = b;
}

void mixed_stats_reset() {
  OHX_CHECK(hipMemsetAsync(stat_counters(), 0, 2 * STAT_WORDS * sizeof(unsigned long long), stream()));
  fill(scratch_words() + W_STATS, 1, 0);
}

// one scratch word, read through the mapped-memory gather (one small kernel
// and a wait, cheaper than a device-to-host copy)
static u32 read_word(u32 k) {
  u32 const* p = scratch_words() + k;
  u32 v = 0;
  read_many(&p, 1, &v);
  return v;
}
// a new value for the tagged "any" word W_ANY (never 0, the cleared value)
static u32 next_any_tag() {
  static thread_local u32 t = 0;
  t = t + 1 ? t + 1 : 1;
  return t;
}

// ------------------------------------------------------- independent set
// One Jacobi round of the deterministic Luby variant (indset.cpp:55-84):
// an undecided entity leaves the set if a neighbour is in it, waits if a
// live neighbour has larger goodness or equal goodness and a lower index,
// and joins otherwise.  flag is set if anything is still undecided.
enum { NOT_IN_SET = 0, IN_SET = 1, UNKNOWN = 2 };

__global__ __launch_bounds__(BLOCK) void indset_round(u32 n, u32 const* __restrict__ offs,
                                                      u32 const* __restrict__ adj,
                                                      double const* __restrict__ good,
                                                      u32 const* __restrict__ old, u32* __restrict__ state,
                                                      u32* __restrict__ flag) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  bool undecided = false;
  if (i < n) {
    u32 s = old[i];
    if (s == UNKNOWN) {
      // one walk over the neighbours: a neighbour in the set decides at
      // once; otherwise a live neighbour with larger goodness (or equal
      // goodness and a lower index) makes this one wait (goodness is read
      // only until the first such neighbour)
      u32 f = offs[i], e = offs[i + 1];
      double const myg = good[i];
      bool wait = false, out = false;
      for (u32 j = f; j < e; ++j) {
        u32 o = adj[j];
        u32 so = old[o];
        if (so == IN_SET) {
          out = true;
          break;
        }
        if (so == NOT_IN_SET || wait) continue;
        double og = good[o];
        if ((myg == og && o < i) || myg < og) wait = true;
      }
      s = out ? (u32) NOT_IN_SET : (wait ? (u32) UNKNOWN : (u32) IN_SET);
      undecided = !out && wait;
    }
    state[i] = s;
  }
  wave_flag(flag, undecided);
}

// The same round over the edges of a mesh with the neighbours taken from the
// elements around each edge (up(1,dim), down(dim,1); NE edges per element):
// an edge's neighbours are the other edges of its elements, which as a set
// is the edge star star(1,dim) (in 3D the two other edges of every triangle
// through the edge and the opposite edge of every tet through it); the rule
// depends only on that set, so the star itself, which would need up(1,2) in
// 3D, is not built.  Bound by the gathers around undecided edges; the walk
// meets a neighbour once per shared element, about twice the star's reads,
// but a split pass saves the star, which cost far more than its rounds
// (384,000 tets, 5 split passes: up(1,2) and the star 1.9 ms of 9.5 ms).
template <u32 NE>
__global__ __launch_bounds__(BLOCK) void indset_round_elems(u32 n, u32 const* __restrict__ uo,
                                                            u32 const* __restrict__ ua, u32 const* __restrict__ ud,
                                                            u32 const* __restrict__ er,
                                                            double const* __restrict__ good,
                                                            u32 const* __restrict__ old, u32* __restrict__ state,
                                                            u32* __restrict__ flag) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  bool undecided = false;
  if (i < n) {
    u32 s = old[i];
    if (s == UNKNOWN) {
      double const myg = good[i];
      bool wait = false, out = false;
      for (u32 j = uo[i]; j < uo[i + 1] && !out; ++j) {
        u32 t = ua[j], d = ud[j];
        for (u32 l = 0; l < NE; ++l) {
          if (l == d) continue;
          u32 o = er[NE * (size_t) t + l];
          u32 so = old[o];
          if (so == IN_SET) {
            out = true;
            break;
          }
          if (so == NOT_IN_SET || wait) continue;
          double og = good[o];
          if ((myg == og && o < i) || myg < og) wait = true;
        }
      }
      s = out ? (u32) NOT_IN_SET : (wait ? (u32) UNKNOWN : (u32) IN_SET);
      undecided = !out && wait;
    }
    state[i] = s;
  }
  wave_flag(flag, undecided);
}

// The same round over the vertices, with the neighbours taken from the
// edges (up(0,1), down(1,0)): in a simplicial mesh two vertices share an
// element exactly when they share an edge, so the other ends of a vertex's
// edges are, as a set, its star star(0,dim), which is then not built.
__global__ __launch_bounds__(BLOCK) void indset_round_verts(u32 n, u32 const* __restrict__ uo,
                                                            u32 const* __restrict__ ua, u32 const* __restrict__ ud,
                                                            u32 const* __restrict__ ev,
                                                            double const* __restrict__ good,
                                                            u32 const* __restrict__ old, u32* __restrict__ state,
                                                            u32* __restrict__ flag) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  bool undecided = false;
  if (i < n) {
    u32 s = old[i];
    if (s == UNKNOWN) {
      double const myg = good[i];
      bool wait = false, out = false;
      for (u32 j = uo[i]; j < uo[i + 1]; ++j) {
        u32 o = ev[2 * (size_t) ua[j] + (1 - ud[j])];
        u32 so = old[o];
        if (so == IN_SET) {
          out = true;
          break;
        }
        if (so == NOT_IN_SET || wait) continue;
        double og = good[o];
        if ((myg == og && o < i) || myg < og) wait = true;
      }
      s = out ? (u32) NOT_IN_SET : (wait ? (u32) UNKNOWN : (u32) IN_SET);
      undecided = !out && wait;
    }
    state[i] = s;
  }
  wave_flag(flag, undecided);
}

// rounds == 0: rounds in batches with a host check after each, up to the
// limit (the reference's loop); rounds > 0: exactly that many rounds and no
// host check, *last_flag then points at the device word that is nonzero if
// entities were still undecided after the last round
// start (with start_done rounds already run): the checked loop continues
// from that state instead of from the filter (rounds are a function of the
// state alone, so the result and the round count are those of a run from
// the start)
static void note_rounds(u32 used) {
  u32 seen = g_indset_rounds_seen.load();
  while (used > seen && !g_indset_rounds_seen.compare_exchange_weak(seen, used)) {
  }
}

static Buf<u32> indset_rounds(Mesh& m, u32 ent_dim, u32 const* filter, double const* good, u32 rounds,
                              u32 const** last_flag, Buf<u32>* start = nullptr, u32 start_done = 0) {
  u32 n = count(m, ent_dim);
  // vertices: neighbours through the edges (indset_round_verts); edges:
  // through the elements (indset_round_elems), unless the star, which holds
  // each neighbour once, is there already (set of a 162,000-tet mesh's edges:
  // 343 us by the star, 415 through the elements)
  bool const via_edges = ent_dim == 0 && m.dim >= 2;
  bool const via_elems = ent_dim == 1 && m.dim >= 2 && !m.star[1][m.dim];
  Graph empty;
  Graph const& g = (via_elems || via_edges) ? empty : ask_star(m, ent_dim, m.dim);
  Up const* ut = via_elems ? &ask_up(m, 1, m.dim) : via_edges ? &ask_up(m, 0, 1) : nullptr;
  u32 const* er = via_elems ? ask_down(m, m.dim, 1) : via_edges ? ask_down(m, 1, 0) : nullptr;
  auto round = [&](u32 const* in, u32* outs, u32* fl, double bytes) {
    if (via_elems)
      launch_timed("indset_round", bytes, m.dim == 3 ? indset_round_elems<6> : indset_round_elems<3>, dim3(nblocks(n)),
                   dim3(BLOCK), n, ut->offsets.get(), ut->adj.get(), ut->dirs.get(), er, good, in, outs, fl);
    else if (via_edges)
      launch_timed("indset_round", bytes, indset_round_verts, dim3(nblocks(n)), dim3(BLOCK), n, ut->offsets.get(),
                   ut->adj.get(), ut->dirs.get(), er, good, in, outs, fl);
    else
      launch_timed("indset_round", bytes, indset_round, dim3(nblocks(n)), dim3(BLOCK), n, g.offsets.get(),
                   g.adj.get(), good, in, outs, fl);
  };
  bool const resume = start && *start;
  Buf<u32> a = resume ? std::move(*start) : Buf<u32>(n), b(n);
  constexpr u32 BATCH = 8;
  u32* flags = scratch_words() + W_FLAGS;
  if (!resume) {
    // the states, and the first batch's round flags cleared on the way
    u32* s = a.get();
    parallel_for(n, OHX_LAMBDA(u32 i) {
      s[i] = filter[i] ? UNKNOWN : NOT_IN_SET;
      if (i < BATCH) flags[i] = 0;
    });
  }
  if (!n) {
    if (rounds) {
      fill(flags, 1, 0);
      *last_flag = flags;
    }
    return a;
  }
  // compulsory bytes per round: every state read and written once (the
  // goodness and the star are read only around undecided entities, a count
  // the host does not know, so they are left out: a lower bound)
  double round_bytes = (double) n * 8;
  // rounds are launched in batches; a round after convergence copies the
  // state unchanged, so running past the converged round is harmless
  // rounds per host check: most sets settle within 8 rounds
  u32 const MAX_ROUNDS = g_indset_max_rounds;
  if (rounds) {
    u32 nr = rounds < BATCH ? rounds : BATCH;
    if (n < nr) fill(flags, nr, 0);  // the set-up kernel cleared flags [0, n)
    for (u32 r = 0; r < nr; ++r) {
      round(a.get(), b.get(), flags + r, round_bytes);
      std::swap(a, b);
    }
    *last_flag = flags + nr - 1;
    return a;
  }
  for (u32 done = resume ? start_done : 0; done < MAX_ROUNDS; done += BATCH) {
    // the last batch stops at the limit, as the reference's loop does
    u32 nr = MAX_ROUNDS - done < BATCH ? MAX_ROUNDS - done : BATCH;
    if (done || n < nr) fill(flags, nr, 0);
    for (u32 r = 0; r < nr; ++r) {
      round(a.get(), b.get(), flags + r, round_bytes);
      std::swap(a, b);
    }
    u32 h[BATCH];
    u32 const* fp[BATCH];
    for (u32 r = 0; r < nr; ++r) fp[r] = flags + r;
    read_many(fp, nr, h);
    if (!h[nr - 1]) {
      // h[r]: entities still undecided after round r of this batch
      u32 k = 0;
      while (h[k]) ++k;
      note_rounds(done + k + 1);
      return a;
    }
  }
  fail("independent set did not converge within the round limit (indset.cpp:107-116)", __FILE__, __LINE__);
  return a;
}

Buf<u32> find_indset(Mesh& m, u32 ent_dim, u32 const* filter, double const* good) {
  return indset_rounds(m, ent_dim, filter, good, 0, nullptr);
}


// a first batch of rounds with no host check; if the set has not settled
// the caller goes on from its state with the checked loop
// (find_indset_resume: same rounds, same result).  The batch never runs
// more rounds than the limit allows, so a set that needs more than the
// limit always reaches the checked loop's failure.
// Four rounds: measured on the 64^3 x 6 anisotropic box (8 cycles), 87 % of the vertex sets and
// 95 % of the edge sets settle within four rounds (most within two), so a
// longer first batch mostly launches rounds that only copy a settled state.
static u32 first_batch_rounds() { return g_indset_max_rounds < 4 ? g_indset_max_rounds : 4; }
static Buf<u32> find_indset_bounded(Mesh& m, u32 ent_dim, u32 const* filter, double const* good,
                                    u32 const** last_flag) {
  return indset_rounds(m, ent_dim, filter, good, first_batch_rounds(), last_flag);
}
// the same from states that are set up already (UNKNOWN or NOT_IN_SET, the
// round flags cleared): the kernels that decide the candidates write them
static Buf<u32> find_indset_from(Mesh& m, u32 ent_dim, Buf<u32>&& state, double const* good,
                                 u32 const** last_flag) {
  return indset_rounds(m, ent_dim, nullptr, good, first_batch_rounds(), last_flag, &state);
}
constexpr u32 INDSET_FLAGS = 8;
// the checked loop from the first batch's state
static Buf<u32> find_indset_resume(Mesh& m, u32 ent_dim, double const* good, Buf<u32>&& state) {
  return indset_rounds(m, ent_dim, nullptr, good, 0, nullptr, &state, first_batch_rounds());
}

struct UpPatchCounts;
static std::unique_ptr<Up> up_patch(u32 deg, Up const& old, u32 nl_old, u32 const* soff_l, u32 nsame_l,
                                    u32 ngen_l, u32 const* soff_h, u32 nsame_h, u32 ngen_h, u32 const* dn,
                                    UpPatchCounts* keep = nullptr);

// ------------------------------------------------------------- inherit
// Class tags (class_dim, class_id) of products come from the entity they
// were made from (inherit.cpp:14-232); the fused output kernels of each
// pass write them next to the connectivity.

// --------------------------------------------------------------- refine
// the minimum over a group of G lanes (it does not depend on the order, so
// the result is the serial loop's)
template <u32 G>
__device__ inline double group_min(double v) {
#pragma unroll
  for (u32 d = G / 2; d >= 1; d >>= 1) {
    double o = __shfl_xor(v, d, G);
    if (o < v) v = o;
  }
  return v;
}

// Worst child quality of every candidate edge split
// (refine_qualities.cpp:16-82); rejected candidates are cleared, the others
// become UNKNOWN: cand is then the independent set's first state, and the
// flags of its rounds are cleared on the way.
//
// FP64 arithmetic bounds it, and the lanes that take part in it: with a
// thread per edge, of which a few are candidates with rings of 3 to 12, a
// wave ran at 8 to 12 of its 64 lanes and a small mesh's call was as long as
// ten child qualities in a row.  A block lists the candidates of `per` edges
// and a group of four lanes takes each, a child per lane (a ring of five tets
// has ten): a call at 55 thousand tets 187 -> 111 us, in a box of 384 thousand
// 60 -> 35 us, at 3 thousand 23 -> 14 us (groups of 8: 218, 47 and 17 us, of
// 2: 208, 43 and 18 us, both with a quarter of the blocks).
constexpr u32 RQ_EDGES = 1024, RQ_BLOCKS = 4096;

template <u32 DIM>
struct SplitRing {
  V3 split;
  Sym msplit;
};

// the child t of a split: 2 to an element of the edge's ring
template <u32 DIM, bool F32>
__device__ inline double split_child_q(SplitRing<DIM> const& r, u32 e, u32 dir, u32 k, u32 const* __restrict__ ve,
                                       double const* __restrict__ x, double const* __restrict__ mt) {
  constexpr u32 VPE = DIM + 1;
  u32 const* bv = canon(DIM, DIM - 1, 0, opp(DIM, 0)[canon(DIM, 1, 0, dir)[k]]);
  V3 p[VPE];
#pragma unroll
  for (u32 l = 0; l + 1 < VPE; ++l) p[l] = ld3(x + 3 * (size_t) ve[(size_t) e * VPE + bv[l]]);
  p[VPE - 1] = r.split;
  if (mt) {
    Sym pm[VPE];
#pragma unroll
    for (u32 l = 0; l + 1 < VPE; ++l) pm[l] = ld6(mt + 6 * (size_t) ve[(size_t) e * VPE + bv[l]]);
    pm[VPE - 1] = r.msplit;
    return F32 ? (double) quality32<DIM>(p, pm, false) : metric_quality<DIM>(p, pm, false);
  }
  return F32 ? (double) quality32<DIM>(p, nullptr, false) : entity_quality(DIM, p);
}

// per: edges per block, at most RQ_EDGES
template <u32 DIM, bool MIXED>
__global__ __launch_bounds__(BLOCK) void refine_quality_f64(
    u32 ns, u32 per, u32 const* __restrict__ vs, u32 const* __restrict__ uo, u32 const* __restrict__ ua,
    u32 const* __restrict__ ud, u32 const* __restrict__ ve, double const* __restrict__ x,
    double const* __restrict__ mt, double const* __restrict__ eq, double qual_floor_all,
    double const* __restrict__ qfe, u32* __restrict__ cand, double* __restrict__ out, u32* __restrict__ words,
    u32* __restrict__ err, ScreenStats st) {
  constexpr u32 G = 4;
  __shared__ u32 list[RQ_EDGES], nlist;
  if (blockIdx.x == 0 && threadIdx.x < INDSET_FLAGS) words[W_FLAGS + threadIdx.x] = 0;
  if (threadIdx.x == 0) nlist = 0;
  __syncthreads();
  u32 const first = xcd_block() * per;
  for (u32 k = threadIdx.x; k < per && first + k < ns; k += BLOCK)
    if (cand[first + k]) list[atomicAdd(&nlist, 1u)] = first + k;
  __syncthreads();
  u32 const lane = threadIdx.x % G, n = nlist;
  for (u32 c = threadIdx.x / G; c < n; c += BLOCK / G) {
    u32 const i = list[c];
    // one floor for the mesh, or its component's in a batch
    double const qual_floor = qfe ? qfe[i] : qual_floor_all;
    u32 const v0 = vs[2 * (size_t) i], v1 = vs[2 * (size_t) i + 1];
    V3 a = ld3(x + 3 * (size_t) v0), b = ld3(x + 3 * (size_t) v1);
    // average_element_field (element_field.hpp:8-25): ((0 + a) + b) / 2
    SplitRing<DIM> r;
    {
      double s;
      s = 0; s += a.x; s += b.x; s /= 2; r.split.x = s;
      s = 0; s += a.y; s += b.y; s /= 2; r.split.y = s;
      s = 0; s += a.z; s += b.z; s /= 2; r.split.z = s;
    }
    // the new vertex's metric is the average its field would get on refinement
    if (mt) {
      Sym ma = ld6(mt + 6 * (size_t) v0), mb = ld6(mt + 6 * (size_t) v1);
      for (int k = 0; k < 6; ++k) {
        double s = 0;
        s += ma.m[k];
        s += mb.m[k];
        s /= 2;
        r.msplit.m[k] = s;
      }
    }
    u32 const begin = uo[i], nchild = 2 * (uo[i + 1] - begin);
    double minq32 = 1;
    if (MIXED && !eq) {
      // FP32 screen: a split certainly below the floor is rejected here; one
      // with a child near zero goes to FP64, which also checks q > 0
      bool sure = true;
      for (u32 t = lane; t < nchild; t += G) {
        u32 const j = begin + t / 2;
        double const q = split_child_q<DIM, true>(r, ua[j], ud[j], t & 1u, ve, x, mt);
        if (!(q > (double) SCREEN_MARGIN)) sure = false;
        if (q < minq32) minq32 = q;
      }
      minq32 = group_min<G>(minq32);
#pragma unroll
      for (u32 d = G / 2; d >= 1; d >>= 1) sure = __shfl_xor((int) sure, d, G) && sure;
      bool const reject = sure && ((float) minq32 < (float) qual_floor - SCREEN_MARGIN);
      if (lane == 0) wave_count(st.screened, reject);
      if (reject) {
        if (lane == 0) cand[i] = 0;
        continue;
      }
      if (lane == 0) wave_count(st.reeval, true);
    }
    double minq = 1, old_minq = 1;
    for (u32 t = lane; t < nchild; t += G) {
      u32 const j = begin + t / 2, e = ua[j];
      if (eq && eq[e] < old_minq) old_minq = eq[e];
      double const q = split_child_q<DIM, false>(r, e, ud[j], t & 1u, ve, x, mt);
      if (!(q > 0)) *err = ERR_REFINE_QUALITY;
      if (q < minq) minq = q;
    }
    minq = group_min<G>(minq);
    if (eq) old_minq = group_min<G>(old_minq);
    if (lane != 0) continue;
    if (MIXED && !eq && minq == minq) {
      float const d = (float) minq - (float) minq32;
      note_max_err(st.max_err, d < 0 ? -d : d);
    }
    if ((minq < qual_floor) || (eq && (minq <= old_minq))) {
      cand[i] = 0;
    } else {
      out[i] = minq;
      cand[i] = UNKNOWN;
    }
  }
}

// candidates of refine_by_size (refine.cpp:11-15), fused with measure_edge
__global__ __launch_bounds__(BLOCK) void refine_candidate_f64(u32 n, u32 const* __restrict__ ev,
                                                              double const* __restrict__ x,
                                                              double const* __restrict__ h,
                                                              double const* __restrict__ mt,
                                                              u32* __restrict__ cand, u32* __restrict__ words,
                                                              u32 tag) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  if (i >= n) return;
  u32 c = edge_size(ev[2 * i], ev[2 * i + 1], x, h, mt) > 1.0 ? 1u : 0u;
  cand[i] = c;
  wave_flag_value(words + W_ANY, c != 0, tag);
}

static Buf<double> refine_qualities(Mesh& m, u32* cand, double qual_floor, bool require_better,
                                    double const* qfe) {
  u32 dim = m.dim;
  u32 ns = count(m, 1);
  u32 const* vs = ask_down(m, 1, 0);
  u32 const* ve = ask_down(m, dim, 0);
  Up const& u = ask_up(m, 1, dim);
  Buf<double> eq;
  if (require_better) eq = mesh_qualities(m);
  Buf<double> out(ns);
  double prof_bytes = (double) ns * 20 + (double) u.adj.size() * 8 + (double) count(m, dim) * (dim + 1) * 4 + (double) count(m, 0) * 24;
  ScreenStats sst = screen_stats();
  // in the mixed mode the FP32 screen is a variant chosen online (it pays
  // only where it rejects enough splits); both give identical results
  static thread_local Tuner tuners[2] = {Tuner("refine_quality_2d_mixed", {0, 1}), Tuner("refine_quality_3d_mixed", {0, 1})};
  // a block's edges: as few as fill the chip (16 blocks per CU: the
  // candidates lie close together, and many small blocks even that out)
  u32 per = 32;
  while (per < RQ_EDGES && (u64) per * RQ_BLOCKS < ns) per *= 2;
  dim3 const grid((ns + per - 1) / per);
  auto go = [&](auto kernel, char const* kn, hipEvent_t ea, hipEvent_t eb) {
    if (ea) {
      hipExtLaunchKernelGGL(kernel, grid, dim3(BLOCK), 0, stream(), ea, eb, 0, ns, per, vs, u.offsets.get(),
                            u.adj.get(), u.dirs.get(), ve, coords(m), metric_of(m), eq.get(), qual_floor, qfe,
                            cand, out.get(), scratch_words(), dev_error_word(), sst);
      check_launch(kn);
    } else {
      launch_timed(kn, prof_bytes, kernel, grid, dim3(BLOCK), ns, per, vs, u.offsets.get(), u.adj.get(),
                   u.dirs.get(), ve, coords(m), metric_of(m), eq.get(), qual_floor, qfe, cand, out.get(),
                   scratch_words(), dev_error_word(), sst);
    }
  };
  auto run = [&](u32 screen, hipEvent_t ea, hipEvent_t eb) {
    if (dim == 3)
      screen ? go(refine_quality_f64<3, true>, "refine_quality_mixed", ea, eb)
             : go(refine_quality_f64<3, false>, "refine_quality_f64", ea, eb);
    else
      screen ? go(refine_quality_f64<2, true>, "refine_quality_mixed", ea, eb)
             : go(refine_quality_f64<2, false>, "refine_quality_f64", ea, eb);
  };
  if (g_mixed)
    tuned(tuners[dim == 3], ns, run);
  else
    run(0, nullptr, nullptr);
  return out;
}

// Up to 8 tag arrays handled by one kernel (FP64 or u32 components).
struct TagList {
  u32 n = 0;
  u32 ncomps[8];
  u32 f64[8];
  void const* src[8];
  void* dst[8];
};

static void tag_list_add(TagList& L, Tag& t, void* dst) {
  OHX_REQUIRE(L.n < 8, "too many vertex tags for one fused kernel");
  L.ncomps[L.n] = t.ncomps;
  L.f64[L.n] = t.type == TagType::F64;
  L.src[L.n] = t.raw();
  L.dst[L.n] = dst;
  ++L.n;
}

// refine_verts + refine_node (refine_common.cpp:29-54, refine_nodal.cpp:10-46):
// every FP64 vertex tag keeps its old values (v0 == v1) and gets, for each
// split edge in order, the average ((0 + f(v0)) + f(v1)) / 2 of its vertices.
__device__ inline void refine_vertex_tags(u32 v0, u32 v1, u32 o, TagList const& L) {
  for (u32 t = 0; t < L.n; ++t) {
    u32 w = L.ncomps[t];
    double const* f = static_cast<double const*>(L.src[t]);
    double* d = static_cast<double*>(L.dst[t]);
    for (u32 c = 0; c < w; ++c) {
      double const f0 = f[(size_t) v0 * w + c];
      if (v0 != v1) {
        double sum = 0;
        sum += f0;
        sum += f[(size_t) v1 * w + c];
        sum /= 2;
        d[(size_t) o * w + c] = sum;
      } else {
        d[(size_t) o * w + c] = f0;
      }
    }
  }
}

// whether the mesh has element fields that the passes transfer
static bool has_element_transfer(Mesh& m) {
  for (auto& t : m.tags[m.dim])
    if (t->transfer == 1 || t->transfer == 2) return true;  // OSH_TRANSFER_POINTWISE, _CONSERVE
  return false;
}

static u32 prods_per_dom(u32 dom_dim, u32 src_dim, u32 prod_dim) {  // refine_topology.cpp:110-121
  if (prod_dim == 0) return (dom_dim == src_dim) ? 1 : 0;
  u32 base_dim = prod_dim - 1;
  u32 opp_dim = dom_dim - 1 - base_dim;
  if (src_dim < opp_dim) return 0;
  return h_down_deg[src_dim][opp_dim];
}

// Arguments of the fused refine product kernel.
struct RefineArgs {
  u32 dim;
  u32 nv;
  u32 n[4];                // entity counts
  u32 const* off[4];       // split offsets of domains of each dim (off[1] = edge split offsets)
  u32 const* verts_of[4];  // down(d, 0)
  u32 const* edges_of[4];  // down(d, 1), d >= 2
  u32 const* faces_of;     // down(3, 2), when maps are carried
  u32 const* cd[4];        // class_dim / class_id per dim (may be null)
  u32 const* ci[4];
  u32 block0[4];           // first blocks of the domains of dim, dim - 1, ..., 0
  TagList tags;            // the vertices' FP64 tags
  struct Prod {            // one product dimension
    u32 ppd[4];            // products per splitting domain of dim d
    u32 go[4];             // output base of the products of domains of dim d
    u32* out_verts;        // pd >= 1
    u32* out_cd;
    u32* out_ci;
    u32* out_edges;        // the new down(pd, 1), pd >= 2, when carried
    u32* out_faces;        // the new down(3, 2), when carried
    u32* soff;             // survivor offsets of dim pd, when wanted
  } p[4];
};

// local vertices of a tet's edge d (of a triangle's for d < 3), its opposite
// edge, the face opposite a local vertex, the edge between two local vertices
// (k_r_e_v, k_f_e_v, k_o_r_e, k_o_r_v), a digit each
__device__ inline u32 tet_ev0(u32 d) { return (0x210210u >> (4 * d)) & 3u; }
__device__ inline u32 tet_ev1(u32 d) { return (0x333021u >> (4 * d)) & 3u; }
__device__ inline u32 tet_oe(u32 d) { return (0x021435u >> (4 * d)) & 7u; }
__device__ inline u32 tet_face_without(u32 v) { return (0x0132u >> (4 * v)) & 3u; }
__device__ inline u32 tet_edge_of(u32 a, u32 b) {
  return a == 3 ? 3 + b : b == 3 ? 3 + a : a + b == 1 ? 0u : a + b == 3 ? 1u : 2u;
}

// The sides of the entities a split pass makes, without looking them up.  A
// domain entity has one split edge (the set's edges share no element), at
// vertex v, with ends p and q.  A side of a product without v is a side of
// the domain that keeps one end, so it survives; one with v and the end E
// is the half, on E's side, of the domain's side on both ends; one with v
// and no end is what the domain's side on both ends and the others makes
// inside.
struct RefineSides {
  RefineArgs const& a;
  __device__ u32 survivor(u32 d, u32 i) const { return i - a.off[d][i]; }
  // the half of split edge e without vertex x; of split face f (its split
  // edge e)
  __device__ u32 half_edge(u32 e, u32 x) const {
    return a.p[1].go[1] + 2 * a.off[1][e] + (a.verts_of[1][2 * (size_t) e] == x ? 0u : 1u);
  }
  __device__ u32 half_face(u32 f, u32 e, u32 x) const {
    u32 const* fe = a.edges_of[2] + 3 * (size_t) f;
    u32 const k = fe[0] == e ? 0u : fe[1] == e ? 1u : 2u;
    return a.p[2].go[2] + 2 * a.off[2][f] + (a.verts_of[2][3 * (size_t) f + k] == x ? 0u : 1u);
  }
  __device__ u32 inner_edge(u32 f) const { return a.p[1].go[2] + a.off[2][f]; }
  __device__ u32 inner_face(u32 t) const { return a.p[2].go[3] + a.off[3][t]; }

  // product j of triangle i, split edge dir: (b0, b1, v) with the edge b0 b1
  // opposite the end that goes
  __device__ void tri(u32 i, u32 dir, u32 j, u32 const* vd, u32* out) const {
    u32 const* e = a.edges_of[2] + 3 * (size_t) i;
    u32 const ends[2] = {tet_ev0(dir), tet_ev1(dir)};
    u32 const gone = ends[j], kept = ends[1 - j];
    u32 const opp_e = (gone + 1) % 3, b0 = opp_e, b1 = (opp_e + 1) % 3;
    u32 const half = half_edge(e[dir], vd[gone]), inner = inner_edge(i);
    out[0] = survivor(1, e[opp_e]);
    out[1] = b1 == kept ? half : inner;
    out[2] = b0 == kept ? half : inner;
  }
  // the face a split tet makes inside: (c0, c1, v) on the edge opposite
  __device__ void tet_inner(u32 i, u32 dir, u32* out) const {
    u32 const* e = a.edges_of[3] + 6 * (size_t) i;
    u32 const* f = a.faces_of + 4 * (size_t) i;
    u32 const o = tet_oe(dir), c0 = tet_ev0(o), c1 = tet_ev1(o);
    out[0] = survivor(1, e[o]);
    // the face on both ends and c is the one without the other
    out[1] = inner_edge(f[tet_face_without(c0)]);
    out[2] = inner_edge(f[tet_face_without(c1)]);
  }
  // product j of tet i: (b0, b1, b2, v) with the face b0 b1 b2 opposite the
  // end that goes
  __device__ void tet(u32 i, u32 dir, u32 j, u32 const* vd, u32* oe, u32* of) const {
    u32 const* e = a.edges_of[3] + 6 * (size_t) i;
    u32 const* f = a.faces_of + 4 * (size_t) i;
    u32 const p = tet_ev0(dir), q = tet_ev1(dir);
    u32 const gone = j == 0 ? p : q, kept = j == 0 ? q : p;
    u32 const base = tet_face_without(gone);
    u32 const* b = k_r_f_v[base];
    u32 const x = vd[gone], half = half_edge(e[dir], x), inner = inner_face(i);
    // the face on both ends and local vertex s
    auto on = [&](u32 s) { return f[tet_face_without(6 - p - q - s)]; };
    for (u32 k = 0; k < 3; ++k) {
      u32 const u = b[k], w = b[(k + 1) % 3];
      oe[k] = survivor(1, e[tet_edge_of(u, w)]);
      oe[3 + k] = u == kept ? half : inner_edge(on(u));
      // the face of v and the edge u w: local faces 1, 2, 3 are on the
      // base's edges 0-1, 1-2, 2-0
      of[1 + k] = u == kept ? half_face(on(w), e[dir], x) : w == kept ? half_face(on(u), e[dir], x) : inner;
    }
    of[0] = survivor(2, f[base]);
  }
};

// refine_ents (refine_common.cpp:64-129) by domain, every dimension in one
// launch (a range of blocks each, the elements first): an entity that does
// not split keeps its vertices and class (inherit.cpp:104-138); one that does
// (split_to_domain, splits_to_domains.cpp:13-56: along its one split edge)
// emits its products of every dimension (refine_domain_entity,
// refine_topology.cpp:26-107: the base opposite each of the edge's
// opposite-dim entities + the new vertex), classified like it: the halves on
// the base opposite each end, and what it makes inside.  With maps carried,
// survivors and products also get their sides (RefineSides): looking them up
// again in hash tables and counting the elements around the edges anew cost
// 2.6 of 6.9 ms of the kernel time of refining 384,000 tets to 1.76 million.
// Bound by bandwidth and the gathers of the renumbering; each entity is read
// once (a thread per product dimension and domain read a tet three times:
// 263 us a pass there, this 194).
template <u32 D>
__device__ inline void refine_entity(RefineArgs const& a, u32 i) {
  if (i >= a.n[D]) return;
  RefineArgs::Prod const& P = a.p[D];
  RefineSides const S{a};
  constexpr u32 NE = D == 3 ? 6 : 3;
  u32 vd[D + 1];
#pragma unroll
  for (u32 k = 0; k <= D; ++k) vd[k] = a.verts_of[D][(size_t) i * (D + 1) + k];
  u32 const k0 = a.off[D][i], k1 = a.off[D][i + 1];
  u32 const cd = P.out_cd ? a.cd[D][i] : 0u, ci = P.out_ci ? a.ci[D][i] : 0u;
  u32 const s = i - k0;
  if (P.soff) {
    P.soff[i] = s;
    if (i + 1 == a.n[D]) P.soff[i + 1] = i + 1 - k1;
  }
  if (k0 == k1) {
#pragma unroll
    for (u32 k = 0; k <= D; ++k) P.out_verts[(size_t) s * (D + 1) + k] = vd[k];
    if (D >= 2 && P.out_edges) {
      u32 e[NE];
#pragma unroll
      for (u32 k = 0; k < NE; ++k) e[k] = a.edges_of[D][(size_t) i * NE + k];
#pragma unroll
      for (u32 k = 0; k < NE; ++k) P.out_edges[(size_t) s * NE + k] = S.survivor(1, e[k]);
    }
    if (D == 3 && P.out_faces) {
      u32 f[4];
#pragma unroll
      for (u32 k = 0; k < 4; ++k) f[k] = a.faces_of[4 * (size_t) i + k];
#pragma unroll
      for (u32 k = 0; k < 4; ++k) P.out_faces[4 * (size_t) s + k] = S.survivor(2, f[k]);
    }
    if (P.out_cd) P.out_cd[s] = cd;
    if (P.out_ci) P.out_ci[s] = ci;
    return;
  }
  // the split edge: its place in the entity, its vertex, its ends
  u32 dir = 0, edge = i;
  if (D >= 2) {
    for (u32 j = 0; j < NE; ++j) {
      u32 const e = a.edges_of[D][(size_t) i * NE + j];
      if (a.off[1][e] != a.off[1][e + 1]) {
        dir = j;
        edge = e;
        break;
      }
    }
  }
  u32 const at = a.off[1][edge], vert = a.nv + at;
  for (u32 j = 0; j < 2; ++j) {
    u32 const o = P.go[D] + 2 * k0 + j;
    u32* q = P.out_verts + (size_t) o * (D + 1);
    if (D == 1) {
      q[0] = vd[1 - j];
    } else if (D == 2) {
      u32 const b = ((j == 0 ? tet_ev0(dir) : tet_ev1(dir)) + 1) % 3;
      q[0] = a.verts_of[2][3 * (size_t) i + b];
      q[1] = a.verts_of[2][3 * (size_t) i + (b + 1) % 3];
      if (P.out_edges) S.tri(i, dir, j, a.verts_of[2] + 3 * (size_t) i, P.out_edges + 3 * (size_t) o);
    } else {
      u32 const* b = k_r_f_v[tet_face_without(j == 0 ? tet_ev0(dir) : tet_ev1(dir))];
      for (u32 k = 0; k < 3; ++k) q[k] = a.verts_of[3][4 * (size_t) i + b[k]];
      if (P.out_edges)
        S.tet(i, dir, j, a.verts_of[3] + 4 * (size_t) i, P.out_edges + 6 * (size_t) o,
              P.out_faces + 4 * (size_t) o);
    }
    q[D] = vert;
    if (P.out_cd) P.out_cd[o] = cd;
    if (P.out_ci) P.out_ci[o] = ci;
  }
  // what it makes inside: an edge its vertex, a face an edge, a tet a face
  RefineArgs::Prod const& I = a.p[D - 1];
  u32 const o = I.go[D] + k0;
  if (D == 1) {
    refine_vertex_tags(vd[0], vd[1], vert, a.tags);
  } else if (D == 2) {
    I.out_verts[2 * (size_t) o] = a.verts_of[2][3 * (size_t) i + k_o_f_e[dir]];
    I.out_verts[2 * (size_t) o + 1] = vert;
  } else {
    u32 const oe = tet_oe(dir);
    I.out_verts[3 * (size_t) o] = a.verts_of[3][4 * (size_t) i + tet_ev0(oe)];
    I.out_verts[3 * (size_t) o + 1] = a.verts_of[3][4 * (size_t) i + tet_ev1(oe)];
    I.out_verts[3 * (size_t) o + 2] = vert;
    if (I.out_edges) S.tet_inner(i, dir, I.out_edges + 3 * (size_t) o);
  }
  if (I.out_cd) I.out_cd[o] = cd;
  if (I.out_ci) I.out_ci[o] = ci;
}

__global__ __launch_bounds__(BLOCK) void refine_products(RefineArgs a) {
  u32 part = 0;
  while (part < a.dim && blockIdx.x >= a.block0[part + 1]) ++part;
  u32 const i = (blockIdx.x - a.block0[part]) * BLOCK + threadIdx.x, d = a.dim - part;
  if (d == 3) {
    refine_entity<3>(a, i);
  } else if (d == 2) {
    refine_entity<2>(a, i);
  } else if (d == 1) {
    refine_entity<1>(a, i);
  } else if (i < a.n[0]) {
    refine_vertex_tags(i, i, i, a.tags);
    if (a.p[0].out_cd) a.p[0].out_cd[i] = a.cd[0][i];
    if (a.p[0].out_ci) a.p[0].out_ci[i] = a.ci[0][i];
  }
}

// nsplit[d]: splitting domains of dimension d (from the offsets' totals);
// carry: the new mesh gets the maps the next split pass reads
static void refine_ents(Mesh& m, Mesh& mo, u32 const* gen_off, Buf<u32>* off, u32 const* nsplit, bool carry) {
  OHX_REQUIRE(m.full, "refine needs a full-topology mesh");
  u32 dim = m.dim;
  RefineArgs a{};
  a.dim = dim;
  a.nv = count(m, 0);
  a.off[1] = gen_off;  // an edge splits iff it is in the independent set
  for (u32 d = 0; d <= dim; ++d) {
    a.n[d] = count(m, d);
    a.verts_of[d] = d ? ask_down(m, d, 0) : nullptr;
  }
  for (u32 d = 2; d <= dim; ++d) {
    a.edges_of[d] = ask_down(m, d, 1);
    a.off[d] = off[d].get();
  }
  if (carry && dim == 3) a.faces_of = ask_down(m, 3, 2);
  bool has_class = find_tag(m, 0, "class_dim") != nullptr;
  bool has_id = find_tag(m, 0, "class_id") != nullptr;
  if (has_class)
    for (u32 d = 0; d <= dim; ++d) {
      a.cd[d] = u32_tag(m, d, "class_dim");
      a.ci[d] = has_id ? u32_tag(m, d, "class_id") : nullptr;
    }
  bool const transfers = has_element_transfer(m);
  Buf<u32> verts[4], cdo[4], cio[4], edges[4], faces, soff[4];
  u32 total[4], nsame[4], blocks = 0;
  for (u32 pd = 0; pd <= dim; ++pd) {
    RefineArgs::Prod& P = a.p[pd];
    nsame[pd] = a.n[pd] - (pd ? nsplit[pd] : 0);
    total[pd] = nsame[pd];
    for (u32 d = 1; d <= 3; ++d) {
      bool live = d <= dim && d >= (pd > 1 ? pd : 1);
      P.ppd[d] = live ? prods_per_dom(d, 1, pd) : 0;
      P.go[d] = total[pd];
      total[pd] += P.ppd[d] * nsplit[d];
    }
    if (pd) {
      verts[pd] = Buf<u32>((size_t) total[pd] * (pd + 1));
      P.out_verts = verts[pd].get();
    }
    if (has_class) {
      cdo[pd] = Buf<u32>(total[pd]);
      P.out_cd = cdo[pd].get();
      if (has_id) {
        cio[pd] = Buf<u32>(total[pd]);
        P.out_ci = cio[pd].get();
      }
    }
    if (carry && pd >= 2) {
      edges[pd] = Buf<u32>((size_t) total[pd] * (pd == 3 ? 6 : 3));
      P.out_edges = edges[pd].get();
    }
    if (carry && pd == 3) {
      faces = Buf<u32>((size_t) total[pd] * 4);
      P.out_faces = faces.get();
    }
    if ((carry && pd == 1) || (pd == dim && (carry || transfers))) {
      soff[pd] = Buf<u32>((size_t) a.n[pd] + 1);
      P.soff = soff[pd].get();
    }
  }
  // the vertices and every FP64 vertex tag
  set_ents(mo, 0, total[0], Buf<u32>());
  for (auto& tp : m.tags[0]) {
    Tag& t = *tp;
    if (t.type != TagType::F64) continue;
    Tag& nt = add_tag_f64(mo, 0, t.name.c_str(), t.ncomps, Buf<double>((size_t) total[0] * t.ncomps), t.transfer);
    tag_list_add(a.tags, t, nt.f.get());
  }
  for (u32 k = 0; k < 4; ++k) {
    a.block0[k] = blocks;
    if (k <= dim) blocks += nblocks(a.n[dim - k]);
  }
  hipLaunchKernelGGL(refine_products, dim3(blocks), dim3(BLOCK), 0, stream(), a);
  check_launch("refine_products");
  for (u32 pd = 0; pd <= dim; ++pd) {
    if (pd) set_ents(mo, pd, total[pd], std::move(verts[pd]));
    if (has_class) {
      add_tag_u32(mo, pd, "class_dim", 1, std::move(cdo[pd]));
      if (has_id) add_tag_u32(mo, pd, "class_id", 1, std::move(cio[pd]));
    }
  }
  if (transfers)
    refine_transfer(m, mo, soff[dim].get(), a.off[dim], a.p[dim].ppd[dim], a.p[dim].go[dim], total[dim]);
  if (!carry) return;
  // the elements around the edges from the old ones: survivors of both
  // dimensions come first and the products are numbered after them
  mo.up[1][dim] = up_patch(h_down_deg[dim][1], ask_up(m, 1, dim), a.n[1], soff[1].get(), nsame[1],
                           total[1] - nsame[1], soff[dim].get(), nsame[dim], total[dim] - nsame[dim],
                           edges[dim].get());
  for (u32 d = 2; d <= dim; ++d) mo.down[d][1] = std::move(edges[d]);
  if (dim == 3) mo.down[3][2] = std::move(faces);
}

static void say(char const* verb, u32 n, u32 d) {
  static char const* const names[4][2] = {{"vertex", "vertices"}, {"edge", "edges"},
                                          {"triangle", "triangles"}, {"tet", "tets"}};
  if (g_verbose) std::printf("%s %10u %s\n", verb, n, names[d][n != 1]);
}

// refine_common (refine_common.cpp:131-190) for edges
// Every adjacency CSR uses 32-bit offsets, as the reference's.  The largest
// one a pass builds is the edge star (3D: 2 uses(1,2) + uses(1,3) = 6F + 6T;
// 2D: 2 uses(1,2) = 6T), and a refine pass can at most double the element
// count; refuse a mesh that could overflow 32 bits instead of wrapping.
static void check_index_space(Mesh& m) {
  size_t t = count(m, m.dim);
  // faces not derived yet: at most 4 per tet
  size_t f = m.dim == 3 ? (has_dim(m, 2) ? (size_t) m.counts[2] : 4 * t) : 0;
  size_t star = m.dim == 3 ? 6 * f + 6 * t : 6 * t;
  if (2 * star >= ((size_t) 1 << 32))
    fail("mesh too large for 32-bit adjacency offsets", __FILE__, __LINE__);
}

static u32 refine_common(Mesh& m, Buf<u32>& cand, double qual_floor, bool require_better,
                         double const* qfe = nullptr, bool carry = false) {
  check_index_space(m);
  u32 ns = count(m, 1), dim = m.dim;
  Buf<double> q = refine_qualities(m, cand.get(), qual_floor, require_better, qfe);
  // one synchronisation for the whole decision: a first batch of indset
  // rounds, the split offsets of every dimension, then one read of the
  // convergence flag and the totals (a candidate-free call ends with an
  // empty set and returns 0)
  u32 const* flag = nullptr;
  Buf<u32> indset = find_indset_from(m, 1, std::move(cand), q.get(), &flag);
  Buf<u32> gen_off(ns + 1);
  Buf<u32> off[4], splits[4];
  u32 got[3] = {0, 0, 0}, open = 0;
  auto offsets_and_totals = [&] {
    // a face or tet splits iff one of its edges does: both dimensions'
    // flags in one launch, then every scan in one
    scan_detail::ScanJobs J{};
    scan_job(J, ns, indset.get(), IN_SET, gen_off.get());
    u32 n[4] = {0, 0, 0, 0};
    u32 const* ed[4] = {nullptr, nullptr, nullptr, nullptr};
    for (u32 d = 2; d <= dim; ++d) {
      n[d] = count(m, d);
      ed[d] = ask_down(m, d, 1);
      off[d] = Buf<u32>(n[d] + 1);
      splits[d] = Buf<u32>(n[d]);
      scan_job(J, n[d], splits[d].get(), 1, off[d].get());
    }
    u32 const* is = indset.get();
    u32 const n2 = n[2], n3 = n[3];
    u32 const *e2 = ed[2], *e3 = ed[3];
    u32 *s2 = splits[2].get(), *s3 = splits[3].get();
    parallel_for(n2 > n3 ? n2 : n3, OHX_LAMBDA(u32 i) {
      if (i < n2) {
        u32 const* e = e2 + 3 * (size_t) i;
        s2[i] = is[e[0]] == IN_SET || is[e[1]] == IN_SET || is[e[2]] == IN_SET ? 1u : 0u;
      }
      if (i < n3) {
        u32 const* e = e3 + 6 * (size_t) i;
        u32 any = 0;
#pragma unroll
        for (u32 j = 0; j < 6; ++j) any |= is[e[j]] == IN_SET ? 1u : 0u;
        s3[i] = any;
      }
    });
    exscan_jobs(J, flag, got, &open);
  };
  offsets_and_totals();
  if (open) {  // not settled in the first batch: the checked loop from there
    indset = find_indset_resume(m, 1, q.get(), std::move(indset));
    flag = nullptr;
    offsets_and_totals();
  }
  if (g_batch) batch_note_changed(m, 1, indset.get());
  q.release();
  indset.release();
  u32 total = got[0];
  if (!total) return 0;
  u32 nsplit[4] = {0, total, got[1], got[2]};
  Mesh mo(m.dim, m.full);
  // maps are carried only through mesh_adapt's loop of split passes: a pass
  // on its own would make maps of the new mesh that its caller may not read
  // (384,000 tets with all their maps split once: 375 us, 668 with maps carried)
  refine_ents(m, mo, gen_off.get(), off, nsplit, carry);
  say("split", total, 1);
  overwrite(m, std::move(mo));
  return 1;
}

u32 refine_by_size(Mesh& m, double qual_floor, bool carry) {
  u32 ne = count(m, 1);
  double const* h = size_of(m);
  double const* mt = metric_of(m);
  Buf<u32> cand(ne);
  u32 tag = next_any_tag();
  if (ne) {
    double prof_bytes = (double) ne * 12 + (double) count(m, 0) * 32;
    launch_timed("refine_candidate_f64", prof_bytes, refine_candidate_f64, dim3(nblocks(ne)), dim3(BLOCK), ne,
                       ask_down(m, 1, 0), coords(m), h, mt, cand.get(), scratch_words(), tag);
  }
  if (read_word(W_ANY) != tag) return 0;
  if (g_batch) {
    batch_mask(m, 1, cand.get());
    Buf<double> qfe = batch_floors(m, 1);
    return refine_common(m, cand, qual_floor, false, qfe.get());
  }
  return refine_common(m, cand, qual_floor, false, nullptr, carry);
}

void uniformly_refine(Mesh& m) {
  Buf<u32> cand = filled(count(m, 1), 1);
  if (!count(m, 1)) return;
  refine_common(m, cand, 0.0, false);
}

// -------------------------------------------------------------- coarsen
enum { DONT_COLLAPSE = 0, COLLAPSE_BOTH = 3 };  // collapse_codes.hpp:8-31
__host__ __device__ inline u32 collapses(u32 c, u32 d) { return (c & (1u << d)) != 0; }
__host__ __device__ inline u32 dont_collapse(u32 c, u32 d) { return c & ~(1u << d); }

// check_basic_edge_class (check_collapse_class.cpp:12-55)
static void check_basic_class(Mesh& m, u32* codes) {
  u32 const* ev = ask_down(m, 1, 0);
  u32 const* vcd = u32_tag(m, 0, "class_dim");
  u32 const* ecd = u32_tag(m, 1, "class_dim");
  parallel_for(count(m, 1), OHX_LAMBDA(u32 i) {
    u32 c = codes[i];
    if (c == DONT_COLLAPSE) return;
    u32 c0 = vcd[ev[2 * i]], c1 = vcd[ev[2 * i + 1]], ce = ecd[i];
    if (c0 == c1) {
      if (c0 != ce) codes[i] = DONT_COLLAPSE;
      return;
    }
    if (collapses(c, 0) && c0 != ce) c = dont_collapse(c, 0);
    if (collapses(c, 1) && c1 != ce) c = dont_collapse(c, 1);
    codes[i] = c;
  });
}

// check_for_exposed_side (check_collapse_class.cpp:57-140), from the
// entities' side: every face (ED = 2) or tet (ED = 3) visits its edges that
// still have a collapse direction and clears the directions it forbids.
// The reference walks each edge's upward adjacency instead; the result is
// an AND over the adjacent entities either way, so the order does not
// matter, and the upward maps up(1,2), up(1,3) and the reflection
// down(3,1) that the walk needs are not built here (a tet's edges come
// from its faces' edges: the edge (a, b) lies in the face opposite a third
// vertex).
template <u32 ED>
__global__ __launch_bounds__(BLOCK) void exposed_sides_k(u32 n, u32 const* __restrict__ vent,
                                                         u32 const* __restrict__ sent,
                                                         u32 const* __restrict__ e_of_f,
                                                         u32 const* __restrict__ v_of_f,
                                                         u32 const* __restrict__ ev, u32 const* __restrict__ ecd,
                                                         u32 const* __restrict__ scd, u32* __restrict__ codes) {
  u32 E = xcd_block() * BLOCK + threadIdx.x;
  if (E >= n) return;
  constexpr u32 VPE = ED + 1, SPE = ED + 1, NE = ED == 3 ? 6 : 3;
  u32 v[VPE], sd[SPE];
#pragma unroll
  for (u32 k = 0; k < SPE; ++k) sd[k] = sent[(size_t) E * SPE + k];
  u32 const cE = ecd[E];
  // a direction is forbidden only through a side classified on a lower
  // dimension than the entity; an entity whose sides all share its class
  // (every interior one) forbids nothing and stops here
  bool exposed = false;
#pragma unroll
  for (u32 k = 0; k < SPE; ++k) exposed = exposed || scd[sd[k]] != cE;
  if (!exposed) return;
#pragma unroll
  for (u32 k = 0; k < VPE; ++k) v[k] = vent[(size_t) E * VPE + k];
  u32 const* so = opp(ED, 0);
#pragma unroll
  for (u32 le = 0; le < NE; ++le) {
    u32 const* lv = canon(ED, 1, 0, le);
    u32 edge;
    if (ED == 2) {
      edge = e_of_f[(size_t) E * 3 + le];
    } else {
      // the face opposite the first tet vertex off the edge holds it
      u32 c3 = (lv[0] != 0 && lv[1] != 0) ? 0u : ((lv[0] != 1 && lv[1] != 1) ? 1u : 2u);
      u32 f = sd[so[c3]];
      u32 const* fv = v_of_f + 3 * (size_t) f;
      u32 va = v[lv[0]], vb = v[lv[1]];
      u32 m = 0;
#pragma unroll
      for (u32 q = 0; q < 3; ++q) {
        u32 a = fv[q], b = fv[(q + 1) % 3];
        if ((a == va && b == vb) || (a == vb && b == va)) m = q;
      }
      edge = e_of_f[3 * (size_t) f + m];
    }
    u32 c = codes[edge];
    if (c == DONT_COLLAPSE) continue;
    u32 mask = 0;
    for (u32 k = 0; k < 2; ++k) {
      if (!collapses(c, k)) continue;
      u32 va = ev[2 * (size_t) edge + (1 - k)];
      u32 l = v[lv[0]] == va ? 0u : 1u;
      if (scd[sd[so[lv[l]]]] != cE) mask |= 1u << k;
    }
    if (mask) atomicAnd(&codes[edge], ~mask);
  }
}

static void check_exposed_sides(Mesh& m, u32 ed, u32* codes) {
  u32 n = count(m, ed);
  if (!n) return;
  u32 const* vent = ask_down(m, ed, 0);
  u32 const* sent = ask_down(m, ed, ed - 1);
  u32 const* e_of_f = ask_down(m, 2, 1);
  u32 const* v_of_f = ask_down(m, 2, 0);
  u32 const* ev = ask_down(m, 1, 0);
  u32 const* ecd = u32_tag(m, ed, "class_dim");
  u32 const* scd = u32_tag(m, ed - 1, "class_dim");
  if (ed == 2)
    hipLaunchKernelGGL(exposed_sides_k<2>, dim3(nblocks(n)), dim3(BLOCK), 0, stream(), n, vent, sent, e_of_f, v_of_f,
                       ev, ecd, scd, codes);
  else
    hipLaunchKernelGGL(exposed_sides_k<3>, dim3(nblocks(n)), dim3(BLOCK), 0, stream(), n, vent, sent, e_of_f, v_of_f,
                       ev, ecd, scd, codes);
  check_launch("exposed_sides");
}

// coarsen_quality (coarsen_qualities.cpp:12-79)
// G lanes per edge: the elements around the collapsing vertex are split
// over the group
// Modes of the collapse-quality kernel.  CQ_F64: the reference's
// arithmetic.  CQ_SCREEN: an FP32 pass rejects the directions certainly
// below the floor, every other direction is measured again in FP64.
// CQ_CERTIFIED: the FP32 pass settles every direction whose FP32 minimum is
// farther than the margin from the floor -- rejected, or accepted with the
// FP32 minimum as its goodness, marked inexact (bit 2 + direction of the
// code) -- and measures only the rest in FP64.  An inexact goodness is used
// only where every comparison it takes part in is certified (see
// coarsen_certify); CQ_FORCE then measures in FP64 the inexact directions
// of the vertices that need exact values.
enum CqMode : u32 { CQ_F64 = 0, CQ_SCREEN = 1, CQ_CERTIFIED = 2, CQ_FORCE = 3 };
__host__ __device__ inline u32 inexact_bit(u32 d) { return 4u << d; }
// further bits of a code word: the direction's quality is known from an
// earlier pass (accepted), and it was measured in this one and rejected
__host__ __device__ inline u32 known_bit(u32 d) { return 16u << d; }
__host__ __device__ inline u32 rejected_bit(u32 d) { return 64u << d; }
// SizeCodeCache::known: accepted (1 << d), rejected, inexact
__host__ __device__ inline u32 was_rejected(u32 d) { return 4u << d; }
__host__ __device__ inline u32 was_inexact(u32 d) { return 16u << d; }

template <u32 DIM, bool F32>
__device__ inline double collapse_elem_q(u32 e, u32 dir, u32 gen, V3 const& pg, Sym const& mg,
                                         u32 const* __restrict__ vel, double const* __restrict__ x,
                                         double const* __restrict__ mt, bool* adj) {
  constexpr u32 VPE = DIM + 1;
  u32 const* v = vel + (size_t) e * VPE;
  bool a = false;
#pragma unroll
  for (u32 l = 0; l < VPE; ++l)
    if (v[l] == gen) a = true;
  *adj = a;
  if (a) return 1.0;
  u32 const* bv = canon(DIM, DIM - 1, 0, opp(DIM, 0)[dir]);
  V3 p[VPE];
  p[VPE - 1] = pg;
#pragma unroll
  for (u32 l = 0; l + 1 < VPE; ++l) p[l] = ld3(x + 3 * (size_t) v[bv[l]]);
  if (mt) {
    Sym pm[VPE];
    pm[VPE - 1] = mg;
#pragma unroll
    for (u32 l = 0; l + 1 < VPE; ++l) pm[l] = ld6(mt + 6 * (size_t) v[bv[l]]);
    return F32 ? (double) quality32<DIM>(p, pm, true) : metric_quality<DIM>(p, pm, true);
  }
  return F32 ? (double) quality32<DIM>(p, nullptr, true) : element_quality(DIM, p);
}

struct CqArgs {
  u32 ncand;
  u32 chunk;        // directions per block, at most CQ_CHUNK
  u32 const* list;  // candidate directions 2 e + j, grouped by collapsing vertex
  u32 const* ev;
  u32 const* uo;    // up(0, dim)
  u32 const* ua;
  u32 const* ud;
  u32 const* vel;   // down(dim, 0)
  double const* x;
  double const* mt;
  double const* eq;  // element qualities (require_better) or null
  double qual_floor;
  double const* qfe;  // per-edge floors (batch) or null
  u32* codes;
  double* out;
  u32 const* vmark;  // CQ_FORCE: vertices that need exact goodness
  ScreenStats st;
};

// Collapse directions, a group of G lanes each.  The directions come
// grouped by collapsing vertex (the list is built from each vertex's edges
// in turn), so the groups of one block share the vertex's element star and
// its vertices in the caches: measured on C3, the edge-ordered form fetched
// about seven times the arrays' size from beyond L2 per launch.  Both
// directions of an edge may be in flight at once, so the code bits are
// cleared (or the inexact bit set) with atomics on the edge's word.
//
// FP64 arithmetic bounds it, and how many of a wave's lanes take part: a
// direction ends at its first element below the floor or after a whole star
// of about 20, so with one direction per group a wave ran at 20 of its 64
// lanes.  A block takes a.chunk directions instead, and a group whose
// direction has ended takes the block's next one (once a quarter of the
// wave's groups wait, as taking one is a chain of loads): 541 -> 422 us for a
// call at 55 thousand tets in FP64, at 32 lanes, and 3405 -> 3194 us for a
// certified one at 511 thousand, at 48 (2048 blocks instead of 1024: 487 us).
// The directions that FP32 leaves open are listed and follow in FP64 in the
// same way.
constexpr u32 CQ_CHUNK = 1024, CQ_BLOCKS = 1024;

// a group's direction
struct CqDir {
  u32 i, j, gen, k, end;
  double floor_;
  V3 pg;
  Sym mg;
};

// Evaluates directions get(0) ... get(n - 1), shared by the block's groups
// through the LDS counter *next (zero).  A direction ends early once its
// minimum is below d.floor_ - margin, where STOP allows it; done(d, minimum,
// minimum of the elements' present quality, NaN seen) is called by the
// group's first lane.
template <u32 DIM, u32 G, bool F32, bool STOP, class Get, class Done>
__device__ inline void cq_directions(CqArgs const& A, u32 n, u32* next, double margin, Get get, Done done) {
  constexpr u32 ENOUGH = G < 16 ? 16 / G : 1;
  u32 const lane = threadIdx.x & 63u, gl = lane % G, lead = lane - gl;
  u64 const group = (G == 64 ? ~0ull : ((1ull << G) - 1)) << lead;
  double const* __restrict__ eq = F32 ? nullptr : A.eq;
  CqDir d{};
  bool has = false, more = true;
  double minq = 1, old_minq = 1;
  bool nan = false;
  for (;;) {
    u64 const waiting = __ballot(!has && gl == 0);
    u32 const nwait = (u32) __popcll(waiting);
    if (more && nwait >= ENOUGH) {
      u32 at = 0;
      if (lane == 0) at = atomicAdd(next, nwait);
      at = (u32) __builtin_amdgcn_readfirstlane((int) at);
      more = at + nwait < n;
      if (!has) {
        at += (u32) __popcll(waiting & ((1ull << lead) - 1));
        u32 dir;
        if (at < n && get(at, &dir)) {
          d.i = dir >> 1;
          d.j = dir & 1u;
          u32 const col = A.ev[2 * (size_t) d.i + d.j];
          d.gen = A.ev[2 * (size_t) d.i + (1 - d.j)];
          // one floor for the mesh, or its component's in a batch
          d.floor_ = A.qfe ? A.qfe[d.i] : A.qual_floor;
          d.pg = ld3(A.x + 3 * (size_t) d.gen);
          if (A.mt) d.mg = ld6(A.mt + 6 * (size_t) d.gen);
          d.k = A.uo[col] + gl;
          d.end = A.uo[col + 1];
          minq = old_minq = 1;
          nan = false;
          has = true;
        }
      }
    }
    if (!__ballot(has)) {
      if (more) continue;
      break;
    }
    bool ended = true, low = false;
    if (has) {
      if (d.k < d.end) {
        u32 const e = A.ua[d.k];
        if (eq && eq[e] < old_minq) old_minq = eq[e];
        bool adj;
        double const q = collapse_elem_q<DIM, F32>(e, A.ud[d.k], d.gen, d.pg, d.mg, A.vel, A.x, A.mt, &adj);
        if (!adj) {
          if (F32 && !(q == q)) nan = true;
          if (q < minq) minq = q;
        }
        d.k += G;
      }
      ended = d.k >= d.end;
      // below the floor the direction is rejected whatever the remaining
      // elements give (the minimum only falls)
      low = STOP && minq < d.floor_ - margin;
    }
    if (G == 1) {
      if (has && (ended || low)) {
        done(d, minq, old_minq, nan);
        has = false;
      }
    } else {
      bool const fin = has && ((__ballot(ended) & group) == group || (__ballot(low) & group) != 0);
      if (__ballot(fin)) {
        double const gm = group_min<G>(minq), go = eq ? group_min<G>(old_minq) : 1;
        bool const gn = F32 && (__ballot(nan) & group) != 0;
        if (fin && gl == 0) done(d, gm, go, gn);
        if (fin) has = false;
      }
    }
  }
}

template <u32 DIM, u32 G, u32 MODE>
__global__ __launch_bounds__(BLOCK) void coarsen_quality_f64(CqArgs A) {
  constexpr bool SCREENED = MODE == CQ_SCREEN || MODE == CQ_CERTIFIED;
  __shared__ u32 next[2], nopen;
  __shared__ u32 open[SCREENED ? CQ_CHUNK : 1];
  u32 const first = xcd_block() * A.chunk;
  if (first >= A.ncand) return;  // the whole block
  u32 n = A.ncand - first < A.chunk ? A.ncand - first : A.chunk;
  if (threadIdx.x < 2) next[threadIdx.x] = 0;
  if (threadIdx.x == 2) nopen = 0;
  __syncthreads();
  u32* __restrict__ codes = A.codes;
  double* __restrict__ out = A.out;
  ScreenStats const st = A.st;
  u32 const* list = A.list + first;
  bool const f32 = SCREENED && !A.eq;
  if (f32) {
    // FP32: a direction certainly below the floor is rejected at its first
    // element below it; CQ_CERTIFIED also accepts one certainly above
    double const m = (double) SCREEN_MARGIN;
    cq_directions<DIM, G, true, true>(
        A, n, next, m,
        [&](u32 at, u32* dir) {
          *dir = list[at];
          return true;
        },
        [&](CqDir const& d, double minq, double, bool nan) {
          bool const reject = !nan && minq < d.floor_ - m;
          bool const accept = MODE == CQ_CERTIFIED && !nan && minq > d.floor_ + m;
          wave_count(st.screened, reject || accept);
          if (reject) {
            atomicXor(&codes[d.i], (1u << d.j) | rejected_bit(d.j));
            return;
          }
          out[2 * (size_t) d.i + d.j] = minq;
          if (accept) {
            atomicOr(&codes[d.i], inexact_bit(d.j));
            return;
          }
          wave_count(st.reeval, true);
          open[atomicAdd(&nopen, 1u)] = 2 * d.i + d.j;
        });
    __syncthreads();
    n = nopen;
    list = open;
  }
  // the screened kernels keep the full minimum for their error statistic
  cq_directions<DIM, G, false, MODE == CQ_F64>(
      A, n, next + 1, 0.0,
      [&](u32 at, u32* dir) {
        u32 const ed = list[at];
        *dir = ed;
        if (MODE != CQ_FORCE) return true;
        bool const wanted =
            (codes[ed >> 1] & inexact_bit(ed & 1u)) && A.vmark[A.ev[2 * (size_t) (ed >> 1) + (ed & 1u)]];
        return wanted;
      },
      [&](CqDir const& d, double minq, double old_minq, bool) {
        if (MODE == CQ_FORCE) wave_count(st.reeval, true);
        if ((f32 || MODE == CQ_FORCE) && minq == minq) {
          double const e = minq - out[2 * (size_t) d.i + d.j];
          note_max_err(st.max_err, (float) (e < 0 ? -e : e));
        }
        if ((minq < d.floor_) || (A.eq && (minq <= old_minq))) {
          // the direction's bit is set and its rejected bit is not, and the
          // inexact bit is set exactly where an FP32 value is measured again
          atomicXor(&codes[d.i], (1u << d.j) | rejected_bit(d.j) | (MODE == CQ_FORCE ? inexact_bit(d.j) : 0u));
        } else {
          out[2 * (size_t) d.i + d.j] = minq;
          if (MODE == CQ_FORCE) atomicAnd(&codes[d.i], ~inexact_bit(d.j));
        }
      });
}

// collapse_to_vert (collapses_to_verts.cpp:13-42): whether each vertex
// collapses and the best goodness of its collapse directions; inex (when
// given) says whether that goodness is an FP32 value.  cand is the
// independent set's first state, and the flags of its rounds are cleared.
__global__ __launch_bounds__(BLOCK) void collapse_to_vert_k(u32 nv, u32 const* __restrict__ uo,
                                                            u32 const* __restrict__ ua, u32 const* __restrict__ ud,
                                                            u32 const* __restrict__ cd, double const* __restrict__ q,
                                                            u32 const* __restrict__ vo, u32* __restrict__ cand,
                                                            double* __restrict__ vq, u32* __restrict__ inex,
                                                            u32* __restrict__ flags) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  if (i < INDSET_FLAGS) flags[i] = 0;
  if (i >= nv) return;
  double maxq = 0;
  u32 is = 0, mi = 0;
  // vo: the candidate directions' offsets per vertex; a vertex that had
  // none has none left and reads nothing
  u32 const jb = (vo && vo[i] == vo[i + 1]) ? uo[i + 1] : uo[i];
  for (u32 j = jb; j < uo[i + 1]; ++j) {
    u32 e = ua[j], d = ud[j];
    u32 c = cd[e];
    if (!collapses(c, d)) continue;
    double qq = q[2 * (size_t) e + d];
    if (!is) {
      is = 1;
      maxq = qq;
      mi = (c & inexact_bit(d)) ? 1u : 0u;
    } else if (qq > maxq) {
      maxq = qq;
      mi = (c & inexact_bit(d)) ? 1u : 0u;
    }
  }
  cand[i] = is ? (u32) UNKNOWN : (u32) NOT_IN_SET;
  vq[i] = is ? maxq : 0.0;
  if (inex) inex[i] = mi;
}

// The comparisons an FP32 goodness takes part in, certified or not: a
// collapsing vertex needs exact goodness (mark[v] = 1) if one of its
// directions within the margin of its best is inexact while another is
// also within it (the destination is the first direction equal to the
// best, collapses_to_verts.cpp:86-101), or if a neighbouring candidate's
// best lies within the margin of its own and either is inexact (the
// independent set compares them with == and <, indset.cpp:72-83).  FP32
// values are within half the margin of their FP64 values, so every
// comparison left unmarked has the FP64 outcome.
__global__ __launch_bounds__(BLOCK) void coarsen_certify(u32 nv, u32 const* __restrict__ uo,
                                                         u32 const* __restrict__ ua, u32 const* __restrict__ ud,
                                                         u32 const* __restrict__ cd, double const* __restrict__ q,
                                                         u32 const* __restrict__ ev,
                                                         u32 const* __restrict__ cand, double const* __restrict__ vq,
                                                         u32 const* __restrict__ inex, u32* __restrict__ mark) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  if (i >= nv) return;
  u32 mk = 0;
  if (cand[i]) {
    double const m = (double) SCREEN_MARGIN;
    double const best = vq[i];
    u32 near = 0, near_inex = 0;
    for (u32 j = uo[i]; j < uo[i + 1]; ++j) {
      u32 e = ua[j], d = ud[j];
      u32 c = cd[e];
      if (!collapses(c, d)) continue;
      double qq = q[2 * (size_t) e + d];
      if (!(qq < best - m)) {
        ++near;
        if (c & inexact_bit(d)) near_inex = 1;
      }
    }
    if (near > 1 && near_inex) mk = 1;
    // the neighbours the independent set compares: the other ends of the
    // vertex's edges (the vertex star, as a set)
    u32 const mine = inex[i];
    for (u32 k = uo[i]; !mk && k < uo[i + 1]; ++k) {
      u32 o = ev[2 * (size_t) ua[k] + (1 - ud[k])];
      if (!cand[o]) continue;
      double dd = vq[o] - best;
      if (!(dd > m || dd < -m) && (mine || inex[o])) mk = 1;
    }
  }
  mark[i] = mk;
}

// coarsen_size_code (coarsen.cpp:13-21), fused with measure_edge
__global__ __launch_bounds__(BLOCK) void coarsen_size_code_f64(u32 n, u32 const* __restrict__ ev,
                                                               double const* __restrict__ x,
                                                               double const* __restrict__ h,
                                                               double const* __restrict__ mt, double floor_,
                                                               u32* __restrict__ codes, u32* __restrict__ words,
                                                               u32 tag) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  if (i >= n) return;
  double sz = edge_size(ev[2 * i], ev[2 * i + 1], x, h, mt);
  u32 c = (sz < floor_) ? (u32) COLLAPSE_BOTH : (u32) DONT_COLLAPSE;
  codes[i] = c;
  wave_flag_value(words + W_ANY, c != 0, tag);
}

// size codes carried to a collapse pass's new mesh: threads [0, ne_old)
// give a surviving edge its old code; the next ngen measure a product edge.
// A surviving edge's direction whose collapsing vertex kept all its elements
// and gained none also keeps what is known of its quality: the quality reads
// those elements, their vertices and the target's position, and a collapse
// moves no vertex.
struct CarryCodes {
  u32 ne_old, ngen, nsame;
  u32 const* soff;
  u32 const* old_codes;
  u32 const* ev;  // the new mesh's
  double const* x;
  double const* h;
  double const* mt;
  double floor_;
  u32* codes;
  u32 const* now;        // the pass's code words
  u32 const* old_known;  // or null
  double const* q;
  u32 const* old_ev;
  u32 const* vsoff;
  u32 const* full;  // per new vertex (UpPatchCounts)
  u32 const* cnt;
  u32 const* cnt_s;
  u32* known;
  double* new_q;
};
__global__ __launch_bounds__(BLOCK) void carry_size_codes_k(CarryCodes a) {
  u32 t = xcd_block() * BLOCK + threadIdx.x;
  if (t < a.ne_old) {
    u32 o = a.soff[t];
    if (o == a.soff[t + 1]) return;
    a.codes[o] = a.old_codes[t];
    u32 const c = a.now[t], was = a.old_known ? a.old_known[t] : 0u;
    u32 k = 0;
    for (u32 d = 0; d < 2; ++d) {
      u32 b = was & ((1u << d) | was_rejected(d) | was_inexact(d));
      if (collapses(c, d))
        b = (1u << d) | ((c & inexact_bit(d)) ? was_inexact(d) : 0u);
      else if (c & rejected_bit(d))
        b = was_rejected(d);
      if (!b) continue;
      u32 const v = a.vsoff[a.old_ev[2 * (size_t) t + d]];
      if (!a.full[v] || a.cnt[v] != a.cnt_s[v]) continue;
      k |= b;
      if (b & (1u << d)) a.new_q[2 * (size_t) o + d] = a.q[2 * (size_t) t + d];
    }
    a.known[o] = k;
  } else if (t - a.ne_old < a.ngen) {
    u32 i = a.nsame + (t - a.ne_old);
    double sz = edge_size(a.ev[2 * i], a.ev[2 * i + 1], a.x, a.h, a.mt);
    a.codes[i] = (sz < a.floor_) ? (u32) COLLAPSE_BOTH : (u32) DONT_COLLAPSE;
    a.known[i] = 0;
  }
}

// tags_subset (subset.cpp:15-43): every tag of old vertex i if it survives
__device__ inline void subset_tags(u32 i, u32 n, u32 const* __restrict__ soff, TagList const& L) {
  if (i >= n) return;
  u32 o = soff[i];
  if (o == soff[i + 1]) return;
  for (u32 t = 0; t < L.n; ++t) {
    u32 w = L.ncomps[t];
    if (L.f64[t]) {
      double const* f = static_cast<double const*>(L.src[t]);
      double* dd = static_cast<double*>(L.dst[t]);
      for (u32 c = 0; c < w; ++c) dd[(size_t) o * w + c] = f[(size_t) i * w + c];
    } else {
      u32 const* f = static_cast<u32 const*>(L.src[t]);
      u32* dd = static_cast<u32*>(L.dst[t]);
      for (u32 c = 0; c < w; ++c) dd[(size_t) o * w + c] = f[(size_t) i * w + c];
    }
  }
}

// The new entities' sides of dimension l (0 < l < d), carried from the old
// map instead of reflected (reflect_down.cpp:13-81 gives the same map: an
// entity's lows are unique in a conforming mesh).  A survivor keeps its
// sides, renumbered.  A product is the old entity with its collapsing vertex
// replaced by the target; a side without that vertex survives, and one with
// it is either rebuilt on the target itself (a product of dimension l) or
// fused into the side that already joins the target to the same vertices.
struct CoarsenSides {
  u32* out;            // new entities x sides (null: not built)
  u32 const* old;      // the old entities' sides
  u32 const* soff;     // old side -> its index among the surviving sides
  u32 const* egoff;    // old side -> its index among the product sides
  u32 const* fused_to; // fused old side -> the old side it merges into
  u32 nsame, l;        // surviving sides, their dimension
  u32 nold;            // old sides
  u32* err;
};

struct CoarsenArgs {
  u32 d, n, nsame;
  u32 const* vent;
  u32 const* esoff;  // survivor offsets
  u32 const* egoff;  // generated offsets
  u32 const* gv;     // target vertex of generating entities
  u32 const* gd;     // local index of their collapsing vertex
  u32 const* vsoff;  // vertex renumbering (survivor offsets of vertices)
  u32* out;
  u32 const* cd;
  u32 const* ci;
  u32* out_cd;
  u32* out_ci;
  CoarsenSides sides, edges;  // down(d, d-1); the tets' edges (sliver passes)
};

// sides of dimension l of a d-simplex
__host__ __device__ inline u32 simplex_sides(u32 d, u32 l) { return d == 3 ? (l == 1 ? 6u : 4u) : 3u; }

// the new id of side c (dimension s.l) of a product: the old entity's
// sides in row, its collapsing vertex at old local index gd; the product's
// local vertices are the base opposite gd in canonical order, then the
// target in gd's place
template <u32 D, u32 L>
__device__ inline u32 coarsen_product_side(u32 c, u32 gd, u32 const* row, CoarsenSides const& s) {
  u32 const* bv = canon(D, D - 1, 0, opp(D, 0)[gd]);
  u32 const* cs = canon(D, L, 0, c);
  u32 mask = 0;
  bool on_target = false;
#pragma unroll
  for (u32 q = 0; q <= L; ++q) {
    u32 const nl = cs[q];
    on_target = on_target || nl == D;
    mask |= 1u << (nl < D ? bv[nl] : gd);
  }
  u32 k = 0;
#pragma unroll
  for (u32 j = 0; j < simplex_sides(D, L); ++j) {
    u32 const* os = canon(D, L, 0, j);
    u32 mj = 0;
#pragma unroll
    for (u32 q = 0; q <= L; ++q) mj |= 1u << os[q];
    if (mj == mask) k = j;
  }
  u32 const side = row[k];
  if (!on_target) return s.soff[side];
  if (s.egoff[side] != s.egoff[side + 1]) return s.nsame + s.egoff[side];
  u32 const into = s.fused_to[side];
  if (into < s.nold) return s.soff[into];
  *s.err = ERR_REFLECT_NOT_FOUND;  // a side on the target that is neither rebuilt nor fused
  return INVALID;
}

// the sides of dimension L of old entity i, as entity o
template <u32 D, u32 L>
__device__ inline void coarsen_sides(CoarsenSides const& s, u32 i, u32 o, bool same, u32 gd) {
  constexpr u32 NS = D == 3 ? (L == 1 ? 6 : 4) : 3;
  u32 row[NS];
#pragma unroll
  for (u32 c = 0; c < NS; ++c) row[c] = s.old[(size_t) i * NS + c];
  u32* const out = s.out + (size_t) o * NS;
  if (same) {
#pragma unroll
    for (u32 c = 0; c < NS; ++c) row[c] = s.soff[row[c]];
#pragma unroll
    for (u32 c = 0; c < NS; ++c) out[c] = row[c];
  } else {
    for (u32 c = 0; c < NS; ++c) out[c] = coarsen_product_side<D, L>(c, gd, s.old + (size_t) i * NS, s);
  }
}

// concat_verts_of_ents (inherit.cpp:234-255) + coarsen_elem
// (coarsen_topology.cpp:9-44) + remap_conn (coarsen_common.cpp:29-33) +
// setup_coarsen class inheritance (inherit.cpp:140-156), fused: survivors
// first, then the entities rebuilt on the collapse target (the base
// opposite the collapsing vertex, then the target), vertex ids renumbered.
// Every dimension and the vertices' tags in one launch, a range of blocks
// each: the elements first, which take longest.
// The dimension is a template parameter: an entity's loads and the gathers
// of its renumbering then go out together (with loops of the dimension's
// length one after another, 4.4 million entities took 178 us, this way 120).
template <u32 D>
__device__ inline void coarsen_entity(CoarsenArgs const& a, u32 i) {
  if (i >= a.n) return;
  u32 v[D + 1];
#pragma unroll
  for (u32 j = 0; j <= D; ++j) v[j] = a.vent[(size_t) i * (D + 1) + j];
  u32 const s0 = a.esoff[i], s1 = a.esoff[i + 1], g0 = a.egoff[i], g1 = a.egoff[i + 1];
  bool const same = s0 != s1;
  if (!same && g0 == g1) return;
  u32 const o = same ? s0 : a.nsame + g0;
  u32 const cd = a.out_cd ? a.cd[i] : 0u, ci = a.out_ci ? a.ci[i] : 0u;
  u32* const out = a.out + (size_t) o * (D + 1);
  u32 gd = 0;
  if (same) {
#pragma unroll
    for (u32 j = 0; j <= D; ++j) v[j] = a.vsoff[v[j]];
#pragma unroll
    for (u32 j = 0; j <= D; ++j) out[j] = v[j];
  } else {
    gd = a.gd[i];
    u32 const* bv = canon(D, D - 1, 0, opp(D, 0)[gd]);
    for (u32 j = 0; j < D; ++j) out[j] = a.vsoff[a.vent[(size_t) i * (D + 1) + bv[j]]];
    out[D] = a.vsoff[a.gv[i]];
  }
  if (D >= 2 && a.sides.out) coarsen_sides<D, (D >= 2 ? D - 1 : 1)>(a.sides, i, o, same, gd);
  if (D == 3 && a.edges.out) coarsen_sides<3, 1>(a.edges, i, o, same, gd);
  if (a.out_cd) a.out_cd[o] = cd;
  if (a.out_ci) a.out_ci[o] = ci;
}
struct CoarsenOutputs {
  CoarsenArgs a[3];
  u32 block0[4];  // first blocks of a[0..2] and of the vertices
  u32 nv;
  u32 const* soff;
  TagList tags;
};
__global__ __launch_bounds__(BLOCK) void coarsen_outputs(CoarsenOutputs O) {
  if (blockIdx.x >= O.block0[3]) {
    subset_tags((blockIdx.x - O.block0[3]) * BLOCK + threadIdx.x, O.nv, O.soff, O.tags);
    return;
  }
  u32 part = 0;
  while (part < 2 && blockIdx.x >= O.block0[part + 1]) ++part;
  CoarsenArgs const& a = O.a[part];
  u32 const i = (blockIdx.x - O.block0[part]) * BLOCK + threadIdx.x;
  if (a.d == 3) coarsen_entity<3>(a, i);
  else if (a.d == 2) coarsen_entity<2>(a, i);
  else coarsen_entity<1>(a, i);
}

// collapse_to_ent (collapses_to_ents.cpp:11-82) for the entities of one
// dimension: what becomes of each (those without a collapsing vertex survive
// unchanged), and for each fused side the side it merges into (the one
// opposite the collapsing vertex), which the maps carried to the new mesh read
enum Fate : u32 { REMOVED = 0, SAME = 1, REBUILT = 2 };
struct CollapseEnts {
  u32 n;
  u32 const* vent;
  u32 const* sent;
  u32 const* is;  // per vertex: collapses
  u32 const* g;   // its target
  u32 const* fe;  // fused_to of this dimension (null: elements), read
  u32* ft;        // fused_to of the sides, written (null: vertices)
  u32* fate;
  u32* gv;
  u32* gd;
};
template <u32 D>
__global__ __launch_bounds__(BLOCK) void collapse_ents_k(CollapseEnts a) {
  u32 const i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= a.n) return;
  constexpr u32 SPE = D == 1 ? 2 : D + 1;
  u32 v[D + 1], in[D + 1];
#pragma unroll
  for (u32 j = 0; j <= D; ++j) v[j] = a.vent[(size_t) i * (D + 1) + j];
#pragma unroll
  for (u32 j = 0; j <= D; ++j) in[j] = a.is[v[j]];
  u32 col = INVALID, dir = INVALID;
#pragma unroll
  for (u32 j = 0; j <= D; ++j)
    if (in[j]) {
      col = v[j];
      dir = j;
    }
  u32 w = SAME;
  if (dir != INVALID) {
    w = REMOVED;
    u32 const target = a.g[col];
    u32 gdir = INVALID;
#pragma unroll
    for (u32 j = 0; j <= D; ++j)
      if (v[j] == target) gdir = j;
    if (gdir != INVALID) {
      if (a.ft)
        a.ft[a.sent[(size_t) i * SPE + opp(D, 0)[gdir]]] = a.sent[(size_t) i * SPE + opp(D, 0)[dir]];
    } else if (!(a.fe && a.fe[i] != INVALID)) {
      w = REBUILT;
      a.gv[i] = target;
      a.gd[i] = dir;
    }
  }
  a.fate[i] = w;
}

static char const* cq_name(u32 mode) {
  return mode == CQ_F64 ? "coarsen_quality_f64"
                        : mode == CQ_SCREEN ? "coarsen_quality_mixed"
                                            : mode == CQ_CERTIFIED ? "coarsen_quality_certified" : "coarsen_quality_force";
}

template <u32 DIM, u32 MODE>
static void cq_launch(u32 g, CqArgs a, double bytes, hipEvent_t ea, hipEvent_t eb) {
  // a block's share: at least a direction per group, and more as soon as
  // that fills the chip (four blocks per CU)
  u32 const share = (a.ncand + CQ_BLOCKS - 1) / CQ_BLOCKS, least = BLOCK / g;
  a.chunk = share < least ? least : share < CQ_CHUNK ? share : CQ_CHUNK;
  dim3 grid((a.ncand + a.chunk - 1) / a.chunk);
  char const* kn = cq_name(MODE);
  auto one = [&](auto kernel) {
    if (ea) {
      hipExtLaunchKernelGGL(kernel, grid, dim3(BLOCK), 0, stream(), ea, eb, 0, a);
      check_launch(kn);
    } else {
      launch_timed(kn, bytes, kernel, grid, dim3(BLOCK), a);
    }
  };
  if (g == 1) one(coarsen_quality_f64<DIM, 1, MODE>);
  else if (g == 2) one(coarsen_quality_f64<DIM, 2, MODE>);
  else if (g == 4) one(coarsen_quality_f64<DIM, 4, MODE>);
  else one(coarsen_quality_f64<DIM, 8, MODE>);
}

template <u32 DIM>
static void cq_launch_mode(u32 mode, u32 g, CqArgs const& a, double bytes, hipEvent_t ea, hipEvent_t eb) {
  switch (mode) {
    case CQ_F64: cq_launch<DIM, CQ_F64>(g, a, bytes, ea, eb); break;
    case CQ_SCREEN: cq_launch<DIM, CQ_SCREEN>(g, a, bytes, ea, eb); break;
    case CQ_CERTIFIED: cq_launch<DIM, CQ_CERTIFIED>(g, a, bytes, ea, eb); break;
    default: cq_launch<DIM, CQ_FORCE>(g, a, bytes, ea, eb); break;
  }
}

// ------------------------------------------------ maps carried across a pass
// A pass numbers the surviving entities of every dimension first, in their
// old relative order and vertex order, and appends its products; the lows
// of a surviving entity survive too.  So the new mesh's upward adjacency of
// a (low, high) pair follows from the old one (up_from_down.cpp:9-47 gives
// the same lists: per low, its uses in increasing use index high * deg +
// local index): a surviving low's list is its old list without the removed
// highs, renumbered, followed by its uses in product highs; a product low
// has product uses only.  Only the product uses (a few per cavity) take
// atomics and a sort.
struct UpPatch {
  u32 deg, nl_old, nsame_l, ngen_l, nsame_h, ngen_h;
  u32 nuse;           // (nsame_h + ngen_h) * deg: writes stay below it
  u32 const* uo;      // old up(l,h): offsets, highs, local indices
  u32 const* ua;
  u32 const* ud;
  u32 const* soff_l;  // old low / high -> index among the survivors
  u32 const* soff_h;
  u32 const* dn;      // the new down(h,l)
  u32* cnt;           // per new low: its uses (surviving, then + product)
  u32* cnt_s;         // per new low: its uses in surviving highs
  u32* full;          // per new low: 1 if it kept every old use (null: not kept)
  u32* slot;          // per product use: its place in its low's list
  u32 const* off;     // the new offsets
  u32* key;           // product use indices at their unsorted places
  u32* adj;
  u32* dirs;
};

// G lanes per old low (a group): a surviving low counts its surviving
// highs, G uses at a time; groups past nl_old start the product lows at
// zero (lane 0 of each)
template <u32 G>
__global__ __launch_bounds__(BLOCK) void up_patch_count_k(UpPatch a) {
  size_t gid = (size_t) xcd_block() * BLOCK + threadIdx.x;
  u32 const t = (u32) (gid / G), lane = (u32) (gid % G);
  if (t < a.nl_old) {
    u32 n = a.soff_l[t];
    if (n == a.soff_l[t + 1]) return;
    u32 c = 0;
    for (u32 k = a.uo[t] + lane; k < a.uo[t + 1]; k += G) {
      u32 h = a.ua[k];
      c += a.soff_h[h] != a.soff_h[h + 1] ? 1u : 0u;
    }
#pragma unroll
    for (u32 d = G / 2; d >= 1; d >>= 1) c += (u32) __shfl_xor((int) c, (int) d, (int) G);
    if (lane == 0) {
      a.cnt[n] = c;
      a.cnt_s[n] = c;
      if (a.full) a.full[n] = c == a.uo[t + 1] - a.uo[t] ? 1u : 0u;
    }
  } else if (t - a.nl_old < a.ngen_l && lane == 0) {
    u32 n = a.nsame_l + (t - a.nl_old);
    a.cnt[n] = 0;
    a.cnt_s[n] = 0;
    if (a.full) a.full[n] = 0;
  }
}

// a product use's low, or INVALID where the product's lows were not found
// (reported where they were built)
__device__ inline u32 up_patch_low(UpPatch const& a, u32 u) {
  u32 e = a.dn[(size_t) a.nsame_h * a.deg + u];
  return e < a.nsame_l + a.ngen_l ? e : INVALID;
}

// each product use takes a place after its low's surviving uses.  Bound by the
// atomics' rate; the products of a cavity share their lows (the 60 edge uses of
// ten tets around a new vertex have 22), so a wave combines its adds: a split
// adaptation of 384 thousand tets 5.33 -> 5.18 ms, of 3 thousand 2.40 -> 2.31.
__global__ __launch_bounds__(BLOCK) void up_patch_slot_k(UpPatch a) {
  u32 const u = xcd_block() * BLOCK + threadIdx.x;
  bool const in = u < a.ngen_h * a.deg;
  u32 const e = in ? up_patch_low(a, u) : INVALID;
  u32 const s = wave_slot_add(a.cnt, e == INVALID ? 0u : e, e != INVALID);
  if (e != INVALID) a.slot[u] = s;
}

// after the scan of the counts: groups of G lanes over the old lows write
// a surviving low's surviving uses in order (G at a time, placed by a
// prefix count over the group's ballot); the ngen_h * deg threads after
// them put each product use's index at its place
template <u32 G>
__global__ __launch_bounds__(BLOCK) void up_patch_fill_k(UpPatch a) {
  size_t gid = (size_t) xcd_block() * BLOCK + threadIdx.x;
  size_t const ngroups_lanes = (size_t) a.nl_old * G;
  if (gid < ngroups_lanes) {
    u32 const t = (u32) (gid / G), lane = (u32) (gid % G);
    u32 n = a.soff_l[t];
    if (n == a.soff_l[t + 1]) return;
    u32 const first = (u32) (threadIdx.x & 63u) & ~(G - 1u);  // the group's first lane in the wave
    unsigned long long const below = ((1ull << lane) - 1ull) << first;
    u32 p = a.off[n];
    for (u32 k0 = a.uo[t]; k0 < a.uo[t + 1]; k0 += G) {
      u32 const k = k0 + lane;
      bool keep = false;
      u32 s = 0;
      if (k < a.uo[t + 1]) {
        u32 h = a.ua[k];
        s = a.soff_h[h];
        keep = s != a.soff_h[h + 1];
      }
      unsigned long long const m = __ballot(keep);
      u32 const q = p + (u32) __popcll(m & below);
      if (keep && q < a.nuse) {
        a.adj[q] = s;
        a.dirs[q] = a.ud[k];
      }
      p += (u32) __popcll((m >> first) & ((G == 64 ? ~0ull : (1ull << G) - 1ull)));
    }
  } else if (gid - ngroups_lanes < (size_t) a.ngen_h * a.deg) {
    u32 u = (u32) (gid - ngroups_lanes);
    u32 e = up_patch_low(a, u);
    if (e == INVALID) return;
    u32 const p = a.off[e] + a.slot[u];
    if (p < a.nuse) a.key[p] = a.nsame_h * a.deg + u;
  }
}

// each product use's final place: its rank by use index among its low's
// product uses
__global__ __launch_bounds__(BLOCK) void up_patch_sort_k(UpPatch a) {
  u32 u = xcd_block() * BLOCK + threadIdx.x;
  if (u >= a.ngen_h * a.deg) return;
  u32 e = up_patch_low(a, u);
  if (e == INVALID) return;
  u32 const b = a.off[e] + a.cnt_s[e], end = a.off[e + 1] < a.nuse ? a.off[e + 1] : a.nuse;
  u32 const me = a.nsame_h * a.deg + u;
  u32 r = 0;
  for (u32 k = b; k < end; ++k) r += a.key[k] < me ? 1u : 0u;
  if (b + r >= a.nuse) return;
  u32 const h = me / a.deg;
  a.adj[b + r] = h;
  a.dirs[b + r] = me - a.deg * h;
}

// per new low, kept for the caller: all its uses (cnt), those in surviving
// highs (cnt_s), and whether those are all its old ones (full); a low with
// full set and cnt == cnt_s has exactly its old highs
struct UpPatchCounts {
  Buf<u32> cnt, cnt_s, full;
};

// the new mesh's up(l,h) from the old mesh's: nl_old old lows, survivors
// of both dimensions given by their offsets over the old entities, dn the
// new down(h,l) (its product rows are read)
static std::unique_ptr<Up> up_patch(u32 deg, Up const& old, u32 nl_old, u32 const* soff_l, u32 nsame_l,
                                    u32 ngen_l, u32 const* soff_h, u32 nsame_h, u32 ngen_h, u32 const* dn,
                                    UpPatchCounts* keep) {
  u32 const nl = nsame_l + ngen_l, nuse = (nsame_h + ngen_h) * deg, nprod = ngen_h * deg;
  auto up = std::make_unique<Up>();
  up->offsets = Buf<u32>(nl + 1);
  up->adj = Buf<u32>(nuse);
  up->dirs = Buf<u32>(nuse);
  Buf<u32> cnt(nl), cnt_s(nl), slot(nprod), key(nuse), full;
  if (keep) full = Buf<u32>(nl);
  UpPatch a{};
  a.deg = deg;
  a.nuse = nuse;
  a.nl_old = nl_old;
  a.nsame_l = nsame_l;
  a.ngen_l = ngen_l;
  a.nsame_h = nsame_h;
  a.ngen_h = ngen_h;
  a.uo = old.offsets.get();
  a.ua = old.adj.get();
  a.ud = old.dirs.get();
  a.soff_l = soff_l;
  a.soff_h = soff_h;
  a.dn = dn;
  a.cnt = cnt.get();
  a.cnt_s = cnt_s.get();
  a.full = full.get();
  a.slot = slot.get();
  a.off = up->offsets.get();
  a.key = key.get();
  a.adj = up->adj.get();
  a.dirs = up->dirs.get();
  // compulsory bytes: the old lists and the highs' survivor flags read
  double const old_bytes = (double) nl_old * 12 + (double) old.adj.size() * 12;
  // lanes per old low: about its mean list length (edges in tets ~5,
  // vertices in edges ~14, vertices in tets ~24)
  size_t const mean = nl_old ? old.adj.size() / nl_old : 0;
  u32 const G = mean <= 6 ? 4u : mean <= 16 ? 8u : 16u;
  auto groups = [&](auto count_k, auto fill_k) {
    size_t const nc = ((size_t) nl_old + ngen_l) * G;
    if (nc) launch_timed("up_patch_count", old_bytes, count_k, dim3(nblocks(nc)), dim3(BLOCK), a);
    if (nprod) {
      hipLaunchKernelGGL(up_patch_slot_k, dim3(nblocks(nprod)), dim3(BLOCK), 0, stream(), a);
      check_launch("up_patch_slot");
    }
    exscan(cnt.get(), nl, up->offsets.get());
    size_t const nf = (size_t) nl_old * G + nprod;
    if (nf) launch_timed("up_patch_fill", old_bytes + (double) nuse * 8, fill_k, dim3(nblocks(nf)), dim3(BLOCK), a);
  };
  if (G == 4) groups(up_patch_count_k<4>, up_patch_fill_k<4>);
  else if (G == 8) groups(up_patch_count_k<8>, up_patch_fill_k<8>);
  else groups(up_patch_count_k<16>, up_patch_fill_k<16>);
  if (nprod) {
    hipLaunchKernelGGL(up_patch_sort_k, dim3(nblocks(nprod)), dim3(BLOCK), 0, stream(), a);
    check_launch("up_patch_sort");
  }
  if (keep) {
    keep->cnt = std::move(cnt);
    keep->cnt_s = std::move(cnt_s);
    keep->full = std::move(full);
  }
  return up;
}

static u32 coarsen_common(Mesh& m, Buf<u32>& codes, double qual_floor, bool require_better,
                          double const* qfe = nullptr, double const* eq_given = nullptr,
                          SizeCodeCache* sizes = nullptr, double size_floor = 0) {
  check_index_space(m);
  u32 dim = m.dim;
  u32 ne = count(m, 1);
  check_basic_class(m, codes.get());
  for (u32 d = 2; d <= dim; ++d) check_exposed_sides(m, d, codes.get());
  // the collapse directions left, listed vertex by vertex (each vertex's
  // edges in up(0,1) order): the quality kernel's groups then all have
  // work, and neighbouring groups share a vertex's star (the count, read
  // once, is also the early return when the class checks leave nothing).
  // The list is the uses of up(0,1) that collapse, in use order, so one
  // flat scan over the uses numbers them (no per-vertex loop), and a
  // vertex's first direction is the scan at its first use.
  // Where the loop carries known qualities, only the directions without one
  // are measured: a second list, from a second scan before the same read.
  u32 ncand, neval;
  Buf<u32> clist, elist, voff;
  u32 const nv0 = count(m, 0);
  bool const some_known = sizes && sizes->known;
  {
    Up const& uv = ask_up(m, 0, 1);
    u32 const* uo = uv.offsets.get();
    u32 const* ua = uv.adj.get();
    u32 const* ud = uv.dirs.get();
    u32 const* cp = codes.get();
    u32 const nuse = 2 * ne;
    Buf<u32> uoff(nuse + 1), eoff;
    auto listed = OHX_LAMBDA(u32 k) { return collapses(cp[ua[k]], ud[k]); };
    if (some_known) {
      eoff = Buf<u32>(nuse + 1);
      exscan_fn(nuse, listed, uoff.get());
      exscan_fn(nuse, OHX_LAMBDA(u32 k) {
        u32 const c = cp[ua[k]], d = ud[k];
        return collapses(c, d) && !(c & known_bit(d)) ? 1u : 0u;
      }, eoff.get());
      u32 const* ptrs[2] = {uoff.get() + nuse, eoff.get() + nuse};
      u32 n[2];
      read_many(ptrs, 2, n);
      ncand = n[0];
      neval = n[1];
    } else {
      ncand = neval = exscan_fn_total(nuse, listed, uoff.get());
    }
    if (!ncand) return 0;
    clist = Buf<u32>(ncand);
    if (some_known) elist = Buf<u32>(neval);
    voff = Buf<u32>(nv0 + 1);
    u32 const* uf = uoff.get();
    u32 const* ef = eoff.get();
    u32* cl = clist.get();
    u32* el = elist.get();
    u32* vo = voff.get();
    parallel_for(nuse > nv0 ? nuse : nv0 + 1, OHX_LAMBDA(u32 k) {
      if (k < nuse && uf[k] != uf[k + 1]) cl[uf[k]] = 2 * ua[k] + ud[k];
      if (ef && k < nuse && ef[k] != ef[k + 1]) el[ef[k]] = 2 * ua[k] + ud[k];
      if (k <= nv0) vo[k] = uf[uo[k]];
    });
  }
  Buf<double> eq;
  u32 const* ev = ask_down(m, 1, 0);
  u32 const* vel = ask_down(m, dim, 0);
  Up const& ue = ask_up(m, 0, dim);
  // the element qualities of this mesh: the caller's (the adapt loop
  // computes them once per mesh) or evaluated here
  double const* eqp = nullptr;
  if (require_better) {
    if (!eq_given) eq = element_qualities(dim, count(m, dim), vel, coords(m), count(m, 0), metric_of(m));
    eqp = eq_given ? eq_given : eq.get();
  }
  Buf<double> cq = some_known ? std::move(sizes->q) : Buf<double>((size_t) 2 * ne);
  Buf<u32> cand;
  Buf<double> vq;
  {
    // compulsory bytes: of each direction measured its list entry, its edge's
    // ends, code and value; and of the elements around the collapsing
    // vertices, their vertices and coordinates at least the share of the
    // mesh's that the directions are of all directions (a vertex's are mostly
    // listed together).  The directions measured again in FP64 are chosen on
    // the device among all: what is read to choose them.
    double const share = (double) neval / (2.0 * ne);
    double const prof_bytes =
        (double) neval * 24 + share * ((double) ue.adj.size() * 8 + (double) count(m, dim) * (dim + 1) * 4 +
                                       (double) count(m, 0) * (metric_of(m) ? 76 : 28));
    double const force_bytes = (double) ncand * 16;
    // variants, chosen online per size class of the directions measured: lanes
    // per edge (1, 2, 4 or 8) and, in the mixed mode, the FP32 screen (+16) or
    // the certified FP32 pass (+32); all give identical results.  The mixed
    // mode takes an FP32 form from CQ_CERTIFIED_MIN directions up (below that
    // the certified pass's three extra small launches cost more than the FP64
    // work it saves).  Above it the FP32 forms no longer win: since a block's
    // directions are handed on as they end, 8 cycles of the 64^3 x 6
    // anisotropic box spend 134 ms on these kernels in FP64 and 180 ms in the
    // mixed mode, which has no FP64 variant there (192 ms with every variant
    // timed anew on live launches, the trials included).
    static thread_local Tuner tuners[2][3] = {
        {Tuner("coarsen_quality_2d_f64", {1, 2, 4, 8}),
         Tuner("coarsen_quality_2d_mixed", {33, 34, 36, 40, 17, 18, 20, 24}),
         Tuner("coarsen_quality_2d_mixed_small", {1, 2, 4, 8})},
        {Tuner("coarsen_quality_3d_f64", {1, 2, 4, 8}),
         Tuner("coarsen_quality_3d_mixed", {33, 34, 36, 40, 17, 18, 20, 24}),
         Tuner("coarsen_quality_3d_mixed_small", {1, 2, 4, 8})}};
    constexpr u32 CQ_CERTIFIED_MIN = 4096;
    bool const big = neval >= CQ_CERTIFIED_MIN || tuners[dim == 3][1].forced();
    Tuner& tuner = tuners[dim == 3][g_mixed ? (big ? 1 : 2) : 0];
    CqArgs a{};
    a.ncand = neval;
    a.list = some_known ? elist.get() : clist.get();
    a.ev = ev;
    a.uo = ue.offsets.get();
    a.ua = ue.adj.get();
    a.ud = ue.dirs.get();
    a.vel = vel;
    a.x = coords(m);
    a.mt = metric_of(m);
    a.eq = eqp;
    a.qual_floor = qual_floor;
    a.qfe = qfe;
    a.codes = codes.get();
    a.out = cq.get();
    a.vmark = nullptr;
    a.st = screen_stats();
    // collapse_to_vert (collapses_to_verts.cpp:13-70) belongs to the timed
    // variant: the certified pass adds its certification, the FP64
    // measurement of what it could not certify and a second collapse_to_vert,
    // so a trial times the whole sequence (events recorded on the stream
    // around it) and the tuner weighs the variants by what they cost
    u32 const nv = count(m, 0);
    Up const& uv = ask_up(m, 0, 1);
    cand = Buf<u32>(nv);
    vq = Buf<double>(nv);
    auto measure = [&](u32 var, hipEvent_t ea, hipEvent_t eb) {
      u32 g = var & 15u;
      u32 mode = (var & 32u) ? (u32) CQ_CERTIFIED : (var & 16u) ? (u32) CQ_SCREEN : (u32) CQ_F64;
      bool const measures32 = mode == CQ_CERTIFIED && !require_better;
      if (sizes && measures32) sizes->inexact = true;
      // FP32 values may also come from an earlier pass
      bool const certified = measures32 || (sizes && sizes->inexact);
      if (ea) OHX_CHECK(hipEventRecord(ea, stream()));
      if (neval)
        dim == 3 ? cq_launch_mode<3>(mode, g, a, prof_bytes, nullptr, nullptr)
                 : cq_launch_mode<2>(mode, g, a, prof_bytes, nullptr, nullptr);
      Buf<u32> vinex, vmark;
      if (certified) vinex = Buf<u32>(nv);
      auto to_vert = [&] {
        if (!nv) return;
        hipLaunchKernelGGL(collapse_to_vert_k, dim3(nblocks(nv)), dim3(BLOCK), 0, stream(), nv, uv.offsets.get(),
                           uv.adj.get(), uv.dirs.get(), codes.get(), cq.get(), voff.get(), cand.get(), vq.get(),
                           certified ? vinex.get() : nullptr, scratch_words() + W_FLAGS);
        check_launch("collapse_to_vert");
      };
      to_vert();
      if (certified && nv) {
        // the comparisons the FP32 goodness takes part in: the vertices
        // whose choices are not certified get exact values (their inexact
        // directions measured in FP64), then their best again
        vmark = Buf<u32>(nv);
        hipLaunchKernelGGL(coarsen_certify, dim3(nblocks(nv)), dim3(BLOCK), 0, stream(), nv, uv.offsets.get(),
                           uv.adj.get(), uv.dirs.get(), codes.get(), cq.get(), ev, cand.get(), vq.get(), vinex.get(),
                           vmark.get());
        check_launch("coarsen_certify");
        CqArgs f = a;
        f.ncand = ncand;
        f.list = clist.get();
        f.vmark = vmark.get();
        dim == 3 ? cq_launch_mode<3>(CQ_FORCE, g, f, force_bytes, nullptr, nullptr)
                 : cq_launch_mode<2>(CQ_FORCE, g, f, force_bytes, nullptr, nullptr);
        to_vert();
      }
      if (eb) OHX_CHECK(hipEventRecord(eb, stream()));
    };
    if (neval)
      tuned(tuner, neval, measure);
    else
      measure(1, nullptr, nullptr);
  }
  // no host check here: if the quality check left no collapse, the
  // candidates below are empty, the independent set settles at once and the
  // one read of its total returns 0 (check_coarsen_quality's early return)
  u32 nv = count(m, 0);
  Up const& uv = ask_up(m, 0, 1);
  eq.release();
  // a first batch of indset rounds, the collapse destinations and the
  // vertex offsets, then one read of the convergence flag and the total
  u32 const* flag = nullptr;
  Buf<u32> indset = find_indset_from(m, 0, std::move(cand), vq.get(), &flag);
  Buf<u32> gvv(nv);
  // coarsen_all_ents (coarsen_common.cpp:91-107), top dimension first.
  // Phase 1 decides every dimension's survivors and products on the device
  // (a dimension's fused sides feed the next lower one, no host decision
  // needed), right after the destinations; one launch scans them all and one
  // read then brings the set's convergence flag, the collapse count and all
  // the totals; phase 2 writes the outputs.
  bool has_class = find_tag(m, 0, "class_dim") != nullptr;
  bool has_id = find_tag(m, 0, "class_id") != nullptr;
  bool const transfers = has_element_transfer(m);
  Buf<u32> fused_to[4], goff, soff(nv + 1);
  struct DimPlan {
    Buf<u32> gv, gd, egoff, esoff, fate;
  };
  DimPlan plan[4];
  u32 got[scan_detail::MAX_JOBS], open = 0;
  auto dest_and_total = [&] {
    // vertex_dest (collapses_to_verts.cpp:72-135); the sides' fusions are
    // cleared on the way
    u32 const* uo = uv.offsets.get();
    u32 const* ua = uv.adj.get();
    u32 const* ud = uv.dirs.get();
    u32 const* cd = codes.get();
    double const* q = cq.get();
    double const* vqp = vq.get();
    u32 const* is = indset.get();
    u32* g = gvv.get();
    u32* err = dev_error_word();
    u32 const* fl = flag;
    u32 const nf1 = dim >= 2 ? count(m, 1) : 0, nf2 = dim == 3 ? count(m, 2) : 0;
    for (u32 d = 1; d < dim; ++d) fused_to[d] = Buf<u32>(count(m, d));
    u32 *ft1 = fused_to[1].get(), *ft2 = fused_to[2].get();
    u32 const nmost = nf2 > nf1 ? nf2 : nf1;
    parallel_for(nmost > nv ? nmost : nv, OHX_LAMBDA(u32 i) {
      if (i < nf1) ft1[i] = INVALID;
      if (i < nf2) ft2[i] = INVALID;
      if (i >= nv) return;
      if (!is[i] || (fl && *fl)) {  // not in the set, or the set is not settled yet
        g[i] = INVALID;
        return;
      }
      double maxq = vqp[i];
      if (maxq == 1e10) maxq = -1e10;
      u32 gv = INVALID;
      for (u32 j = uo[i]; j < uo[i + 1]; ++j) {
        u32 e = ua[j], d = ud[j];
        if (!collapses(cd[e], d)) continue;
        double qq = q[2 * (size_t) e + d];
        if (qq == 1e10) qq = -1e10;
        if (qq == maxq) {
          gv = ev[2 * (size_t) e + (1 - d)];
          break;
        }
      }
      if (gv == INVALID) *err = ERR_NO_DESTINATION;
      g[i] = gv;
    });
    // coarsen_interior (coarsen_common.cpp:191-219)
    scan_detail::ScanJobs J{};
    scan_job(J, nv, is, NOT_IN_SET, soff.get());
    for (u32 dd = 0; dd < dim; ++dd) {
      u32 d = dim - dd;
      u32 n = count(m, d);
      u32 const* vent = ask_down(m, d, 0);
      u32 const* sent = ask_down(m, d, d - 1);
      DimPlan& pl = plan[d];
      pl.gv = Buf<u32>(n);
      pl.gd = Buf<u32>(n);
      pl.fate = Buf<u32>(n);
      pl.egoff = Buf<u32>(n + 1);
      pl.esoff = Buf<u32>(n + 1);
      {
        CollapseEnts a{};
        a.n = n;
        a.vent = vent;
        a.sent = sent;
        a.is = is;
        a.g = g;
        a.fe = fused_to[d].get();  // null for elements
        a.ft = d >= 2 ? fused_to[d - 1].get() : nullptr;
        a.fate = pl.fate.get();
        a.gv = pl.gv.get();
        a.gd = pl.gd.get();
        auto go = [&](auto kernel) {
          hipLaunchKernelGGL(kernel, dim3(nblocks(n)), dim3(BLOCK), 0, stream(), a);
          check_launch("collapse_ents");
        };
        if (n) d == 3 ? go(collapse_ents_k<3>) : d == 2 ? go(collapse_ents_k<2>) : go(collapse_ents_k<1>);
      }
    }
    for (u32 d = 1; d <= dim; ++d) {
      u32 const n = count(m, d);
      scan_job(J, n, plan[d].fate.get(), REBUILT, plan[d].egoff.get());
      scan_job(J, n, plan[d].fate.get(), SAME, plan[d].esoff.get());
    }
    if (transfers) {  // the only reader of the collapsing vertices' own numbering
      goff = Buf<u32>(nv + 1);
      scan_job(J, nv, is, IN_SET, goff.get());
    }
    exscan_jobs(J, flag, got, &open);
  };
  // got: surviving vertices, then per dimension the rebuilt and the same
  dest_and_total();
  if (open) {  // not settled in the first batch: the checked loop from there
    indset = find_indset_resume(m, 0, vq.get(), std::move(indset));
    flag = nullptr;
    dest_and_total();
  }
  if (g_batch) batch_note_changed(m, 0, indset.get());
  if (!sizes) {
    codes.release();
    cq.release();
  }
  vq.release();
  u32 const nv_out = got[0], total = nv - nv_out;
  if (!total) return 0;
  indset.release();
  auto const rebuilt = [&](u32 d) { return got[1 + 2 * (d - 1)]; };
  auto const same = [&](u32 d) { return got[2 + 2 * (d - 1)]; };
  Mesh mo(dim, m.full);
  set_ents(mo, 0, nv_out, Buf<u32>());
  CoarsenOutputs out{};
  out.nv = nv;
  out.soff = soff.get();
  // tags_subset (subset.cpp:15-43): every vertex tag
  for (auto& tp : m.tags[0]) {
    Tag& t = *tp;
    void* dst;
    if (t.type == TagType::F64)
      dst = add_tag_f64(mo, 0, t.name.c_str(), t.ncomps, Buf<double>((size_t) nv_out * t.ncomps), t.transfer).f.get();
    else
      dst = add_tag_u32(mo, 0, t.name.c_str(), t.ncomps, Buf<u32>((size_t) nv_out * t.ncomps), t.transfer).u.get();
    tag_list_add(out.tags, t, dst);
  }
  double out_bytes = 0;
  u32 blocks = 0;
  // the maps this pass read and the next collapse pass reads again,
  // carried to the new mesh instead of derived again: each entity's sides
  // (down(d, d-1)) here, the vertices' upward adjacencies below.  The tets'
  // edges and up(1,3) are carried by the sliver collapse passes only: a swap
  // pass reads them, and carrying them through the collapse-by-size loop
  // as well cost more than one reflection before the swap (64^3 x 6
  // anisotropic box: 2.87 against 2.82 s per 8 cycles)
  Buf<u32> side_maps[4][4];
  for (u32 dd = 0; dd < dim; ++dd) {
    u32 d = dim - dd;
    u32 n = count(m, d);
    u32 vpe = d + 1;
    u32 ngen = rebuilt(d), nsame = same(d);
    DimPlan& pl = plan[d];
    Buf<u32> vout((size_t) (nsame + ngen) * vpe);
    Buf<u32> cdo, cio;
    CoarsenArgs& a = out.a[dd];
    out.block0[dd] = blocks;
    blocks += nblocks(n);
    auto carry_sides = [&](u32 l, CoarsenSides& cs) {
      u32 const ns = simplex_sides(d, l);
      side_maps[d][l] = Buf<u32>((size_t) (nsame + ngen) * ns);
      cs.out = side_maps[d][l].get();
      cs.old = m.down[d][l].get();
      cs.soff = plan[l].esoff.get();
      cs.egoff = plan[l].egoff.get();
      cs.fused_to = fused_to[l].get();
      cs.nsame = same(l);
      cs.l = l;
      cs.nold = m.counts[l];
      cs.err = dev_error_word();
    };
    if (d >= 2 && m.down[d][d - 1]) carry_sides(d - 1, a.sides);
    // a sliver collapse pass is followed by a swap pass, which reads the
    // tets' edges (and up(1,3), carried below)
    if (require_better && d == 3 && m.down[3][1]) carry_sides(1, a.edges);
    a.d = d;
    a.n = n;
    a.nsame = nsame;
    a.vent = ask_down(m, d, 0);
    a.esoff = pl.esoff.get();
    a.egoff = pl.egoff.get();
    a.gv = pl.gv.get();
    a.gd = pl.gd.get();
    a.vsoff = soff.get();
    a.out = vout.get();
    if (has_class) {
      cdo = Buf<u32>(nsame + ngen);
      a.cd = u32_tag(m, d, "class_dim");
      a.out_cd = cdo.get();
      if (has_id) {
        cio = Buf<u32>(nsame + ngen);
        a.ci = u32_tag(m, d, "class_id");
        a.out_ci = cio.get();
      }
    }
    // compulsory bytes per old entity: its vertices in, their new numbers
    // gathered and written, its survivor and product offsets, target and
    // direction, class tags in and out, and the carried sides (old ids in,
    // new ids gathered and written)
    u32 const ns = (a.sides.out ? simplex_sides(d, d - 1) : 0u) + (a.edges.out ? 6u : 0u);
    out_bytes += (double) n * (vpe * 12 + 32 + ns * 12);
    set_ents(mo, d, nsame + ngen, std::move(vout));
    if (has_class) {
      add_tag_u32(mo, d, "class_dim", 1, std::move(cdo));
      if (has_id) add_tag_u32(mo, d, "class_id", 1, std::move(cio));
    }
  }
  for (u32 k = dim; k < 4; ++k) out.block0[k] = blocks;
  launch_timed("coarsen_outputs", out_bytes, coarsen_outputs, dim3(blocks + nblocks(nv)), dim3(BLOCK), out);
  if (transfers)
    coarsen_transfer(m, mo, goff.get(), total, plan[dim].egoff.get(), plan[dim].esoff.get(), same(dim), rebuilt(dim));
  for (u32 h = 2; h <= dim; ++h)
    for (u32 l = 1; l < h; ++l)
      if (side_maps[h][l]) mo.down[h][l] = std::move(side_maps[h][l]);
  // the vertices' upward adjacencies this pass read (to edges, to
  // elements), carried too (vertices survive or are removed, none is new)
  UpPatchCounts elems;  // which vertices kept their elements
  auto carry_up = [&](u32 h) {
    if (!m.up[0][h]) return;
    mo.up[0][h] = up_patch(h_down_deg[h][0], *m.up[0][h], m.counts[0], soff.get(), nv_out, 0, plan[h].esoff.get(),
                           same(h), rebuilt(h), mo.down[h][0].get(), h == dim && sizes ? &elems : nullptr);
  };
  carry_up(1);
  carry_up(dim);
  if (sizes && sizes->ne == m.counts[1]) {
    // the new mesh's size codes: survivors' carried, products measured;
    // and what is known of the survivors' qualities
    u32 const ne_old = m.counts[1], ngen1 = rebuilt(1), nsame1 = same(1), ne_new = nsame1 + ngen1;
    Buf<u32> nc(ne_new), nk(ne_new);
    Buf<double> nq((size_t) 2 * ne_new);
    CarryCodes a{};
    a.ne_old = ne_old;
    a.ngen = ngen1;
    a.nsame = nsame1;
    a.soff = plan[1].esoff.get();
    a.old_codes = sizes->codes.get();
    a.ev = mo.down[1][0].get();
    a.x = coords(mo);
    a.h = size_of(mo);
    a.mt = metric_of(mo);
    a.floor_ = size_floor;
    a.codes = nc.get();
    a.now = codes.get();
    a.old_known = sizes->known.get();
    a.q = cq.get();
    a.old_ev = ev;
    a.vsoff = soff.get();
    a.full = elems.full.get();
    a.cnt = elems.cnt.get();
    a.cnt_s = elems.cnt_s.get();
    a.known = nk.get();
    a.new_q = nq.get();
    hipLaunchKernelGGL(carry_size_codes_k, dim3(nblocks((size_t) ne_old + ngen1)), dim3(BLOCK), 0, stream(), a);
    check_launch("carry_size_codes");
    sizes->ne = ne_new;
    sizes->codes = std::move(nc);
    sizes->known = std::move(nk);
    sizes->q = std::move(nq);
  } else if (sizes) {
    sizes->clear();
  }
  if (require_better && dim == 3 && m.up[1][3] && mo.down[3][1])
    mo.up[1][3] = up_patch(6, *m.up[1][3], m.counts[1], plan[1].esoff.get(), same(1), rebuilt(1),
                           plan[3].esoff.get(), same(3), rebuilt(3), mo.down[3][1].get());
  say("collapsed", total, 1);
  overwrite(m, std::move(mo));
  return 1;
}

u32 coarsen_by_size(Mesh& m, double qual_floor, double size_floor, SizeCodeCache* cache) {
  u32 ne = count(m, 1);
  double const* h = size_of(m);
  double const* mt = metric_of(m);
  Buf<u32> codes(ne);
  u32 tag = next_any_tag();
  if (g_batch && cache) cache->clear();
  if (cache && cache->ne != ne) cache->clear();
  if (ne && cache && cache->ne) {
    // the codes carried from the pass before (the pass consumes its copy)
    // -- without the directions known to be rejected, the accepted ones
    // marked so that they are not measured again
    u32* c = codes.get();
    u32 const* cc = cache->codes.get();
    u32 const* kn = cache->known.get();
    u32* words = scratch_words();
    parallel_for(ne, OHX_LAMBDA(u32 i) {
      u32 v = cc[i];
      u32 const k = kn && v ? kn[i] : 0u;
      for (u32 d = 0; d < 2; ++d) {
        if (k & was_rejected(d)) v = dont_collapse(v, d);
        if (k & (1u << d)) v |= known_bit(d) | ((k & was_inexact(d)) ? inexact_bit(d) : 0u);
      }
      c[i] = v;
      wave_flag_value(words + W_ANY, (v & (u32) COLLAPSE_BOTH) != 0, tag);
    });
  } else if (ne) {
    double prof_bytes = (double) ne * 12 + (double) count(m, 0) * 32;
    launch_timed("coarsen_size_code_f64", prof_bytes, coarsen_size_code_f64, dim3(nblocks(ne)), dim3(BLOCK), ne,
                       ask_down(m, 1, 0), coords(m), h, mt, size_floor, codes.get(), scratch_words(), tag);
    if (cache && !g_batch) {
      cache->ne = ne;
      cache->codes = copy(codes.get(), ne);
    }
  }
  // check_coarsen_noop (coarsen_common.cpp:109-118), kept as its own read:
  // without it the last, unproductive pass of every coarsening loop would
  // derive the maps of the class checks for nothing, which on small meshes
  // costs more than the host wait it saves on each productive pass
  if (read_word(W_ANY) != tag) return 0;
  if (g_batch) {
    batch_mask(m, 1, codes.get());
    Buf<double> qfe = batch_floors(m, 1);
    return coarsen_common(m, codes, qual_floor, false, qfe.get());
  }
  return coarsen_common(m, codes, qual_floor, false, nullptr, nullptr, cache, size_floor);
}

// coarsen_slivers (coarsen.cpp:38-70)
u32 coarsen_slivers(Mesh& m, double qual_floor, u32 nlayers, double const* eq) {
  u32 dim = m.dim;
  Buf<u32> sl = mark_slivers(m, qual_floor, nlayers, eq);
  Buf<u32> mv = mark_down(m, dim, 0, sl.get());
  sl.release();
  u32 ne = count(m, 1);
  u32 const* ev = ask_down(m, 1, 0);
  Buf<u32> codes(ne);
  u32* c = codes.get();
  u32 const* mk = mv.get();
  parallel_for(ne, OHX_LAMBDA(u32 i) {
    u32 r = 0;
    if (mk[ev[2 * i]]) r |= 1u;
    if (mk[ev[2 * i + 1]]) r |= 2u;
    c[i] = r;
  });
  if (g_batch) batch_mask(m, 1, c);
  // check_coarsen_noop (coarsen_common.cpp:109-118) is coarsen_common's
  // count of the directions left (its first host read)
  return coarsen_common(m, codes, 0.0, true, nullptr, eq);
}

// ----------------------------------------------------------------- swap
// Triangulations of an N-gon (N = 3..7), their unique triangles
// (edge_swap.cpp:21-200) and, generated on first use, the interior edges of
// each triangulation.  The triangulation index is the swap code; ties in
// quality keep the lowest code, so the order must equal the reference's.
static u32 const h_sw_sizes[8] = {0, 0, 0, 1, 2, 3, 4, 5};
static u32 const h_sw_counts[8] = {0, 0, 0, 1, 2, 5, 14, 42};
static u32 const h_sw_tri_off[8] = {0, 0, 0, 0, 1, 5, 15, 35};
static u32 const h_sw_mesh_off[8] = {0, 0, 0, 0, 1, 5, 20, 76};
static unsigned char const h_sw_tris[70][3] = {
    {0, 1, 2},  // N = 3
    {0, 1, 2}, {0, 2, 3}, {0, 1, 3}, {1, 2, 3},  // N = 4
    {0, 1, 2}, {0, 2, 3}, {0, 3, 4}, {0, 1, 4}, {1, 3, 4}, {1, 2, 3}, {2, 3, 4}, {0, 2, 4}, {0, 1, 3},
    {1, 2, 4},  // N = 5
    {0, 1, 2}, {0, 2, 3}, {0, 3, 4}, {0, 4, 5}, {0, 2, 5}, {2, 4, 5}, {2, 3, 4}, {0, 3, 5}, {3, 4, 5},
    {0, 2, 4}, {2, 3, 5}, {1, 2, 3}, {0, 1, 3}, {0, 1, 5}, {1, 4, 5}, {1, 3, 4}, {0, 1, 4}, {1, 3, 5},
    {1, 2, 4}, {1, 2, 5},  // N = 6
    {0, 1, 2}, {0, 2, 3}, {0, 3, 4}, {0, 4, 5}, {0, 5, 6}, {0, 3, 6}, {3, 5, 6}, {3, 4, 5}, {0, 4, 6},
    {4, 5, 6}, {0, 3, 5}, {3, 4, 6}, {0, 2, 4}, {2, 3, 4}, {0, 2, 6}, {2, 5, 6}, {2, 4, 5}, {0, 2, 5},
    {2, 4, 6}, {2, 3, 5}, {2, 3, 6}, {0, 1, 3}, {1, 2, 3}, {0, 1, 4}, {1, 3, 4}, {0, 1, 6}, {1, 5, 6},
    {1, 4, 5}, {0, 1, 5}, {1, 4, 6}, {1, 3, 5}, {1, 3, 6}, {1, 2, 4}, {1, 2, 5}, {1, 2, 6}};  // N = 7
static unsigned char const h_sw_meshes[286] = {
    0,                                                                             // N = 3
    0, 1, 2, 3,                                                                    // N = 4
    0, 1, 2, 3, 4, 5, 0, 6, 7, 2, 5, 8, 3, 6, 9,                                   // N = 5
    0, 1, 2, 3, 0, 4, 5, 6, 0, 1, 7, 8, 0, 3, 6, 9, 0, 4, 8, 10, 2, 3, 11, 12, 11, 13, 14, 15, 7, 8, 11, 12,
    3, 11, 15, 16, 8, 11, 13, 17, 6, 13, 14, 18, 3, 6, 16, 18, 5, 6, 13, 19, 8, 10, 13, 19,  // N = 6
    0, 1, 2, 3, 4, 0, 1, 5, 6, 7, 0, 1, 2, 8, 9, 0, 1, 4, 7, 10, 0, 1, 5, 9, 11, 0, 3, 4, 12, 13, 0, 13, 14,
    15, 16, 0, 8, 9, 12, 13, 0, 4, 13, 16, 17, 0, 9, 13, 14, 18, 0, 7, 14, 15, 19, 0, 4, 7, 17, 19, 0, 6, 7,
    14, 20, 0, 9, 11, 14, 20, 2, 3, 4, 21, 22, 5, 6, 7, 21, 22, 2, 8, 9, 21, 22, 4, 7, 10, 21, 22, 5, 9, 11,
    21, 22, 3, 4, 22, 23, 24, 22, 24, 25, 26, 27, 8, 9, 22, 23, 24, 4, 22, 24, 27, 28, 9, 22, 24, 25, 29, 7,
    22, 25, 26, 30, 4, 7, 22, 28, 30, 6, 7, 22, 25, 31, 9, 11, 22, 25, 31, 3, 4, 13, 23, 32, 13, 25, 26, 27,
    32, 8, 9, 13, 23, 32, 4, 13, 27, 28, 32, 9, 13, 25, 29, 32, 13, 16, 25, 26, 33, 4, 13, 16, 28, 33, 13,
    15, 16, 25, 34, 9, 13, 18, 25, 34, 7, 19, 25, 26, 33, 4, 7, 19, 28, 33, 7, 15, 19, 25, 34, 6, 7, 20, 25,
    34, 9, 11, 20, 25, 34};  // N = 7

static __constant__ u32 k_sw_sizes[8] = {0, 0, 0, 1, 2, 3, 4, 5};
static __constant__ u32 k_sw_counts[8] = {0, 0, 0, 1, 2, 5, 14, 42};
static __constant__ u32 k_sw_tri_off[8] = {0, 0, 0, 0, 1, 5, 15, 35};
static __constant__ u32 k_sw_mesh_off[8] = {0, 0, 0, 0, 1, 5, 20, 76};
static __constant__ unsigned char k_sw_tris[70][3];
static __constant__ unsigned char k_sw_meshes[286];
// interior edges: offsets per ring size, then [code][edge][2]
static __constant__ u32 k_sw_nint[8];
static __constant__ u32 k_sw_int_off[8];
static __constant__ unsigned char k_sw_int[444];

static u32 h_sw_nint[8];
static u32 h_sw_int_off[8];
static unsigned char h_sw_int[444];
static bool g_swap_ready = false;
static std::mutex g_swap_mu;

// The interior edges of each triangulation, derived the way the
// reference's generator does (test_print_swap_edges.cpp:29-64): the
// triangulation as a reduced 2D mesh, its derived edges, the non-boundary
// ones in edge order.  All triangulations of one N form one mesh of
// disjoint components; side derivation numbers each component's edges
// contiguously and in the same order as a mesh of its own would.
static void make_swap_tables() {
  std::lock_guard<std::mutex> lock(g_swap_mu);
  if (g_swap_ready) return;
  u32 off = 0;
  for (u32 n = 0; n < 4; ++n) {
    h_sw_nint[n] = 0;
    h_sw_int_off[n] = 0;
  }
  for (u32 n = 4; n <= MAX_EDGE_SWAP; ++n) {
    u32 nm = h_sw_counts[n], nt = h_sw_sizes[n];
    std::vector<u32> conn((size_t) nm * nt * 3);
    for (u32 c = 0; c < nm; ++c)
      for (u32 k = 0; k < nt; ++k)
        for (u32 l = 0; l < 3; ++l)
          conn[((size_t) c * nt + k) * 3 + l] = c * n + h_sw_tris[h_sw_tri_off[n] + h_sw_meshes[h_sw_mesh_off[n] + c * nt + k]][l];
    Mesh m(2, false);
    set_ents(m, 0, nm * n, Buf<u32>());
    set_ents(m, 2, nm * nt, to_device(conn.data(), conn.size()));
    Buf<u32> bd = mark_part_boundary(m);
    u32 ne = count(m, 1);
    std::vector<u32> hb = host_copy(bd.get(), ne);
    std::vector<u32> ev = host_copy(ask_down(m, 1, 0), (size_t) 2 * ne);
    u32 nint_total = 0;
    for (u32 k = 0; k < ne; ++k) nint_total += !hb[k];
    OHX_REQUIRE(nint_total % nm == 0, "swap tables: uneven interior edge counts");
    u32 nint = nint_total / nm;
    h_sw_nint[n] = nint;
    h_sw_int_off[n] = off;
    std::vector<u32> seen(nm, 0);
    for (u32 k = 0; k < ne; ++k) {
      if (hb[k]) continue;
      u32 c = ev[2 * k] / n;
      OHX_REQUIRE(ev[2 * k + 1] / n == c && seen[c] < nint, "swap tables: bad interior edge");
      u32 slot = off + (c * nint + seen[c]) * 2;
      h_sw_int[slot] = (unsigned char) (ev[2 * k] - c * n);
      h_sw_int[slot + 1] = (unsigned char) (ev[2 * k + 1] - c * n);
      ++seen[c];
    }
    off += nm * nint * 2;
  }
  OHX_REQUIRE(off == 444, "swap tables: unexpected size");
  OHX_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(k_sw_tris), h_sw_tris, sizeof(h_sw_tris)));
  OHX_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(k_sw_meshes), h_sw_meshes, sizeof(h_sw_meshes)));
  OHX_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(k_sw_nint), h_sw_nint, sizeof(h_sw_nint)));
  OHX_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(k_sw_int_off), h_sw_int_off, sizeof(h_sw_int_off)));
  OHX_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(k_sw_int), h_sw_int, sizeof(h_sw_int)));
  g_swap_ready = true;
}

u32 swap_nint_edges(u32 rs) {
  make_swap_tables();
  return h_sw_nint[rs];
}

void swap_int_edges_host(u32 rs, u32 code, u32* out) {
  make_swap_tables();
  u32 k = h_sw_nint[rs];
  for (u32 i = 0; i < 2 * k; ++i) out[i] = h_sw_int[h_sw_int_off[rs] + code * k * 2 + i];
}

// find_edge_ring (edge_ring.cpp:12-74): ring vertices ordered by chaining
// each tet's opposite edge (a -> b), insertion style, <= 7 entries
__device__ inline u32 edge_ring(u32 edge, u32 f, u32 e, u32 const* ua, u32 const* ud, u32 const* ev,
                                u32 const* vt, u32* edge_v, u32* ring_v) {
  u32 rs = e - f;
  if (rs > MAX_EDGE_SWAP || rs < 3) return rs;
  u32 const* oe = opp(3, 1);
  edge_v[0] = ev[2 * (size_t) edge];
  edge_v[1] = ev[2 * (size_t) edge + 1];
  u32 ra[MAX_EDGE_SWAP], rb[MAX_EDGE_SWAP];
  for (u32 i = f; i < e; ++i) {
    u32 const* tv = vt + 4 * (size_t) ua[i];
    u32 te = ud[i];
    u32 const* tve = canon(3, 1, 0, te);
    u32 al = (tv[tve[0]] != edge_v[0]) ? 1u : 0u;
    u32 const* tvo = canon(3, 1, 0, oe[te]);
    ra[i - f] = tv[tvo[al]];
    rb[i - f] = tv[tvo[al ^ 1u]];
  }
  for (u32 i = 0; i + 1 < rs; ++i) {
    u32 j;
    for (j = i + 1; j < rs; ++j)
      if (ra[j] == rb[i]) break;
    if (j == rs) return 0;  // ring does not close: reported by the caller
    u32 ta = ra[j], tb = rb[j];
    ra[j] = ra[i + 1];
    rb[j] = rb[i + 1];
    ra[i + 1] = ta;
    rb[i + 1] = tb;
  }
  for (u32 i = 0; i < rs; ++i) ring_v[i] = ra[i];
  return rs;
}

// swap_quality (swap_qualities.cpp:13-65) with choose_edge_swap
// (edge_swap.cpp:230-280), SW_G lanes per edge.  One lane per edge would
// hold the ring's coordinates and metrics and the quality of every unique
// triangle (up to 35) in registers, which spills; here a group of lanes
// shares them in LDS:
//   A. lane j < ring size reads the edge's j-th tet: its opposite edge
//      (a, b) oriented as find_edge_ring orients it, and its quality
//      (old_minq is the minimum over the group);
//   B. lane 0 chains the pairs into the ring (edge_ring.cpp:12-74);
//   C. lane j stages ring vertex j (or edge vertex j - ring size): its
//      coordinates and metric;
//   D. two neighbouring lanes measure a unique triangle: the two tets it
//      forms with the edge's ends, as choose_edge_swap does (a ring of 4 has
//      4 triangles: its 8 tets take the group's 8 lanes once; with both of a
//      triangle's tets on one lane half the lanes waited);
//   E. lane l takes triangulations l, l + SW_G, ...: the running minimum of
//      its triangles, stopped at the first negative one as the reference's
//      loop stops, and the lane's best with a strict > in triangulation
//      order; the group combines them keeping the higher value and, on
//      ties, the lower triangulation index -- the reference's sequential
//      strict > choice.
// FP32-mixed (MIXED): D and E run first with the FP32 quality; a candidate
// whose FP32 best lies more than the margin below old_minq (and none of
// whose triangles is within the margin of zero, where the reference's
// early stop could fall elsewhere) is rejected there, every other one is
// measured again in FP64, so every accepted value and code is the FP64
// path's.  Accepted candidates store the value (goodness), the ring size
// and the triangulation code, which swap_cavity uses.  The kernel is built
// for 4 waves per SIMD (at most 128 VGPRs; its 33 KB of LDS per block allow
// 4 blocks per CU): with both tets of a triangle on one lane that cost 28
// bytes of scratch per lane and measured 4 % less time on the 64^3 x 6
// anisotropic box than 3 waves without spills; with a tet per lane it takes
// 98 VGPRs and no scratch.
constexpr u32 SW_G = 8;
constexpr u32 SW_EDGES = BLOCK / SW_G;
constexpr u32 SW_MAXTRI = 35;
static __constant__ u32 k_sw_ntri[8] = {0, 0, 0, 1, 4, 10, 20, 35};

template <bool MT>
struct SwapLds {
  u32 ra[SW_EDGES][MAX_EDGE_SWAP], rb[SW_EDGES][MAX_EDGE_SWAP];
  u32 ring[SW_EDGES][MAX_EDGE_SWAP];
  u32 rs[SW_EDGES];      // ring size of an active edge, else 0
  u32 again[SW_EDGES];   // FP32-mixed: measure again in FP64
  double old_minq[SW_EDGES];
  double x[SW_EDGES][MAX_EDGE_SWAP + 2][3];          // ring, then edge vertices
  double m[MT ? SW_EDGES : 1][MAX_EDGE_SWAP + 2][6];  // their metrics
  double tq[SW_EDGES][SW_MAXTRI];
};

template <bool MT, bool F32>
__device__ inline double swap_tet_q(SwapLds<MT> const& L, u32 g, u32 a0, u32 a1, u32 a2, u32 e) {
  V3 p[4];
  u32 const idx[4] = {a0, a1, a2, e};
#pragma unroll
  for (u32 k = 0; k < 4; ++k) p[k] = V3{L.x[g][idx[k]][0], L.x[g][idx[k]][1], L.x[g][idx[k]][2]};
  if (MT) {
    Sym pm[4];
#pragma unroll
    for (u32 k = 0; k < 4; ++k)
#pragma unroll
      for (u32 c = 0; c < 6; ++c) pm[k].m[c] = L.m[g][idx[k]][c];
    return F32 ? (double) quality32<3>(p, pm, true) : metric_quality<3>(p, pm, true);
  }
  return F32 ? (double) quality32<3>(p, nullptr, true) : tet_quality(p[0], p[1], p[2], p[3]);
}

// phases D and E for the group of this lane; returns the group's (best,
// code) in every lane of the group, *near0 set if any triangle's quality is
// within SCREEN_MARGIN of zero
template <bool MT, bool F32>
__device__ inline void swap_choose(SwapLds<MT>& L, u32 g, u32 lane, bool active, double* best, u32* code,
                                   bool* near0) {
  u32 rs = active ? L.rs[g] : 0u;
  bool nz = false;
  if (rs) {
    u32 ntri = k_sw_ntri[rs];
    unsigned char const(*tris)[3] = k_sw_tris + k_sw_tri_off[rs];
    u32 const E0 = rs, E1 = rs + 1;  // edge vertices follow the ring in LDS
    for (u32 k = lane; k < 2 * ntri; k += SW_G) {
      // the triangle with edge end 1, then with the first two corners
      // exchanged and edge end 0 (choose_edge_swap's two tets), on two
      // neighbouring lanes
      u32 const t = k / 2, end = k & 1u;
      double const q = swap_tet_q<MT, F32>(L, g, tris[t][end], tris[t][1 - end], tris[t][2], end ? E0 : E1);
      double tmin = q < 1 ? q : 1;
      double const other = __shfl_xor(tmin, 1, SW_G);
      if (other < tmin) tmin = other;
      if (F32 && !(tmin > (double) SCREEN_MARGIN || tmin < -(double) SCREEN_MARGIN)) nz = true;
      if (!end) L.tq[g][t] = tmin;
    }
  }
  __syncthreads();
  double b = -1;
  u32 c = INVALID;
  if (rs) {
    u32 tpm = k_sw_sizes[rs], nm = k_sw_counts[rs];
    unsigned char const* meshes = k_sw_meshes + k_sw_mesh_off[rs];
    for (u32 k = lane; k < nm; k += SW_G) {
      double mq = 1;
      for (u32 j = 0; j < tpm; ++j) {
        double tq = L.tq[g][meshes[k * tpm + j]];
        if (tq < mq) mq = tq;
        if (mq < 0) break;
      }
      if (mq > b) {
        b = mq;
        c = k;
      }
    }
  }
  // combine over the group: higher value, then lower triangulation index
#pragma unroll
  for (u32 d = SW_G / 2; d >= 1; d >>= 1) {
    double ob = __shfl_xor(b, d, SW_G);
    u32 oc = (u32) __shfl_xor((int) c, d, SW_G);
    if (ob > b || (ob == b && oc < c)) {
      b = ob;
      c = oc;
    }
    nz = nz || __shfl_xor((int) nz, d, SW_G);
  }
  *best = b;
  *code = c;
  *near0 = nz;
}

// one batch of SW_EDGES candidates, group g of the block takes list[slot];
// returns whether the group's candidate is accepted, with its value, ring
// size and triangulation code; settled: the group had a candidate whose
// choice is now known
template <bool MT, bool MIXED>
__device__ inline bool swap_quality_batch(SwapLds<MT>& L, u32 ncand, u32 slot, u32 const* __restrict__ list,
                                          u32 const* __restrict__ uo, u32 const* __restrict__ un,
                                          u32 const* __restrict__ ua, u32 const* __restrict__ ud,
                                          u32 const* __restrict__ ev, u32 const* __restrict__ vt,
                                          double const* __restrict__ x, double const* __restrict__ mt,
                                          double const* __restrict__ eq, u32* __restrict__ err, ScreenStats st,
                                          u32* edge, bool* settled, double* value, u32* ring_size, u32* choice) {
  u32 const g = threadIdx.x / SW_G, lane = threadIdx.x % SW_G;
  bool active = slot < ncand;
  u32 const i = active ? list[slot] : 0u;
  *edge = i;
  *settled = active;
  // A: the tets around the edge
  u32 f = 0, rs = 0, e0 = 0, e1 = 0;
  double qmin = 1;
  if (active) {
    f = uo[i];
    rs = un ? un[i] : uo[i + 1] - f;
    e0 = ev[2 * (size_t) i];
    e1 = ev[2 * (size_t) i + 1];
    if (rs > MAX_EDGE_SWAP || rs < 3) {
      if (lane == 0 && rs < 3) *err = ERR_EDGE_RING;
      active = false;
    } else if (lane < rs) {
      u32 tet = ua[f + lane], te = ud[f + lane];
      u32 const* tv = vt + 4 * (size_t) tet;
      u32 const* tve = canon(3, 1, 0, te);
      u32 al = (tv[tve[0]] != e0) ? 1u : 0u;
      u32 const* tvo = canon(3, 1, 0, opp(3, 1)[te]);
      L.ra[g][lane] = tv[tvo[al]];
      L.rb[g][lane] = tv[tvo[al ^ 1u]];
      double q = eq[tet];
      if (q < qmin) qmin = q;
    }
  }
#pragma unroll
  for (u32 d = SW_G / 2; d >= 1; d >>= 1) {
    double o = __shfl_xor(qmin, d, SW_G);
    if (o < qmin) qmin = o;
  }
  __syncthreads();
  // B: the ring, chained as find_edge_ring does
  if (active && lane == 0) {
    u32* ra = L.ra[g];
    u32* rb = L.rb[g];
    bool closed = true;
    for (u32 a = 0; a + 1 < rs; ++a) {
      u32 j;
      for (j = a + 1; j < rs; ++j)
        if (ra[j] == rb[a]) break;
      if (j == rs) {
        closed = false;
        break;
      }
      u32 ta = ra[j], tb = rb[j];
      ra[j] = ra[a + 1];
      rb[j] = rb[a + 1];
      ra[a + 1] = ta;
      rb[a + 1] = tb;
    }
    if (!closed) *err = ERR_EDGE_RING;
    L.rs[g] = closed ? rs : 0u;
    L.old_minq[g] = qmin;
    for (u32 a = 0; a < rs; ++a) L.ring[g][a] = ra[a];
  } else if (lane == 0) {
    L.rs[g] = 0;
  }
  __syncthreads();
  // C: the ring's and the edge's vertices
  rs = active ? L.rs[g] : 0u;
  active = rs != 0;
  // (a 7-ring has 9 vertices: more than the group's lanes)
  for (u32 k = lane; active && k < rs + 2; k += SW_G) {
    u32 v = k < rs ? L.ring[g][k] : (k == rs ? e0 : e1);
#pragma unroll
    for (u32 c = 0; c < 3; ++c) L.x[g][k][c] = x[3 * (size_t) v + c];
    if (MT)
#pragma unroll
      for (u32 c = 0; c < 6; ++c) L.m[g][k][c] = mt[6 * (size_t) v + c];
  }
  if (lane == 0) L.again[g] = 0;
  // the block's work needs the staged data and every lane of the group
  // (and of the block: the phases below are separated by barriers)
  __syncthreads();
  double best;
  u32 code;
  bool near0;
  double const old_minq = active ? L.old_minq[g] : 1.0;
  if (MIXED) {
    swap_choose<MT, true>(L, g, lane, active, &best, &code, &near0);
    bool reject = active && !near0 && best + (double) SCREEN_MARGIN <= old_minq;
    if (lane == 0) {
      if (active) L.again[g] = reject ? 0u : 1u;
    }
    wave_count(st.screened, lane == 0 && reject);
    wave_count(st.reeval, lane == 0 && active && !reject);
    __syncthreads();
    double best32 = best;
    bool const valid32 = !near0;  // no triangle near zero: best32 is the FP64 choice's, rounded
    bool again = active && L.again[g] != 0;
    swap_choose<MT, false>(L, g, lane, again, &best, &code, &near0);
    if (again && valid32 && lane == 0 && best == best) {
      double dd = best - best32;
      note_max_err(st.max_err, (float) (dd < 0 ? -dd : dd));
    }
    active = again;
  } else {
    swap_choose<MT, false>(L, g, lane, active, &best, &code, &near0);
  }
  *value = best;
  *ring_size = rs;
  *choice = code;
  return active && best > old_minq;
}

template <bool MT, bool MIXED>
__global__ __launch_bounds__(BLOCK, 4) void swap_quality_k(
    u32 ncand, u32 const* __restrict__ list, u32 const* __restrict__ uo, u32 const* __restrict__ ua,
    u32 const* __restrict__ ud, u32 const* __restrict__ ev, u32 const* __restrict__ vt,
    double const* __restrict__ x, double const* __restrict__ mt, double const* __restrict__ eq,
    u32* __restrict__ cand, double* __restrict__ out, u32* __restrict__ rsz, u32* __restrict__ codes,
    u32* __restrict__ words, u32 tag, u32* __restrict__ err, ScreenStats st) {
  __shared__ SwapLds<MT> L;
  u32 i, rs, code;
  bool settled;
  double best;
  bool const accept = swap_quality_batch<MT, MIXED>(L, ncand, xcd_block() * SW_EDGES + threadIdx.x / SW_G, list, uo,
                                                    nullptr, ua, ud, ev, vt, x, mt, eq, err, st, &i, &settled, &best,
                                                    &rs, &code);
  if (settled && threadIdx.x % SW_G == 0) {
    if (accept) {
      out[i] = best;
      rsz[i] = rs;
      codes[i] = code;
    } else {
      cand[i] = 0;
    }
  }
  wave_flag_value(words + W_ANY, accept, tag);
}

// count_swap_ents (edge_swap.cpp:375-386)
static inline __host__ __device__ u32 count_swap_ents(u32 rs, u32 d, u32 nint, u32 tpm) {
  return d == 1 ? nint : (d == 2 ? tpm + 2 * nint : 2 * tpm);
}

// The swapped mesh's tet-to-edge map, built from the old one instead of by
// reflection (reflect_down.cpp:13-81 gives the same map: an entity's lows
// are unique in a conforming mesh).  A surviving tet is adjacent to no
// swapped edge, so its six edges survive too and it keeps them, renumbered.
// A product tet's edges are its cavity's: ring edges and spokes (ring
// vertex to an end of the swapped edge), both edges of the old tets around
// the swapped edge, and the new interior edges.  out null: not built.
struct SwapEdgesOf {
  u32* out;            // (surviving + product tets) x 6 new edge ids
  u32 const* old;      // the old tets' edges
  u32 const* soff1;    // old edge -> its index among the surviving edges
  u32 nsame1, nsame3;  // surviving edges, surviving tets
  u32* err;
  // the element dual carried too (dual null: not built): the old dual,
  // the tets' survivor offsets, per old tet face the product now across it
  // (written for the cavities' outer faces), and per product face whose
  // outside tet is in another cavity the old (tet, face) to resolve
  u32* dual;
  u32 const* old_dual;
  u32 const* soff3;
  u32* face_prod;
  u32* deferred;
};

constexpr u32 DUAL_PENDING = 0xfffffffeu;

// local face of a tet (vertices tv) with the vertices a, b, c
__device__ inline u32 tet_face_of(u32 const* tv, u32 a, u32 b, u32 c) {
  for (u32 f = 0; f < 4; ++f) {
    u32 const* fv = canon(3, 2, 0, f);
    u32 hits = 0;
    for (u32 q = 0; q < 3; ++q) {
      u32 v = tv[fv[q]];
      hits += (v == a || v == b || v == c) ? 1u : 0u;
    }
    if (hits == 3) return f;
  }
  return 0;
}

// local edge of a tet between local vertices a and b
__device__ inline u32 tet_edge_between(u32 a, u32 b) {
  for (u32 j = 0; j < 6; ++j) {
    u32 const* c = canon(3, 1, 0, j);
    if ((c[0] == a && c[1] == b) || (c[0] == b && c[1] == a)) return j;
  }
  return 0;
}

// swap_cavity (swap_topology.cpp:46-75) with get_swap_ents
// (edge_swap.cpp:282-373), every dimension in one launch: the ring again
// (integer work) and the triangulation code that swap_quality chose, then
// the products' vertices (interior edges, their faces, the tets: triangle t
// of the triangulation with edge end 1, then with its first two corners
// exchanged and edge end 0), written where out_d is given.  With E.out, the
// product tets' edges too: a product tet's vertices are labelled by where
// they come from (ring slot, or edge end); an edge between adjacent ring
// slots is a ring edge, one between a slot and an edge end a spoke, both
// edges of the old tet at that ring slot (the one holding ring vertices k
// and k + 1), and any other is one of the new interior edges.  The cavity's
// ring edges and spokes are staged in LDS per thread (indexed by slot).
__global__ __launch_bounds__(BLOCK) void swap_products_k(
    u32 ne, u32 const* __restrict__ indset, u32 const* __restrict__ goff1, u32 const* __restrict__ goff2,
    u32 const* __restrict__ goff3, u32 const* __restrict__ uo, u32 const* __restrict__ ua,
    u32 const* __restrict__ ud, u32 const* __restrict__ ev, u32 const* __restrict__ vt,
    u32 const* __restrict__ codes, u32* __restrict__ out1, u32* __restrict__ out2, u32* __restrict__ out3,
    SwapEdgesOf E) {
  __shared__ u32 s_ring[MAX_EDGE_SWAP][BLOCK];
  __shared__ u32 s_spoke[2][MAX_EDGE_SWAP][BLOCK];
  __shared__ u32 s_tet[MAX_EDGE_SWAP][BLOCK];
  u32 const tid = threadIdx.x;
  u32 i = xcd_block() * BLOCK + tid;
  if (i >= ne || !indset[i]) return;  // no barrier follows
  u32 const g1 = goff1[i], g2 = goff2[i], g3 = goff3[i];
  u32 const f = uo[i], e = uo[i + 1];
  u32 edge_v[2], ring_v[MAX_EDGE_SWAP];
  u32 rs = edge_ring(i, f, e, ua, ud, ev, vt, edge_v, ring_v);
  if (rs < 3 || rs > MAX_EDGE_SWAP) return;  // cannot happen for an indset edge
  u32 const code = codes[i];
  u32 const tpm = k_sw_sizes[rs];
  unsigned char const* mesh = k_sw_meshes + k_sw_mesh_off[rs] + code * tpm;
  unsigned char const(*tris)[3] = k_sw_tris + k_sw_tri_off[rs];
  u32 const nint = k_sw_nint[rs];
  unsigned char const* ie = k_sw_int + k_sw_int_off[rs] + code * nint * 2;
  if (out1) {
    u32* o = out1 + (size_t) g1 * 2;
    for (u32 k = 0; k < nint; ++k) {
      o[2 * k] = ring_v[ie[2 * k]];
      o[2 * k + 1] = ring_v[ie[2 * k + 1]];
    }
  }
  if (out2) {
    u32* o = out2 + (size_t) g2 * 3;
    for (u32 k = 0; k < nint; ++k)
      for (u32 j = 0; j < 2; ++j) {
        o[k * 6 + j * 3 + 0] = ring_v[ie[2 * k]];
        o[k * 6 + j * 3 + 1] = ring_v[ie[2 * k + 1]];
        o[k * 6 + j * 3 + 2] = edge_v[j];
      }
    o += nint * 6;
    for (u32 t = 0; t < tpm; ++t)
      for (u32 j = 0; j < 3; ++j) o[t * 3 + j] = ring_v[tris[mesh[t]][j]];
  }
  for (u32 k = 0; E.out && k < rs; ++k) {
    u32 const a = ring_v[k], b = ring_v[k + 1 < rs ? k + 1 : 0];
    u32 tet = INVALID;
    for (u32 q = f; q < e && tet == INVALID; ++q) {
      u32 const* tv = vt + 4 * (size_t) ua[q];
      bool ha = false, hb = false;
      for (u32 c = 0; c < 4; ++c) {
        ha = ha || tv[c] == a;
        hb = hb || tv[c] == b;
      }
      if (ha && hb) tet = ua[q];
    }
    if (tet == INVALID) {
      *E.err = ERR_REFLECT_NOT_FOUND;
      return;
    }
    u32 const* tv = vt + 4 * (size_t) tet;
    u32 const* te = E.old + 6 * (size_t) tet;
    u32 la = 0, lb = 0, l0 = 0, l1 = 0;
    for (u32 c = 0; c < 4; ++c) {
      if (tv[c] == a) la = c;
      if (tv[c] == b) lb = c;
      if (tv[c] == edge_v[0]) l0 = c;
      if (tv[c] == edge_v[1]) l1 = c;
    }
    s_tet[k][tid] = tet;
    s_ring[k][tid] = E.soff1[te[tet_edge_between(la, lb)]];
    s_spoke[0][k][tid] = E.soff1[te[tet_edge_between(la, l0)]];
    s_spoke[1][k][tid] = E.soff1[te[tet_edge_between(la, l1)]];
  }
  if (!out3) return;
  u32* o3 = out3 + (size_t) g3 * 4;
  u32 const first = E.nsame3 + g3;
  for (u32 t = 0; t < tpm; ++t) {
    u32 lab[4], tv[4];  // labels: ring slot, or 8 + edge end; vertices
    for (u32 j = 0; j < 3; ++j) {
      lab[j] = tris[mesh[t]][j];
      tv[j] = ring_v[lab[j]];
    }
    for (u32 j = 0; j < 2; ++j) {
      lab[3] = 8 + (1 - j);
      tv[3] = edge_v[1 - j];
      for (u32 k = 0; k < 4; ++k) *o3++ = tv[k];
      if (!E.out) {
        u32 tmp = tv[0];
        tv[0] = tv[1];
        tv[1] = tmp;
        tmp = lab[0];
        lab[0] = lab[1];
        lab[1] = tmp;
        continue;
      }
      u32* eo = E.out + 6 * (size_t) (first + 2 * t + j);
      for (u32 le = 0; le < 6; ++le) {
        u32 const* c = canon(3, 1, 0, le);
        u32 a = lab[c[0]], b = lab[c[1]];
        u32 id = INVALID;
        if (a >= 8 || b >= 8) {
          if (a < 8) id = s_spoke[b - 8][a][tid];
          else if (b < 8) id = s_spoke[a - 8][b][tid];
        } else if (a + 1 == b || a == b + rs - 1) {
          id = s_ring[a][tid];
        } else if (b + 1 == a || b == a + rs - 1) {
          id = s_ring[b][tid];
        } else {
          for (u32 k = 0; k < nint; ++k)
            if ((ie[2 * k] == a && ie[2 * k + 1] == b) || (ie[2 * k] == b && ie[2 * k + 1] == a))
              id = E.nsame1 + g1 + k;
        }
        if (id == INVALID) *E.err = ERR_REFLECT_NOT_FOUND;
        eo[le] = id;
      }
      if (E.dual) {
        // the tet across each face: the twin (same triangle, other end)
        // across the triangle; across a face on a ring edge, the tet
        // outside the ring tet's face there; across a face on an interior
        // edge, the product of the other triangle holding that edge
        u32 const self = first + 2 * t + j;
        u32* dd = E.dual + 4 * (size_t) self;
        for (u32 f = 0; f < 4; ++f) {
          u32 const* fv = canon(3, 2, 0, f);
          u32 r[2], nr = 0;
          bool has_end = false;
          for (u32 q = 0; q < 3; ++q) {
            u32 l = lab[fv[q]];
            if (l >= 8)
              has_end = true;
            else if (nr < 2)
              r[nr++] = l;
          }
          u32 nb = INVALID;
          if (!has_end) {
            nb = first + 2 * t + (1 - j);
          } else {
            u32 const a = r[0], b = r[1];
            bool const ring = a + 1 == b || a == b + rs - 1 || b + 1 == a || b == a + rs - 1;
            if (ring) {
              u32 const k = (a + 1 == b || a == b + rs - 1) ? a : b;
              u32 const tk = s_tet[k][tid];
              u32 const x = 1 - j;  // this tet's edge end
              u32 const lf = tet_face_of(vt + 4 * (size_t) tk, edge_v[x], ring_v[k], ring_v[k + 1 < rs ? k + 1 : 0]);
              E.face_prod[4 * (size_t) tk + lf] = self;
              u32 const o = E.old_dual[4 * (size_t) tk + lf];
              if (o == INVALID) {
                nb = INVALID;
              } else if (E.soff3[o] != E.soff3[o + 1]) {
                nb = E.soff3[o];
              } else {
                nb = DUAL_PENDING;
                E.deferred[4 * (size_t) (self - E.nsame3) + f] = 4 * tk + lf;
              }
            } else {
              for (u32 t2 = 0; t2 < tpm; ++t2) {
                if (t2 == t) continue;
                unsigned char const* tr = tris[mesh[t2]];
                bool ha = tr[0] == a || tr[1] == a || tr[2] == a;
                bool hb = tr[0] == b || tr[1] == b || tr[2] == b;
                if (ha && hb) nb = first + 2 * t2 + j;
              }
              if (nb == INVALID) *E.err = ERR_REFLECT_NOT_FOUND;
            }
          }
          dd[f] = nb;
        }
      }
      u32 tmp = tv[0];
      tv[0] = tv[1];
      tv[1] = tmp;
      tmp = lab[0];
      lab[0] = lab[1];
      lab[1] = tmp;
    }
  }
}

// The new dual's remaining entries: threads [0, nt_old) give a surviving
// tet its neighbours (a surviving one renumbered, a removed one replaced by
// the product now across that face); the ngen3 * 4 after them resolve a
// product face whose outside tet was removed by another cavity.
__global__ __launch_bounds__(BLOCK) void swap_dual_k(u32 nt_old, u32 ngen3, SwapEdgesOf E) {
  u32 const s = xcd_block() * BLOCK + threadIdx.x;
  auto across = [&](u32 n, u32 from) -> u32 {  // the product across n's face shared with from
    for (u32 g = 0; g < 4; ++g)
      if (E.old_dual[4 * (size_t) n + g] == from) return E.face_prod[4 * (size_t) n + g];
    *E.err = ERR_REFLECT_NOT_FOUND;
    return INVALID;
  };
  if (s < nt_old) {
    u32 const o = E.soff3[s];
    if (o == E.soff3[s + 1]) return;
    for (u32 f = 0; f < 4; ++f) {
      u32 const n = E.old_dual[4 * (size_t) s + f];
      u32 r = INVALID;
      if (n != INVALID) r = E.soff3[n] != E.soff3[n + 1] ? E.soff3[n] : across(n, s);
      E.dual[4 * (size_t) o + f] = r;
    }
  } else if (s - nt_old < 4 * ngen3) {
    u32 const q = s - nt_old;
    u32* d = E.dual + 4 * (size_t) E.nsame3 + q;
    if (*d != DUAL_PENDING) return;
    u32 const key = E.deferred[q];
    u32 const tk = key / 4;
    u32 const n = E.old_dual[key];
    *d = across(n, tk);
  }
}

__global__ __launch_bounds__(BLOCK) void copy_tags(u32 n, TagList L) {
  u32 i = xcd_block() * BLOCK + threadIdx.x;
  if (i >= n) return;
  for (u32 t = 0; t < L.n; ++t) {
    u32 w = L.ncomps[t];
    if (L.f64[t]) {
      double const* f = static_cast<double const*>(L.src[t]);
      double* dd = static_cast<double*>(L.dst[t]);
      for (u32 c = 0; c < w; ++c) dd[(size_t) i * w + c] = f[(size_t) i * w + c];
    } else {
      u32 const* f = static_cast<u32 const*>(L.src[t]);
      u32* dd = static_cast<u32*>(L.dst[t]);
      for (u32 c = 0; c < w; ++c) dd[(size_t) i * w + c] = f[(size_t) i * w + c];
    }
  }
}

struct SwapKeepArgs {
  u32 n, ne, vpe, nsame;
  u32 const* soff;
  u32 const* goff;
  u32 const* vent;
  u32* out;
  SwapEdgesOf E;  // tets: the survivors' edges (E.out null: not built)
  u32 const* cd;
  u32 const* ci;
  u32 const* ecd;
  u32 const* eci;
  u32* out_cd;
  u32* out_ci;
};

// concat_verts_of_ents for the survivors of a swap, and the class tags of
// survivors (their own) and of products (their edge's, setup_swap,
// inherit.cpp:158-166): threads [0, n) are entities, [n, n + ne) edges
__global__ __launch_bounds__(BLOCK) void swap_keep(SwapKeepArgs a) {
  u32 t = xcd_block() * BLOCK + threadIdx.x;
  if (t < a.n) {
    u32 o = a.soff[t];
    if (o == a.soff[t + 1]) return;
    for (u32 j = 0; j < a.vpe; ++j) a.out[(size_t) o * a.vpe + j] = a.vent[(size_t) t * a.vpe + j];
    if (a.E.out)
      for (u32 j = 0; j < 6; ++j) a.E.out[(size_t) o * 6 + j] = a.E.soff1[a.E.old[(size_t) t * 6 + j]];
    if (a.out_cd) a.out_cd[o] = a.cd[t];
    if (a.out_ci) a.out_ci[o] = a.ci[t];
    return;
  }
  u32 e = t - a.n;
  if (e >= a.ne) return;
  for (u32 k = a.goff[e]; k < a.goff[e + 1]; ++k) {
    if (a.out_cd) a.out_cd[a.nsame + k] = a.ecd[e];
    if (a.out_ci) a.out_ci[a.nsame + k] = a.eci[e];
  }
}

// a vertex pair as one key (smaller vertex in the high word) and its home
// slot in a table of mask + 1 slots
__host__ __device__ inline unsigned long long swap_pair_key(u32 a, u32 b) {
  return a < b ? ((unsigned long long) a << 32) | b : ((unsigned long long) b << 32) | a;
}
__host__ __device__ inline u32 swap_pair_slot(unsigned long long key, u32 mask) {
  key ^= key >> 29;
  key *= 0xBF58476D1CE4E5B9ull;
  key ^= key >> 32;
  return (u32) key & mask;
}

// in the mixed mode the FP32 screen is a variant chosen online: it pays only
// where it rejects enough candidates (most swap candidates improve their
// cavity and need their exact FP64 value anyway)
static Tuner& swap_tuner() {
  static thread_local Tuner tuner("swap_quality_3d_mixed", {0, 1});
  return tuner;
}
static bool swap_screen_pinned() {
  u32 const* v = swap_tuner().forced_variant();
  return v && *v == 1;
}

// swap_common + swap_interior + swap_ents (swap.cpp:27-136)
static u32 swap_common(Mesh& m, Buf<u32>& cand, double const* eq_given = nullptr, SwapCache* cache = nullptr) {
  check_index_space(m);
  u32 ne = count(m, 1);
  unmark_boundary(m, 1, cand.get());
  Buf<double> q(ne);
  Buf<u32> rsz = filled(ne, 0);
  Buf<u32> codes(ne);
  // candidates with a cached choice (their edge's tets unchanged since an
  // earlier swap pass of this shape loop evaluated it) take it: a rejected
  // one leaves the candidates, an accepted one keeps its value, ring size
  // and triangulation; they are counted on the device
  if (cache && cache->ne != ne) cache->clear();
  SwapCache* const cc = cache && cache->ne ? cache : nullptr;
  u32 const* inf = cc ? cc->info.get() : nullptr;
  if (cc) {
    fill(scratch_words() + W_CACHED, 1, 0);
    u32* cp = cand.get();
    double const* cq = cc->q.get();
    double* qo = q.get();
    u32* rs = rsz.get();
    u32* cd = codes.get();
    u32* nacc = scratch_words() + W_CACHED;
    parallel_for(ne, OHX_LAMBDA(u32 i) {
      bool hit = false;
      u32 const f = inf[i];
      if (cp[i] && (f >> 31)) {
        if ((f >> 30) & 1u) {
          qo[i] = cq[i];
          rs[i] = (f >> 16) & 0xffu;
          cd[i] = f & 0xffffu;
          hit = true;
        } else {
          cp[i] = 0;
        }
      }
      unsigned long long const b = __ballot(hit), act = __ballot(1);
      if (b && (u32) __lane_id() == (u32) (__ffsll((long long) act) - 1)) atomicAdd(nacc, (u32) __popcll(b));
    });
  }
  // the candidates to evaluate, compacted (with the cached ones accepted,
  // their count is the reference's early return, swap.cpp:103-106, in one
  // read)
  Buf<u32> coff(ne + 1);
  u32 ncand, ncached = 0;
  {
    u32 const* cp = cand.get();
    auto f = OHX_LAMBDA(u32 i) { return cp[i] && !(inf && (inf[i] >> 31)) ? 1u : 0u; };
    if (cc) {
      exscan_fn(ne, f, coff.get());
      u32 const* ptrs[2] = {coff.get() + ne, scratch_words() + W_CACHED};
      u32 got[2];
      read_many(ptrs, 2, got);
      ncand = got[0];
      ncached = got[1];
    } else {
      ncand = exscan_fn_total(ne, f, coff.get());
    }
  }
  if (!ncand && !ncached) return 0;
  Buf<u32> clist(ncand);
  if (ncand) {
    u32 const* co = coff.get();
    u32* cl = clist.get();
    parallel_for(ne, OHX_LAMBDA(u32 i) {
      if (co[i] != co[i + 1]) cl[co[i]] = i;
    });
  }
  coff.release();
  make_swap_tables();
  Up const& u = ask_up(m, 1, 3);
  u32 const* ev = ask_down(m, 1, 0);
  u32 const* vt = ask_down(m, 3, 0);
  Buf<double> eq;
  if (!eq_given) eq = mesh_qualities(m);
  double const* eqp = eq_given ? eq_given : eq.get();
  u32 tag = next_any_tag();
  if (ncand) {
    // compulsory bytes: the edges' candidate flags, vertices and outputs,
    // the tets around them (uses + directions), their qualities and
    // vertices, and the vertex coordinates (and metrics)
    double const* mts = metric_of(m);
    double prof_bytes = (double) ne * 24 + (double) u.adj.size() * 8 + (double) count(m, 3) * 24 +
                        (double) count(m, 0) * (mts ? 72 : 24);
    ScreenStats sst = screen_stats();
    dim3 grid((unsigned) ((ncand + SW_EDGES - 1) / SW_EDGES));
    auto go = [&](auto kernel, char const* kn, hipEvent_t ea, hipEvent_t eb) {
      if (ea) {
        hipExtLaunchKernelGGL(kernel, grid, dim3(BLOCK), 0, stream(), ea, eb, 0, ncand, clist.get(), u.offsets.get(),
                              u.adj.get(), u.dirs.get(), ev, vt, coords(m), mts, eqp, cand.get(), q.get(),
                              rsz.get(), codes.get(), scratch_words(), tag, dev_error_word(), sst);
        check_launch(kn);
      } else {
        launch_timed(kn, prof_bytes, kernel, grid, dim3(BLOCK), ncand, clist.get(), u.offsets.get(), u.adj.get(),
                     u.dirs.get(), ev, vt, coords(m), mts, eqp, cand.get(), q.get(), rsz.get(), codes.get(),
                     scratch_words(), tag, dev_error_word(), sst);
      }
    };
    auto run = [&](u32 screen, hipEvent_t ea, hipEvent_t eb) {
      if (screen)
        mts ? go(swap_quality_k<true, true>, "swap_quality_mixed", ea, eb)
            : go(swap_quality_k<false, true>, "swap_quality_mixed", ea, eb);
      else
        mts ? go(swap_quality_k<true, false>, "swap_quality_f64", ea, eb)
            : go(swap_quality_k<false, false>, "swap_quality_f64", ea, eb);
    };
    if (g_mixed)
      tuned(swap_tuner(), ncand, run);
    else
      run(0, nullptr, nullptr);
  }
  eq.release();
  // the evaluated candidates' choices go into the cache (this mesh's
  // numbering; the swap below carries the cache to the new mesh)
  if (cache) {
    if (!cc) {
      cache->ne = ne;
      cache->q = Buf<double>(ne);
      cache->info = filled(ne, 0);
    }
    if (ncand) {
      u32 const* cl = clist.get();
      u32 const* cp = cand.get();
      double const* qi = q.get();
      u32 const* rs = rsz.get();
      u32 const* cd = codes.get();
      double* cq = cache->q.get();
      u32* ci = cache->info.get();
      parallel_for(ncand, OHX_LAMBDA(u32 k) {
        u32 const i = cl[k];
        ci[i] = (1u << 31) | (cp[i] ? (1u << 30) | (rs[i] << 16) | cd[i] : 0u);
        cq[i] = qi[i];
      });
    }
  }
  // the early return after the qualities (swap.cpp:119-124) is the totals
  // read below: the quality kernel clears every rejected candidate, so
  // with none accepted the set is empty and no element is generated
  // a first batch of indset rounds with no host check, every dimension's
  // product and survivor offsets, then one read of the convergence flag
  // and all the totals (a set not settled in the first batch goes on from
  // there with the checked loop, same rounds, same result)
  u32 const* flag = nullptr;
  Buf<u32> indset = find_indset_bounded(m, 1, cand.get(), q.get(), &flag);
  u32 dlo = m.full ? 1 : m.dim;
  Buf<u32> goffs[4], soffs[4];
  u32 tots[8];
  // the faces that survive are those holding no swapped edge; a face holds
  // an edge exactly when it holds both of the edge's vertices, so when the
  // face-to-edge map is not derived (it is needed for nothing else here) the
  // swapped edges' vertex pairs go into a small hash table and each face
  // looks its three vertex pairs up, instead of hashing every edge of the
  // mesh to build down(2,1)
  bool const faces_by_pairs = m.dim == 3 && m.full && !m.down[2][1];
  u32 pcap = 64;
  while (pcap < 4 * ((size_t) ncand + ncached)) pcap *= 2;
  Buf<unsigned long long> pairs(faces_by_pairs ? pcap : 0);
  auto offsets_and_totals = [&] {
    u32 const* is = indset.get();
    u32 const* rs = rsz.get();
    u32 const* pt[8];
    u32 k = 0;
    pt[k++] = flag;
    if (faces_by_pairs) {
      unsigned long long* tb = pairs.get();
      u32 const mask = pcap - 1;
      parallel_for(pcap, OHX_LAMBDA(u32 i) { tb[i] = ~0ull; });
      u32* err = dev_error_word();
      parallel_for(ne, OHX_LAMBDA(u32 e) {
        if (!is[e]) return;
        unsigned long long key = swap_pair_key(ev[2 * (size_t) e], ev[2 * (size_t) e + 1]);
        u32 h = swap_pair_slot(key, mask);
        for (u32 probe = 0; probe <= mask; ++probe, h = (h + 1) & mask)
          if (atomicCAS(&tb[h], ~0ull, key) == ~0ull) return;
        *err = ERR_REFLECT_NOT_FOUND;
      });
    }
    for (u32 d = dlo; d <= m.dim; ++d) {
      u32 n = count(m, d);
      // products per swapped edge (edge_topo_offset, swap_topology.cpp:16-44)
      // and survivors: entities adjacent to no swapped edge (swap.cpp:41-45)
      goffs[d] = Buf<u32>(ne + 1);
      soffs[d] = Buf<u32>(n + 1);
      exscan_fn(ne, OHX_LAMBDA(u32 i) {
        return is[i] ? count_swap_ents(rs[i], d, k_sw_nint[rs[i]], k_sw_sizes[rs[i]]) : 0u;
      }, goffs[d].get());
      if (d == 2 && faces_by_pairs) {
        u32 const* fv = ask_down(m, 2, 0);
        unsigned long long const* tb = pairs.get();
        u32 const mask = pcap - 1;
        exscan_fn_heavy(n, OHX_LAMBDA(u32 i) {
          u32 const* v = fv + 3 * (size_t) i;
          for (u32 j = 0; j < 3; ++j) {
            unsigned long long key = swap_pair_key(v[j], v[(j + 1) % 3]);
            for (u32 probe = 0, h = swap_pair_slot(key, mask); probe <= mask; ++probe, h = (h + 1) & mask) {
              unsigned long long t = tb[h];
              if (t == key) return 0u;
              if (t == ~0ull) break;
            }
          }
          return 1u;
        }, soffs[d].get());
      } else {
        u32 lpe = h_down_deg[d][1];
        u32 const* le = ask_down(m, d, 1);
        exscan_fn_heavy(n, OHX_LAMBDA(u32 i) {
          for (u32 j = 0; j < lpe; ++j)
            if (is[le[(size_t) i * lpe + j]]) return 0u;
          return 1u;
        }, soffs[d].get());
      }
      pt[k++] = goffs[d].get() + ne;
      pt[k++] = soffs[d].get() + n;
    }
    read_many(pt, k, tots);
  };
  offsets_and_totals();
  if (tots[0]) {  // not settled in the first batch: the checked loop from there
    indset = find_indset_resume(m, 1, q.get(), std::move(indset));
    flag = nullptr;
    offsets_and_totals();
  }
  if (g_batch) batch_note_changed(m, 1, indset.get());
  cand.release();
  q.release();
  // every swapped edge generates elements, so none generated: nothing swapped
  if (!tots[1 + 2 * (m.dim - dlo)]) return 0;
  u32 total = g_verbose ? sum_u32(indset.get(), ne) : 0u;
  u32 nv = count(m, 0);
  Mesh mo(m.dim, m.full);
  set_ents(mo, 0, nv, Buf<u32>());
  {
    // copy_tags (tag.cpp): the vertices are unchanged, one launch for all tags
    TagList L;
    for (auto& tp : m.tags[0]) {
      Tag& t = *tp;
      void* dst;
      if (t.type == TagType::F64)
        dst = add_tag_f64(mo, 0, t.name.c_str(), t.ncomps, Buf<double>((size_t) nv * t.ncomps), t.transfer).f.get();
      else
        dst = add_tag_u32(mo, 0, t.name.c_str(), t.ncomps, Buf<u32>((size_t) nv * t.ncomps), t.transfer).u.get();
      tag_list_add(L, t, dst);
    }
    if (L.n) {
      hipLaunchKernelGGL(copy_tags, dim3(nblocks(nv)), dim3(BLOCK), 0, stream(), nv, L);
      check_launch("copy_tags");
    }
  }
  u32 const* is = indset.get();
  bool has_class = m.full && find_tag(m, 0, "class_dim") != nullptr;
  bool has_id = has_class && find_tag(m, 0, "class_id") != nullptr;
  // the tets' edges of the new mesh, from the old map (the old one exists:
  // the rings above read up(1,3)); the next pass asks for them first
  bool const edges_of_tets = m.dim == 3 && dlo == 1;
  Buf<u32> d31, dual_new, face_prod, deferred;
  // every dimension's products in one launch (the ring of each swapped edge
  // found once), then the survivors dimension by dimension
  Buf<u32> vouts[4];
  u32* pouts[4] = {nullptr, nullptr, nullptr, nullptr};
  double prof_bytes = (double) ne * 12;
  for (u32 d = dlo; d <= m.dim; ++d) {
    u32 ngen = tots[1 + 2 * (d - dlo)], nsame = tots[2 + 2 * (d - dlo)];
    vouts[d] = Buf<u32>((size_t) (nsame + ngen) * (d + 1));
    pouts[d] = vouts[d].get() + (size_t) nsame * (d + 1);
    prof_bytes += (double) ngen * (d + 1) * 4;
  }
  SwapEdgesOf E{};
  u32 const nt_old = count(m, 3), ngen3 = tots[1 + 2 * (3 - dlo)], nsame3 = tots[2 + 2 * (3 - dlo)];
  if (edges_of_tets) {
    d31 = Buf<u32>((size_t) (nsame3 + ngen3) * 6);
    E.out = d31.get();
    E.old = ask_down(m, 3, 1);
    E.soff1 = soffs[1].get();
    E.nsame1 = tots[2];
    E.nsame3 = nsame3;
    E.err = dev_error_word();
    if (m.dual) {
      // the dual this pass's sliver marks read, carried to the next mesh
      dual_new = Buf<u32>((size_t) (nsame3 + ngen3) * 4);
      face_prod = Buf<u32>((size_t) nt_old * 4);
      deferred = Buf<u32>((size_t) ngen3 * 4);
      E.dual = dual_new.get();
      E.old_dual = m.dual.get();
      E.soff3 = soffs[3].get();
      E.face_prod = face_prod.get();
      E.deferred = deferred.get();
    }
  }
  launch_timed("swap_cavity", prof_bytes, swap_products_k, dim3(nblocks(ne)), dim3(BLOCK), ne, is,
               goffs[1].get(), goffs[2].get(), goffs[3].get(), u.offsets.get(), u.adj.get(), u.dirs.get(), ev, vt,
               codes.get(), pouts[1], pouts[2], pouts[3], E);
  if (E.dual) {
    hipLaunchKernelGGL(swap_dual_k, dim3(nblocks((size_t) nt_old + (size_t) ngen3 * 4)), dim3(BLOCK), 0, stream(),
                       nt_old, ngen3, E);
    check_launch("swap_dual");
  }
  for (u32 d = dlo; d <= m.dim; ++d) {
    u32 n = count(m, d);
    u32 vpe = d + 1;
    Buf<u32>& goff = goffs[d];
    Buf<u32>& soff = soffs[d];
    u32 ngen = tots[1 + 2 * (d - dlo)], nsame = tots[2 + 2 * (d - dlo)];
    Buf<u32> vout = std::move(vouts[d]);
    Buf<u32> cdo, cio;
    SwapKeepArgs a{};
    if (d == 3) a.E = E;
    a.n = n;
    a.ne = ne;
    a.vpe = vpe;
    a.nsame = nsame;
    a.soff = soff.get();
    a.goff = goff.get();
    a.vent = ask_down(m, d, 0);
    a.out = vout.get();
    if (has_class) {
      cdo = Buf<u32>(nsame + ngen);
      a.cd = u32_tag(m, d, "class_dim");
      a.ecd = u32_tag(m, 1, "class_dim");
      a.out_cd = cdo.get();
      if (has_id) {
        cio = Buf<u32>(nsame + ngen);
        a.ci = u32_tag(m, d, "class_id");
        a.eci = u32_tag(m, 1, "class_id");
        a.out_ci = cio.get();
      }
    }
    hipLaunchKernelGGL(swap_keep, dim3(nblocks(n + ne)), dim3(BLOCK), 0, stream(), a);
    check_launch("swap_keep");
    set_ents(mo, d, nsame + ngen, std::move(vout));
    if (has_class) {
      add_tag_u32(mo, d, "class_dim", 1, std::move(cdo));
      if (has_id) add_tag_u32(mo, d, "class_id", 1, std::move(cio));
    }
    if (d == m.dim) swap_transfer(m, mo, goff.get(), soff.get(), nsame, ngen);
    if (d == m.dim && cache && eq_given) {
      // the new mesh's element qualities: a survivor's is its old one, a
      // product's is evaluated (the same kernel mesh_qualities runs)
      Buf<double> neq = element_qualities(d, ngen, mo.down[d][0].get() + (size_t) nsame * vpe, coords(m),
                                          count(m, 0), metric_of(m));
      Buf<double> all((size_t) nsame + ngen);
      double* ap = all.get();
      double const* np = neq.get();
      u32 const* so = soff.get();
      double const* oq = eq_given;
      parallel_for(n, OHX_LAMBDA(u32 t) {
        u32 const o = so[t];
        if (o != so[t + 1]) ap[o] = oq[t];
      });
      if (ngen) d2d(ap + nsame, np, ngen);
      cache->eq = std::move(all);
    }
  }
  if (d31) {
    // the edge-to-tet adjacency from the old one (the rings above read it)
    UpPatchCounts pc;
    mo.up[1][3] = up_patch(6, u, ne, soffs[1].get(), tots[2], tots[1], soffs[3].get(), tots[6], tots[5], d31.get(),
                           cache ? &pc : nullptr);
    mo.down[3][1] = std::move(d31);
    if (dual_new) mo.dual = std::move(dual_new);
    if (cache) {
      // the cache in the new numbering: a surviving edge that kept all its
      // tets and gained none keeps its entry
      u32 const ne_new = tots[2] + tots[1];
      Buf<double> nq(ne_new);
      Buf<u32> ninfo = filled(ne_new, 0);
      u32 const* so = soffs[1].get();
      u32 const* full = pc.full.get();
      u32 const* cnt = pc.cnt.get();
      u32 const* cnt_s = pc.cnt_s.get();
      u32 const* ci = cache->info.get();
      double const* cq = cache->q.get();
      u32* ni = ninfo.get();
      double* nqp = nq.get();
      parallel_for(ne, OHX_LAMBDA(u32 e) {
        u32 const n = so[e];
        if (n == so[e + 1] || !full[n] || cnt[n] != cnt_s[n]) return;
        ni[n] = ci[e];
        nqp[n] = cq[e];
      });
      cache->ne = ne_new;
      cache->q = std::move(nq);
      cache->info = std::move(ninfo);
    }
  } else if (cache) {
    cache->clear();
  }
  say("swapped", total, 1);
  overwrite(m, std::move(mo));
  return 1;
}

u32 swap_slivers(Mesh& m, double good_qual, u32 nlayers, double const* eq, double const* gate, SwapCache* cache) {
  OHX_REQUIRE(m.dim == 3, "swap_slivers needs a 3D mesh");
  // the pass reads up(1,3) (the edge marks below, the rings, the quality
  // kernel); derived first, it also gives the sliver layers' element dual
  // from the rings (dual_edges_k) instead of a hash table of the faces
  (void) ask_up(m, 1, 3);
  Buf<u32> sl = mark_slivers(m, good_qual, nlayers, eq, gate);
  Buf<u32> c = mark_down(m, m.dim, 1, sl.get());
  sl.release();
  if (g_batch) batch_mask(m, 1, c.get());
  return swap_common(m, c, eq, cache);
}

// ------------------------------------------------- swap passes in place
// The shape loop's consecutive swap passes (adapt.cpp:58-80) on one copy of
// the mesh that is changed in place.  A pass through swap_common writes a
// whole new mesh, although it changes only its cavities and the passes of a
// run change ever fewer: on the 44^3 x 6 anisotropic box (2.2 to 4 million
// tets) a run's passes swap 412936, 276154, ... 11, 5, 1 edges, and each
// cost 2.4 ms of rewriting, renumbering and patching everything (all swap
// passes of that adapt: about 650 of 1309 ms of kernel time; in place 290 of 907).  Here
// entities keep their places: a pass marks what it removes, appends its
// products, and rewrites the tet lists of the edges around its cavities.
// swap_common's numbering (survivors in order, then products in the order of
// their swapped edges) is the order of the places in use, so every comparison
// of indices (ties in the independent set, the order of a list, where a ring
// starts) comes out the same, and closing the gaps once, after the run's
// last pass, gives the mesh that pass by pass rewriting gives.
//
// What is left per pass over the whole mesh is bound by bandwidth and small:
// the sliver marks (a byte per tet, their layers through the dual: 17 bytes
// read per tet and layer, the bytes gathered from L2), the edges' words (4
// bytes each; the tets of an edge are visited only where its swap is accepted
// or not yet known) and the states (a byte per edge).  The rest is as long as
// the pass's candidates or cavities.  One wait of the host per pass.
//
// A face survives a swap pass unless it holds the swapped edge, that is,
// both its vertices (swap.cpp:41-45), and the passes do not read faces, so
// the faces are settled once: each removed edge's vertex pair goes into a
// hash table with the last pass that removed it, and a face is gone if one
// of its pairs was removed in a pass after the one that made the face.

// Words of a swap run (SwapRunView::words).  RW_ERR: the error code of a
// kernel that changes the run's mesh, which is then of no use; an error found
// while a pass is only decided goes into the error word of every sync().
enum { RW_ACC = 0, RW_AFF = 2, RW_POOL = 3, RW_FIRST = 4, RW_ERR = 5, RW_FLAGS = 8, RW_EVAL = 16, RW_WORDS = 24 };
// ring sizes 3 to MAX_EDGE_SWAP: the candidates to evaluate are listed by
// ring size
constexpr u32 RUN_RINGS = MAX_EDGE_SWAP - 2;
// an edge's word in a run: its choice is known, it is accepted, then ring
// size and triangulation code as in the swap cache; a dead or boundary edge
// is known and rejected for good
constexpr u32 RI_KNOWN = 1u << 31, RI_ACCEPT = 1u << 30;

// The mesh of a run of swap passes (see "swap passes in place"), as slots.
struct SwapRunView {
  u32 nE, nF, nT, nF0;  // slots in use before the pass's products; faces at the start
  u32 pass;             // 1, 2, ...
  u32* ev;              // edges: vertices, class, the pass that removed it (0: alive), choice and its
  u32* ecd;             // value, first place and length of its list in (ua, ud), product uses
  u32* eci;
  u32* death;
  u32* info;
  double* q;
  u32* lb;
  u32* ln;
  u32* cnt;
  unsigned char* sa;  // independent-set state before / after a round
  unsigned char* sb;
  u32* ua;  // tets around the edges and the edges' places in them, ascending per edge
  u32* ud;
  u32* vt;  // tets: vertices, edges, dual, class, removed
  u32* te;
  u32* dual;
  u32* tcd;
  u32* tci;
  unsigned char* dead;
  u32* fv;  // faces: vertices, class, the pass that made a product face (from slot nF0 on)
  u32* fcd;
  u32* fci;
  u32* fbirth;
  u32* acc;  // accepted candidates (any order)
  u32* eval; // candidates to evaluate (any order), a list of ecap places per ring size
  u32 ecap;
  u32* sw;   // swapped edges in order, their first products of each dimension
  u32* o1;
  u32* o2;
  u32* o3;
  u32* words;
};

// Appending to a run's lists: blocks of RUN_AB threads, RUN_AI items each, one
// atomic per block and list.  Same-address atomics retire about one per 12 ns
// on this part, so one per wave held these kernels up (candidates of 3.7
// million edges 149 us, 36 us with one per 4096 edges and list).
constexpr u32 RUN_AB = 1024, RUN_AI = 4, RUN_AT = RUN_AB * RUN_AI;
// exclusive prefix of c over the block, the block's sum in *total; every
// thread of the block must call it
__device__ inline u32 run_block_prefix(u32 c, u32* lds, u32* total) {
  u32 const lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  u32 x = c;
#pragma unroll
  for (u32 d = 1; d < 64; d <<= 1) {
    u32 const y = (u32) __shfl_up((int) x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63u) lds[wave] = x;
  __syncthreads();
  u32 off = 0, all = 0;
  for (u32 w = 0; w < RUN_AB / 64; ++w) {
    u32 const v = lds[w];
    if (w < wave) off += v;
    all += v;
  }
  __syncthreads();
  *total = all;
  return off + x - c;
}
// the first list place of this thread's c items
__device__ inline u32 run_append(u32* counter, u32 c, u32* lds) {
  u32 total;
  u32 const p = run_block_prefix(c, lds, &total);
  if (threadIdx.x == 0) lds[0] = total ? atomicAdd(counter, total) : 0u;
  __syncthreads();
  u32 const base = lds[0];
  __syncthreads();
  return base + p;
}

constexpr u32 RUN_RED_BLOCKS = 1024;

// slivers (marks a byte per tet, mark.cpp:202-232) and the quality minimum
// over the live tets but the first (the serial doubles_min starts at 1);
// block 0 clears the pass's counters
__global__ __launch_bounds__(BLOCK) void run_slivers_k(SwapRunView R, double const* __restrict__ tq, double good,
                                                       unsigned char* __restrict__ marks,
                                                       double* __restrict__ part) {
  __shared__ double lds[BLOCK / 64];
  if (blockIdx.x == 0 && threadIdx.x < RW_WORDS && threadIdx.x != RW_POOL && threadIdx.x != RW_FIRST &&
      threadIdx.x != RW_ERR)
    R.words[threadIdx.x] = 0;
  u32 const first = R.words[RW_FIRST];
  double v = 1.7976931348623157e308;
  for (u32 t = blockIdx.x * BLOCK + threadIdx.x; t < R.nT; t += gridDim.x * BLOCK) {
    bool const live = !R.dead[t];
    double const q = tq[t];
    marks[t] = live && q < good ? 1 : 0;
    if (live && t != first && q < v) v = q;
  }
#pragma unroll
  for (u32 d = 32; d >= 1; d >>= 1) {
    double o = __shfl_down(v, d, 64);
    if (o < v) v = o;
  }
  if ((threadIdx.x & 63u) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = lds[0];
    for (u32 w = 1; w < BLOCK / 64; ++w)
      if (lds[w] < r) r = lds[w];
    part[blockIdx.x] = r;
  }
}

// one layer of mesh_mark_dual_layers (mark.cpp:90-126)
__global__ __launch_bounds__(BLOCK) void run_layer_k(u32 n, uint4 const* __restrict__ dual,
                                                     unsigned char const* __restrict__ in,
                                                     unsigned char* __restrict__ out) {
  u32 const t = blockIdx.x * BLOCK + threadIdx.x;
  if (t >= n) return;
  unsigned char r = in[t];
  if (!r) {
    uint4 const d = dual[t];
    r = ((d.x != INVALID && in[d.x]) || (d.y != INVALID && in[d.y]) || (d.z != INVALID && in[d.z]) ||
         (d.w != INVALID && in[d.w]))
            ? 1
            : 0;
  }
  out[t] = r;
}

// the candidates: live interior edges of marked tets whose swap is accepted
// (they enter the independent set) or not yet known (to be evaluated, listed
// by ring size: a ring of 7 has 35 triangles and one of 4 has 4, and a wave
// takes as long as its longest); a ring too large is rejected here
__global__ __launch_bounds__(RUN_AB) void run_candidates_k(SwapRunView R, unsigned char const* __restrict__ marks) {
  __shared__ u32 lds[RUN_AB / 64];
  constexpr u32 LISTS = 1 + RUN_RINGS;  // the accepted, then the rings
  u32 const e0 = blockIdx.x * RUN_AT + threadIdx.x;
  u32 list[RUN_AI];  // each edge's list, LISTS: none
  u32 count[(LISTS + 1) / 2] = {};  // two lists' counts a word: a block has at most 4096 of each
#pragma unroll
  for (u32 k = 0; k < RUN_AI; ++k) {
    list[k] = LISTS;
    u32 const e = e0 + k * RUN_AB;
    if (e >= R.nE) continue;
    u32 const w = R.info[e];
    if ((w & RI_KNOWN) && !(w & RI_ACCEPT)) continue;
    bool in = false;
    u32 const f = R.lb[e], n = R.ln[e];
    for (u32 j = 0; j < n && !in; ++j) in = marks[R.ua[f + j]] != 0;
    if (!in) continue;
    if (w & RI_KNOWN)
      list[k] = 0;
    else if (n > MAX_EDGE_SWAP)
      R.info[e] = RI_KNOWN;
    else
      list[k] = n < 3 ? 1 : n - 2;  // (below 3: the evaluation reports it)
  }
#pragma unroll
  for (u32 k = 0; k < RUN_AI; ++k)
#pragma unroll
    for (u32 l = 0; l < LISTS; ++l)
      if (list[k] == l) count[l / 2] += 1u << (16 * (l % 2));
#pragma unroll
  for (u32 p = 0; p < (LISTS + 1) / 2; ++p) {
    u32 total;
    u32 const mine = run_block_prefix(count[p], lds, &total);
    if (threadIdx.x < 2) {
      u32 const l = 2 * p + threadIdx.x, n = (total >> (16 * threadIdx.x)) & 0xffffu;
      lds[threadIdx.x] = n ? atomicAdd(R.words + (l == 0 ? (u32) RW_ACC : RW_EVAL + l - 1), n) : 0u;
    }
    __syncthreads();
    u32 at[2] = {lds[0] + (mine & 0xffffu), lds[1] + (mine >> 16)};
    __syncthreads();
#pragma unroll
    for (u32 k = 0; k < RUN_AI; ++k) {
      if (list[k] / 2 != p || list[k] == LISTS) continue;
      u32 const e = e0 + k * RUN_AB;
      if (list[k] == 0) {
        R.acc[at[0]++] = e;
        R.sa[e] = UNKNOWN;
      } else if (list[k] % 2 == 0) {
        R.eval[(size_t) (list[k] - 1) * R.ecap + at[0]++] = e;
      } else {
        R.eval[(size_t) (list[k] - 1) * R.ecap + at[1]++] = e;
      }
    }
  }
}

// swap qualities of the candidates to evaluate: the choice goes into the
// edge's word.  Bound by FP64 arithmetic with a wave's groups in step, so a
// batch holds one ring size: with the rings mixed as they came and both tets
// of a triangle on one lane, a call took 420 us where it now takes 247 us
// (mean of the 302 calls of an adaptation to 511 thousand tets), 101 us where
// it now takes 62 us at 55 thousand.
template <bool MT, bool MIXED>
__global__ __launch_bounds__(BLOCK, 4) void run_quality_k(SwapRunView R, double const* __restrict__ x,
                                                          double const* __restrict__ mt,
                                                          double const* __restrict__ tq, u32* __restrict__ err,
                                                          ScreenStats st) {
  __shared__ SwapLds<MT> L;
  u32 const group = threadIdx.x / SW_G;
  bool const lead = threadIdx.x % SW_G == 0;
  // batches of one ring size, the largest rings first
  u32 before[RUN_RINGS + 1];
  before[0] = 0;
#pragma unroll
  for (u32 c = 0; c < RUN_RINGS; ++c)
    before[c + 1] = before[c] + (R.words[RW_EVAL + RUN_RINGS - 1 - c] + SW_EDGES - 1) / SW_EDGES;
  for (u32 batch = blockIdx.x; batch < before[RUN_RINGS]; batch += gridDim.x) {
    u32 c = 0, first = 0;
#pragma unroll
    for (u32 k = 1; k < RUN_RINGS; ++k)
      if (batch >= before[k]) {
        c = k;
        first = before[k];
      }
    u32 const ring = RUN_RINGS - 1 - c, n = R.words[RW_EVAL + ring], base = (batch - first) * SW_EDGES;
    u32 e, rs, code;
    bool settled;
    double best;
    bool const accept = swap_quality_batch<MT, MIXED>(L, n, base + group, R.eval + (size_t) ring * R.ecap, R.lb, R.ln, R.ua, R.ud, R.ev, R.vt,
                                                      x, mt, tq, err, st, &e, &settled, &best, &rs, &code);
    if (settled && lead) {
      R.info[e] = accept ? RI_KNOWN | RI_ACCEPT | (rs << 16) | code : RI_KNOWN;
      if (accept) R.q[e] = best;
    }
    __syncthreads();  // the next batch reuses the staging
  }
}

// the evaluated candidates that are accepted join the accepted ones
__global__ __launch_bounds__(RUN_AB) void run_accept_k(SwapRunView R) {
  __shared__ u32 lds[RUN_AB / 64];
  u32 const ring = blockIdx.y;
  u32 const n = R.words[RW_EVAL + ring];
  for (u32 base = blockIdx.x * RUN_AT; base < n; base += gridDim.x * RUN_AT) {
    u32 e[RUN_AI], in = 0;
#pragma unroll
    for (u32 k = 0; k < RUN_AI; ++k) {
      u32 const i = base + k * RUN_AB + threadIdx.x;
      e[k] = i < n ? R.eval[(size_t) ring * R.ecap + i] : INVALID;
    }
#pragma unroll
    for (u32 k = 0; k < RUN_AI; ++k)
      if (e[k] != INVALID && (R.info[e[k]] & RI_ACCEPT)) in |= 1u << k;
    u32 a = run_append(R.words + RW_ACC, (u32) __popc(in), lds);
#pragma unroll
    for (u32 k = 0; k < RUN_AI; ++k)
      if ((in >> k) & 1u) {
        R.acc[a++] = e[k];
        R.sa[e[k]] = UNKNOWN;
      }
  }
}

// indset_round_elems over the accepted candidates (every other edge is out,
// in both states)
__global__ __launch_bounds__(BLOCK) void run_round_k(SwapRunView R, unsigned char const* __restrict__ old,
                                                     unsigned char* __restrict__ state, u32* __restrict__ flag) {
  u32 const n = R.words[RW_ACC];
  bool undecided = false;
  for (u32 k = blockIdx.x * BLOCK + threadIdx.x; k < n; k += gridDim.x * BLOCK) {
    u32 const i = R.acc[k];
    u32 s = old[i];
    if (s == UNKNOWN) {
      double const myg = R.q[i];
      bool wait = false, out = false;
      u32 const f = R.lb[i], l = R.ln[i];
      for (u32 j = f; j < f + l && !out; ++j) {
        // a tet's edges and their states in two round trips
        u32 const t = R.ua[j];
        u32 o[6], so[6];
#pragma unroll
        for (u32 c = 0; c < 6; ++c) o[c] = R.te[6 * (size_t) t + c];
#pragma unroll
        for (u32 c = 0; c < 6; ++c)  // (INVALID: a product's edge that was not found, reported)
          so[c] = o[c] == i || o[c] >= R.nE ? (u32) NOT_IN_SET : old[o[c]];
#pragma unroll
        for (u32 c = 0; c < 6; ++c) {
          if (so[c] == IN_SET) out = true;
          if (so[c] != UNKNOWN || wait) continue;
          double const og = R.q[o[c]];
          if ((myg == og && o[c] < i) || myg < og) wait = true;
        }
      }
      s = out ? (u32) NOT_IN_SET : (wait ? (u32) UNKNOWN : (u32) IN_SET);
      undecided = undecided || (!out && wait);
    }
    state[i] = (unsigned char) s;
  }
  wave_flag(flag, undecided);
}

// What a swapped edge makes: itself, product edges, faces and tets
struct RunCount {
  u32 v[4];
};
constexpr u32 RUN_PER = 8;  // edges per thread of the two counting kernels

__device__ inline void run_count_edge(SwapRunView const& R, u32 e, RunCount& c) {
  u32 const w = R.info[e], rs = (w >> 16) & 0xffu;
  u32 const nint = k_sw_nint[rs], tpm = k_sw_sizes[rs];
  c.v[0] += 1;
  c.v[1] += nint;
  c.v[2] += count_swap_ents(rs, 2, nint, tpm);
  c.v[3] += count_swap_ents(rs, 3, nint, tpm);
}

// exclusive prefix of c over the block's threads, totals in *tot
__device__ inline void run_block_scan(RunCount& c, RunCount* tot, u32 (*lds)[4]) {
  u32 const lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (u32 k = 0; k < 4; ++k) {
    u32 const mine = c.v[k];
    u32 x = mine;
#pragma unroll
    for (u32 d = 1; d < 64; d <<= 1) {
      u32 const y = (u32) __shfl_up((int) x, d, 64);
      if (lane >= d) x += y;
    }
    if (lane == 63u) lds[wave][k] = x;
    c.v[k] = x - mine;
  }
  __syncthreads();
#pragma unroll
  for (u32 k = 0; k < 4; ++k) {
    u32 off = 0, all = 0;
    for (u32 w = 0; w < nw; ++w) {
      if (w < wave) off += lds[w][k];
      all += lds[w][k];
    }
    c.v[k] += off;
    tot->v[k] = all;
  }
  __syncthreads();
}

// per block of BLOCK * RUN_PER edges: the totals of its swapped edges
__global__ __launch_bounds__(BLOCK) void run_count_k(SwapRunView R, unsigned char const* __restrict__ state,
                                                     RunCount* __restrict__ part) {
  __shared__ u32 lds[BLOCK / 64][4];
  u32 const e0 = (blockIdx.x * BLOCK + threadIdx.x) * RUN_PER;
  RunCount c{}, tot;
  if (e0 < R.nE) {
    // the states are padded with zeros to a multiple of RUN_PER
    unsigned long long const w = *reinterpret_cast<unsigned long long const*>(state + e0);
    if (w)
      for (u32 k = 0; k < RUN_PER; ++k)
        if (((w >> (8 * k)) & 0xffu) == IN_SET) run_count_edge(R, e0 + k, c);
  }
  run_block_scan(c, &tot, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// one block: the blocks' totals become their first products, and the totals,
// the pool's top, the set's flag, the run's error, the counts of candidates
// and the quality minimum go to the host
__global__ __launch_bounds__(1024) void run_offsets_k(u32 nb, RunCount* __restrict__ part, u32 npart,
                                                      double const* __restrict__ qpart, SwapRunView R,
                                                      u32 const* __restrict__ flag, u32* __restrict__ host,
                                                      double* __restrict__ host_min) {
  __shared__ u32 lds[16][4];
  __shared__ double mins[16];
  // candidates in the set's rounds; evaluated ones, and the tets around them
  u32 const accepted = R.words[RW_ACC];
  u32 evals = 0, tets = 0;
#pragma unroll
  for (u32 r = 0; r < RUN_RINGS; ++r) {
    u32 const n = R.words[RW_EVAL + r];
    evals += n;
    tets += (r + 3) * n;
  }
  u32 const per = (nb + 1023) / 1024, b = threadIdx.x * per, e = b + per < nb ? b + per : nb;
  RunCount c{}, tot;
  for (u32 i = b; i < e; ++i)
    for (u32 k = 0; k < 4; ++k) c.v[k] += part[i].v[k];
  run_block_scan(c, &tot, lds);
  for (u32 i = b; i < e; ++i)
    for (u32 k = 0; k < 4; ++k) {
      u32 const n = part[i].v[k];
      part[i].v[k] = c.v[k];
      c.v[k] += n;
    }
  double v = 1.7976931348623157e308;
  for (u32 i = threadIdx.x; i < npart; i += 1024)
    if (qpart[i] < v) v = qpart[i];
#pragma unroll
  for (u32 d = 32; d >= 1; d >>= 1) {
    double o = __shfl_down(v, d, 64);
    if (o < v) v = o;
  }
  if ((threadIdx.x & 63u) == 0) mins[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (u32 w = 1; w < 16; ++w)
    if (mins[w] < v) v = mins[w];
  for (u32 k = 0; k < 4; ++k) host[k] = tot.v[k];
  host[4] = R.words[RW_POOL];
  host[5] = *flag;
  host[6] = R.words[RW_ERR];
  host[7] = accepted;
  host[8] = evals;
  host[9] = tets;
  *host_min = v;
}

// the swapped edges in order with their first products; each is removed
// with the tets around it
__global__ __launch_bounds__(BLOCK) void run_list_k(SwapRunView R, unsigned char const* __restrict__ state,
                                                    RunCount const* __restrict__ part) {
  __shared__ u32 lds[BLOCK / 64][4];
  u32 const e0 = (blockIdx.x * BLOCK + threadIdx.x) * RUN_PER;
  RunCount c{}, tot;
  unsigned long long w = 0;
  if (e0 < R.nE) w = *reinterpret_cast<unsigned long long const*>(state + e0);
  if (w)
    for (u32 k = 0; k < RUN_PER; ++k)
      if (((w >> (8 * k)) & 0xffu) == IN_SET) run_count_edge(R, e0 + k, c);
  run_block_scan(c, &tot, lds);
  if (!w) return;
  RunCount const base = part[blockIdx.x];
  for (u32 k = 0; k < 4; ++k) c.v[k] += base.v[k];
  for (u32 k = 0; k < RUN_PER; ++k) {
    if (((w >> (8 * k)) & 0xffu) != IN_SET) continue;
    u32 const e = e0 + k, s = c.v[0];
    R.sw[s] = e;
    R.o1[s] = c.v[1];
    R.o2[s] = c.v[2];
    R.o3[s] = c.v[3];
    run_count_edge(R, e, c);
    R.death[e] = R.pass;
    R.info[e] &= ~RI_ACCEPT;  // the ring size and triangulation stay for the products
    u32 const f = R.lb[e], n = R.ln[e];
    for (u32 j = f; j < f + n; ++j) R.dead[R.ua[j]] = 1;
  }
}

// The products of the pass's cavities (swap_products_k's, unnumbered), RUN_G
// lanes per swapped edge: lane j reads the edge's j-th tet, the lanes chain
// the ring together (edge_ring.cpp:12-74 follows each tet's opposite edge a
// -> b from the first tet; here the lane whose a is the current b is found by
// ballot), and each writes an edge, faces and a tet with its edges and dual.
// A thread per cavity took 99 us on the 21^3 x 6 anisotropic box whether a
// pass had 60,000 cavities or one: a serial chain of its loads and of the
// products' bookkeeping, which a cavity's lanes now share.
constexpr u32 RUN_G = 16;
struct RunCavity {
  // by ring slot k: the vertex, the tet around (k, k + 1), its ring edge, the
  // edges from the vertex to the swapped edge's ends, and where the ends are
  // in the tet
  u32 ring[8], tet[8], redge[8], spoke[2][8], loc[8];
};
__global__ __launch_bounds__(BLOCK) void run_products_k(SwapRunView R, u32 ns, u32* __restrict__ face_prod,
                                                        u32* __restrict__ deferred, u32* __restrict__ err) {
  __shared__ RunCavity cavities[BLOCK / RUN_G];
  u32 const g = threadIdx.x / RUN_G, lane = threadIdx.x % RUN_G;
  RunCavity& C = cavities[g];
  u32 const s = blockIdx.x * (BLOCK / RUN_G) + g;
  u32 e = 0, f = 0, rs = 0, ends[2] = {0, 0}, code = 0, g1 = 0, g2 = 0, g3 = 0, cd = 0, ci = 0;
  if (s < ns) {
    e = R.sw[s];
    f = R.lb[e];
    rs = R.ln[e];
    ends[0] = R.ev[2 * (size_t) e];
    ends[1] = R.ev[2 * (size_t) e + 1];
    code = R.info[e] & 0xffffu;
    g1 = R.o1[s];
    g2 = R.o2[s];
    g3 = R.o3[s];
    cd = R.ecd[e];
    if (R.eci) ci = R.eci[e];
    if (rs < 3 || rs > MAX_EDGE_SWAP) rs = 0;  // cannot happen for an accepted edge
  }
  // the edge's tets
  u32 a = INVALID, b = INVALID, t = 0, redge = 0, sp0 = 0, sp1 = 0, loc = 0;
  if (lane < rs) {
    t = R.ua[f + lane];
    u32 const d = R.ud[f + lane];
    u32 v[4], le[6];
#pragma unroll
    for (u32 k = 0; k < 4; ++k) v[k] = R.vt[4 * (size_t) t + k];
#pragma unroll
    for (u32 k = 0; k < 6; ++k) le[k] = R.te[6 * (size_t) t + k];
    auto vert = [&](u32 l) { return l == 0 ? v[0] : l == 1 ? v[1] : l == 2 ? v[2] : v[3]; };
    auto edge = [&](u32 l) { return l == 0 ? le[0] : l == 1 ? le[1] : l == 2 ? le[2] : l == 3 ? le[3] : l == 4 ? le[4] : le[5]; };
    u32 const o = tet_oe(d);
    bool const turned = vert(tet_ev0(d)) != ends[0];
    u32 const l0 = turned ? tet_ev1(d) : tet_ev0(d), l1 = turned ? tet_ev0(d) : tet_ev1(d);
    u32 const la = turned ? tet_ev1(o) : tet_ev0(o), lb = turned ? tet_ev0(o) : tet_ev1(o);
    a = vert(la);
    b = vert(lb);
    redge = edge(o);
    sp0 = edge(tet_edge_of(la, l0));
    sp1 = edge(tet_edge_of(la, l1));
    loc = l0 | (l1 << 2);
  }
  // the ring: each lane's slot
  u32 const shift = (threadIdx.x & 63u) & ~(RUN_G - 1u);
  u32 slot = lane == 0 ? 0u : INVALID, cur = 0;
  for (u32 k = 1; k < MAX_EDGE_SWAP; ++k) {
    u32 const want = (u32) __shfl((int) b, (int) cur, (int) RUN_G);
    u32 const m = (u32) (__ballot(lane < rs && a == want) >> shift) & ((1u << RUN_G) - 1u);
    cur = m ? (u32) (__ffs((int) m) - 1) : 0u;
    if (m && k < rs && lane == cur) slot = k;
  }
  if (lane < rs) {
    if (slot == INVALID) {
      *err = ERR_EDGE_RING;  // cannot happen: the ring closed when it was evaluated
      slot = lane;
    }
    C.ring[slot] = a;
    C.tet[slot] = t;
    C.redge[slot] = redge;
    C.spoke[0][slot] = sp0;
    C.spoke[1][slot] = sp1;
    C.loc[slot] = loc;
  }
  __syncthreads();
  if (!rs) return;  // no barrier follows
  u32 const tpm = k_sw_sizes[rs], nint = k_sw_nint[rs];
  unsigned char const* mesh = k_sw_meshes + k_sw_mesh_off[rs] + code * tpm;
  unsigned char const(*tris)[3] = k_sw_tris + k_sw_tri_off[rs];
  unsigned char const* ie = k_sw_int + k_sw_int_off[rs] + code * nint * 2;
  if (lane < nint) {
    u32 const n = R.nE + g1 + lane;
    R.ev[2 * (size_t) n] = C.ring[ie[2 * lane]];
    R.ev[2 * (size_t) n + 1] = C.ring[ie[2 * lane + 1]];
    R.ecd[n] = cd;
    if (R.eci) R.eci[n] = ci;
    R.death[n] = 0;
    R.info[n] = cd == 3 ? 0u : RI_KNOWN;
    R.lb[n] = 0;
    R.ln[n] = 0;
    R.cnt[n] = 0;
    R.sa[n] = 0;
    R.sb[n] = 0;
  }
  u32 const nf = tpm + 2 * nint;  // at most 13: a lane each
  if (lane < nf) {
    u32 const n = R.nF + g2 + lane;
    u32* o = R.fv + 3 * (size_t) n;
    if (lane < 2 * nint) {
      o[0] = C.ring[ie[2 * (lane / 2)]];
      o[1] = C.ring[ie[2 * (lane / 2) + 1]];
      o[2] = ends[lane & 1u];
    } else {
      for (u32 j = 0; j < 3; ++j) o[j] = C.ring[tris[mesh[lane - 2 * nint]][j]];
    }
    R.fcd[n] = cd;
    if (R.fci) R.fci[n] = ci;
    R.fbirth[n - R.nF0] = R.pass;
  }
  if (lane >= 2 * tpm) return;  // at most 10 tets
  // the tet of triangle p and edge end 1, then with its first two corners
  // exchanged and edge end 0
  u32 const p = lane / 2, j = lane & 1u, x = 1 - j;
  u32 const first = R.nT + g3, self = first + lane;
  u32 lab[3] = {tris[mesh[p]][j], tris[mesh[p]][1 - j], tris[mesh[p]][2]};
  for (u32 k = 0; k < 3; ++k) R.vt[4 * (size_t) self + k] = C.ring[lab[k]];
  R.vt[4 * (size_t) self + 3] = ends[x];
  R.tcd[self] = cd;
  if (R.tci) R.tci[self] = ci;
  R.dead[self] = 0;
  // adjacent ring slots: the slot their ring edge and tet have, else INVALID
  auto beside = [&](u32 u, u32 v) {
    return u + 1 == v || u == v + rs - 1 ? u : v + 1 == u || v == u + rs - 1 ? v : INVALID;
  };
#pragma unroll
  for (u32 k = 0; k < 3; ++k) {
    // edges 0-1, 1-2, 2-0 and the faces on them (1, 2, 3); spokes 3, 4, 5
    u32 const u = lab[k], v = lab[(k + 1) % 3], r = beside(u, v);
    u32 id = INVALID, across = INVALID;
    if (r != INVALID) {
      id = C.redge[r];
      u32 const tk = C.tet[r], lf = tet_face_without((C.loc[r] >> (2 * (1 - x))) & 3u);
      size_t const key = 4 * (size_t) tk + lf;
      face_prod[key] = self;
      u32 const o = R.dual[key];
      if (o != INVALID && !R.dead[o]) {
        across = o;
        for (u32 q = 0; q < 4; ++q)
          if (R.dual[4 * (size_t) o + q] == tk) R.dual[4 * (size_t) o + q] = self;
      } else if (o != INVALID) {
        across = DUAL_PENDING;  // another cavity's: known once its products are written
        deferred[4 * (size_t) (g3 + lane) + 1 + k] = (u32) key;
      }
    } else {
      for (u32 q = 0; q < nint; ++q)
        if ((ie[2 * q] == u && ie[2 * q + 1] == v) || (ie[2 * q] == v && ie[2 * q + 1] == u)) id = R.nE + g1 + q;
      for (u32 t2 = 0; t2 < tpm; ++t2) {
        if (t2 == p) continue;
        unsigned char const* tr = tris[mesh[t2]];
        if ((tr[0] == u || tr[1] == u || tr[2] == u) && (tr[0] == v || tr[1] == v || tr[2] == v))
          across = first + 2 * t2 + j;
      }
      if (across == INVALID) *err = ERR_REFLECT_NOT_FOUND;
    }
    if (id == INVALID) *err = ERR_REFLECT_NOT_FOUND;
    R.te[6 * (size_t) self + k] = id;
    R.te[6 * (size_t) self + 3 + k] = C.spoke[x][u];
    R.dual[4 * (size_t) self + 1 + k] = across;
  }
  R.dual[4 * (size_t) self] = first + 2 * p + x;  // the twin: the same triangle, the other end
}

// every use of an edge by a product tet takes a place among its edge's
// product uses; the edge's first one puts the edge on the list of changed
// edges
__global__ __launch_bounds__(RUN_AB) void run_touch_k(SwapRunView R, u32 nuse, u32* __restrict__ slot,
                                                      u32* __restrict__ changed) {
  __shared__ u32 lds[RUN_AB / 64];
  u32 const u0 = blockIdx.x * RUN_AT + threadIdx.x;
  u32 e[RUN_AI], first = 0;
#pragma unroll
  for (u32 k = 0; k < RUN_AI; ++k) {
    u32 const u = u0 + k * RUN_AB;
    e[k] = u < nuse ? R.te[6 * (size_t) R.nT + u] : INVALID;
  }
#pragma unroll
  for (u32 k = 0; k < RUN_AI; ++k) {
    u32 const u = u0 + k * RUN_AB;
    if (u >= nuse) continue;
    u32 const s = e[k] != INVALID ? atomicAdd(&R.cnt[e[k]], 1u) : 1u;
    slot[u] = s;
    if (s == 0) first |= 1u << k;
  }
  u32 a = run_append(R.words + RW_AFF, (u32) __popc(first), lds);
#pragma unroll
  for (u32 k = 0; k < RUN_AI; ++k)
    if ((first >> k) & 1u) changed[a++] = e[k];
}

// a changed edge's new list: a place in the pool for its surviving and its
// product uses, the survivors copied in order; cnt is then the survivors'
// number.  Its swap is not known any more.
__global__ __launch_bounds__(RUN_AB) void run_lists_k(SwapRunView R, u32 const* __restrict__ changed) {
  __shared__ u32 lds[RUN_AB / 64];
  u32 const i = blockIdx.x * RUN_AB + threadIdx.x;
  u32 const n = R.words[RW_AFF];
  u32 e = 0, f = 0, l = 0, s = 0, len = 0;
  // the first RUN_L uses in registers, their loads in flight together
  constexpr u32 RUN_L = 8;
  u32 t[RUN_L];
  bool live[RUN_L];
  if (i < n) {
    e = changed[i];
    f = R.lb[e];
    l = R.ln[e];
#pragma unroll
    for (u32 k = 0; k < RUN_L; ++k) t[k] = k < l ? R.ua[f + k] : INVALID;
#pragma unroll
    for (u32 k = 0; k < RUN_L; ++k) {
      live[k] = t[k] != INVALID && !R.dead[t[k]];
      s += live[k] ? 1u : 0u;
    }
    for (u32 k = f + RUN_L; k < f + l; ++k) s += R.dead[R.ua[k]] ? 0u : 1u;
    len = s + R.cnt[e];
  }
  u32 const base = run_append(R.words + RW_POOL, len, lds);
  if (i >= n) return;
  u32 p = base;
#pragma unroll
  for (u32 k = 0; k < RUN_L; ++k)
    if (live[k]) {
      R.ua[p] = t[k];
      R.ud[p] = R.ud[f + k];
      ++p;
    }
  for (u32 k = f + RUN_L; k < f + l; ++k) {
    u32 const v = R.ua[k];
    if (R.dead[v]) continue;
    R.ua[p] = v;
    R.ud[p] = R.ud[k];
    ++p;
  }
  R.lb[e] = base;
  R.ln[e] = len;
  R.cnt[e] = s;
  R.info[e] = R.ecd[e] == 3 ? 0u : RI_KNOWN;
}

__global__ __launch_bounds__(BLOCK) void run_place_k(SwapRunView R, u32 nuse, u32 const* __restrict__ slot) {
  u32 const u = blockIdx.x * BLOCK + threadIdx.x;
  if (u >= nuse) return;
  u32 const key = 6 * R.nT + u, e = R.te[key];
  if (e != INVALID) R.ua[R.lb[e] + R.cnt[e] + slot[u]] = key;
}

// a changed edge's product uses in ascending order (a few: insertion sort)
__global__ __launch_bounds__(BLOCK) void run_sort_k(SwapRunView R, u32 const* __restrict__ changed) {
  u32 const i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= R.words[RW_AFF]) return;
  u32 const e = changed[i];
  u32 const b = R.lb[e] + R.cnt[e], end = R.lb[e] + R.ln[e];
  for (u32 k = b + 1; k < end; ++k) {
    u32 const v = R.ua[k];
    u32 j = k;
    for (; j > b && R.ua[j - 1] > v; --j) R.ua[j] = R.ua[j - 1];
    R.ua[j] = v;
  }
  for (u32 k = b; k < end; ++k) {
    u32 const v = R.ua[k], t = v / 6;
    R.ua[k] = t;
    R.ud[k] = v - 6 * t;
  }
  R.cnt[e] = 0;
}

// product faces between two cavities of the pass (swap_dual_k); the accepted
// candidates' states are cleared and the first live tet is found again
__global__ __launch_bounds__(BLOCK) void run_settle_k(SwapRunView R, u32 n3, u32 const* __restrict__ face_prod,
                                                      u32 const* __restrict__ deferred, u32* __restrict__ err) {
  u32 const i = blockIdx.x * BLOCK + threadIdx.x;
  if (i < 4 * n3) {
    u32* d = R.dual + 4 * (size_t) R.nT + i;
    if (*d == DUAL_PENDING) {
      u32 const key = deferred[i], n = R.dual[key];
      u32 r = INVALID;
      for (u32 g = 0; g < 4; ++g)
        if (R.dual[4 * (size_t) n + g] == key / 4) r = face_prod[4 * (size_t) n + g];
      if (r == INVALID) *err = ERR_REFLECT_NOT_FOUND;
      *d = r;
    }
  }
  u32 const n = R.words[RW_ACC];
  for (u32 k = i; k < n; k += gridDim.x * BLOCK) {
    u32 const e = R.acc[k];
    R.sa[e] = 0;
    R.sb[e] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    u32 f = R.words[RW_FIRST];
    u32 const nt = R.nT + n3;
    for (;;) {
      u32 const t = f + threadIdx.x;
      unsigned long long const m = __ballot(t < nt && !R.dead[t]);
      if (m) {
        f += (u32) (__ffsll((long long) m) - 1);
        break;
      }
      f += 64;
      if (f >= nt) break;
    }
    if (threadIdx.x == 0) R.words[RW_FIRST] = f;
  }
}

// the last pass that removed each vertex pair
__global__ __launch_bounds__(BLOCK) void run_pairs_k(SwapRunView R, u32 mask, unsigned long long* __restrict__ keys,
                                                     u32* __restrict__ when, u32* __restrict__ err) {
  u32 const e = blockIdx.x * BLOCK + threadIdx.x;
  if (e >= R.nE) return;
  u32 const p = R.death[e];
  if (!p) return;
  unsigned long long const key = swap_pair_key(R.ev[2 * (size_t) e], R.ev[2 * (size_t) e + 1]);
  u32 h = swap_pair_slot(key, mask);
  for (u32 probe = 0; probe <= mask; ++probe, h = (h + 1) & mask) {
    unsigned long long const k = atomicCAS(&keys[h], ~0ull, key);
    if (k == ~0ull || k == key) {
      atomicMax(&when[h], p);
      return;
    }
  }
  *err = ERR_REFLECT_NOT_FOUND;
}

// the live entities of one dimension, renumbered into the new mesh
struct RunOut {
  u32 n, vpe;
  u32 const* rank;  // n + 1
  u32 const* v;
  u32 const* cd;
  u32 const* ci;
  u32* out;
  u32* out_cd;
  u32* out_ci;
  // edges: choices and values, and the lists' lengths
  u32 const* info;
  double const* q;
  u32 const* ln;
  u32* out_info;
  double* out_q;
  u32* out_ln;
  // tets: edges, dual, qualities
  u32 const* te;
  u32 const* dual;
  double const* tq;
  u32 const* erank;
  u32* out_te;
  u32* out_dual;
  double* out_tq;
};
__global__ __launch_bounds__(BLOCK) void run_out_k(RunOut a) {
  u32 const i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= a.n) return;
  u32 const o = a.rank[i];
  if (o == a.rank[i + 1]) return;
  for (u32 j = 0; j < a.vpe; ++j) a.out[(size_t) o * a.vpe + j] = a.v[(size_t) i * a.vpe + j];
  a.out_cd[o] = a.cd[i];
  if (a.out_ci) a.out_ci[o] = a.ci[i];
  if (a.out_ln) a.out_ln[o] = a.ln[i];
  if (a.out_info) {
    a.out_info[o] = a.info[i];
    a.out_q[o] = a.q[i];
  }
  if (a.out_te) {
    for (u32 j = 0; j < 6; ++j) a.out_te[6 * (size_t) o + j] = a.erank[a.te[6 * (size_t) i + j]];
    for (u32 j = 0; j < 4; ++j) {
      u32 const d = a.dual[4 * (size_t) i + j];
      a.out_dual[4 * (size_t) o + j] = d == INVALID ? INVALID : a.rank[d];
    }
    a.out_tq[o] = a.tq[i];
  }
}

// the live edges' lists in the new mesh's numbering (RUN_LG lanes an edge)
constexpr u32 RUN_LG = 4;
__global__ __launch_bounds__(BLOCK) void run_up_k(SwapRunView R, u32 const* __restrict__ erank,
                                                  u32 const* __restrict__ trank, u32 const* __restrict__ off,
                                                  u32* __restrict__ adj, u32* __restrict__ dirs) {
  size_t const gid = (size_t) blockIdx.x * BLOCK + threadIdx.x;
  u32 const e = (u32) (gid / RUN_LG), lane = (u32) (gid % RUN_LG);
  if (e >= R.nE) return;
  u32 const o = erank[e];
  if (o == erank[e + 1]) return;
  u32 const f = R.lb[e], n = R.ln[e], p = off[o];
  for (u32 k = lane; k < n; k += RUN_LG) {
    adj[p + k] = trank[R.ua[f + k]];
    dirs[p + k] = R.ud[f + k];
  }
}

namespace {
struct SwapRun {
  Mesh& m;
  Buf<u32> ev, ecd, eci, death, info, lb, ln, cnt, ua, ud, vt, te, dual, tcd, tci, fv, fcd, fci, fbirth, face_prod;
  Buf<u32> acc, eval, words;
  Buf<double> q, tq, qpart;
  Buf<unsigned char> sa, sb, dead, marks, marks2;
  Buf<RunCount> part;
  u32 nE = 0, nF = 0, nT = 0, nF0 = 0, aE = 0, aF = 0, aT = 0, pass = 0;
  size_t pool = 0;  // at most so many list places are in use
  static constexpr size_t MAX_USES = (size_t) 1 << 32;
  bool has_id = false;
  bool intact = true;  // the mesh in the arrays is that of the passes so far
  u32 got[10];
  double min_q = 0;

  explicit SwapRun(Mesh& mesh) : m(mesh) {}

  template <class T>
  static void need(Buf<T>& b, size_t used, size_t want) {
    if (b && b.size() >= want) return;
    Buf<T> n(want + want / 2);
    if (b) d2d(n.get(), b.get(), used);
    b = std::move(n);
  }
  static size_t room(size_t n) { return n + n / 4 + 1024; }
  template <class T>
  static Buf<T> taken(T const* a, size_t n, size_t cap) {
    Buf<T> b(cap);
    d2d(b.get(), a, n);
    return b;
  }
  void clear_states(size_t from) {
    // zero beyond the edges in use: products start out of the set, and the
    // counting kernels read whole words
    unsigned char *a = sa.get(), *b = sb.get();
    u32 const n = (u32) (sa.size() - from);
    parallel_for(n, OHX_LAMBDA(u32 i) {
      a[from + i] = 0;
      b[from + i] = 0;
    });
  }
  void edge_room(u32 want) {
    if (ev && info.size() >= want) return;
    size_t const old = sa.size();
    need(ev, 2 * (size_t) nE, 2 * (size_t) want);
    need(ecd, nE, want);
    if (has_id) need(eci, nE, want);
    need(death, nE, want);
    need(info, nE, want);
    need(q, nE, want);
    need(lb, nE, want);
    need(ln, nE, want);
    need(cnt, nE, want);
    need(acc, nE, want);  // still read: its edges' states are cleared at the pass's end
    eval = Buf<u32>(RUN_RINGS * info.size());
    size_t const states = (info.size() + RUN_PER) / RUN_PER * RUN_PER;
    Buf<unsigned char> a2(states), b2(states);
    if (old) {
      d2d(a2.get(), sa.get(), old);
      d2d(b2.get(), sb.get(), old);
    }
    sa = std::move(a2);
    sb = std::move(b2);
    clear_states(old);
  }
  void tet_room(u32 want) {
    if (dead && dead.size() >= want) return;
    need(vt, 4 * (size_t) nT, 4 * (size_t) want);
    need(te, 6 * (size_t) nT, 6 * (size_t) want);
    need(dual, 4 * (size_t) nT, 4 * (size_t) want);
    need(tcd, nT, want);
    if (has_id) need(tci, nT, want);
    need(tq, nT, want);
    need(dead, nT, want);
    face_prod = Buf<u32>(4 * dead.size());
    marks = Buf<unsigned char>(dead.size());
    marks2 = Buf<unsigned char>(dead.size());
  }

  // room for the lists of a pass that leaves so many tets: the changed edges'
  // new lists are some of the lists of the mesh it leaves, which have 6 uses a
  // tet (counting around the cavities instead took a wait and, as an edge was
  // counted once for each tet that goes, found several times as many)
  void list_room(u32 tets) {
    size_t const want = got[4] + 6 * (size_t) tets;
    if (want >= MAX_USES) fail("swap: more than 2^32 uses", __FILE__, __LINE__);
    need(ua, got[4], want);
    need(ud, got[4], want);
  }
  // whether the next pass could run out of places that 32 bits can number: a
  // pass replaces a ring of 7 tets with 10 at most, so its lists take fewer
  // than 9 places for each tet before it.  Lists in use take 6 a tet, and
  // check_index_space keeps a mesh below 2^32 / 36 tets: with the gaps closed
  // there is always room.
  bool lists_full() const { return pool + 9 * (size_t) aT >= MAX_USES; }

  SwapRunView view() const {
    SwapRunView R{};
    R.nE = nE;
    R.nF = nF;
    R.nT = nT;
    R.nF0 = nF0;
    R.pass = pass;
    R.ev = ev.get();
    R.ecd = ecd.get();
    R.eci = eci.get();
    R.death = death.get();
    R.info = info.get();
    R.q = q.get();
    R.lb = lb.get();
    R.ln = ln.get();
    R.cnt = cnt.get();
    R.sa = sa.get();
    R.sb = sb.get();
    R.ua = ua.get();
    R.ud = ud.get();
    R.vt = vt.get();
    R.te = te.get();
    R.dual = dual.get();
    R.tcd = tcd.get();
    R.tci = tci.get();
    R.dead = dead.get();
    R.fv = fv.get();
    R.fcd = fcd.get();
    R.fci = fci.get();
    R.fbirth = fbirth.get();
    R.acc = acc.get();
    R.eval = eval.get();
    R.ecap = (u32) info.size();
    R.words = words.get();
    return R;
  }

  // the mesh's arrays, with room for products; choices: the edges' words and
  // values when a run on the same mesh has them already (else null)
  void begin(double const* qualities, u32 const* known, double const* values) {
    Up const& u = ask_up(m, 1, 3);
    u32 const* d31 = ask_down(m, 3, 1);
    u32 const* du = ask_dual(m);
    has_id = find_tag(m, 0, "class_id") != nullptr;
    nE = aE = count(m, 1);
    nF = aF = nF0 = count(m, 2);
    nT = aT = count(m, 3);
    pass = 0;
    pool = u.adj.size();
    size_t const cE = room(nE), cF = room(nF), cT = room(nT), cL = 2 * pool + pool / 4 + 4096;
    ev = taken(ask_down(m, 1, 0), 2 * (size_t) nE, 2 * cE);
    ecd = taken(u32_tag(m, 1, "class_dim"), nE, cE);
    vt = taken(ask_down(m, 3, 0), 4 * (size_t) nT, 4 * cT);
    te = taken(d31, 6 * (size_t) nT, 6 * cT);
    dual = taken(du, 4 * (size_t) nT, 4 * cT);
    tcd = taken(u32_tag(m, 3, "class_dim"), nT, cT);
    fv = taken(ask_down(m, 2, 0), 3 * (size_t) nF, 3 * cF);
    fcd = taken(u32_tag(m, 2, "class_dim"), nF, cF);
    if (has_id) {
      eci = taken(u32_tag(m, 1, "class_id"), nE, cE);
      tci = taken(u32_tag(m, 3, "class_id"), nT, cT);
      fci = taken(u32_tag(m, 2, "class_id"), nF, cF);
    }
    fbirth = Buf<u32>(cF - nF);
    tq = taken(qualities, nT, cT);
    ua = taken(u.adj.get(), pool, cL);
    ud = taken(u.dirs.get(), pool, cL);
    dead = Buf<unsigned char>(cT);
    marks = Buf<unsigned char>(cT);
    marks2 = Buf<unsigned char>(cT);
    face_prod = Buf<u32>(4 * cT);
    death = Buf<u32>(cE);
    info = Buf<u32>(cE);
    q = Buf<double>(cE);
    lb = Buf<u32>(cE);
    ln = Buf<u32>(cE);
    cnt = Buf<u32>(cE);
    acc = Buf<u32>(cE);
    eval = Buf<u32>(RUN_RINGS * cE);
    size_t const states = (cE + RUN_PER) / RUN_PER * RUN_PER;
    sa = Buf<unsigned char>(states);
    sb = Buf<unsigned char>(states);
    qpart = Buf<double>(RUN_RED_BLOCKS);
    words = Buf<u32>(RW_WORDS);
    // every array's start values, one launch over the states (the edges and
    // their room) and the tets
    SwapRunView R = view();
    u32 const* off = u.offsets.get();
    u32 const p0 = (u32) pool, ns = (u32) states;
    parallel_for(ns > nT ? ns : nT, OHX_LAMBDA(u32 i) {
      if (i < ns) {
        R.sa[i] = 0;
        R.sb[i] = 0;
      }
      if (i < R.nE) {
        R.death[i] = 0;
        R.cnt[i] = 0;
        R.lb[i] = off[i];
        R.ln[i] = off[i + 1] - off[i];
        R.info[i] = R.ecd[i] != 3 ? RI_KNOWN : known ? known[i] : 0u;
        if (known) R.q[i] = values[i];
      }
      if (i < R.nT) R.dead[i] = 0;
      if (i < RW_WORDS) R.words[i] = i == RW_POOL ? p0 : 0u;
    });
  }

  // one swap pass; returns whether it changed the mesh, and sets min_q, the
  // quality minimum of the mesh before the pass (at least good: no pass)
  bool step(double good, u32 nlayers) {
    {
      // as check_index_space, from the live counts
      size_t const star = 6 * (size_t) aF + 6 * (size_t) aT;
      if (2 * star >= ((size_t) 1 << 32)) fail("mesh too large for 32-bit adjacency offsets", __FILE__, __LINE__);
    }
    make_swap_tables();
    ++pass;
    SwapRunView R = view();
    u32 const rb = nblocks(nT) < RUN_RED_BLOCKS ? nblocks(nT) : RUN_RED_BLOCKS;
    hipLaunchKernelGGL(run_slivers_k, dim3(rb), dim3(BLOCK), 0, stream(), R, tq.get(), good, marks.get(),
                       qpart.get());
    check_launch("run_slivers");
    for (u32 l = 0; l < nlayers; ++l) {
      hipLaunchKernelGGL(run_layer_k, dim3(nblocks(nT)), dim3(BLOCK), 0, stream(), nT,
                         reinterpret_cast<uint4 const*>(dual.get()), marks.get(), marks2.get());
      check_launch("run_layer");
      std::swap(marks, marks2);
    }
    hipLaunchKernelGGL(run_candidates_k, dim3(nblocks(nE, RUN_AT)), dim3(RUN_AB), 0, stream(), R, marks.get());
    check_launch("run_candidates");
    evaluate(R);
    // a first batch of rounds with no host check, as the other passes
    u32 const first = first_batch_rounds();
    u32 const gr = nblocks(nE) < 512 ? nblocks(nE) : 512;
    unsigned char *a = sa.get(), *b = sb.get();
    u32* flags = words.get() + RW_FLAGS;
    auto round = [&](u32* fl) {
      launch_timed("indset_round", 0, run_round_k, dim3(gr), dim3(BLOCK), R, a, b, fl);
      std::swap(a, b);
    };
    // the first rounds' bytes at least: each candidate's list entry, state in
    // and out, and in the first round its value
    auto count_rounds = [&] { prof_add_bytes("indset_round", (6.0 * first + 8) * got[7]); };
    for (u32 r = 0; r < first; ++r) round(flags + r);
    u32 const nb = nblocks(nE, BLOCK * RUN_PER);
    if (!part || part.size() < nb) part = Buf<RunCount>(nb + nb / 2);
    u32* hs = host_slot<u32>(SLOT_RUN);
    u32* ds = dev_slot<u32>(SLOT_RUN);
    u32 const* flag = flags + first - 1;
    auto totals = [&] {
      hipLaunchKernelGGL(run_count_k, dim3(nb), dim3(BLOCK), 0, stream(), R, a, part.get());
      hipLaunchKernelGGL(run_offsets_k, dim3(1), dim3(1024), 0, stream(), nb, part.get(), rb, qpart.get(), R, flag,
                         ds, dev_slot<double>(SLOT_RUN_MIN));
      check_launch("run_offsets");
      hs[6] = 0;
      try {
        sync();
      } catch (Error const&) {
        intact = !hs[6];
        throw;
      }
      for (u32 k = 0; k < 10; ++k) got[k] = hs[k];
      if (got[6]) {
        intact = false;
        fail_device(got[6]);
      }
    };
    totals();
    count_rounds();
    // of each evaluated candidate its list entry, ends, list place and length,
    // choice and value, and the tets around it and its places in them
    prof_add_bytes(quality_name(), 36.0 * got[8] + 8.0 * got[9]);
    min_q = *host_slot<double>(SLOT_RUN_MIN);
    if (min_q >= good) return false;
    if (got[5]) {
      // not settled in the first batch: checked batches up to the limit
      rounds_to_the_end(round, flags);
      flag = words.get() + RW_AFF;  // zero: settled
      totals();
    }
    if (!got[0]) return false;
    swap(R, a, nb);
    return true;
  }

  char const* quality_name() const {
    return g_mixed && swap_screen_pinned() ? "swap_quality_mixed" : "swap_quality_f64";
  }
  void evaluate(SwapRunView const& R) {
    double const* mt = metric_of(m);
    double const* x = coords(m);
    u32 const need = (aE + SW_EDGES - 1) / SW_EDGES;
    dim3 const grid(need < 2048 ? (need ? need : 1) : 2048);
    ScreenStats st = screen_stats();
    auto go = [&](auto kernel) {
      launch_timed(quality_name(), 0, kernel, grid, dim3(BLOCK), R, x, mt, tq.get(), dev_error_word(), st);
    };
    // the FP32 screen runs only where it is pinned on: timed on live
    // launches it lost to FP64 at every size class of the shipped table
    if (g_mixed && swap_screen_pinned())
      mt ? go(run_quality_k<true, true>) : go(run_quality_k<false, true>);
    else
      mt ? go(run_quality_k<true, false>) : go(run_quality_k<false, false>);
    u32 const ab = nblocks(aE, RUN_AT);
    hipLaunchKernelGGL(run_accept_k, dim3(ab < 64 ? ab : 64, RUN_RINGS), dim3(RUN_AB), 0, stream(), R);
    check_launch("run_accept");
  }

  template <class F>
  void rounds_to_the_end(F&& round, u32* flags) {
    constexpr u32 BATCH = 8;
    u32 const limit = g_indset_max_rounds;
    for (u32 done = first_batch_rounds(); done < limit; done += BATCH) {
      u32 const nr = limit - done < BATCH ? limit - done : BATCH;
      fill(flags, nr, 0);
      for (u32 r = 0; r < nr; ++r) round(flags + r);
      u32 h[BATCH];
      u32 const* fp[BATCH];
      for (u32 r = 0; r < nr; ++r) fp[r] = flags + r;
      read_many(fp, nr, h);
      if (!h[nr - 1]) {
        u32 k = 0;
        while (h[k]) ++k;
        note_rounds(done + k + 1);
        return;
      }
    }
    fail("independent set did not converge within the round limit (indset.cpp:107-116)", __FILE__, __LINE__);
  }

  // the run's mesh, gaps closed, becomes m; eq its element qualities, and
  // known and values (when wanted) its edges' words and values
  void finish(Buf<double>& eq, Buf<u32>* known, Buf<double>* values) {
    // what only the passes need goes first, and the maps of the mesh that
    // goes: there is room then also where a pass found too little
    for (auto* b : {&face_prod, &acc, &eval, &cnt}) b->release();
    for (auto* b : {&sa, &sb, &marks, &marks2}) b->release();
    part.release();
    qpart.release();
    m.up[1][3].reset();
    m.down[3][1].release();
    m.dual.release();
    SwapRunView R = view();
    Buf<u32> er(nE + 1), tr(nT + 1), fr(nF + 1);
    exscan_fn(nE, OHX_LAMBDA(u32 i) { return R.death[i] ? 0u : 1u; }, er.get());
    exscan_fn(nT, OHX_LAMBDA(u32 i) { return R.dead[i] ? 0u : 1u; }, tr.get());
    u32 cap = 64;
    while (cap < 4 * (size_t) (nE - aE)) cap *= 2;
    u32 const mask = cap - 1;
    Buf<unsigned long long> keys(cap);
    Buf<u32> when(cap);
    unsigned long long* kp = keys.get();
    u32* wp = when.get();
    parallel_for(cap, OHX_LAMBDA(u32 i) {
      kp[i] = ~0ull;
      wp[i] = 0;
    });
    hipLaunchKernelGGL(run_pairs_k, dim3(nblocks(nE)), dim3(BLOCK), 0, stream(), R, mask, kp, wp, dev_error_word());
    check_launch("run_pairs");
    exscan_fn_heavy(nF, OHX_LAMBDA(u32 i) {
      u32 const* v = R.fv + 3 * (size_t) i;
      u32 const born = i < R.nF0 ? 0u : R.fbirth[i - R.nF0];
      for (u32 j = 0; j < 3; ++j) {
        unsigned long long const key = swap_pair_key(v[j], v[(j + 1) % 3]);
        for (u32 probe = 0, h = swap_pair_slot(key, mask); probe <= mask; ++probe, h = (h + 1) & mask) {
          unsigned long long const t = kp[h];
          if (t == ~0ull) break;
          if (t != key) continue;
          if (wp[h] > born) return 0u;
          break;
        }
      }
      return 1u;
    }, fr.get());
    // an error of the last pass's kernels shows here, before its output is
    // followed, and how many entities are left.  The faces are counted: around
    // inverted tets a swap can make an edge whose vertices another edge has,
    // and the pair rule then takes the faces of both
    u32 const* ends[4] = {words.get() + RW_ERR, er.get() + nE, tr.get() + nT, fr.get() + nF};
    u32 left[4];
    read_many(ends, 4, left);
    if (left[0]) fail_device(left[0]);
    OHX_REQUIRE(left[1] == aE && left[2] == aT, "swap run: edges or tets miscounted");
    aF = left[3];
    Mesh mo(3, true);
    set_ents(mo, 0, m.counts[0], Buf<u32>());
    u32 const alive[4] = {0, aE, aF, aT};
    Buf<u32> lens(aE), nd31((size_t) 6 * aT), ndual((size_t) 4 * aT);
    Buf<double> neq(aT);
    if (known) {
      *known = Buf<u32>(aE);
      *values = Buf<double>(aE);
    }
    for (u32 d = 1; d <= 3; ++d) {
      RunOut o{};
      o.n = d == 1 ? nE : d == 2 ? nF : nT;
      o.vpe = d + 1;
      o.rank = d == 1 ? er.get() : d == 2 ? fr.get() : tr.get();
      o.v = d == 1 ? ev.get() : d == 2 ? fv.get() : vt.get();
      o.cd = d == 1 ? ecd.get() : d == 2 ? fcd.get() : tcd.get();
      o.ci = !has_id ? nullptr : d == 1 ? eci.get() : d == 2 ? fci.get() : tci.get();
      Buf<u32> verts((size_t) alive[d] * (d + 1)), cdo(alive[d]), cio;
      if (has_id) cio = Buf<u32>(alive[d]);
      o.out = verts.get();
      o.out_cd = cdo.get();
      o.out_ci = cio.get();
      if (d == 1) {
        o.ln = ln.get();
        o.out_ln = lens.get();
        if (known) {
          o.info = info.get();
          o.q = q.get();
          o.out_info = known->get();
          o.out_q = values->get();
        }
      }
      if (d == 3) {
        o.te = te.get();
        o.dual = dual.get();
        o.tq = tq.get();
        o.erank = er.get();
        o.out_te = nd31.get();
        o.out_dual = ndual.get();
        o.out_tq = neq.get();
      }
      hipLaunchKernelGGL(run_out_k, dim3(nblocks(o.n)), dim3(BLOCK), 0, stream(), o);
      check_launch("run_out");
      set_ents(mo, d, alive[d], std::move(verts));
      add_tag_u32(mo, d, "class_dim", 1, std::move(cdo));
      if (has_id) add_tag_u32(mo, d, "class_id", 1, std::move(cio));
    }
    auto up = std::make_unique<Up>();
    up->offsets = exscan(lens.get(), aE);
    up->adj = Buf<u32>((size_t) 6 * aT);
    up->dirs = Buf<u32>((size_t) 6 * aT);
    hipLaunchKernelGGL(run_up_k, dim3(nblocks((size_t) nE * RUN_LG)), dim3(BLOCK), 0, stream(), R, er.get(), tr.get(),
                       up->offsets.get(), up->adj.get(), up->dirs.get());
    check_launch("run_up");
    mo.up[1][3] = std::move(up);
    mo.down[3][1] = std::move(nd31);
    mo.dual = std::move(ndual);
    // nothing below fails: until here m is the mesh the run began with
    mo.tags[0] = std::move(m.tags[0]);
    overwrite(m, std::move(mo));
    eq = std::move(neq);
  }

  void swap(SwapRunView R, unsigned char const* state, u32 nb) {
    u32 const ns = got[0], n1 = got[1], n2 = got[2], n3 = got[3];
    if (6 * ((size_t) nT + n3) >= MAX_USES) fail("swap: more than 2^32 uses", __FILE__, __LINE__);
    edge_room(nE + n1);
    tet_room(nT + n3);
    need(fv, 3 * (size_t) nF, 3 * ((size_t) nF + n2));
    need(fcd, nF, (size_t) nF + n2);
    if (has_id) need(fci, nF, (size_t) nF + n2);
    need(fbirth, nF - nF0, (size_t) nF - nF0 + n2);
    // a ring of rs tets and faces goes, 2 (rs - 2) tets come
    u32 const ring = n3 / 2 + 2 * ns;
    list_room(aT + n3 - ring);
    Buf<u32> lists((size_t) 4 * ns), uses((size_t) 12 * n3), deferred((size_t) 4 * n3);
    // the states may have moved: the round's result is in sa or sb as before
    bool const in_a = state == R.sa;
    R = view();
    state = in_a ? R.sa : R.sb;
    R.sw = lists.get();
    R.o1 = R.sw + ns;
    R.o2 = R.o1 + ns;
    R.o3 = R.o2 + ns;
    u32 const nuse = 6 * n3;
    u32 *slot = uses.get(), *changed = slot + nuse;
    intact = false;  // until the pass is whole
    hipLaunchKernelGGL(run_list_k, dim3(nb), dim3(BLOCK), 0, stream(), R, state, part.get());
    check_launch("run_list");
    launch_timed("swap_cavity", (double) n1 * 8 + (double) n2 * 12 + (double) n3 * 16 + (double) ns * 12,
                 run_products_k, dim3(nblocks((size_t) ns * RUN_G)), dim3(BLOCK), R, ns, face_prod.get(),
                 deferred.get(), R.words + RW_ERR);
    element_qualities_into(3, n3, R.vt + 4 * (size_t) nT, coords(m), 0, metric_of(m), tq.get() + nT);
    hipLaunchKernelGGL(run_touch_k, dim3(nblocks(nuse, RUN_AT)), dim3(RUN_AB), 0, stream(), R, nuse, slot, changed);
    hipLaunchKernelGGL(run_lists_k, dim3(nblocks(nuse, RUN_AB)), dim3(RUN_AB), 0, stream(), R, changed);
    hipLaunchKernelGGL(run_place_k, dim3(nblocks(nuse)), dim3(BLOCK), 0, stream(), R, nuse, slot);
    hipLaunchKernelGGL(run_sort_k, dim3(nblocks(nuse)), dim3(BLOCK), 0, stream(), R, changed);
    hipLaunchKernelGGL(run_settle_k, dim3(nblocks(4 * (size_t) n3)), dim3(BLOCK), 0, stream(), R, n3,
                       face_prod.get(), deferred.get(), R.words + RW_ERR);
    check_launch("run_settle");
    intact = true;
    nE += n1;
    nF += n2;
    nT += n3;
    aE = aE + n1 - ns;
    aF = aF + n2 - ring;
    aT = aT + n3 - ring;
    pool = got[4] + 6 * (size_t) aT;
  }
};
}  // namespace

// ---------------------------------------------------------------- adapt
// mesh_adapt (adapt.cpp:19-94)
namespace {
struct Ctx {
  u32 ops = 0, max_ops = 0;
  AdaptStats st;
  SwapCache swap_cache;  // the shape loop's swap choices (cleared by other passes)
  SizeCodeCache size_codes;  // the collapse loop's size codes (cleared by other passes)
  // passes that changed the mesh: events around them on the stream, read
  // once at the end (a pass's time is the stream's, from the end of the work
  // before it to the end of its own, host waits included)
  struct Timed {
    hipEvent_t a, b;
    double tin;  // input elements, or less than 0: part of the passes, but no pass
  };
  std::vector<Timed> timed;
  std::vector<hipEvent_t> pool;
  bool timing = false;  // the caller wants the statistics
  hipEvent_t event() {
    if (!pool.empty()) {
      hipEvent_t e = pool.back();
      pool.pop_back();
      return e;
    }
    hipEvent_t e;
    OHX_CHECK(hipEventCreate(&e));
    return e;
  }
  Timed start(double tin) {
    Timed t{nullptr, nullptr, tin};
    if (timing) {
      t.a = event();
      t.b = event();
      OHX_CHECK(hipEventRecord(t.a, stream()));
    }
    return t;
  }
  void stop(Timed const& t, bool changed) {
    if (!timing) return;
    OHX_CHECK(hipEventRecord(t.b, stream()));
    if (changed) {
      timed.push_back(t);
    } else {
      pool.push_back(t.a);
      pool.push_back(t.b);
    }
  }
  void finish() {
    for (Timed& t : timed) {
      float ms = 0;
      OHX_CHECK(hipEventElapsedTime(&ms, t.a, t.b));
      if (t.tin >= 0) {
        st.npass += 1;
        st.nelems += t.tin;
      }
      st.tpass += ms * 1e-3;
      pool.push_back(t.a);
      pool.push_back(t.b);
    }
    timed.clear();
    for (hipEvent_t e : pool) (void) hipEventDestroy(e);
    pool.clear();
  }
};
// adapt_summary (adapt.cpp:22-34) only prints: it reads the mesh and changes
// nothing, so it runs only when the per-pass lines are printed
void adapt_summary(Mesh& m) {
  if (!g_verbose) return;
  u32 nel = count(m, m.dim);
  double mq = mesh_min_quality(m);
  u32 ne = count(m, 1);
  Buf<double> s = measure_edges(m);
  double lo = min_f64(s.get(), ne, 1), hi = max_f64(s.get(), ne, 1);
  std::printf("%10u elements, min quality %.0f%%, metric range %.2f - %.2f\n", nel, mq * 100.0, lo, hi);
}
bool incr_op(Mesh& m, Ctx& c) {  // adapt.cpp:36-45
  if (c.ops > c.max_ops) return false;
  ++c.ops;
  adapt_summary(m);
  return true;
}
enum Kind { REFINE, COARSEN, SWAP, COARSEN_SLIVERS };
u32 run_pass(Mesh& m, Ctx& c, Kind k, double a, double b, u32 n, double const* eq = nullptr,
             double const* gate = nullptr) {
  double tin = count(m, m.dim);
  static bool const trace = std::getenv("OHX_TRACE_DERIVE") && std::getenv("OHX_TRACE_DERIVE")[0] == '1';
  if (trace) std::fprintf(stderr, "pass %s n=%.0f\n", k == REFINE ? "refine" : k == COARSEN ? "coarsen" : k == SWAP ? "swap" : "csliv", tin);
  u32 ok = 0;
  Ctx::Timed const t = c.start(tin);
  if (k != SWAP) c.swap_cache.clear();
  if (k != COARSEN) c.size_codes.clear();
  switch (k) {
    case REFINE: ok = refine_by_size(m, a, true); break;
    case COARSEN: ok = coarsen_by_size(m, a, b, &c.size_codes); break;
    case SWAP: ok = swap_slivers(m, a, n, eq, gate, &c.swap_cache); break;
    case COARSEN_SLIVERS: ok = coarsen_slivers(m, a, n, eq); break;
  }
  c.stop(t, ok != 0);
  return ok;
}

// the meshes the in-place swap passes serve: no element field to transfer, no
// batch, nothing to print per pass, classified in every dimension
bool swap_run_fits(Mesh& m) {
  if (m.dim != 3 || !m.full || g_batch || g_verbose) return false;
  bool const has_id = find_tag(m, 0, "class_id") != nullptr;
  for (u32 d = 0; d <= 3; ++d)
    for (char const* name : {"class_dim", "class_id"}) {
      Tag* t = find_tag(m, d, name);
      bool const wanted = name[6] == 'd' || has_id;
      if (wanted && !(t && t->type == TagType::U32 && t->ncomps == 1)) return false;
    }
  return !has_element_transfer(m);
}

// swap passes until one changes nothing; eq: the element qualities of m,
// before and after.  *good_now: the last one found every quality good.
// Returns whether the operation limit was reached.
bool swap_passes(Mesh& m, Ctx& c, double good_qual, u32 nlayers, Buf<double>& eq, bool* good_now) {
  SwapRun run(m);
  bool changed = false, limited = false;
  *good_now = false;
  // copying the mesh is part of the first pass, closing the gaps of them all
  Ctx::Timed t = c.start(count(m, 3));
  run.begin(eq.get(), nullptr, nullptr);
  for (;;) {
    bool ok;
    try {
      ok = run.step(good_qual, nlayers);
    } catch (Error const&) {
      // a pass that fails before it changes anything leaves the mesh of the
      // passes before, as the pass through a whole mesh does
      if (run.intact && changed) {
        try {
          run.finish(eq, nullptr, nullptr);
        } catch (Error const&) {  // the pass's own error is the one to report
        }
      }
      throw;
    }
    c.stop(t, ok);
    if (!ok) {
      *good_now = run.min_q >= good_qual;
      break;
    }
    changed = true;
    if (!incr_op(m, c)) {
      limited = true;
      break;
    }
    // more gaps than tets: close them, so that what each pass reads of the
    // whole mesh stays below twice the mesh
    if (run.nT - run.aT > run.aT || run.lists_full()) {
      Ctx::Timed const gaps = c.start(-1);
      Buf<u32> known;
      Buf<double> values;
      run.finish(eq, &known, &values);
      run.begin(eq.get(), known.get(), values.get());
      c.stop(gaps, true);
      changed = false;
    }
    t = c.start(run.aT);
  }
  if (changed) {
    Ctx::Timed const gaps = c.start(-1);
    run.finish(eq, nullptr, nullptr);
    c.stop(gaps, true);
  }
  return limited;
}
}  // namespace

int adapt(Mesh& m, double size_floor, double good_qual, u32 nlayers, u32 max_ops, AdaptStats* st) {
  Ctx c;
  c.max_ops = max_ops;
  c.timing = st != nullptr;
  double t0 = now_s();
  int result = 0;
  adapt_summary(m);
  double qf = mesh_min_quality(m);  // satisfy_size (adapt.cpp:47-56)
  if (good_qual < qf) qf = good_qual;
  bool aborted = false;
  while (!aborted && run_pass(m, c, REFINE, qf, 0, 0))
    if (!incr_op(m, c)) aborted = true;
  while (!aborted && run_pass(m, c, COARSEN, qf, size_floor, 0))
    if (!incr_op(m, c)) aborted = true;
  while (!aborted) {  // satisfy_shape (adapt.cpp:58-80)
    // the element qualities of this mesh, evaluated once: its minimum, the
    // sliver marks and the comparisons of the swap and collapse passes all
    // read them (a pass that changes nothing leaves them valid for the next)
    u32 const nel = count(m, m.dim);
    Buf<double> eq = c.swap_cache.eq ? std::move(c.swap_cache.eq) : mesh_qualities(m);
    if (swap_run_fits(m)) {
      // the minimum first, in a wait of its own: a mesh of good quality then
      // needs none of the maps a swap pass derives
      double const prev = nel > 1 ? min_f64(eq.get(), nel, 1) : 1.7976931348623157e308;
      if (prev >= good_qual) break;
      c.size_codes.clear();
      c.swap_cache.clear();
      bool good_now = false;
      aborted = swap_passes(m, c, good_qual, nlayers, eq, &good_now);
      if (aborted || good_now) break;
    } else if (m.dim == 3) {
      // the minimum (over elements 1..n-1, as the serial doubles_min)
      // reaches the host with the swap pass's first wait instead of a wait
      // of its own: the pass's sliver marks are gated on it on the device,
      // so when it is at least good_qual the pass marks nothing, changes
      // nothing, and the loop stops where the reference's stops
      Buf<double> mq(1);
      min_f64_async(eq.get(), nel, 1, mq.get());
      u32 const swapped = run_pass(m, c, SWAP, good_qual, 0, nlayers, eq.get(), mq.get());
      double const prev = min_f64_async_result();
      if (prev >= good_qual) {
        OHX_REQUIRE(!swapped, "shape loop: a swap pass ran on a mesh of good quality");
        break;
      }
      if (swapped) {
        if (!incr_op(m, c)) aborted = true;
        continue;
      }
    } else {
      double prev = nel > 1 ? min_f64(eq.get(), nel, 1) : 1.7976931348623157e308;
      if (prev >= good_qual) break;
    }
    if (run_pass(m, c, COARSEN_SLIVERS, good_qual, 0, nlayers, eq.get())) {
      if (!incr_op(m, c)) aborted = true;
      continue;
    }
    if (g_verbose) std::printf("warning: shape quality could not be satisfied\n");
    break;
  }
  result = aborted ? -1 : (c.ops > 0 ? 1 : 0);
  sync();
  c.finish();
  c.st.ttotal = now_s() - t0;
  if (st) *st = c.st;
  return result;
}

// mesh_warp_to_limit (warp_to_limit.cpp:14-81)
u32 warp_to_limit(Mesh& m, double qual_floor) {
  u32 dim = m.dim;
  u32 nv = count(m, 0), ne = count(m, dim);
  u32 const* ev = ask_down(m, dim, 0);
  double const* x = coords(m);
  Tag* wt = find_tag(m, 0, "warp");
  OHX_REQUIRE(wt && wt->type == TagType::F64 && wt->ncomps == 3, "mesh has no 3-component warp field");
  double const* w = wt->f.get();
  Buf<double> xo((size_t) 3 * nv);
  double* xp = xo.get();
  double f = 1;
  bool hit = false;
  auto axpy = [&](double a) {  // doubles_axpy (doubles.cpp:133-145): a*x + y, unfused
    parallel_for(3 * nv, OHX_LAMBDA(u32 i) { xp[i] = a * w[i] + x[i]; });
  };
  axpy(f);
  while (true) {
    double mq = min_element_quality(dim, ne, ev, xp, nv, metric_of(m));
    if (!(mq < qual_floor)) break;
    if (g_verbose) std::printf("quality %f exceeds limit\n", mq);
    hit = true;
    f /= 2;
    axpy(f);
  }
  Buf<double> wo((size_t) 3 * nv);
  double* wp = wo.get();
  double nf = -f;
  parallel_for(3 * nv, OHX_LAMBDA(u32 i) { wp[i] = nf * w[i] + w[i]; });
  remove_tag(m, 0, "coordinates");
  remove_tag(m, 0, "warp");
  add_tag_f64(m, 0, "coordinates", 3, std::move(xo));
  add_tag_f64(m, 0, "warp", 3, std::move(wo));
  return hit ? 0 : 1;
}

}  // namespace ohx
