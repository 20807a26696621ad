// Flag-complex edge collapse (model bit 1) — host part of libssq.
//
// Produces exactly the kept-edge set of GUDHI's sequential collapser as SpecSeq++ calls
// it (specseq.h:209-212,410-424 -> Flag_complex_edge_collapser.h:416-482; edge i has
// filtration i).  The algorithm is split in two:
//
//  1. Main-loop decisions.  When the sequential loop tests edge i, every critical edge has
//     index < i, so "valid" (:148-152) reduces to "index < i": the test is a pure function
//     of the graph of edges < i.  These tests are independent and run on all host threads.
//  2. Cascades (set_edge_critical, :326-359).  For each edge that the main loop finds
//     critical, in index order, the non-critical edges of its 3-cliques are re-tested in
//     decreasing index order with the critical set of that moment.  This part is
//     inherently sequential and runs on one thread.  A re-test is first decided from the
//     edge's last witness: the valid edges only grow, so the common neighbours of an edge
//     only grow and its witness's valid neighbourhood only grows; every new common neighbour
//     comes from an edge turned critical, whose 3-clique pass records it for the re-tested
//     edge.  If the witness is adjacent by a valid edge to every recorded vertex that is now a
//     valid common neighbour, the edge is still dominated; otherwise the full test runs.
//     This part is bound by loads from memory and by branches that cannot be predicted.  With
//     one list of id pairs per edge in large pages, no branch on validity, ids found from one
//     line of the bit sets, and the triangles of a failed test used again, 163,840 edges of 4096
//     rotations (235,000 re-tests) take 47 ms in all on 16 threads, 77 ms before.
//
// The domination predicate (:224-303) is: with I the common valid neighbours of (a,b),
// the edge is dominated iff |I| == 1 or some w in I has I inside its closed valid
// neighbourhood.  It does not depend on vertex labels, so vertices are compacted.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <new>
#include <queue>
#include <thread>
#include <vector>

#include <sys/mman.h>

#include "ssq_internal.h"

// This file is built twice.  The tests count bits throughout, so the second build, with
// SSQ_COLLAPSE_POPCNT defined, may use the processor's instruction for it; the first one has the entry
// points and calls the second's collapse where it is linked in and the processor has that instruction
// (4096 rotations at mean degree 80: 47 ms in all with it, 57.5 without).
namespace ssq {
#ifdef SSQ_COLLAPSE_POPCNT
#define SSQ_COLLAPSE collapse_edges_popcnt
#else
#define SSQ_COLLAPSE collapse_edges_plain
static
#endif
void SSQ_COLLAPSE(int64_t ne, const int32_t* u, const int32_t* v, uint8_t* kept, int threads);
}

namespace {

// Uninitialised storage in large pages where the system has them, grown as needed.
template <typename T>
struct Pages {
  T* p = nullptr;
  size_t cap = 0;
  Pages() = default;
  Pages(const Pages&) = delete;
  Pages& operator=(const Pages&) = delete;
  ~Pages() { release(); }
  void release() {
    std::free(p);
    p = nullptr;
    cap = 0;
  }
  void reserve(size_t n) {
    if (n <= cap) return;
    constexpr size_t kPage = size_t(1) << 21;
    const size_t bytes = ((n + n / 4) * sizeof(T) + kPage - 1) / kPage * kPage;
    release();
    p = (T*)std::aligned_alloc(kPage, bytes);
    if (!p) throw std::bad_alloc();
    madvise(p, bytes, MADV_HUGEPAGE);  // a hint: without it only slower
    cap = bytes / sizeof(T);
  }
};

struct Tri {
  int32_t ea, eb;
};
struct Graph {
  std::vector<int64_t> off;
  std::vector<int32_t> nbr, eid;
  std::vector<uint8_t> crit;
  // Per edge e = (a, b): the ids of (a, x) and (b, x) for its common neighbours x in the whole
  // graph, ascending -- the edge's triangles.  The valid common neighbours of a test are
  // a filter of this list, not a merge of two adjacency lists.  Empty when too large.
  // The lists are far larger than the caches and a test reads one of them from memory (about
  // 9 of 44 triangles are valid in the tests of 4096 rotations at mean degree 80), so they hold
  // both ids side by side and not x, which is read off (a, x) for the valid ones.
  std::vector<int64_t> toff;
  Pages<Tri> own;      // the lists, where they are not kept between calls
  Tri* tri = nullptr;  // edge e's triangles: [toff[e], toff[e] + tcnt[e])
  std::vector<int32_t> tcnt;
  // No loops and no two edges with the same ends.  Otherwise the tables have more than one answer
  // for a pair of vertices (edge_id(x, w) need not be edge_id(w, x)), the third vertices are kept in tx,
  // and candidates are tried one by one: such lists keep the edges that the merges of adjacency
  // lists, or the bit sets, give for them.
  bool simple = true;
  std::vector<int32_t> tx;
  std::vector<int32_t> eu, ev, ex;  // ends, and their exclusive or
  // With at most kBitsetVertices vertices: each neighbourhood as a bit set, W words per vertex.
  // Each word has beside it where its first neighbour stands in nbr and eid, so that finding
  // an edge's id reads one line of this table and one of eid.
  struct Word {
    uint64_t bits;
    int64_t pos;
  };
  Pages<Word> nb;
  int64_t W = 0;
};
constexpr int64_t kTriListMax = int64_t(1) << 28;  // entries (8 bytes each)
constexpr size_t kTriKeep = size_t(1) << 25;       // of them kept by a thread between calls (256 MB)
constexpr int64_t kBitsetVertices = 16384;          // neighbourhood bit sets up to 64 MB

template <typename Valid>
int64_t common(const Graph& g, int32_t a, int32_t b, Valid valid, int32_t* out, int32_t* ea,
               int32_t* eb);

// ... without triangle lists, or of a list that is not simple (out of line: the ordinary test is short).
template <typename Valid>
__attribute__((noinline)) int64_t common_any(const Graph& g, int32_t e, Valid valid, int32_t* out, int32_t* ea,
                                             int32_t* eb, bool ids) {
  if (g.toff.empty()) return common(g, g.eu[e], g.ev[e], valid, out, ids ? ea : nullptr, ids ? eb : nullptr);
  int64_t k = 0;
  const int32_t* tx = g.tx.data() + g.toff[e];
  const Tri* tri = g.tri + g.toff[e];
  for (int32_t t = 0, nt = g.tcnt[e]; t < nt; t++) {
    const int32_t e1 = tri[t].ea, e2 = tri[t].eb;
    if (!valid(e1) || !valid(e2)) continue;
    ea[k] = e1;
    eb[k] = e2;
    out[k++] = tx[t];
  }
  return k;
}

// Valid common neighbours of edge e (ascending), with the two edge ids (not in every case without ids).
template <typename Valid>
int64_t common_e(const Graph& g, int32_t e, Valid valid, int32_t* out, int32_t* ea, int32_t* eb, bool ids) {
  if (__builtin_expect(g.toff.empty() | !g.simple, 0)) return common_any(g, e, valid, out, ea, eb, ids);
  int64_t k = 0;
  const Tri* tri = g.tri + g.toff[e];
  const int32_t nt = g.tcnt[e], a = g.eu[e];
  // No branch on what is valid, which cannot be predicted: every entry is written, and k stands
  // still for those that are not (an edge has fewer triangles than the arrays have room).
  for (int32_t t = 0; t < nt; t++) {
    const int32_t e1 = tri[t].ea, e2 = tri[t].eb;
    ea[k] = e1;
    eb[k] = e2;
    k += (int)valid(e1) & (int)valid(e2);
  }
  for (int64_t t = 0; t < k; t++) out[t] = g.ex[ea[t]] ^ a;
  return k;
}

template <typename Valid>
int64_t common(const Graph& g, int32_t a, int32_t b, Valid valid, int32_t* out, int32_t* ea,
               int32_t* eb) {
  int64_t i = g.off[a], ie = g.off[a + 1], j = g.off[b], je = g.off[b + 1], k = 0;
  while (i < ie && j < je) {
    if (!valid(g.eid[i])) { i++; continue; }
    if (!valid(g.eid[j])) { j++; continue; }
    int32_t x = g.nbr[i], y = g.nbr[j];
    if (x < y) i++;
    else if (x > y) j++;
    else {
      if (ea) {
        ea[k] = g.eid[i];
        eb[k] = g.eid[j];
      }
      if (out) out[k] = x;
      k++;
      i++;
      j++;
    }
  }
  return k;
}

// id of edge (u, v), or -1 (neighbours are ascending)
inline int32_t edge_id(const Graph& g, int32_t u, int32_t v) {
  if (g.W) {
    const Graph::Word& word = g.nb.p[u * g.W + (v >> 6)];
    const uint64_t bit = 1ull << (v & 63);
    if (!(word.bits & bit)) return -1;
    return g.eid[word.pos + __builtin_popcountll(word.bits & (bit - 1))];
  }
  const int32_t* b = g.nbr.data() + g.off[u];
  const int32_t* e = g.nbr.data() + g.off[u + 1];
  const int32_t* p = std::lower_bound(b, e, v);
  return (p != e && *p == v) ? g.eid[p - g.nbr.data()] : -1;
}

// The first of I[0:m) that is not in w's closed valid neighbourhood, or -1.
template <typename Valid>
inline int32_t uncovered(const Graph& g, int32_t w, const int32_t* I, int64_t m, Valid valid) {
  if (g.W) {
    for (int64_t t = 0; t < m; t++) {
      if (I[t] == w) continue;
      const int32_t e = edge_id(g, w, I[t]);
      if (e < 0 || !valid(e)) return I[t];
    }
    return -1;
  }
  int64_t p = g.off[w], pe = g.off[w + 1];
  for (int64_t t = 0; t < m; t++) {
    const int32_t x = I[t];
    if (x == w) continue;
    while (p < pe && g.nbr[p] < x) p++;
    if (!(p < pe && g.nbr[p] == x && valid(g.eid[p]))) return x;
  }
  return -1;
}

// The predicate of edge_is_dominated: |I| == 1 or some w in I covers I.  *witness is tried
// first and receives the dominating vertex found (the answer does not depend on the order
// in which candidates are tried).  A vertex x that one candidate does not cover is checked
// against all candidates left before the next is tried: it is usually a vertex with few
// neighbours in I, so that most candidates go with it, and the checks read x's row only.  `missed`,
// if it is one of I, is such a vertex known beforehand.  The workspace holds I and its edges
// afterwards.
struct Work {
  std::vector<int32_t> I, C, ea, eb;
  int64_t m = 0;
  bool ids;  // the edges are read afterwards
  Work(int64_t maxdeg, bool ids_read) : I((size_t)maxdeg), C((size_t)maxdeg), ea((size_t)maxdeg), eb((size_t)maxdeg), ids(ids_read) {}
};
template <typename Valid>
__attribute__((noinline)) bool dominated_in_turn(const Graph& g, const int32_t* I, int64_t m, Valid valid,
                                                 int32_t* witness) {
  const int32_t hint = *witness;
  if (hint >= 0 && std::binary_search(I, I + m, hint) && uncovered(g, hint, I, m, valid) < 0) return true;
  for (int64_t c = 0; c < m; c++) {
    if (I[c] == hint || uncovered(g, I[c], I, m, valid) >= 0) continue;
    *witness = I[c];
    return true;
  }
  return false;
}
template <typename Valid>
bool dominated(const Graph& g, int32_t e, Valid valid, Work& wk, int32_t* witness, int32_t missed) {
  int32_t *I = wk.I.data(), *C = wk.C.data();
  const int64_t m = wk.m = common_e(g, e, valid, I, wk.ea.data(), wk.eb.data(), wk.ids);
  if (m <= 1) {
    if (m == 1) *witness = I[0];
    return m == 1;
  }
  // Striking relies on an edge having one id from both its ends, and on the bit sets: without them an id
  // is a binary search, and it pays to read one candidate's list after the other (17,000 vertices of
  // mean degree 300: 5.6 s with the searches, 5.2 s this way, on 8 threads; in the plane 2.3 and 1.7 s).
  if (__builtin_expect(!g.simple | !g.W, 0)) return dominated_in_turn(g, I, m, valid, witness);
  int64_t n = m;
  std::copy(I, I + m, C);
  auto strike = [&](int32_t x) {  // x stays a candidate, and those joined to it by a valid edge
    int64_t k = 0;
    for (int64_t c = 0; c < n; c++) {
      const int32_t w = C[c];
      if (w != x) {
        const int32_t id = edge_id(g, x, w);
        if (id < 0 || !valid(id)) continue;
      }
      C[k++] = w;
    }
    n = k;
  };
  int32_t w = *witness;
  if (missed >= 0 && std::binary_search(I, I + m, missed)) {
    strike(missed);
  } else if (w >= 0 && std::binary_search(I, I + m, w)) {
    const int32_t x = uncovered(g, w, I, m, valid);
    if (x < 0) return true;
    strike(x);
  }
  while (n > 0) {
    w = C[0];
    const int32_t x = uncovered(g, w, I, m, valid);
    if (x < 0) {
      *witness = w;
      return true;
    }
    strike(x);  // at least w goes
  }
  return false;
}

}  // namespace

namespace ssq {

void SSQ_COLLAPSE(int64_t ne, const int32_t* u, const int32_t* v, uint8_t* kept, int threads) {
  if (ne <= 0) return;
  // compact vertex labels to 0..nv-1 in increasing label order
  int32_t lmin = u[0], lmax = u[0];
  for (int64_t i = 0; i < ne; i++) {
    lmin = std::min(lmin, std::min(u[i], v[i]));
    lmax = std::max(lmax, std::max(u[i], v[i]));
  }
  std::vector<int32_t> eu((size_t)ne), ev((size_t)ne);
  int64_t nv = 0;
  const int64_t range = (int64_t)lmax - lmin + 1;
  if (range <= 8 * ne + 1024) {  // labels in a small range: a direct table
    std::vector<int32_t> id((size_t)range, -1);
    for (int64_t i = 0; i < ne; i++) id[(size_t)(u[i] - lmin)] = id[(size_t)(v[i] - lmin)] = 0;
    for (int64_t x = 0; x < range; x++)
      if (id[(size_t)x] == 0) id[(size_t)x] = (int32_t)nv++;
    for (int64_t i = 0; i < ne; i++) {
      eu[i] = id[(size_t)(u[i] - lmin)];
      ev[i] = id[(size_t)(v[i] - lmin)];
    }
  } else {
    std::vector<int32_t> lab((size_t)(2 * ne));
    for (int64_t i = 0; i < ne; i++) { lab[2 * i] = u[i]; lab[2 * i + 1] = v[i]; }
    std::sort(lab.begin(), lab.end());
    lab.erase(std::unique(lab.begin(), lab.end()), lab.end());
    nv = (int64_t)lab.size();
    for (int64_t i = 0; i < ne; i++) {
      eu[i] = (int32_t)(std::lower_bound(lab.begin(), lab.end(), u[i]) - lab.begin());
      ev[i] = (int32_t)(std::lower_bound(lab.begin(), lab.end(), v[i]) - lab.begin());
    }
  }
  Graph g;
  g.off.assign((size_t)nv + 1, 0);
  for (int64_t i = 0; i < ne; i++) { g.off[eu[i] + 1]++; g.off[ev[i] + 1]++; }
  for (int64_t i = 0; i < nv; i++) g.off[i + 1] += g.off[i];
  g.nbr.resize((size_t)(2 * ne));
  g.eid.resize((size_t)(2 * ne));
  {
    std::vector<int64_t> fill(g.off.begin(), g.off.end() - 1);
    for (int64_t i = 0; i < ne; i++) {
      int64_t p = fill[eu[i]]++;
      g.nbr[p] = ev[i]; g.eid[p] = (int32_t)i;
      p = fill[ev[i]]++;
      g.nbr[p] = eu[i]; g.eid[p] = (int32_t)i;
    }
  }
  if (threads < 1) threads = 1;
  // body(i) for i in [0, count), chunks of `chunk` taken by all threads
  auto parallel_range = [&](int64_t count, int64_t chunk, auto&& body) {
    std::atomic<int64_t> next{0};
    auto work = [&]() {
      for (;;) {
        const int64_t s0 = next.fetch_add(chunk);
        if (s0 >= count) break;
        for (int64_t i = s0; i < std::min(count, s0 + chunk); i++) body(i);
      }
    };
    std::vector<std::thread> pool;
    for (int t = 1; t < threads; t++) pool.emplace_back(work);
    work();
    for (auto& t : pool) t.join();
  };
  auto parallel_edges = [&](auto&& body) { parallel_range(ne, 1024, body); };
  // each vertex's neighbours ascending (they were filled in edge order)
  std::atomic<bool> simple{true};
  parallel_range(nv, 16, [&](int64_t a) {
    thread_local std::vector<std::pair<int32_t, int32_t>> tmp;
    tmp.clear();
    for (int64_t p = g.off[a]; p < g.off[a + 1]; p++) tmp.emplace_back(g.nbr[p], g.eid[p]);
    std::sort(tmp.begin(), tmp.end());
    for (int64_t p = g.off[a], k = 0; p < g.off[a + 1]; p++, k++) {
      g.nbr[p] = tmp[k].first;
      g.eid[p] = tmp[k].second;
      if (tmp[k].first == a || (k > 0 && tmp[k].first == tmp[k - 1].first))
        simple.store(false, std::memory_order_relaxed);
    }
  });
  g.simple = simple;
  int64_t maxdeg = 1;
  for (int64_t a = 0; a < nv; a++) maxdeg = std::max(maxdeg, g.off[a + 1] - g.off[a]);
  g.eu = eu;
  g.ev = ev;
  g.ex.resize((size_t)ne);
  for (int64_t e = 0; e < ne; e++) g.ex[e] = eu[e] ^ ev[e];
  {  // triangle lists of every edge
    std::vector<int64_t> cap((size_t)ne + 1, 0);
    g.tcnt.assign((size_t)ne, 0);
    const int64_t W = (nv + 63) / 64;
    // f(x, id of (a, x), id of (b, x)) for the common neighbours x of e = (a, b), ascending, by the bit
    // sets: the set bits of one AND per word, or the shorter list's neighbours looked up in the other
    // row where they are fewer than the words (16,000 vertices of mean degree 37: 340 ms in all on
    // one thread by the words alone, 150 ms this way).
    const auto each_common = [&](int64_t e, auto&& f) {
      const int32_t a = eu[e], b = ev[e];
      const Graph::Word *ra = g.nb.p + (int64_t)a * W, *rb = g.nb.p + (int64_t)b * W;
      const auto id = [&](const Graph::Word& word, int bit) {
        return g.eid[word.pos + __builtin_popcountll(word.bits & ((1ull << bit) - 1))];
      };
      const bool first = g.off[a + 1] - g.off[a] <= g.off[b + 1] - g.off[b];
      const int32_t s = first ? a : b;
      if (g.simple && g.off[s + 1] - g.off[s] < W) {
        const Graph::Word* other = first ? rb : ra;
        for (int64_t p = g.off[s]; p < g.off[s + 1]; p++) {
          const int32_t x = g.nbr[p];
          const Graph::Word& word = other[x >> 6];
          if (!((word.bits >> (x & 63)) & 1)) continue;
          const int32_t there = id(word, x & 63);
          f(x, first ? g.eid[p] : there, first ? there : g.eid[p]);
        }
        return;
      }
      for (int64_t w = 0; w < W; w++)
        for (uint64_t m = ra[w].bits & rb[w].bits; m; m &= m - 1) {
          const int bit = __builtin_ctzll(m);
          f(w * 64 + bit, id(ra[w], bit), id(rb[w], bit));
        }
    };
    if (nv <= kBitsetVertices) {
      g.W = W;
      // neighbourhoods as bit sets: a neighbour's position in a sorted adjacency list is the
      // popcount of the set bits below it (a prefix count per word plus one word)
      g.nb.reserve((size_t)(nv * W));
      parallel_range(nv, 16, [&](int64_t a) {
        Graph::Word* row = g.nb.p + a * W;
        std::fill(row, row + W, Graph::Word{0, 0});
        for (int64_t p = g.off[a]; p < g.off[a + 1]; p++) row[g.nbr[p] >> 6].bits |= 1ull << (g.nbr[p] & 63);
        int64_t run = g.off[a];
        for (int64_t w = 0; w < W; w++) {
          row[w].pos = run;
          run += __builtin_popcountll(row[w].bits);
        }
      });
      parallel_edges([&](int64_t e) {  // exact counts first
        int32_t k = 0;
        each_common(e, [&](int64_t, int32_t, int32_t) { k++; });
        g.tcnt[e] = k;
      });
      for (int64_t e = 0; e < ne; e++) cap[e + 1] = cap[e] + g.tcnt[e];
    } else {  // merges: edge e gets min(deg a, deg b) slots
      for (int64_t e = 0; e < ne; e++)
        cap[e + 1] = cap[e] + std::min(g.off[eu[e] + 1] - g.off[eu[e]], g.off[ev[e] + 1] - g.off[ev[e]]);
    }
    if (cap[ne] <= kTriListMax) {
      // Kept by the calling thread between calls, as fresh pages cost more than filling them; above
      // kTriKeep the search takes so much longer that the pages are given back at the end of the call.
      thread_local Pages<Tri> keep;
      Pages<Tri>& lists = (size_t)cap[ne] <= kTriKeep ? keep : g.own;
      lists.reserve((size_t)cap[ne]);
      g.tri = lists.p;
      if (!g.simple) g.tx.resize((size_t)cap[ne]);
      if (nv <= kBitsetVertices) {
        parallel_edges([&](int64_t e) {
          Tri* tri = g.tri + cap[e];
          each_common(e, [&](int64_t x, int32_t ea, int32_t eb) {
            if (!g.simple) g.tx[(size_t)(tri - g.tri)] = (int32_t)x;
            *tri++ = Tri{ea, eb};
          });
        });
      } else {
        parallel_edges([&](int64_t e) {
          thread_local std::vector<int32_t> ta, tb;
          ta.resize((size_t)maxdeg);
          tb.resize((size_t)maxdeg);
          int32_t* tx = g.simple ? nullptr : g.tx.data() + cap[e];
          const int32_t k = (int32_t)common(g, eu[e], ev[e], [](int32_t) { return true; }, tx, ta.data(), tb.data());
          for (int32_t t = 0; t < k; t++) g.tri[cap[e] + t] = Tri{ta[t], tb[t]};
          g.tcnt[e] = k;
        });
      }
      g.toff.swap(cap);
    }
  }

  // 1. main-loop decisions, in parallel
  std::vector<uint8_t> main_crit((size_t)ne, 0);
  std::vector<int32_t> witness((size_t)ne, -1);
  main_crit[0] = 1;
  {
    std::atomic<int64_t> next{1};
    auto work = [&]() {
      Work wk(maxdeg, false);
      for (;;) {
        int64_t s = next.fetch_add(256);
        if (s >= ne) break;
        int64_t e = std::min(ne, s + 256);
        for (int64_t i = s; i < e; i++) {
          int32_t idx = (int32_t)i;
          main_crit[i] = !dominated(g, idx, [idx](int32_t x) { return x < idx; }, wk, &witness[i], -1);
        }
      }
    };
    std::vector<std::thread> pool;
    for (int t = 1; t < threads; t++) pool.emplace_back(work);
    work();
    for (auto& t : pool) t.join();
  }

  // 2. sequential cascades
  g.crit.assign((size_t)ne, 0);
  Work wk(maxdeg, true);
  std::priority_queue<int32_t> heap;
  // vertices that may have become common neighbours of a pushed edge since its last test: a
  // list per edge in a pool that lives for one cascade (every pushed edge is popped in it)
  struct Head {
    int32_t sid, at;  // the cascade that pushed the edge last, and its list's first entry
  };
  struct Cand {
    int32_t next, x;
  };
  std::vector<Head> head((size_t)ne, Head{-1, -1});
  std::vector<Cand> pool;
  auto add_cand = [&](int32_t e, int32_t x, int32_t sid) {
    Head& h = head[e];
    if (h.sid != sid) {
      h = Head{sid, -1};
      heap.push(e);
    }
    pool.push_back(Cand{h.at, x});
    h.at = (int32_t)pool.size() - 1;
  };
  // the valid triangles of e, now critical, in wk: their other edges are tested again
  auto three_clique = [&](int32_t thresh, int32_t e, int32_t sid) {
    const uint8_t* crit = g.crit.data();
    if (!g.simple)  // an edge may be in a triangle of its own: the test before did not see it as critical
      wk.m = common_e(g, e, [thresh, crit](int32_t x) { return (x < thresh) | crit[x]; }, wk.I.data(), wk.ea.data(),
                      wk.eb.data(), true);
    const int32_t p = g.eu[e], q = g.ev[e];
    for (int64_t k = 0; k < wk.m; k++) {
      const int32_t e1 = wk.ea[k], e2 = wk.eb[k];  // e1 = (p, x) gains q, e2 = (q, x) gains p
      if (!crit[e1] && e1 < thresh) add_cand(e1, q, sid);
      if (!crit[e2] && e2 < thresh) add_cand(e2, p, sid);
    }
  };
  // still dominated by its last witness: every recorded vertex is the witness, or joined to it
  // by a valid edge, or not a valid common neighbour; if not, *missed is that vertex
  auto witness_holds = [&](int32_t cur, int32_t sid, int32_t* missed) {
    const int32_t w = witness[cur];
    *missed = -1;
    if (w < 0) return false;
    const uint8_t* crit = g.crit.data();
    auto valid = [cur, crit](int32_t x) { return x >= 0 && (x < cur || crit[x]); };
    const int32_t a = g.eu[cur], b = g.ev[cur];
    for (int32_t t = head[cur].sid == sid ? head[cur].at : -1; t >= 0; t = pool[t].next) {
      const int32_t x = pool[t].x;
      if (x == w || valid(edge_id(g, w, x))) continue;
      if (valid(edge_id(g, a, x)) && valid(edge_id(g, b, x))) {
        *missed = x;
        return false;
      }
    }
    return true;
  };
  std::fill(kept, kept + ne, 0);
  g.crit[0] = 1;
  kept[0] = 1;
  for (int32_t idx = 1; idx < (int32_t)ne; idx++) {
    if (!main_crit[idx]) continue;
    pool.clear();
    g.crit[idx] = 1;
    kept[idx] = 1;
    wk.m = common_e(g, idx, [idx, crit = g.crit.data()](int32_t x) { return (x < idx) | crit[x]; }, wk.I.data(),
                    wk.ea.data(), wk.eb.data(), true);
    three_clique(idx, idx, idx);
    while (!heap.empty()) {
      int32_t cur = heap.top();
      heap.pop();
      if (!heap.empty() && g.tri) {  // the next one's list comes from memory meanwhile
        const Tri* t = g.tri + g.toff[heap.top()];
        for (int k = 0; k < 48; k += 8) __builtin_prefetch(t + k);
      }
      if (g.crit[cur]) continue;
      int32_t missed;
      if (witness_holds(cur, idx, &missed)) continue;
      const uint8_t* crit = g.crit.data();
      if (dominated(g, cur, [cur, crit](int32_t x) { return (x < cur) | crit[x]; }, wk, &witness[cur], missed))
        continue;
      g.crit[cur] = 1;
      kept[cur] = 1;
      three_clique(cur, cur, idx);
    }
  }
}

}  // namespace ssq

#ifndef SSQ_COLLAPSE_POPCNT
namespace ssq {
__attribute__((weak)) void collapse_edges_popcnt(int64_t ne, const int32_t* u, const int32_t* v, uint8_t* kept,
                                                 int threads);
}
void ssq::collapse_edges(int64_t ne, const int32_t* u, const int32_t* v, uint8_t* kept, int threads) {
  if (collapse_edges_popcnt && __builtin_cpu_supports("popcnt")) collapse_edges_popcnt(ne, u, v, kept, threads);
  else collapse_edges_plain(ne, u, v, kept, threads);
}

extern "C" int ssq_collapse_edges(int64_t ne, const int32_t* u, const int32_t* v, uint8_t* kept, int threads) {
  if (ne < 0 || (ne > 0 && (!u || !v || !kept))) return SSQ_EINVAL;
  if (threads <= 0) threads = (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  ssq::collapse_edges(ne, u, v, kept, threads);
  return SSQ_OK;
}
#endif
