// Matrix assembly dispatch: offset tables, owner-computes schedules and the
// per-integral launches (CUDAAssembler::assemble_matrix,
// cpp/cudolfinx/fem/CUDAAssembler.h:683-740, and set_diagonal :878-958).
#include <algorithm>
#include <array>
#include <cstdio>
#include <exception>
#include <functional>
#include <numeric>
#include <system_error>
#include <thread>

#include "mf_internal.h"

namespace mf {

struct OwnerPlan {
  int64_t nchunks = 0;
  DevArray<int32_t> chunk_rows, chunk_items, item_cell, chunk_meta, pair_list;
  DevArray<uint32_t> item_mask;
  DevArray<uint8_t> pair_kk;
  DevArray<uint16_t> pair_row;        // simplex kernels: each pair's row in its chunk
  DevArray<uint16_t> pair_pos;        // hexahedral kernel: row-relative position of each column
  DevArray<int32_t> item_geo;         // hexahedral kernel: the 8 vertices of each item's cell
  DevArray<int32_t> diag_pos;         // hexahedral kernel: row-relative position of the diagonal
  int64_t nitems = 0, npairs = 0;
  // host copies used while building schedules
  std::vector<int32_t> h_items, h_cell;
  std::vector<uint64_t> h_mask;
  void drop_host() {                  // with their memory
    std::vector<int32_t>().swap(h_items);
    std::vector<int32_t>().swap(h_cell);
    std::vector<uint64_t>().swap(h_mask);
  }
};

namespace {

constexpr int kTableLanes = 64;

// Items of a row partition: every entity of a cell integral that has a
// row dof in a chunk, with the mask of its local rows the chunk owns (on the
// host; each kernel's schedule holds what that kernel reads).
std::shared_ptr<OwnerPlan> build_items(const std::vector<int32_t>& rows, const Integral& I,
                                       const mf_dofmap* d0) {
  const int nd = d0->nd;
  MF_CHECK(nd <= 64, MF_EUNSUPPORTED, "owner schedules need at most 64 dofs per cell");
  const int64_t nch = static_cast<int64_t>(rows.size()) - 1;
  std::vector<int32_t> row_chunk(d0->num_nodes);
  for (int64_t c = 0; c < nch; ++c)
    for (int32_t r = rows[c]; r < rows[c + 1]; ++r) row_chunk[r] = static_cast<int32_t>(c);
  std::vector<int64_t> cnt(nch + 1, 0);
  std::vector<int32_t> tmp(nd);
  auto cell_chunks = [&](int32_t c, int32_t* out) {
    int n = 0;
    for (int l = 0; l < nd; ++l) {
      int32_t ch = row_chunk[d0->host[(int64_t)c * nd + l]];
      bool dup = false;
      for (int q = 0; q < n; ++q) dup |= out[q] == ch;
      if (!dup) out[n++] = ch;
    }
    return n;
  };
  for (int64_t e = 0; e < I.n; ++e) {
    int n = cell_chunks(I.h_ents[e], tmp.data());
    for (int q = 0; q < n; ++q) cnt[tmp[q] + 1]++;
  }
  for (int64_t c = 0; c < nch; ++c) cnt[c + 1] += cnt[c];
  MF_CHECK(cnt[nch] < INT32_MAX, MF_EUNSUPPORTED, "too many owner items");
  std::vector<int32_t> icell(cnt[nch] + 1, 0);
  std::vector<uint64_t> imask(std::max<int64_t>(1, cnt[nch]));
  std::vector<int64_t> pos(cnt.begin(), cnt.end() - 1);
  for (int64_t e = 0; e < I.n; ++e) {
    const int32_t c = I.h_ents[e];
    int n = cell_chunks(c, tmp.data());
    for (int q = 0; q < n; ++q) {
      uint64_t msk = 0;
      for (int l = 0; l < nd; ++l)
        if (row_chunk[d0->host[(int64_t)c * nd + l]] == tmp[q]) msk |= 1ull << l;
      int64_t p = pos[tmp[q]]++;
      icell[p] = c;
      imask[p] = msk;
    }
  }
  auto plan = std::make_shared<OwnerPlan>();
  plan->nchunks = nch;
  plan->nitems = cnt[nch];
  std::vector<int32_t> ci(nch + 1);
  for (int64_t c = 0; c <= nch; ++c) ci[c] = static_cast<int32_t>(cnt[c]);
  plan->h_items = std::move(ci);
  plan->h_cell = std::move(icell);
  plan->h_mask = std::move(imask);
  return plan;
}

// sum[0 .. 8 V) = init[h ..] + the n rows at[.][h ..] (16-byte aligned)
typedef uint16_t U16x8 __attribute__((vector_size(16), may_alias));
template <int V>
static void add_up(uint16_t* sum, uint16_t* const* at, int n, const uint16_t* init, int h) {
  U16x8 m[V];
  for (int v = 0; v < V; ++v) m[v] = reinterpret_cast<const U16x8*>(init + h)[v];
  for (int i = 0; i < n; ++i)
    for (int v = 0; v < V; ++v) m[v] += reinterpret_cast<const U16x8*>(at[i] + h)[v];
  for (int v = 0; v < V; ++v) reinterpret_cast<U16x8*>(sum)[v] = m[v];
}

// Contiguous blocked-row chunks whose unrolled value segment fits `cap`
// doubles, with at most `maxr` rows and `maxp` (cell, owned row) pairs; then
// the per-chunk pair lists and, for every pair and column j of the cell, the
// position of the column node in the row's blocked column list.
std::shared_ptr<OwnerPlan> build_owner_plan(const mf_form& a, const Integral& I, const mf_matrix& A,
                                            int64_t cap, int maxr, int maxp, bool with_kk,
                                            bool mfma = false) {
  const mf_dofmap* d0 = a.dm[0];
  const mf_dofmap* d1 = a.dm[1];
  const int nd = d0->nd;
  if (nd > (with_kk ? 32 : 64)) return nullptr;
  if (with_kk && d0->num_cells >= (int64_t(1) << 26)) return nullptr;   // cell << 6 | i in 32 bits
  if (!with_kk) maxr = std::min(maxr, 1023), maxp = std::min(maxp, 32767);   // fields of pair_list
  const int bs2 = A.bs0 * A.bs1;
  std::vector<int32_t> ncell(A.nrows_b, 0);
  for (int64_t e = 0; e < I.n; ++e)
    for (int l = 0; l < nd; ++l) ncell[d0->host[(int64_t)I.h_ents[e] * nd + l]]++;
  std::vector<int32_t> rows{0};
  if (with_kk) {
    int64_t seg = 0, pairs = 0;
    int32_t r0 = 0;
    for (int64_t r = 0; r < A.nrows_b; ++r) {
      const int64_t len = (int64_t)bs2 * (A.h_rpb[r + 1] - A.h_rpb[r]);
      if (len > cap || ncell[r] > maxp) return nullptr;   // a single row does not fit
      if (seg + len > cap || r - r0 >= maxr || pairs + ncell[r] > maxp) {
        rows.push_back(static_cast<int32_t>(r));
        r0 = static_cast<int32_t>(r);
        seg = 0;
        pairs = 0;
      }
      seg += len;
      pairs += ncell[r];
    }
  } else {
    // The hexahedral kernel forms the geometry of every cell of a chunk at all
    // its quadrature points, and contracts its pairs in tiles of 16, one per SIMD
    // at a time.  In FP64 a chunk ends where it has the fewest cells per value
    // among the row counts that fill at least 3/4 of it; in FP32 and BF16, where
    // the matrix cores make a tile the longest part, a round of four tiles counts
    // as eight cells, from half of it on (a fifth tile keeps three SIMDs waiting).
    // Q3 24^3: FP32 524 -> 474 us; in FP64 the same rule takes 404 for 380 us.
    std::vector<int64_t> start(A.nrows_b + 1, 0);
    for (int64_t r = 0; r < A.nrows_b; ++r) start[r + 1] = start[r] + ncell[r];
    std::vector<int32_t> cells(std::max<int64_t>(1, start[A.nrows_b]));
    {
      std::vector<int64_t> at(start.begin(), start.end() - 1);
      for (int64_t e = 0; e < I.n; ++e)
        for (int l = 0; l < nd; ++l)
          cells[at[d0->host[(int64_t)I.h_ents[e] * nd + l]]++] = I.h_ents[e];
    }
    std::vector<int32_t> seen(d0->num_cells, -1);
    std::vector<std::array<int64_t, 3>> ends;          // (values, cells, pairs) up to each row
    for (int64_t r0 = 0; r0 < A.nrows_b;) {
      int64_t seg = 0, pairs = 0, items = 0, r = r0;
      ends.clear();
      for (; r < A.nrows_b && r - r0 < maxr; ++r) {
        const int64_t len = (int64_t)bs2 * (A.h_rpb[r + 1] - A.h_rpb[r]);
        if (len > cap || ncell[r] > maxp) return nullptr;
        if (seg + len > cap || pairs + ncell[r] > maxp) break;
        seg += len;
        pairs += ncell[r];
        for (int64_t k = start[r]; k < start[r + 1]; ++k)
          if (seen[cells[k]] != (int32_t)r0) {
            seen[cells[k]] = (int32_t)r0;
            ++items;
          }
        ends.push_back({seg, items, pairs});
      }
      auto cost = [&](size_t k) {
        return double(ends[k][1] + (mfma ? 8 * ((ends[k][2] + 63) / 64) : 0)) / ends[k][0];
      };
      size_t best = ends.size() - 1;
      if (r < A.nrows_b)
        for (size_t k = 0; k + 1 < ends.size(); ++k)
          if (4 * ends[k][0] >= (mfma ? 2 : 3) * seg && cost(k) < cost(best)) best = k;
      r0 += static_cast<int64_t>(best) + 1;
      if (r0 < A.nrows_b) rows.push_back(static_cast<int32_t>(r0));
    }
  }
  rows.push_back(static_cast<int32_t>(A.nrows_b));
  auto plan = build_items(rows, I, d0);
  const int64_t nch = plan->nchunks;
  const auto& ci = plan->h_items;
  // pair offsets per chunk
  std::vector<int64_t> poff(nch + 1, 0);
  for (int64_t c = 0; c < nch; ++c) {
    int64_t n = 0;
    for (int32_t it = ci[c]; it < ci[c + 1]; ++it) n += __builtin_popcountll(plan->h_mask[it]);
    poff[c + 1] = poff[c] + n;
  }
  const int64_t np = poff[nch];
  std::vector<int32_t> plist(np + 1, 0);
  std::vector<uint16_t> prow(with_kk ? np + 1 : 1, 0);
  // column offsets: one 16-byte aligned block of npairs * nd bytes per chunk
  std::vector<int64_t> kkoff(nch + 1, 0);
  for (int64_t c = 0; c < nch; ++c)
    kkoff[c + 1] = kkoff[c] + ((poff[c + 1] - poff[c]) * nd + 15) / 16 * 16;
  MF_CHECK(kkoff[nch] < INT32_MAX, MF_EUNSUPPORTED, "column offset table exceeds int32 indexing");
  std::vector<uint8_t> pkk(with_kk ? std::max<int64_t>(16, kkoff[nch]) : 16, 0);
  // hexahedral kernel: position of each of the nd column nodes within the
  // pair's (scalar) row, relative to the row start, one uint16 per column
  std::vector<uint16_t> ppos(with_kk ? 8 : std::max<int64_t>(8, np * nd), 0);
  std::vector<int> bad(16, 0);
  unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  // Order of a simplex chunk's pairs.  The lanes of a wave add an entry of the same
  // column j of their pairs into LDS at once, 16 lanes at a time (groups of 8, 32
  // and 64 were slower), and adds that meet in a bank (32 of 8 bytes) or at one
  // address wait for each other.  So the pairs are dealt to groups of 16 one by one,
  // each to the group where its addresses meet the fewest so far: first one pair of
  // every row, then the next, a row's local indices in turn.  Vector P2 48^3
  // matrix 742 us with the pairs in the order of the cells, 627 dealt in turn
  // without regard to banks, 610 so; 13^3 30 -> 24 us, P2 25^3 29 -> 27, P3 24^3
  // 74.5 -> 73.5.  P1, 24 pairs to a row, stays in the order of the cells: there it
  // is the records that are scattered then (50^3 48 -> 58 us).
  constexpr int kGroup = 16;
  struct Pair {
    int32_t cell, i, row, turn;
    uint8_t kk[32];
  };
  struct Scratch {                                     // of one thread
    std::vector<int32_t> first, order;                 // order[first[r] ..]: the pairs of row r
    std::vector<int32_t> where;                        // of a column node in the row at hand
    std::vector<uint16_t> load, meet;
    std::vector<int> fill;
    std::vector<uint16_t*> at;
  };
  auto order_pairs = [&](const std::vector<Pair>& P, int64_t c, std::vector<int32_t>& place, Scratch& S) {
    const int np = static_cast<int>(P.size()), nb = (np + kGroup - 1) / kGroup, bs = A.bs0;
    const int nr = rows[c + 1] - rows[c];
    const int64_t cb0 = A.h_rpb[rows[c]];
    place.resize(np);
    // in a row by (turn, local row), which no two pairs of it share
    int most = 0;
    auto key = [&](int k) { return P[k].turn * 64 + P[k].i; };
    for (int r = 0; r < nr; ++r) {
      most = std::max(most, S.first[r + 1] - S.first[r]);
      for (int a = S.first[r] + 1; a < S.first[r + 1]; ++a) {
        const int k = S.order[a];
        int q = a;
        for (; q > S.first[r] && key(S.order[q - 1]) > key(k); --q) S.order[q] = S.order[q - 1];
        S.order[q] = k;
      }
    }
    // The pairs that meet in a bank, by (column, component), bank and group: the
    // groups of one place lie side by side, so a pair is weighed against all of
    // them at once.
    const int NB = (nb + 7) / 8 * 8;
    S.load.assign((static_cast<size_t>(nd) * bs * 32 + 1) * NB, 0);
    S.meet.resize(NB);
    S.at.resize(nd * bs);
    S.fill.assign(nb, 0);
    int dealt = 0;
    for (int turn = 0; turn < most; ++turn)
      for (int r = 0; r < nr; ++r) {
        if (S.first[r] + turn >= S.first[r + 1]) continue;
        const int k = S.order[S.first[r] + turn];
        if (nb == 1) {
          place[k] = dealt++;
          continue;
        }
        const Pair& x = P[k];
        const int64_t R = rows[c] + r, len = A.h_rpb[R + 1] - A.h_rpb[R];
        const int64_t lo = (int64_t)bs2 * (A.h_rpb[R] - cb0);
        for (int j = 0; j < nd; ++j)
          for (int e = 0; e < bs; ++e) {
            const int64_t b = (lo + e * A.bs1 * len + A.bs1 * x.kk[j]) & 31;
            S.at[j * bs + e] = &S.load[((size_t)(j * bs + e) * 32 + b) * NB];
          }
        for (int h = 0; h < NB; h += 32) {
          const int v = std::min(4, (NB - h) / 8);
          (v == 1 ? add_up<1> : v == 2 ? add_up<2> : v == 3 ? add_up<3> : add_up<4>)(&S.meet[h], S.at.data(), nd * bs, &S.load[(size_t)nd * bs * 32 * NB], h);
        }
        int best = -1, least = INT32_MAX;
        for (int h = 0; h < nb; ++h)
          if (S.meet[h] < least) {
            least = S.meet[h];
            best = h;
          }
        for (uint16_t* l : S.at) ++l[best];
        place[k] = kGroup * best + S.fill[best]++;
        // a full group looks worse than any other (at most nd * bs * kGroup = 512 meet)
        if (S.fill[best] == std::min(kGroup, np - kGroup * best)) S.load[(size_t)nd * bs * 32 * NB + best] = 1024;
      }
  };
  auto work = [&](unsigned t) {
    std::vector<Pair> P;
    std::vector<int32_t> place, turn;
    Scratch S;
    for (int64_t c = t; c < nch; c += nt) {
      P.clear();
      turn.assign(with_kk ? static_cast<size_t>(rows[c + 1] - rows[c]) * nd : 0, 0);
      int64_t p = poff[c];
      for (int32_t it = ci[c]; it < ci[c + 1]; ++it) {
        const int32_t cell = plan->h_cell[it];
        for (uint64_t msk = plan->h_mask[it]; msk; msk &= msk - 1) {
          const int i = __builtin_ctzll(msk);
          const int32_t R = d0->host[(int64_t)cell * nd + i];
          const int32_t* rb = A.h_colsb.data() + A.h_rpb[R];
          const int32_t* re = A.h_colsb.data() + A.h_rpb[R + 1];
          if (with_kk) {
            P.push_back({cell, i, R - rows[c], turn[(size_t)(R - rows[c]) * nd + i]++, {}});
            continue;
          }
          for (int j = 0; j < nd; ++j) {
            const int32_t Cn = d1->host[(int64_t)cell * nd + j];
            const int32_t* f = std::lower_bound(rb, re, Cn);
            const bool ok = f != re && *f == Cn && f - rb <= 65535;
            if (!ok) bad[t % 16] = 1;
            ppos[p * nd + j] = ok ? static_cast<uint16_t>(f - rb) : 0;
          }
          // hexahedral kernel: item in the chunk << 16 | row in the chunk << 6 | local row
          plist[p++] = ((it - ci[c]) << 16) | ((R - rows[c]) << 6) | i;
        }
      }
      if (!with_kk) continue;
      // the pairs by row, and a row's column positions for all its pairs from one
      // pass over its columns (a search per pair and column took 40% of the time)
      const int nr = rows[c + 1] - rows[c];
      S.first.assign(nr + 1, 0);
      for (auto& x : P) ++S.first[x.row + 1];
      for (int r = 0; r < nr; ++r) S.first[r + 1] += S.first[r];
      S.order.resize(P.size());
      S.fill.assign(nr, 0);
      for (size_t k = 0; k < P.size(); ++k)
        S.order[S.first[P[k].row] + S.fill[P[k].row]++] = static_cast<int32_t>(k);
      if (S.where.empty()) S.where.assign(d1->num_nodes, 0);
      for (int r = 0; r < nr; ++r) {
        const int32_t* rb = A.h_colsb.data() + A.h_rpb[rows[c] + r];
        const int32_t len = A.h_rpb[rows[c] + r + 1] - A.h_rpb[rows[c] + r];
        for (int32_t q = 0; q < len; ++q) S.where[rb[q]] = q;
        for (int32_t a = S.first[r]; a < S.first[r + 1]; ++a) {
          Pair& x = P[S.order[a]];
          for (int j = 0; j < nd; ++j) {
            const int32_t Cn = d1->host[(int64_t)x.cell * nd + j], q = S.where[Cn];
            const bool ok = q < len && rb[q] == Cn && q <= 255;
            if (!ok) bad[t % 16] = 1;
            x.kk[j] = ok ? static_cast<uint8_t>(q) : 0;
          }
        }
      }
      if (nd > 4) {
        order_pairs(P, c, place, S);
      } else {
        place.resize(P.size());
        std::iota(place.begin(), place.end(), 0);
      }
      uint8_t* kkc = pkk.data() + kkoff[c];
      for (size_t k = 0; k < P.size(); ++k) {
        // simplex kernel (column offsets precomputed): cell id << 6 | local row
        const int64_t q = place[k];
        plist[poff[c] + q] = static_cast<int32_t>((static_cast<uint32_t>(P[k].cell) << 6) | P[k].i);
        prow[poff[c] + q] = static_cast<uint16_t>(P[k].row);
        std::copy_n(P[k].kk, nd, &kkc[q * nd]);
      }
    }
  };
  std::vector<std::thread> th;
  for (unsigned t = 0; t < nt; ++t) th.emplace_back(work, t);
  for (auto& t : th) t.join();
  for (int v : bad)
    if (v) return nullptr;   // entry missing from the pattern or row too long for 8-bit offsets
  std::vector<int32_t> meta(12 * nch, 0);
  for (int64_t c = 0; c < nch; ++c) {
    const int32_t q0 = rows[c], q1 = rows[c + 1];
    const int64_t cb0 = A.h_rpb[q0], cb1 = A.h_rpb[q1];
    const int64_t base = (int64_t)bs2 * cb0;
    MF_CHECK(base + (int64_t)bs2 * (cb1 - cb0) < INT32_MAX, MF_EUNSUPPORTED, "CSR offset overflow");
    int32_t* mc = &meta[12 * c];
    mc[0] = q0; mc[1] = q1; mc[2] = ci[c]; mc[3] = ci[c + 1];
    mc[4] = static_cast<int32_t>(cb0); mc[5] = static_cast<int32_t>(cb1 - cb0);
    mc[6] = static_cast<int32_t>(base); mc[7] = static_cast<int32_t>(bs2 * (cb1 - cb0));
    mc[8] = static_cast<int32_t>(poff[c]); mc[9] = static_cast<int32_t>(poff[c + 1]);
    mc[10] = static_cast<int32_t>(kkoff[c]);
  }
  if (!with_kk) {
    plan->item_cell.upload(plan->h_cell);
    const mf_mesh& M = *a.mesh;
    std::vector<int32_t> geo(M.num_cells * M.nv), ig((plan->nitems + 1) * M.nv, 0);
    MF_HIP(hipMemcpy(geo.data(), M.cells.ptr, sizeof(int32_t) * geo.size(), hipMemcpyDeviceToHost));
    for (int64_t it = 0; it < plan->nitems; ++it)
      std::copy_n(&geo[(int64_t)plan->h_cell[it] * M.nv], M.nv, &ig[it * M.nv]);
    plan->item_geo.upload(ig);
  }
  plan->chunk_meta.upload(meta);
  plan->pair_list.upload(plist);
  plan->pair_kk.upload(pkk);
  plan->pair_row.upload(prow);
  plan->pair_pos.upload(ppos);
  {
    // position of the diagonal block in each blocked row (-1: none): the
    // Dirichlet diagonal of the owner kernels
    std::vector<int32_t> dp(std::max<int64_t>(1, A.nrows_b), -1);
    for (int64_t R = 0; R < A.nrows_b; ++R) {
      const int32_t* rb = A.h_colsb.data() + A.h_rpb[R];
      const int32_t* re = A.h_colsb.data() + A.h_rpb[R + 1];
      const int32_t* f = std::lower_bound(rb, re, static_cast<int32_t>(R));
      if (f != re && *f == R) dp[R] = static_cast<int32_t>(f - rb);
    }
    plan->diag_pos.upload(dp);
  }
  plan->npairs = np;
  plan->drop_host();
  return plan;
}

}  // namespace

std::shared_ptr<OwnerPlan> vector_plan(mf_form* L, Integral& I) {
  auto it = L->vplans.find(I.index);
  if (it != L->vplans.end()) return it->second;
  const mf_dofmap* d0 = L->dm[0];
  std::shared_ptr<OwnerPlan> plan;
  if (d0->nd <= 32) {
    const int64_t per = std::max<int64_t>(1, vector_chunk(*L) / d0->bs);
    std::vector<int32_t> rows;
    for (int64_t r = 0; r < d0->num_nodes; r += per) rows.push_back(static_cast<int32_t>(r));
    rows.push_back(static_cast<int32_t>(d0->num_nodes));
    plan = build_items(rows, I, d0);
    plan->chunk_rows.upload(rows);
    plan->chunk_items.upload(plan->h_items);
    plan->item_cell.upload(plan->h_cell);
    std::vector<uint32_t> m32(plan->h_mask.begin(), plan->h_mask.end());   // 32 nodes at most
    plan->item_mask.upload(m32);
    plan->drop_host();
  }
  L->vplans[I.index] = plan;
  return plan;
}

// Whether blocks of cells (mf_vblk_*) beat the row-owning kernel (mf_vown_*).
// The blocks cost a cleared vector (2.3 us of launch) and their atomics; the
// other repeats cells, which weighs what the body weighs, and the registers it
// needs tell light from heavy bodies.  Cell integral in us, rows / blocks:
//   under 100 registers, line at 300 thousand cells: P1 105 thousand 5.8 / 5.9,
//     384 thousand 12.1 / 7.5; P2 118 thousand 8.4 / 8.8, 280 thousand 15.4 / 14.2;
//     vector P1 216 thousand 9.9 / 9.6; vector P2 280 thousand 24.6 / 25.6, 384
//     thousand 34.7 / 31.0;
//   to 160 registers, 300 cells: P1 residual with 27 points 162 cells 7.9 / 8.9, 384
//     cells 13.2 / 8.9; P3 source (104) 6 cells 9.0 / 6.0, 384 cells 10.8 / 7.7, 83
//     thousand 23.3 / 13.9;
//   above, 9 thousand: P2 residual with 64 points (242) 1.3 thousand 37 / 43, 8.0
//     thousand 37.4 / 40.4, 10.4 thousand 58 / 41, 48 thousand 97 / 48.
// Cells of more than 32 nodes have no row-owning kernel: Q3 source on 14
// thousand hexahedra 50 us, 78 us with one atomic per row, 14 us with a wave per
// cell (mf_hsrc_*).
static bool blocks_pay(const mf_form& L, Integral& I) {
  if (I.k_hsrc || !I.k_vown) return true;
  if (L.options.count("vector_chunk_values") || L.options.count("vector_block")) return false;
  if (I.vown_regs == 0) {
    int regs = 0;
    MF_HIP(hipFuncGetAttribute(&regs, HIP_FUNC_ATTRIBUTE_NUM_REGS, I.k_vown));
    I.vown_regs = std::max(1, regs);
  }
  return I.n >= (I.vown_regs < 100 ? 300000 : I.vown_regs < 160 ? 300 : 9000);
}

// The distinct rows among row[0 .. n), appended to `rows` in ascending order, and
// the place of each among them.  By a bitmap over the rows' range where that is
// no longer than the list (entities that lie together have rows that do), else
// by sorting.
struct RowRanks {
  std::vector<uint64_t> bits;
  std::vector<int32_t> before, seen;
  void operator()(const int32_t* row, size_t n, std::vector<int32_t>& rows, uint16_t* place) {
    if (n == 0) return;
    const auto ends = std::minmax_element(row, row + n);
    const int64_t lo = *ends.first, words = (*ends.second - lo) / 64 + 1;
    if (words > static_cast<int64_t>(n)) {
      seen.assign(row, row + n);
      std::sort(seen.begin(), seen.end());
      seen.erase(std::unique(seen.begin(), seen.end()), seen.end());
      for (size_t p = 0; p < n; ++p)
        place[p] = static_cast<uint16_t>(std::lower_bound(seen.begin(), seen.end(), row[p]) - seen.begin());
      rows.insert(rows.end(), seen.begin(), seen.end());
      return;
    }
    bits.assign(words, 0);
    before.resize(words);
    for (size_t p = 0; p < n; ++p) bits[(row[p] - lo) / 64] |= uint64_t(1) << ((row[p] - lo) % 64);
    int32_t count = 0;
    for (int64_t w = 0; w < words; ++w) {
      before[w] = count;
      count += __builtin_popcountll(bits[w]);
      for (uint64_t b = bits[w]; b; b &= b - 1) rows.push_back(static_cast<int32_t>(lo + 64 * w + __builtin_ctzll(b)));
    }
    for (size_t p = 0; p < n; ++p) {
      const int64_t d = row[p] - lo;
      place[p] = static_cast<uint16_t>(before[d / 64] + __builtin_popcountll(bits[d / 64] & ((uint64_t(1) << (d % 64)) - 1)));
    }
  }
};

// f(begin, end, t) over parts t = 0, 1, ... of [0, n), on threads of their own
// where a part gets at least `grain` (on this one where no thread is to be had);
// returns the number of parts.  What a part throws is thrown here.
template <class F>
static int in_parts(int64_t n, int64_t grain, const F& f) {
  const int64_t cpus = std::max(1u, std::thread::hardware_concurrency());
  const int parts = static_cast<int>(std::max<int64_t>(1, std::min({int64_t(8), cpus, n / grain})));
  std::exception_ptr failed[8];
  auto part = [&](int t) {
    try {
      f(n * t / parts, n * (t + 1) / parts, t);
    } catch (...) {
      failed[t] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(parts);
  for (int t = 1; t < parts; ++t) {
    try {
      th.emplace_back(part, t);
    } catch (const std::system_error&) {
      part(t);
    }
  }
  part(0);
  for (auto& x : th) x.join();
  for (auto& e : failed)
    if (e) std::rethrow_exception(e);
  return parts;
}

// Rows of consecutive blocks: row(k, out) gives the rows of block k's entries, in
// order, place[at(k) ..] gets their places among its distinct rows, and ptr and rows
// get the blocks' distinct rows one after the other.
template <class Row>
static void rank_blocks(int64_t nblk, int64_t grain, const Row& row, const std::function<int64_t(int64_t)>& at,
                        std::vector<uint16_t>& place, std::vector<int32_t>& ptr, std::vector<int32_t>& rows) {
  std::vector<std::vector<int32_t>> part(8);
  ptr.assign(nblk + 1, 0);
  const int parts = in_parts(nblk, grain, [&](int64_t k0, int64_t k1, int t) {
    RowRanks rank;
    std::vector<int32_t> entries;
    for (int64_t k = k0; k < k1; ++k) {
      entries.clear();
      row(k, entries);
      const size_t before = part[t].size();
      rank(entries.data(), entries.size(), part[t], place.data() + at(k));
      ptr[k + 1] = static_cast<int32_t>(part[t].size() - before);
    }
  });
  for (int64_t k = 0; k < nblk; ++k) ptr[k + 1] += ptr[k];
  for (int t = 0; t < parts; ++t) rows.insert(rows.end(), part[t].begin(), part[t].end());
}

// Blocks of at most 256 entities (down to 64 where that leaves fewer than
// three blocks per CU) whose rows fit 64 KB of LDS; null when rows are shared so
// little that the blocks hold fewer than half their entities.  With a wave per
// cell 32 cells (down to 4) and 32 KB, in blocks of 256 threads.  Null also where
// they do not exist yet and s is being captured: the kernels that need no
// schedule serve then.
static VectorBlocks* vector_blocks(mf_form* L, const Integral& I, hipStream_t s) {
  auto it = L->vblocks.find(I.index);
  if (it != L->vblocks.end()) return it->second.get();
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  MF_HIP(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone) return nullptr;
  const mf_dofmap* d0 = L->dm[0];
  const int nd = d0->nd, bs = d0->bs;
  auto B = std::make_unique<VectorBlocks>();
  int most = I.k_hsrc ? kHexSourceCells : 256;
  while (most > (I.k_hsrc ? 4 : 64) && I.n < 3LL * L->ctx->num_cus * most) most /= 2;
  B->threads = I.k_hsrc ? 256 : most;
  const size_t cap = (I.k_hsrc ? 4096 : 8192) / bs;      // nodes per block
  std::vector<int32_t> ent{0}, ptr, row;
  std::vector<uint16_t> slot(static_cast<size_t>(I.n) * nd);
  if (static_cast<size_t>(most) * nd <= cap) {
    for (int64_t e = most; e < I.n + most; e += most) ent.push_back(static_cast<int32_t>(std::min(e, I.n)));
  } else {
    std::vector<int32_t> seen(d0->num_nodes, -1);          // the last block with the node
    for (int64_t e = 0; e < I.n;) {
      const int64_t e0 = e;
      const int32_t blk = static_cast<int32_t>(ent.size());
      size_t nodes = 0;
      for (; e < I.n && e - e0 < most; ++e) {
        const int32_t* dm = &d0->host[(int64_t)I.h_ents[e] * nd];
        for (int i = 0; i < nd; ++i)
          if (seen[dm[i]] != blk) {
            seen[dm[i]] = blk;
            ++nodes;
          }
        if (nodes > cap) break;                            // this entity starts the next block
      }
      if (e == e0) return (L->vblocks[I.index] = nullptr).get();   // one entity's rows exceed a block
      ent.push_back(static_cast<int32_t>(e));
    }
  }
  rank_blocks(static_cast<int64_t>(ent.size()) - 1, std::max(1, 20000 / (most * nd)),
              [&](int64_t k, std::vector<int32_t>& out) {
                for (int32_t q = ent[k]; q < ent[k + 1]; ++q) {
                  const int32_t* dm = &d0->host[(int64_t)I.h_ents[q] * nd];
                  out.insert(out.end(), dm, dm + nd);
                }
              },
              [&](int64_t k) { return (int64_t)ent[k] * nd; }, slot, ptr, row);
  for (size_t k = 0; k + 1 < ptr.size(); ++k)
    B->lds = std::max(B->lds, static_cast<uint32_t>(8 * bs * (ptr[k + 1] - ptr[k])));
  B->n = static_cast<int64_t>(ent.size()) - 1;
  if (!I.k_hsrc && B->n * most > 2 * std::max<int64_t>(I.n, most)) return (L->vblocks[I.index] = nullptr).get();
  B->ent.upload(ent);
  B->ptr.upload(ptr);
  B->row.upload(row);
  B->slot.upload(slot);
  return (L->vblocks[I.index] = std::move(B)).get();
}

LiftList build_lift_list(const mf_form& f, const Integral& I, const mf_bc& bc, hipStream_t s) {
  const mf_dofmap* d0 = f.dm[0];
  const mf_dofmap* d1 = f.dm[1];
  LiftList L;
  DevArray<int32_t> cnt;
  L.list.alloc(std::max<int64_t>(1, I.n));
  cnt.alloc(1);
  k_fill_i32(cnt.ptr, 1, 0, s);
  k_lift_list(L.list.ptr, cnt.ptr, I.d_ents.ptr, I.n, entity_stride(I.type), entity_ncell(I.type),
              d1->dev.ptr, d1->nd, d1->bs, bc.markers.ptr, s);
  int32_t n = 0;
  MF_HIP(hipMemcpyAsync(&n, cnt.ptr, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  MF_HIP(hipStreamSynchronize(s));
  L.n = n;
  if (n == 0) return L;
  std::vector<int32_t> list(n);
  MF_HIP(hipMemcpy(list.data(), L.list.ptr, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
  {                                              // the kernel appends in no particular order
    std::vector<uint64_t> in(I.n / 64 + 1, 0);
    for (int32_t e : list) in[e / 64] |= uint64_t(1) << (e % 64);
    size_t k = 0;
    for (size_t w = 0; w < in.size(); ++w)
      for (uint64_t b = in[w]; b; b &= b - 1) list[k++] = static_cast<int32_t>(64 * w + __builtin_ctzll(b));
  }
  L.list.upload(list);
  const int nd = d0->nd, bs1 = d1->bs;
  if (!I.k_slift || d1->nd * bs1 > 64 || (int64_t)n * nd >= INT32_MAX) return L;
  std::vector<uint8_t> constrained(d1->num_nodes * bs1, 0);
  for (int32_t d : bc.h_dofs) constrained[d] = 1;
  std::vector<uint64_t> mask(n, 0);
  in_parts(n, 2000, [&](int64_t k0, int64_t k1, int) {
    for (int64_t k = k0; k < k1; ++k) {
      const int64_t c = I.h_ents[list[k]];
      uint64_t m = 0;
      for (int j = 0; j < d1->nd * bs1; ++j) {
        const int64_t node = d1->host[c * d1->nd + j / bs1];
        m |= static_cast<uint64_t>(constrained[bs1 * node + j % bs1]) << j;
      }
      mask[k] = m;
    }
  });
  // row of every (cell, local row), in the order the kernel visits them: by cell,
  // or sorted by row
  const bool by_cell = staged_trace(I);
  const int64_t entries = (int64_t)n * nd;
  std::vector<int32_t> row;
  if (!by_cell) {
    row.resize(entries);
    std::vector<int32_t> start(d0->num_nodes + 1, 0), pairs(row.size());
    for (int32_t k = 0; k < n; ++k)
      for (int i = 0; i < nd; ++i) start[d0->host[(int64_t)I.h_ents[list[k]] * nd + i] + 1]++;
    for (int64_t r = 0; r < d0->num_nodes; ++r) start[r + 1] += start[r];
    for (int32_t k = 0; k < n; ++k)
      for (int i = 0; i < nd; ++i) {
        const int32_t r = d0->host[(int64_t)I.h_ents[list[k]] * nd + i];
        row[start[r]] = r;
        pairs[start[r]++] = k * nd + i;
      }
    L.pairs.upload(pairs);
  }
  const int64_t per = by_cell ? 64 * nd : 128;           // contributions per workgroup
  std::vector<int32_t> ptr, rows;
  std::vector<uint16_t> slot(entries);
  rank_blocks((entries + per - 1) / per, std::max<int64_t>(1, 20000 / per),
              [&](int64_t b, std::vector<int32_t>& out) {
                const int64_t p1 = std::min(entries, (b + 1) * per);
                if (!by_cell) {
                  out.insert(out.end(), row.begin() + b * per, row.begin() + p1);
                  return;
                }
                for (int64_t k = b * 64; k * nd < p1; ++k) {
                  const int32_t* dm = &d0->host[(int64_t)I.h_ents[list[k]] * nd];
                  out.insert(out.end(), dm, dm + nd);
                }
              },
              [&](int64_t b) { return b * per; }, slot, ptr, rows);
  L.slot.upload(slot);
  L.blk_ptr.upload(ptr);
  L.blk_row.upload(rows);
  L.mask.upload(mask);
  return L;
}

void staged_lift_shape(const mf_form& f, const Integral& I, int64_t n, uint32_t* grid, uint32_t* block) {
  // 64 cells by four waves of rows, or 128 (cell, row) pairs per workgroup
  const bool by_cell = staged_trace(I);
  *block = by_cell ? 256 : 128;
  *grid = static_cast<uint32_t>(by_cell ? (n + 63) / 64 : (n * f.dm[0]->nd + 127) / 128);
}

namespace {

DevArray<int32_t>& get_table(mf_form* a, Integral& I, mf_matrix* A, hipStream_t s) {
  auto key = std::make_pair(a->uid, I.index);
  auto it = A->tables.find(key);
  if (it != A->tables.end()) return it->second;
  const int ncell = entity_ncell(I.type);
  const int ni = ncell * a->dm[0]->nd, nj = ncell * a->dm[1]->nd;
  const int64_t padded = (I.n + kTableLanes - 1) / kTableLanes * kTableLanes;
  DevArray<int32_t> t;
  t.alloc(std::max<int64_t>(1, padded * ni * nj));
  DevArray<int32_t> missing;
  missing.alloc(1);
  k_fill_i32(missing.ptr, 1, 0, s);
  k_build_table(t.ptr, I.d_ents.ptr, I.n, entity_stride(I.type), ncell, a->dm[0]->dev.ptr,
                a->dm[0]->nd, a->dm[1]->dev.ptr, a->dm[1]->nd, A->bs0, A->bs1, A->row_ptr.ptr,
                A->rpb.ptr, A->colsb.ptr, missing.ptr, s);
  int32_t h_missing = 0;
  MF_HIP(hipMemcpyAsync(&h_missing, missing.ptr, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  MF_HIP(hipStreamSynchronize(s));
  MF_CHECK(h_missing == 0, MF_ENOTFOUND,
           std::to_string(h_missing) + " element entries are missing from the sparsity pattern");
  return A->tables.emplace(key, std::move(t)).first->second;
}

}  // namespace

// Gather plan of one integral (built once per matrix, on the device but for
// the prefix sum), null when the workspace would exceed 4 GiB (its offsets are
// int32, and one matrix holds it for good), when memory is short, when one entry
// sums too many contributions, or when it does not exist yet and s is being captured: the per-entity kernel with its offset table serves then.
// That table is built along, so that any uncaptured call leaves what a captured
// one may need, overwriting or adding.
static GatherPlan* gather_plan(mf_form* a, Integral& I, mf_matrix* A, hipStream_t s) {
  const auto key = std::make_pair(a->uid, I.index);
  auto it = A->gathers.find(key);
  if (it != A->gathers.end()) return it->second.get();
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  MF_HIP(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone) return nullptr;
  const mf_dofmap* d0 = a->dm[0];
  const mf_dofmap* d1 = a->dm[1];
  const int ncell = entity_ncell(I.type), ni = ncell * d0->nd, nj = ncell * d1->nd;
  const int64_t planes = (int64_t)ni * d0->bs * nj * d1->bs, ws = (I.n + 63) / 64 * 64 * planes;
  if (ws > (int64_t(1) << 29) || I.n * ni * nj >= INT32_MAX) return A->gathers[key].get();
  get_table(a, I, A, s);
  auto g = std::make_unique<GatherPlan>();
  DevArray<int32_t> count, missing;
  g->ws = A->gather_ws;
  if (!g->ws || g->ws->n < ws) g->ws = std::make_shared<DevArray<double>>();
  if (!(g->ws->n >= ws || g->ws->try_alloc(std::max<int64_t>(1, ws))) ||
      !g->at.try_alloc(std::max<int64_t>(1, I.n * ni * nj)) ||      // one place per contribution
      !g->pos.try_alloc(std::max<int64_t>(1, A->nnz_b)) || !g->ptr.try_alloc(A->nnz_b + 1) ||
      !count.try_alloc(std::max<int64_t>(1, A->nnz_b)))
    return (A->gathers[key] = nullptr).get();
  missing.alloc(1);
  k_fill_i32(count.ptr, A->nnz_b, 0, s);
  k_fill_i32(missing.ptr, 1, 0, s);
  auto pass = [&](int32_t* fill) {
    k_gather_plan(count.ptr, fill, I.d_ents.ptr, I.n, entity_stride(I.type), ncell, d0->dev.ptr,
                  d0->nd, d1->dev.ptr, d1->nd, d0->bs, d1->bs, A->rpb.ptr, A->colsb.ptr, missing.ptr, s);
  };
  pass(nullptr);
  std::vector<int32_t> ptr(A->nnz_b + 1, 0);
  int32_t h_missing = 0;
  MF_HIP(hipMemcpyAsync(ptr.data(), count.ptr, sizeof(int32_t) * A->nnz_b, hipMemcpyDeviceToHost, s));
  MF_HIP(hipMemcpyAsync(&h_missing, missing.ptr, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  MF_HIP(hipStreamSynchronize(s));
  MF_CHECK(h_missing == 0, MF_ENOTFOUND,
           std::to_string(h_missing) + " element entries are missing from the sparsity pattern");
  // An entry's contributions are put in order and summed by one thread, about 0.09 us
  // each here, which a gather saves per 3,300 element entries against adding each
  // with an atomic (P1 10^3 cubes: equal at 72 contributions to one entry, 20^3 at
  // 256, 30^3 at 780; the ordering is quadratic, 21 ms for 1,540).  Most meshes have
  // at most 32; a node that every cell shares sends the integral to the per-entity
  // kernel.
  const int32_t most = A->nnz_b ? *std::max_element(ptr.begin(), ptr.end()) : 0;
  if (most > std::min<int64_t>(1024, 32 + I.n * ni * nj / 3300)) return (A->gathers[key] = nullptr).get();
  int32_t sum = 0;
  for (int64_t q = 0; q <= A->nnz_b; ++q) {
    const int32_t c = ptr[q];
    ptr[q] = sum;
    sum += c;
  }
  MF_HIP(hipMemcpy(g->ptr.ptr, ptr.data(), sizeof(int32_t) * ptr.size(), hipMemcpyHostToDevice));
  MF_HIP(hipMemcpyAsync(count.ptr, g->ptr.ptr, sizeof(int32_t) * A->nnz_b, hipMemcpyDeviceToDevice, s));
  pass(g->at.ptr);
  k_gather_sort(g->at.ptr, g->ptr.ptr, g->pos.ptr, A->nnz_b, A->nrows_b, A->rpb.ptr, A->row_ptr.ptr,
                d0->bs, d1->bs, s);
  MF_HIP(hipStreamSynchronize(s));                     // count and missing are freed here
  A->gather_ws = g->ws;
  return (A->gathers[key] = std::move(g)).get();
}

// ---------------------------------------------------------------------------
// Cell-owner schedule for discontinuous spaces (kernel: dg_kernel.cpp)
// ---------------------------------------------------------------------------

// The test space must number dofs cell by cell (node(c, i) = c * nd + i) so a
// cell's CSR rows are its own.  With a matrix, each item also carries the
// block positions of the owner and the neighbour inside the owner's rows.
std::shared_ptr<DGPlan> build_dg_plan(const mf_form& f, const mf_matrix* A) {
  const mf_dofmap* d = f.dm[0];
  const int nd = d->nd;
  const int64_t nc = d->num_cells;
  if (f.rank == 2 && f.dm[1] != d) return nullptr;
  if (d->num_nodes != nc * nd) return nullptr;
  for (int64_t k = 0; k < nc * nd; ++k)
    if (d->host[k] != k) return nullptr;
  std::vector<int64_t> count(nc + 1, 0);
  for (auto& I : f.ints) {
    const int st = entity_stride(I->type);
    for (int64_t e = 0; e < I->n; ++e) {
      count[I->h_ents[e * st] + 1]++;
      if (I->type == MF_INTERIOR_FACET) count[I->h_ents[e * st + 2] + 1]++;
    }
  }
  for (int64_t c = 0; c < nc; ++c) count[c + 1] += count[c];
  const int64_t nitems = count[nc];
  MF_CHECK(nitems < (int64_t(1) << 31), MF_EUNSUPPORTED, "too many cell items");
  std::vector<int32_t> items(4 * std::max<int64_t>(nitems, 1), 0);
  std::vector<int64_t> pos(count.begin(), count.end() - 1);
  auto push = [&](int64_t c, int32_t k, int32_t other, int32_t lfs, int32_t lfo, int32_t side) {
    int32_t* it = &items[4 * pos[c]++];
    it[0] = k; it[1] = other; it[2] = lfs | (lfo << 8); it[3] = side;
  };
  for (auto& I : f.ints) {
    const int st = entity_stride(I->type);
    for (int64_t e = 0; e < I->n; ++e) {
      const int32_t* en = &I->h_ents[e * st];
      if (I->type == MF_CELL) push(en[0], I->index, -1, 0, 0, 0);
      else if (I->type == MF_EXTERIOR_FACET) push(en[0], I->index, -1, en[1], 0, 0);
      else {
        push(en[0], I->index, en[2], en[1], en[3], 0);
        push(en[2], I->index, en[0], en[3], en[1], 1);
      }
    }
  }
  if (A) {
    // block positions in the owner's rows; each neighbour block must have one source
    std::vector<int32_t> seen;
    for (int64_t c = 0; c < nc; ++c) {
      if (count[c] == count[c + 1]) continue;
      const int64_t R = c * nd;
      const int32_t* cb = A->h_colsb.data() + A->h_rpb[R];
      const int64_t len = A->h_rpb[R + 1] - A->h_rpb[R];
      if (len % nd) return nullptr;
      auto block_of = [&](int64_t cell) -> int {
        const int32_t key = static_cast<int32_t>(cell * nd);
        const int32_t* p = std::lower_bound(cb, cb + len, key);
        if (p == cb + len || *p != key || (p - cb) % nd) return -1;
        return static_cast<int>((p - cb) / nd);
      };
      const int ps = block_of(c);
      if (ps < 0 || ps > 0xFFF) return nullptr;
      seen.clear();
      for (int64_t t = count[c]; t < count[c + 1]; ++t) {
        int32_t* it = &items[4 * t];
        int po = 0;
        if (it[1] >= 0) {
          po = block_of(it[1]);
          if (po < 0 || po > 0xFFF || po == ps) return nullptr;
          if (std::find(seen.begin(), seen.end(), po) != seen.end()) return nullptr;
          seen.push_back(po);
        }
        it[3] |= (ps << 4) | (po << 16);
      }
      if (len / nd != 1 + static_cast<int64_t>(seen.size())) return nullptr;   // unwritten blocks
    }
  }
  auto plan = std::make_shared<DGPlan>();
  std::vector<int32_t> cp(nc + 1);
  for (int64_t c = 0; c <= nc; ++c) cp[c] = static_cast<int32_t>(count[c]);
  plan->cell_ptr.upload(cp.data(), nc + 1);
  plan->items.upload(items.data(), items.size());
  plan->ncells = nc;
  plan->nitems = nitems;
  return plan;
}

namespace {

DevArray<int32_t>& get_block_table(mf_form* a, Integral& I, mf_matrix* A, hipStream_t s) {
  auto key = std::make_pair(a->uid, I.index);
  auto it = A->tables.find(key);
  if (it != A->tables.end()) return it->second;
  const int ncell = entity_ncell(I.type);
  const int ni = ncell * a->dm[0]->nd, nj = ncell * a->dm[1]->nd;
  const int64_t padded = (I.n + kTableLanes - 1) / kTableLanes * kTableLanes;
  DevArray<int32_t> t;
  t.alloc(std::max<int64_t>(1, padded * ni * nj));
  DevArray<int32_t> missing;
  missing.alloc(1);
  k_fill_i32(missing.ptr, 1, 0, s);
  k_build_block_table(t.ptr, I.d_ents.ptr, I.n, entity_stride(I.type), ncell, a->dm[0]->dev.ptr,
                      a->dm[0]->nd, a->rmap[0].ptr, a->roff[0], a->dm[0]->bs, a->dm[1]->dev.ptr,
                      a->dm[1]->nd, a->rmap[1].ptr, a->roff[1], a->dm[1]->bs, A->row_ptr.ptr,
                      A->cols.ptr, missing.ptr, s);
  int32_t h_missing = 0;
  MF_HIP(hipMemcpyAsync(&h_missing, missing.ptr, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  MF_HIP(hipStreamSynchronize(s));
  MF_CHECK(h_missing == 0, MF_ENOTFOUND,
           std::to_string(h_missing) + " element entries are missing from the block pattern");
  return A->tables.emplace(key, std::move(t)).first->second;
}

// Block member form into a monolithic block matrix (CUDAAssembler's
// assemble_matrix on a restricted CUDAForm; python/cudolfinx/assemble.py:112-134
// calls it per block with zero=False): per-entity kernels with the row node
// map and offset, offset tables against the scalar CSR; for a diagonal block
// the Dirichlet rows get `diagonal` at their global positions.
void assemble_block_matrix(mf_form* a, mf_matrix* A, const mf_bc* bc0, const mf_bc* bc1,
                           double diagonal, int zero, hipStream_t s) {
  MF_CHECK(A->block, MF_EINVAL, "a block/restricted form assembles into a block matrix");
  for (int ax = 0; ax < 2; ++ax) {
    const int64_t kept = a->h_rmap[ax].empty() ? a->dm[ax]->num_nodes : a->rcount[ax];
    MF_CHECK(a->roff[ax] + kept * a->dm[ax]->bs <= (ax == 0 ? A->nrows : A->ncols), MF_ESHAPE,
             "block form does not fit the matrix");
  }
  if (bc0) MF_CHECK(bc0->ndofs == a->dm[0]->num_nodes * a->dm[0]->bs, MF_ESHAPE,
                    "bc0 size does not match the block's test space");
  if (bc1) MF_CHECK(bc1->ndofs == a->dm[1]->num_nodes * a->dm[1]->bs, MF_ESHAPE,
                    "bc1 size does not match the block's trial space");
  const int8_t* m0 = bc0 && bc0->nbc ? bc0->markers.ptr : nullptr;
  const int8_t* m1 = bc1 && bc1->nbc ? bc1->markers.ptr : nullptr;
  if (zero) k_fill(A->values, A->nnz, 0.0, s);
  const uint32_t block = static_cast<uint32_t>(a->opt("block", 128));
  for (auto& I : a->ints) {
    if (I->n == 0) continue;
    auto& table = get_block_table(a, *I, A, s);
    launch(I->k_mat, static_cast<uint32_t>((I->n + block - 1) / block), block, 0, s,
           static_cast<int32_t>(I->n), I->d_ents.ptr, a->mesh->cells.ptr, a->mesh->x.ptr,
           a->packed.ptr, a->consts.ptr, a->dm[0]->dev.ptr, a->dm[1]->dev.ptr, m0, m1,
           table.ptr, A->row_ptr.ptr, A->values, a->mesh->fperm.ptr,
           static_cast<const int32_t*>(a->rmap[0].ptr), static_cast<int64_t>(a->roff[0]));
  }
  const bool diag_block = a->dm[0] == a->dm[1] && a->h_rmap[0] == a->h_rmap[1] &&
                          a->roff[0] == a->roff[1];
  if (diag_block && m0 && bc0->n_owned) {
    auto it = a->block_diag_rows.find(bc0->key);
    if (it == a->block_diag_rows.end()) {
      const int bs = a->dm[0]->bs;
      std::vector<int32_t> rows;
      for (int64_t k = 0; k < bc0->n_owned; ++k) {
        const int32_t d = bc0->h_dofs[k], node = d / bs;
        const int32_t m = a->h_rmap[0].empty() ? node : a->h_rmap[0][node];
        if (m >= 0) rows.push_back(static_cast<int32_t>(a->roff[0] + (int64_t)bs * m + d % bs));
      }
      DevArray<int32_t> dr;
      dr.upload(rows.empty() ? std::vector<int32_t>{0} : rows);
      dr.n = static_cast<int64_t>(rows.size());
      it = a->block_diag_rows.emplace(bc0->key, std::move(dr)).first;
    }
    if (it->second.n)
      k_set_diagonal(A->values, A->row_ptr.ptr, A->cols.ptr, it->second.ptr, it->second.n,
                     A->nrows, diagonal, s);
  }
}

}  // namespace

void assemble_matrix(mf_form* a, mf_matrix* A, const mf_bc* bc0, const mf_bc* bc1,
                     double diagonal, int zero, hipStream_t s) {
  MF_CHECK(a->rank == 2, MF_EINVAL, "assemble_matrix needs a bilinear form");
  MF_CHECK(a->compiled, MF_ESTATE, "form is not compiled");
  if (A->inner) {
    // adopted pattern without block structure: assemble on the form's own
    // pattern, then add into the caller's positions (extra entries stay 0)
    MF_CHECK(a == A->inner->form, MF_EUNSUPPORTED,
             "this adopted matrix assembles the form it was created for");
    assemble_matrix(a, A->inner.get(), bc0, bc1, diagonal, 1, s);
    if (zero) k_fill(A->values, A->nnz, 0.0, s);
    k_scatter_add(A->values, A->inner->values, A->inner_map.ptr, A->inner->nnz, s);
    return;
  }
  if (A->block || a->restricted) {
    assemble_block_matrix(a, A, bc0, bc1, diagonal, zero, s);
    return;
  }
  MF_CHECK(A->nrows == a->dm[0]->num_nodes * a->dm[0]->bs &&
               A->ncols == a->dm[1]->num_nodes * a->dm[1]->bs,
           MF_ESHAPE, "matrix shape does not match the form's spaces");
  const bool square = a->dm[0] == a->dm[1];
  if (bc0) MF_CHECK(bc0->ndofs == A->nrows, MF_ESHAPE, "bc0 size does not match the rows");
  if (bc1) MF_CHECK(bc1->ndofs == A->ncols, MF_ESHAPE, "bc1 size does not match the columns");
  const int8_t* m0 = bc0 && bc0->nbc ? bc0->markers.ptr : nullptr;
  const int8_t* m1 = bc1 && bc1->nbc ? bc1->markers.ptr : nullptr;
  const int64_t mode = a->opt("matrix_kernel", 0);

  // discontinuous spaces: one cell-owner launch over every integral
  if (a->k_dgown && (mode == 0 || mode == 3)) {
    auto it = A->dgplans.find(a->uid);
    std::shared_ptr<DGPlan> dp;
    if (it == A->dgplans.end()) {
      dp = build_dg_plan(*a, A);
      A->dgplans[a->uid] = dp;
    } else {
      dp = it->second;
    }
    if (dp) {
      int flags = zero ? 1 : 0;
      if (m0 && square) flags |= 2;
      const uint32_t blk = static_cast<uint32_t>(a->opt("dg_block", 64));
      launch(a->k_dgown, static_cast<uint32_t>((dp->ncells + blk - 1) / blk), blk, 0, s,
             static_cast<int32_t>(dp->ncells), dp->cell_ptr.ptr,
             reinterpret_cast<const int4*>(dp->items.ptr), a->mesh->cells.ptr, a->mesh->x.ptr,
             a->packed.ptr, a->consts.ptr, A->row_ptr.ptr, m0, m1, A->values, diagonal, flags,
             a->mesh->fperm.ptr);
      return;
    }
  }
  MF_CHECK(mode != 3, MF_EUNSUPPORTED, "cell-owner DG kernel unavailable for this form/matrix");

  // the first cell integral with a staged description may run owner-computes
  Integral* owner = nullptr;
  if (mode != 1)
    for (auto& I : a->ints)
      if (I->type == MF_CELL && (I->k_owner || I->k_hprep)) {
        owner = I.get();
        break;
      }
  std::shared_ptr<OwnerPlan> plan;
  if (owner) {
    // the matrix-core kernels of a hexahedral form have chunks of their own; every
    // kernel takes both schedules, and a captured call the one that exists
    const bool hex = owner->k_hprep != nullptr, mfma = hex && a->opt("precision", 64) != 64;
    const int second = static_cast<int>(a->ints.size());
    auto key = std::make_pair(a->uid, owner->index + (mfma ? second : 0));
    auto it = A->plans.find(key);
    auto usable = [&] { return it != A->plans.end() && it->second.first == a->gen; };
    if (hex && !usable()) {
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      MF_HIP(hipStreamIsCapturing(s, &cs));
      if (cs != hipStreamCaptureStatusNone)
        it = A->plans.find(std::make_pair(a->uid, owner->index + (mfma ? 0 : second)));
    }
    if (!usable()) {
      plan = build_owner_plan(*a, *owner, *A, a->opt("chunk_values", 4096),
                              static_cast<int>(a->opt("chunk_rows", 64)),
                              hex ? static_cast<int>(a->opt("owner_pairs", 384))
                                  : owner_shape(*a, *owner).maxp,
                              !hex, mfma);
      A->plans[key] = std::make_pair(a->gen, plan);
    } else {
      plan = it->second.second;
    }
    if (!plan) owner = nullptr;
  }
  MF_CHECK(!(mode == 2 && !owner), MF_EUNSUPPORTED,
           "owner-computes kernel requested but unavailable for this form/matrix");
  bool diag_done = false;
  if (owner && square && bc0 != bc1 && (m0 || m1)) owner = nullptr;   // records hold one bc
  MF_CHECK(owner || a->opt("precision", 64) == 64, MF_EUNSUPPORTED,
           "precision 32 / 16 runs on the owner-computes kernels only (same Dirichlet set on "
           "rows and columns)");
  MF_CHECK(!(mode == 2 && !owner), MF_EUNSUPPORTED,
           "owner-computes kernel needs the same Dirichlet set on rows and columns");
  if (owner) {
    const int bs = a->dm[0]->bs;
    const uint8_t* n0 = m0 ? bc0->bits_for(bs, s) : nullptr;
    int flags = zero ? 1 : 0;
    if (zero && m0) flags |= 2;
    diag_done = (flags & 2) != 0;
    const int64_t nx = 8, per = (plan->nchunks + nx - 1) / nx;
    if (owner->k_hprep) {
      const int64_t prec = a->opt("precision", 64);
      const int v = prec == 64 ? 0 : (prec == 32 ? 1 : 2);
      MF_CHECK(prec == 64 || prec == 32 || prec == 16, MF_EINVAL, "precision must be 64, 32 or 16");
      uint64_t* cmask = n0 ? reinterpret_cast<uint64_t*>(owner->records.ptr) : nullptr;
      if (cmask)
        launch(owner->k_hprep, static_cast<uint32_t>((owner->n + 3) / 4), 256, 0, s,
               static_cast<int32_t>(owner->n), owner->d_ents.ptr, a->dm[0]->dev.ptr, n0, cmask);
      const uint32_t hblock = static_cast<uint32_t>(hex_block(*a, static_cast<int>(prec)));
      int64_t& hgrid = owner->howner_grid[v];
      if (hgrid == 0) {
        int nblk = 0;
        MF_HIP(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nblk, owner->k_howner[v], hblock, 0));
        hgrid = std::max<int64_t>(nx, (int64_t)std::max(1, nblk) * a->ctx->num_cus / nx * nx);
      }
      const int64_t grid = a->opt("owner_persistent", 1) ? std::min(per * nx, hgrid) : per * nx;
      launch(owner->k_howner[v], static_cast<uint32_t>(grid), hblock, 0, s,
             static_cast<int32_t>(plan->nchunks), plan->chunk_meta.ptr, plan->item_cell.ptr,
             plan->item_geo.ptr, plan->pair_list.ptr, plan->pair_pos.ptr, a->mesh->x.ptr, cmask,
             A->rpb.ptr, plan->diag_pos.ptr, n0, A->values, diagonal, flags);
    } else {
    const uint8_t* cf = n0 ? bc0->cell_flags_for(a->dm[0], s) : nullptr;
    launch(owner->k_prep, static_cast<uint32_t>((owner->n + 255) / 256), 256, 0, s,
           static_cast<int32_t>(owner->n), owner->d_ents.ptr, a->mesh->cells.ptr, a->mesh->x.ptr,
           a->packed.ptr, a->dm[0]->dev.ptr, n0, cf, owner->records.ptr);
    // persistent grid: as many workgroups as fit on the device at once
    // (multiple of 8, one group of chunks per XCD); owner_persistent=0 gives
    // one workgroup per chunk
    const uint32_t oblock = static_cast<uint32_t>(a->opt("owner_block", 256));
    // precision 32: FP32 accumulation (scalar reference-tensor forms only)
    const int64_t prec = a->opt("precision", 64);
    MF_CHECK(prec == 64 || (prec == 32 && owner->k_owner32), MF_EUNSUPPORTED,
             "precision " + std::to_string(prec) +
                 " on simplices needs a scalar reference-tensor form (precision 32) or 64");
    // warp-specialised kernel (owner_pipe = 1): compute waves plus one store
    // wave, double-buffered accumulators
    hipFunction_t kpipe = prec == 32 ? owner->k_ownerp32 : owner->k_ownerp;
    if (kpipe && a->opt("owner_pipe", 0)) {
      int64_t& pgrid = prec == 32 ? owner->owner_gridp32 : owner->owner_gridp;
      const uint32_t pblock = static_cast<uint32_t>(64 * (a->opt("owner_cwaves", 4) + 1));
      if (pgrid == 0) {
        int nblk = 0;
        MF_HIP(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nblk, kpipe, pblock, 0));
        pgrid = std::max<int64_t>(nx, (int64_t)std::max(1, nblk) * a->ctx->num_cus / nx * nx);
      }
      launch(kpipe, static_cast<uint32_t>(std::min<int64_t>(per * nx, pgrid)), pblock, 0, s,
             static_cast<int32_t>(plan->nchunks), plan->chunk_meta.ptr, plan->pair_list.ptr, plan->pair_row.ptr,
             plan->pair_kk.ptr, owner->records.ptr, a->consts.ptr, A->rpb.ptr, plan->diag_pos.ptr,
             n0, A->values, diagonal, flags);
    } else {
    hipFunction_t kown = prec == 32 ? owner->k_owner32 : owner->k_owner;
    int64_t& ogrid = prec == 32 ? owner->owner_grid32 : owner->owner_grid;
    int64_t grid = per * nx;
    if (a->opt("owner_persistent", 1)) {
      if (ogrid == 0) {
        int nblk = 0;
        MF_HIP(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nblk, kown, oblock, 0));
        ogrid = std::max<int64_t>(nx, (int64_t)std::max(1, nblk) * a->ctx->num_cus / nx * nx);
      }
      grid = std::min<int64_t>(grid, ogrid * a->opt("owner_waves", 1));
    }
    launch(kown, static_cast<uint32_t>(grid), oblock, 0, s,
           static_cast<int32_t>(plan->nchunks), plan->chunk_meta.ptr, plan->pair_list.ptr,
           plan->pair_row.ptr, plan->pair_kk.ptr, owner->records.ptr, a->consts.ptr, A->rpb.ptr,
           plan->diag_pos.ptr, n0, A->values, diagonal, flags);
    }
    }
  }
  // Without an owner kernel, an overwriting call takes the integral with the
  // most element entries through the gather: its tensors into a workspace, then
  // one sum and one store per CSR value, where the per-entity kernel zeroes
  // the values and adds every entry with a global atomic.
  Integral* gathered = nullptr;
  if (!owner && zero && mode == 0) {
    auto entries = [&](const Integral& I) {
      return I.n * entity_ncell(I.type) * (int64_t)entity_ncell(I.type);
    };
    for (auto& I : a->ints)
      if (I->n && I->k_ten && (!gathered || entries(*I) > entries(*gathered))) gathered = I.get();
    if (GatherPlan* g = gathered ? gather_plan(a, *gathered, A, s) : nullptr) {
      const Integral& I = *gathered;
      const int nc = entity_ncell(I.type) * a->dm[1]->nd * a->dm[1]->bs;
      launch(I.k_ten, static_cast<uint32_t>((I.n + 63) / 64), 64, 0, s,
             static_cast<int32_t>(I.n), I.d_ents.ptr, a->mesh->cells.ptr, a->mesh->x.ptr,
             a->packed.ptr, a->consts.ptr, a->dm[0]->dev.ptr, a->dm[1]->dev.ptr, m0, m1, g->ws->ptr,
             a->mesh->fperm.ptr);
      k_gather(A->values, g->ws->ptr, g->ptr.ptr, g->at.ptr, g->pos.ptr, A->nnz_b, a->dm[0]->bs,
               a->dm[1]->bs, nc, s);
    } else {
      gathered = nullptr;
    }
  }
  if (!owner && !gathered && zero) k_fill(A->values, A->nnz, 0.0, s);
  const uint32_t block = static_cast<uint32_t>(a->opt("block", 128));
  for (auto& I : a->ints) {
    if (I.get() == owner || I.get() == gathered || I->n == 0) continue;
    auto& table = get_table(a, *I, A, s);
    launch(I->k_mat, static_cast<uint32_t>((I->n + block - 1) / block), block, 0, s,
           static_cast<int32_t>(I->n), I->d_ents.ptr, a->mesh->cells.ptr, a->mesh->x.ptr,
           a->packed.ptr, a->consts.ptr, a->dm[0]->dev.ptr, a->dm[1]->dev.ptr, m0, m1,
           table.ptr, A->row_ptr.ptr, A->values, a->mesh->fperm.ptr,
           static_cast<const int32_t*>(nullptr), static_cast<int64_t>(0));
  }
  if (square && m0 && !diag_done)
    k_set_diagonal(A->values, A->row_ptr.ptr, A->cols.ptr, bc0->dofs.ptr, bc0->n_owned, A->nrows,
                   diagonal, s);
}

}  // namespace mf

namespace mf {

void assemble_vector(mf_form* L, double* b, int64_t n, int zero, hipStream_t s) {
  MF_CHECK(L->rank == 1, MF_EINVAL, "assemble_vector needs a linear form");
  MF_CHECK(L->compiled, MF_ESTATE, "form is not compiled");
  if (L->restricted) {
    // block vector member: per-entity kernels with the node map and offset
    const int64_t kept = L->h_rmap[0].empty() ? L->dm[0]->num_nodes : L->rcount[0];
    MF_CHECK(L->roff[0] + kept * L->dm[0]->bs <= n, MF_ESHAPE, "block form does not fit the vector");
    if (zero) k_fill(b, n, 0.0, s);
    const uint32_t block = static_cast<uint32_t>(L->opt("block", 128));
    for (auto& I : L->ints) {
      if (I->n == 0) continue;
      launch(I->k_vec, static_cast<uint32_t>((I->n + block - 1) / block), block, 0, s,
             static_cast<int32_t>(I->n), I->d_ents.ptr, L->mesh->cells.ptr, L->mesh->x.ptr,
             L->packed.ptr, L->consts.ptr, L->dm[0]->dev.ptr, b, L->mesh->fperm.ptr,
             static_cast<const int32_t*>(L->rmap[0].ptr), static_cast<int64_t>(L->roff[0]));
    }
    return;
  }
  MF_CHECK(n == L->dm[0]->num_nodes * L->dm[0]->bs, MF_ESHAPE, "vector length mismatch");
  const int64_t mode = L->opt("vector_kernel", 0);
  if (L->k_dgown && (mode == 0 || mode == 3)) {
    if (!L->dgvplan_tried) {
      L->dgvplan = build_dg_plan(*L, nullptr);
      L->dgvplan_tried = true;
    }
    if (auto& dp = L->dgvplan) {
      const uint32_t blk = static_cast<uint32_t>(L->opt("dg_block", 64));
      launch(L->k_dgown, static_cast<uint32_t>((dp->ncells + blk - 1) / blk), blk, 0, s,
             static_cast<int32_t>(dp->ncells), dp->cell_ptr.ptr,
             reinterpret_cast<const int4*>(dp->items.ptr), L->mesh->cells.ptr, L->mesh->x.ptr,
             L->packed.ptr, L->consts.ptr, b, zero ? 1 : 0, L->mesh->fperm.ptr);
      return;
    }
  }
  MF_CHECK(mode != 3, MF_EUNSUPPORTED, "cell-owner DG vector kernel unavailable for this form");
  Integral* owner = nullptr;
  std::shared_ptr<OwnerPlan> plan;
  VectorBlocks* blocks = nullptr;
  if (mode == 0 || mode == 4)
    for (auto& I : L->ints)
      if (I->type == MF_CELL && I->n && (I->k_vblk || I->k_hsrc)) {
        if (mode == 4 || blocks_pay(*L, *I)) blocks = vector_blocks(L, *I, s);
        if (blocks) owner = I.get();
        break;
      }
  MF_CHECK(!(mode == 4 && !blocks), MF_EUNSUPPORTED, "no blocks of cells for this form");
  if (mode != 1 && !blocks)
    for (auto& I : L->ints)
      if (I->type == MF_CELL && I->k_vown) {
        plan = vector_plan(L, *I);
        if (plan) owner = I.get();
        break;
      }
  MF_CHECK(!(mode == 2 && !owner), MF_EUNSUPPORTED, "owner-computes vector kernel unavailable");
  if (blocks) {
    if (zero) k_fill(b, n, 0.0, s);
    launch(owner->k_hsrc ? owner->k_hsrc : owner->k_vblk, static_cast<uint32_t>((blocks->n + 7) / 8 * 8), blocks->threads, blocks->lds,
           s, static_cast<int32_t>(blocks->n), blocks->ent.ptr, blocks->ptr.ptr, blocks->row.ptr,
           blocks->slot.ptr, owner->d_ents.ptr, L->mesh->cells.ptr, L->mesh->x.ptr, L->packed.ptr,
           L->consts.ptr, b);
  } else if (owner) {
    const int64_t nx = 8, per = (plan->nchunks + nx - 1) / nx;
    launch(owner->k_vown, static_cast<uint32_t>(per * nx),
           static_cast<uint32_t>(L->opt("vector_block", 256)), 0, s,
           static_cast<int32_t>(plan->nchunks), plan->chunk_rows.ptr, plan->chunk_items.ptr,
           plan->item_cell.ptr, plan->item_mask.ptr, L->mesh->cells.ptr, L->mesh->x.ptr,
           L->packed.ptr, L->consts.ptr, L->dm[0]->dev.ptr, b, zero ? 1 : 0);
  } else if (zero) {
    k_fill(b, n, 0.0, s);
  }
  const uint32_t block = static_cast<uint32_t>(L->opt("block", 128));
  for (auto& I : L->ints) {
    if (I.get() == owner || I->n == 0) continue;
    launch(I->k_vec, static_cast<uint32_t>((I->n + block - 1) / block), block, 0, s,
           static_cast<int32_t>(I->n), I->d_ents.ptr, L->mesh->cells.ptr, L->mesh->x.ptr,
           L->packed.ptr, L->consts.ptr, L->dm[0]->dev.ptr, b, L->mesh->fperm.ptr,
           static_cast<const int32_t*>(nullptr), static_cast<int64_t>(0));
  }
}

// The right-hand sides of several linear forms: every form's cell integral in
// one launch of mf_vown_batch (workgroup k runs chunk k of the form whose
// chunks it falls in), then each form's other integrals with their own
// kernels, accumulating, as assemble_vector does for one form.
void assemble_vbatch(mf_batch* B, double* const* d_b, const int64_t* n_b, int zero, hipStream_t s) {
  struct Args {   // one group's kernel arguments, in the order of kOwnerVectorParams
    int32_t nchunks; int32_t pad; const void* chunk_rows; const void* chunk_items;
    const void* item_cell; const void* item_mask; const void* geo; const void* xg;
    const void* coeffs; const void* consts; const void* dm0; void* b; int32_t flags; int32_t pad2;
  };
  const size_t ng = B->forms.size();
  std::vector<Args> h(ng);
  int64_t total = 0;
  for (size_t g = 0; g < ng; ++g) {
    mf_form* L = B->forms[g];
    Integral* I = B->ints[g];
    MF_CHECK(d_b[g], MF_EINVAL, "batch vector " + std::to_string(g) + " is null");
    MF_CHECK(n_b[g] == L->dm[0]->num_nodes * L->dm[0]->bs, MF_ESHAPE,
             "batch vector " + std::to_string(g) + " does not match its form");
    auto plan = vector_plan(L, *I);
    MF_CHECK(plan != nullptr, MF_EUNSUPPORTED,
             "owner vector schedule unavailable for group " + std::to_string(g));
    h[g] = Args{static_cast<int32_t>(plan->nchunks), 0, plan->chunk_rows.ptr, plan->chunk_items.ptr,
                plan->item_cell.ptr, plan->item_mask.ptr, L->mesh->cells.ptr, L->mesh->x.ptr,
                L->packed.ptr, L->consts.ptr, L->dm[0]->dev.ptr, d_b[g], zero ? 1 : 0, 0};
    total += plan->nchunks;
  }
  MF_CHECK(total < INT32_MAX, MF_EUNSUPPORTED, "too many vector chunks for one launch");
  if (total > 0) {
    std::vector<void*> ptrs;
    for (size_t g = 0; g < ng; ++g) {
      Args& x = h[g];
      for (void* p : {static_cast<void*>(&x.nchunks), static_cast<void*>(&x.chunk_rows),
                      static_cast<void*>(&x.chunk_items), static_cast<void*>(&x.item_cell),
                      static_cast<void*>(&x.item_mask), static_cast<void*>(&x.geo),
                      static_cast<void*>(&x.xg), static_cast<void*>(&x.coeffs),
                      static_cast<void*>(&x.consts), static_cast<void*>(&x.dm0),
                      static_cast<void*>(&x.b), static_cast<void*>(&x.flags)})
        ptrs.push_back(p);
    }
    MF_HIP(hipModuleLaunchKernel(B->k, static_cast<uint32_t>(total), 1, 1,
                                 static_cast<uint32_t>(B->block), 1, 1, 0, s, ptrs.data(), nullptr));
  }
  const uint32_t block = 128;
  for (size_t g = 0; g < ng; ++g) {
    mf_form* L = B->forms[g];
    for (auto& I : L->ints) {
      if (I.get() == B->ints[g] || I->n == 0) continue;
      launch(I->k_vec, static_cast<uint32_t>((I->n + block - 1) / block), block, 0, s,
             static_cast<int32_t>(I->n), I->d_ents.ptr, L->mesh->cells.ptr, L->mesh->x.ptr,
             L->packed.ptr, L->consts.ptr, L->dm[0]->dev.ptr, d_b[g], L->mesh->fperm.ptr,
             static_cast<const int32_t*>(nullptr), static_cast<int64_t>(0));
    }
  }
}

// Several bilinear forms (one element group each, e.g. the degree groups of
// many independent meshes) in one persistent owner-computes launch, after
// one per-cell record pass per group.  Each group's matrix gets exactly what
// assemble_matrix's owner path writes (values overwritten when zero != 0;
// Dirichlet rows/columns of bcs[g] masked and the diagonal set).
void assemble_batch(mf_batch* B, mf_matrix* const* As, const mf_bc* const* bcs, double diag,
                    int zero, hipStream_t s) {
  struct Args {   // one group's kernel arguments (see the pointer list below)
    const void* chunk_meta; const void* pair_list; const void* pair_row; const void* pair_kk;
    const void* rec; const void* consts; const void* rpb; const void* dpos; const void* nb0;
    void* values; int32_t nchunks; int32_t pad;
  };
  static_assert(sizeof(Args) == 88, "batch argument layout");
  const size_t ng = B->forms.size();
  std::vector<Args> h(ng);
  for (size_t g = 0; g < ng; ++g) {
    mf_form* a = B->forms[g];
    Integral* I = B->ints[g];
    mf_matrix* A = As[g];
    const mf_bc* bc = bcs ? bcs[g] : nullptr;
    MF_CHECK(A && A->form && !A->block && A->nrows == a->dm[0]->num_nodes * a->dm[0]->bs,
             MF_ESHAPE, "batch matrix " + std::to_string(g) + " does not match its form");
    if (bc) MF_CHECK(bc->ndofs == A->nrows, MF_ESHAPE, "batch bc size does not match the rows");
    auto key = std::make_pair(a->uid, I->index);
    std::shared_ptr<OwnerPlan> plan;
    auto it = A->plans.find(key);
    if (it == A->plans.end() || it->second.first != a->gen) {
      plan = build_owner_plan(*a, *I, *A, a->opt("chunk_values", 4096),
                              static_cast<int>(a->opt("chunk_rows", 64)), owner_shape(*a, *I).maxp,
                              true);
      A->plans[key] = std::make_pair(a->gen, plan);
    } else {
      plan = it->second.second;
    }
    MF_CHECK(plan != nullptr, MF_EUNSUPPORTED, "owner-computes schedule unavailable for group " +
                                                   std::to_string(g));
    const uint8_t* n0 = bc && bc->nbc ? bc->bits_for(a->dm[0]->bs, s) : nullptr;
    const uint8_t* cf = n0 ? bc->cell_flags_for(a->dm[0], s) : nullptr;
    launch(B->preps[g], static_cast<uint32_t>((I->n + 255) / 256), 256, 0, s,
           static_cast<int32_t>(I->n), I->d_ents.ptr, a->mesh->cells.ptr, a->mesh->x.ptr,
           a->packed.ptr, a->dm[0]->dev.ptr, n0, cf, I->records.ptr);
    h[g] = Args{plan->chunk_meta.ptr, plan->pair_list.ptr, plan->pair_row.ptr, plan->pair_kk.ptr,
                I->records.ptr, a->consts.ptr, A->rpb.ptr, plan->diag_pos.ptr, n0, A->values,
                static_cast<int32_t>(plan->nchunks), 0};
  }
  // kernel arguments, per group in the order of kOwnerParams (nchunks,
  // chunk_meta, ..., values), then diag and flags; hipModuleLaunchKernel
  // copies each from its pointer per the kernel's argument layout
  int flags = zero ? 1 : 0;
  if (zero) flags |= 2;              // Dirichlet diagonal for the groups that have constraints
  std::vector<void*> ptrs;
  for (size_t g = 0; g < ng; ++g) {
    Args& x = h[g];
    for (void* p : {static_cast<void*>(&x.nchunks), static_cast<void*>(&x.chunk_meta),
                    static_cast<void*>(&x.pair_list), static_cast<void*>(&x.pair_row),
                    static_cast<void*>(&x.pair_kk), static_cast<void*>(&x.rec),
                    static_cast<void*>(&x.consts), static_cast<void*>(&x.rpb),
                    static_cast<void*>(&x.dpos), static_cast<void*>(&x.nb0),
                    static_cast<void*>(&x.values)})
      ptrs.push_back(p);
  }
  ptrs.push_back(&diag);
  ptrs.push_back(&flags);
  MF_HIP(hipModuleLaunchKernel(B->k, static_cast<uint32_t>(B->grid), 1, 1,
                               static_cast<uint32_t>(B->block), 1, 1, 0, s, ptrs.data(), nullptr));
}

// Rank-0 assembly (CUDAAssembler.h:296-351, CUDAFormIntegral.cpp:68-266):
// per integral, in cell / exterior / interior order, one partial per
// workgroup; then one fixed-order sum of all partials into d_value.
void assemble_scalar(mf_form* M, double* d_value, int zero, hipStream_t s) {
  MF_CHECK(M->rank == 0, MF_EINVAL, "assemble_scalar needs a functional (rank-0 form)");
  MF_CHECK(M->compiled, MF_ESTATE, "form is not compiled");
  for (auto& I : M->ints)
    launch(I->k_scl, I->scl_grid, 256, 0, s, static_cast<int32_t>(I->n), I->d_ents.ptr,
           M->mesh->cells.ptr, M->mesh->x.ptr, M->packed.ptr, M->consts.ptr,
           M->partials.ptr + I->scl_off, M->mesh->fperm.ptr);
  k_sum_partials(M->partials.ptr, M->partials.n, d_value, zero ? 0 : 1, s);
}

}  // namespace mf

const uint8_t* mf_bc::cell_flags_for(const mf_dofmap* dm, hipStream_t s) const {
  auto it = cell_flags.find(dm->uid);
  if (it != cell_flags.end()) return it->second.ptr;
  const uint8_t* bits = bits_for(dm->bs, s);
  mf::DevArray<uint8_t> f;
  f.alloc(std::max<int64_t>(1, dm->num_cells));
  mf::k_cell_flags(f.ptr, dm->dev.ptr, dm->num_cells, dm->nd, bits, s);
  return cell_flags.emplace(dm->uid, std::move(f)).first->second.ptr;
}

const uint8_t* mf_bc::bits_for(int bs, hipStream_t s) const {
  auto it = node_bits.find(bs);
  if (it != node_bits.end()) return it->second.ptr;
  MF_CHECK(ndofs % bs == 0, MF_ESHAPE, "bc size is not a multiple of the block size");
  mf::DevArray<uint8_t> b;
  b.alloc(ndofs / bs);
  mf::k_node_bits(b.ptr, markers.ptr, ndofs / bs, bs, s);
  return node_bits.emplace(bs, std::move(b)).first->second.ptr;
}
