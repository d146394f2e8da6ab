// Host side of the fused path: tile planning (rod -> workgroup bin packing),
// the FP32 copies of the constants, launches, and the director
// re-orthonormalisation and finiteness checks.
#include <algorithm>
#include <mutex>
#include <vector>

#include "erod_fused_kernel.hpp"

namespace erod {

  // FP32 constants of the FP32-bulk path: whole fields, in this order, packed
  // back to back (each keeps the ghost-padded slot indexing of its stagger)
  static const int kConst32Fields[] = {
      EROD_MASS, EROD_INV_MASS, EROD_REFERENCE_ELEMENT_LENGTH, EROD_REFERENCE_SHEAR_STRETCH_STRAIN,
      EROD_SHEAR_STRETCH_RIGIDITY, EROD_MASS_SECOND_MOMENT_OF_INERTIA, EROD_INV_MASS_SECOND_MOMENT_OF_INERTIA,
      EROD_REFERENCE_VORONOI_LENGTH, EROD_REFERENCE_CURVATURE, EROD_BENDING_TWIST_RIGIDITY,
      EROD_FORCE_DAMPING_RATE, EROD_TORQUE_DAMPING_RATE};
  static constexpr int kNConst32 = sizeof(kConst32Fields) / sizeof(kConst32Fields[0]);

  // offset (in floats) of constant i; const32_offset(b, kNConst32) is the total
  static uint64_t const32_offset(const erod_batch* b, int i) {
    uint64_t off = 0;
    for (int k = 0; k < i; ++k) off += uint64_t(field_info(kConst32Fields[k]).ncomp) * b->field_slots(kConst32Fields[k]);
    return off;
  }

  uint64_t fused_const32_offset(const erod_batch* b, int field) {
    for (int i = 0; i < kNConst32; ++i)
      if (kConst32Fields[i] == field) return const32_offset(b, i);
    return ~uint64_t(0);
  }

  using fused::Consts;

  namespace {
    // FP64 constants -> FP32 copies (same slot indexing)
    __global__ void k_to_f32(float* __restrict__ o, const double* __restrict__ a, uint64_t n) {
      for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        o[i] = static_cast<float>(a[i]);
    }

    // one Newton-Schulz polar step Q <- Q (3 I - Q^T Q) / 2 on element slot k
    __device__ __forceinline__ void reortho_slot(double* __restrict__ Q, uint64_t E, uint64_t k) {
      double q[9], g[9], o[9];
      for (int m = 0; m < 9; ++m) q[m] = Q[m * E + k];
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) g[3 * a + b] = q[a] * q[b] + q[3 + a] * q[3 + b] + q[6 + a] * q[6 + b];
      for (int p = 0; p < 3; ++p)
        for (int r = 0; r < 3; ++r) {
          double s = 0.0;
          for (int c = 0; c < 3; ++c) s += q[3 * p + c] * ((c == r ? 3.0 : 0.0) - g[3 * c + r]);
          o[3 * p + r] = 0.5 * s;
        }
      for (int m = 0; m < 9; ++m) Q[m * E + k] = o[m];
    }

    // every element slot
    __global__ void k_reortho(double* __restrict__ Q, uint64_t E) {
      for (uint64_t k = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; k < E; k += (uint64_t)gridDim.x * blockDim.x)
        reortho_slot(Q, E, k);
    }

    // the active elements of every rod with steps left (steps_left null: all
    // rods); a rod whose budget is spent keeps its state bit for bit
    __global__ void k_reortho_live(double* __restrict__ Q, uint64_t E, const RodInfo* __restrict__ rods, uint64_t n_rods,
                                   const uint32_t* __restrict__ steps_left) {
      for (uint64_t r = blockIdx.x; r < n_rods; r += gridDim.x) {
        if (steps_left && steps_left[r] == 0) continue;
        const RodInfo ri = rods[r];
        for (uint32_t k = threadIdx.x; k < ri.n; k += blockDim.x) reortho_slot(Q, E, ri.start + k);
      }
    }

    template <typename Flag>
    __global__ void k_check_finite(const double* __restrict__ X, const double* __restrict__ Vel, const double* __restrict__ Qd,
                                   const double* __restrict__ W, const RodInfo* __restrict__ rods, uint64_t n_rods,
                                   uint64_t E, Flag* __restrict__ flags) {
      const uint64_t N = E + 1;
      for (uint64_t r = blockIdx.x; r < n_rods; r += gridDim.x) {
        const RodInfo ri = rods[r];
        int bad = 0;
        for (uint32_t k = threadIdx.x; k <= ri.n; k += blockDim.x) {
          const uint64_t s = ri.start + k;
          for (int c = 0; c < 3; ++c) bad |= int(!isfinite(X[c * N + s])) | int(!isfinite(Vel[c * N + s]));
          if (k < ri.n) {
            for (int c = 0; c < 3; ++c) bad |= !isfinite(W[c * E + s]);
            for (int m = 0; m < 9; ++m) bad |= !isfinite(Qd[m * E + s]);
          }
        }
        if (bad) flags[r] = Flag(1);
      }
    }

    __global__ void k_zero_u8(uint8_t* __restrict__ p, uint64_t n) {
      for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0;
    }

  }  // namespace

  // ---- planning: bin-pack rods into tiles --------------------------------------

  int fused_shape_lanes(int si) { return fused::kShapes[si].P * fused::kShapes[si].NT; }
  int fused_shape_epl(int si) { return fused::kShapes[si].P; }

  // rods the fused kernels advance: non-empty slots with steps left
  static bool planned(const erod_batch* b, uint64_t r) {
    return b->n_active[r] != 0 && (!b->budgets || b->steps_left[r] != 0);
  }

  // A rod runs as pieces when it is longer than the main tile, or longer
  // than the pieces' tile when seg_lanes is set.
  static bool cut_rod(const erod_batch* b, uint64_t n, int main_shape) {
    const uint64_t cap = uint64_t(fused_shape_lanes(main_shape));
    return n > cap || (b->plan.seg_lanes > 0 && n > uint64_t(b->plan.seg_lanes));
  }

  // Feasible main shapes: its lanes and elements per thread are the ones
  // requested, and every rod that is not cut has at least P elements (a
  // thread then holds at most one rod end).
  static bool shape_feasible(const erod_batch* b, int si) {
    const fused::Shape sh = fused::kShapes[si];
    const int lanes = b->plan.lanes_per_tile, epl = b->plan.elements_per_thread;
    if (lanes && sh.P * sh.NT != lanes) return false;
    if (epl && sh.P != epl) return false;
    for (uint64_t r = 0; r < b->n_rods; ++r)
      if (planned(b, r) && !cut_rod(b, b->n_active[r], si) && b->n_active[r] < uint64_t(sh.P)) return false;
    return true;
  }

  // whether the caller left the main shape free
  static bool unrequested(const erod_batch* b) { return b->plan.lanes_per_tile == 0 && b->plan.elements_per_thread == 0; }

  // whether neither the caller nor the autotuner chose it
  static bool shapes_free(const erod_batch* b) { return unrequested(b) && b->plan.tuned_shape < 0; }

  constexpr int kShape128 = 1, kShape256 = 2, kShape512 = 3;  // one element per thread
  constexpr int kShape128x2 = 8, kShape512x2 = 4;             // two

  bool shadow_fits(const erod_batch* b) {
    if (b->d_shadow[3]) return true;
    if (b->pool) return false;
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return free / 4 > 18 * sizeof(double) * b->E;
  }

  // whether pieces of 256 lanes leave a part of 64 elements between their halos
  static bool halo_fits_256(const erod_batch* b) { return 2 * b->plan.halo + 64 <= 256; }

  // the longest rod and the elements of those that the plan takes
  struct Extent {
    uint64_t longest = 0, lanes = 0;
  };
  static Extent extent(const erod_batch* b) {
    Extent e;
    for (uint64_t r = 0; r < b->n_rods; ++r)
      if (planned(b, r)) {
        e.longest = std::max<uint64_t>(e.longest, b->n_active[r]);
        e.lanes += b->n_active[r];
      }
    return e;
  }

  // Few FP64 rods of up to 257 to 512 elements, which run as pieces in 256 lanes
  // (see default_shape) where the caller leaves shapes free: the halo has to
  // leave the pieces room, and to pay for their launches (100 steps of 20 rods
  // of 400 elements, us a step: 4.1 whole; 5.4, 4.6, 4.2, 3.8, 3.6 and 2.9 with a
  // halo of 2, 3, 4, 6, 8 and 16).
  static bool few_in_256(const erod_batch* b, const Extent& e, int precision) {
    return precision == EROD_FP64 && b->plan.seg_lanes == 0 && b->plan.halo >= 6 && halo_fits_256(b) && e.longest > 256 &&
           e.longest <= 512 && e.lanes <= 32 * uint64_t(b->cus);
  }

  // Default shape without measurement: the smallest capacity that holds the
  // longest rod; one element per thread up to 256 lanes, two elements per
  // thread for 1024 lanes; rods longer than 1024 elements run as pieces.  (Four
  // elements per thread spill and run one wave per SIMD.)  512 lanes take two
  // elements per thread for FP32-bulk when the tiles fill more than a round of
  // the CUs: two 4-wave workgroups share a CU (1,200 rods of 16 to 512
  // elements: 3.6 us a step against 4.4 in 8-wave workgroups of one element per
  // thread).  While every tile has a CU of its own a step costs its latency,
  // which is shorter at one element per thread (600 such rods: 2.40 against
  // 2.65; 61 rods of up to 301: 2.15 against 2.67); fused FP64 has no registers
  // for two (17.5 against 21.0 for 2,400 rods, 5.7 against 7.1 for 61).
  // FP32-bulk batches of shorter rods take two elements per thread too once
  // they fill the SIMDs, where fewer instructions per element count: rods of up
  // to 128 elements in 128-lane tiles of one wave (8,192 rods of 128: 9.8 us a
  // step against 13.9; 1,024: 1.87 and 1.93; 512: 1.81 and 1.62; rods of 64:
  // 8,192 5.25 and 6.28, 3,072 2.84 and 3.01, 2,048 1.90 and 1.69), rods of up
  // to 256 in 512-lane ones (4,096 of 256: 11.2 and 13.3; 512: 2.41 and 2.02).
  // Fused FP64 pays 8 waves' exchanges in 512-lane tiles: in a batch of few
  // rods those past 256 elements run as pieces in 256 lanes (61 rods of up to
  // 301: 4.6 -> 3.4 us a step; 100 of up to 512, over the line: 4.6 and 4.8).
  // Not for calls whose launches are shorter than a halo, each of which passes
  // over the state twice more (calls on one rod of 300, us: 1 step 16 whole and
  // 25 in pieces, 8 steps 44 and 44, 16 steps 75 and 63, 100 steps 402 and 274).
  // Results are the same, bit by bit; FP32-bulk's depend on where a launch ends,
  // so its rods stay whole.  (Batches with rods of 513 to 1,024 elements would
  // gain more, 13.6 -> 3.5 for 20 of them, but erod_set_fused_config documents
  // 1024 lanes for them: an autotune, or a request for pieces, has them faster.)
  // A shape the autotuner chose is taken again while it stays feasible (a
  // replan after rods changed length keeps it, with its second group).  Tuned
  // for FP32-bulk, 128 lanes may have two elements per thread in one wave, for
  // which FP64 has no registers (8,192 rods of 128 elements 47 us a step, 29 at
  // one): it takes one.
  static int default_shape(const erod_batch* b, int precision, bool brief) {
    static const int pref[] = {0, 1, 2, 4, 5, 3, 7, 6, 8};
    const int tuned = b->plan.tuned_shape;
    if (tuned >= 0 && shape_feasible(b, tuned))
      return tuned == kShape128x2 && precision == EROD_FP64 && shape_feasible(b, kShape128) ? kShape128 : tuned;
    const Extent e = extent(b);
    const uint64_t maxn = e.longest, lanes = e.lanes;
    if (shapes_free(b) && !brief && few_in_256(b, e, precision) && shadow_fits(b)) return kShape256;
    for (int si : pref)
      if (uint64_t(fused_shape_lanes(si)) >= maxn && shape_feasible(b, si)) {
        const bool two = fused_shape_lanes(si) == 512 && fused_shape_epl(si) == 2;
        if (precision != EROD_FP64 && shapes_free(b)) {
          const uint64_t cus = uint64_t(b->cus);
          if (maxn <= 128 && lanes > (maxn <= 64 ? 640 : 512) * cus && shape_feasible(b, kShape128x2)) return kShape128x2;
          if (maxn > 128 && maxn <= 256 && lanes > 1024 * cus && shape_feasible(b, kShape512x2)) return kShape512x2;
        }
        if (two && shape_feasible(b, kShape512) && (precision == EROD_FP64 || lanes <= 512 * uint64_t(b->cus))) return kShape512;
        return si;
      }
    // longer rods than any tile: the largest tiles, the longer rods in pieces
    for (int si : {5, 4, 3, 2, 1, 0, 7, 6, 8})
      if (shape_feasible(b, si)) return si;
    return -1;
  }

  // the shape a requested or tuned second group uses, or -1 (none)
  static int split_shape(const erod_batch* b, int precision) {
    if (b->plan.split_lanes <= 0) return -1;
    if (b->plan.split_tuned && precision == EROD_FP64 && b->plan.split_lanes == 128) return kShape128;
    for (int si : {0, 1, 2, 4, 5, 3, 7, 6, 8})  // the default order of preference
      if (fused::kShapes[si].P * fused::kShapes[si].NT == b->plan.split_lanes &&
          (b->plan.split_epl <= 0 || fused::kShapes[si].P == b->plan.split_epl))
        return si;
    return -2;
  }

  // The shape of the pieces of long rods: the one of seg_lanes lanes (and
  // seg_epl elements per thread when set), or the main shape; -2 if none.
  // With every shape `free` (the caller requested none; the main one may be a
  // tuned one or a trial's), smaller pieces than the main tiles where those
  // would leave CUs idle, and always for fused FP64, whose 1024-lane tiles
  // spill registers.  24 rods of 2,500 to 6,000 elements (107 / 212 / 440
  // pieces of 1024 / 512 / 256 lanes on 256 CUs), us a step: FP32-bulk 6.0 /
  // 4.4 / 4.5, FP64 21.1 / 7.7 / 8.2; 2 rods of 1,200 to 1,500: 4.6 / 3.2 / 2.7
  // and 14.8 / 6.5 / 4.5; 60 rods of 1,100 to 6,000 (206 / 391 / 803): 6.4 / 7.3
  // / 7.0 and 22.8 / 13.7 / 13.1.
  static int piece_shape(const erod_batch* b, int main_shape, int precision, bool free) {
    if (b->plan.seg_lanes > 0) {
      for (int si : {0, 1, 2, 4, 5, 3, 7, 6, 8})  // the default order of preference
        if (fused_shape_lanes(si) == b->plan.seg_lanes && (b->plan.seg_epl <= 0 || fused_shape_epl(si) == b->plan.seg_epl))
          return si;
      return -2;
    }
    const uint64_t halo = uint64_t(b->plan.halo);
    if (!free || !halo_fits_256(b) || fused_shape_lanes(main_shape) != 1024) return main_shape;
    uint64_t pieces256 = 0, pieces512 = 0;
    for (uint64_t r = 0; r < b->n_rods; ++r)
      if (planned(b, r) && cut_rod(b, b->n_active[r], main_shape)) {
        pieces256 += (b->n_active[r] + 255 - 2 * halo) / (256 - 2 * halo);
        pieces512 += (b->n_active[r] + 511 - 2 * halo) / (512 - 2 * halo);
      }
    if (pieces256 <= uint64_t(b->cus)) return kShape256;
    if (pieces512 <= uint64_t(b->cus)) return kShape512;
    return precision == EROD_FP64 ? kShape256 : main_shape;
  }

  // One group of tiles on the host: the tiles, their entries (rods or
  // pieces) in order and each entry's first lane; rods sent on to a second group.
  struct Packed {
    std::vector<Tile> tiles;
    std::vector<uint32_t> trods, tlane0, overflow;
  };

  // Best-fit-decreasing bin packing of entries into tiles of P * NT elements:
  // each entry, longest first, goes to the tile with the least free room that
  // holds it (ties: the tile that reached that room first).  A workgroup costs
  // about the same whether its tile is full or not, so the tile count sets the
  // launch time; on the 4096-rod ragged batch this packs to the lower bound
  // (972 tiles of 1024 lanes, against 1170 for first fit over the 64 newest).
  // Lengths and rooms are at most P * NT, so the sort is a counting sort and
  // the open tiles sit in one FIFO list per room, found through a bitset: a
  // serving pool replans its ~30,000 slots in about 0.5 ms of host time.
  // Here `order` holds the entries, longest first, len[e] their lengths, and
  // cap is P * NT.  With spill_cap > 0, an entry of at most spill_cap
  // elements that finds no room in an open tile goes to `overflow` instead of
  // opening one, provided it has at least spill_min elements (the second
  // group's elements per thread; a shorter rod stays in the main group).
  static void pack(const std::vector<uint32_t>& len, uint64_t cap, const std::vector<uint32_t>& order,
                   uint64_t spill_cap, uint64_t spill_min, Packed& out) {
    // open tiles by free room: FIFO lists (head, tail, next) and a bitset of non-empty rooms
    std::vector<int32_t> head(cap + 1, -1), tail(cap + 1, -1), next;
    std::vector<uint64_t> nonempty(cap / 64 + 1, 0);
    auto open = [&](uint64_t room, uint32_t t) {
      next[t] = -1;
      if (tail[room] < 0) head[room] = int32_t(t);
      else next[tail[room]] = int32_t(t);
      tail[room] = int32_t(t);
      nonempty[room >> 6] |= uint64_t(1) << (room & 63);
    };
    std::vector<uint32_t> placed, tile_of, tile_rods_count;
    for (const uint32_t r : order) {
      const uint64_t n = len[r];
      int64_t room = -1;  // the smallest room >= n that has a tile
      for (uint64_t w = n >> 6; w < nonempty.size() && room < 0; ++w) {
        uint64_t m = nonempty[w];
        if (w == (n >> 6)) m &= ~uint64_t(0) << (n & 63);
        if (m) room = int64_t(w * 64 + uint64_t(__builtin_ctzll(m)));
      }
      uint32_t t;
      if (room < 0) {
        if (n <= spill_cap && n >= spill_min) {
          out.overflow.push_back(r);
          continue;
        }
        t = static_cast<uint32_t>(tile_rods_count.size());
        tile_rods_count.push_back(0);
        next.push_back(-1);
        if (cap > n) open(cap - n, t);
      } else {
        t = static_cast<uint32_t>(head[room]);
        head[room] = next[t];
        if (head[room] < 0) {
          tail[room] = -1;
          nonempty[room >> 6] &= ~(uint64_t(1) << (room & 63));
        }
        if (const uint64_t left = uint64_t(room) - n) open(left, t);
      }
      placed.push_back(r);
      tile_of.push_back(t);
      ++tile_rods_count[t];
    }
    // tiles in creation order, each with its entries in the order they were placed
    const size_t n_tiles = tile_rods_count.size(), n_placed = placed.size();
    out.tiles.assign(n_tiles, Tile{});
    out.trods.assign(n_placed, 0);
    out.tlane0.assign(n_placed, 0);
    std::vector<uint32_t> fill(n_tiles), lane(n_tiles, 0);
    for (uint32_t t = 0, first = 0; t < n_tiles; ++t) {
      out.tiles[t].first = first;
      out.tiles[t].count = tile_rods_count[t];
      out.tiles[t].pad = 0;
      fill[t] = first;
      first += tile_rods_count[t];
    }
    for (size_t i = 0; i < n_placed; ++i) {
      const uint32_t t = tile_of[i], k = fill[t]++;
      out.trods[k] = placed[i];
      out.tlane0[k] = lane[t];
      lane[t] += len[placed[i]];
    }
    for (size_t t = 0; t < n_tiles; ++t) out.tiles[t].lanes = lane[t];
  }

  // entries longest first (stable), by a counting sort over lengths <= cap
  static std::vector<uint32_t> longest_first(const std::vector<uint32_t>& len, const std::vector<uint32_t>& ids,
                                             uint64_t cap) {
    std::vector<uint32_t> count(cap + 2, 0), next_pos(cap + 2, 0), order(ids.size());
    for (const uint32_t e : ids) ++count[len[e]];
    uint32_t k = 0;
    for (uint64_t n = cap + 1; n >= 1; --n) {
      next_pos[n] = k;
      k += count[n];
    }
    for (const uint32_t e : ids) order[next_pos[len[e]]++] = e;
    return order;
  }

  // how many pieces `cut` makes of a rod of n elements: the least number of an
  // even split whose longest piece, a middle part plus two halos, fits
  static uint64_t n_pieces(uint64_t n, uint64_t cap, uint64_t halo) {
    uint64_t m = 2;
    while (true) {
      const uint64_t part = (n + m - 1) / m;
      if (part + 2 * halo <= cap || part <= 1) return m;
      ++m;
    }
  }

  // The pieces of a rod of n elements for tiles of `cap` lanes: owned parts
  // of nearly equal length, each piece loading `halo` more elements on each
  // side that has a neighbouring piece; every piece at most cap long.
  static void cut(uint32_t rod, uint64_t n, uint64_t cap, uint64_t halo, std::vector<Seg>& out) {
    const uint64_t m = n_pieces(n, cap, halo);
    for (uint64_t i = 0; i < m; ++i) {
      const uint64_t a = i * n / m, z = (i + 1) * n / m;  // owned [a, z)
      // (a halo longer than the parts reaches past its neighbours', to the rod's
      // end at most)
      const uint64_t lo = a < halo ? 0 : a - halo, hi = std::min(n, z + halo);
      Seg sg{};
      sg.rod = rod;
      sg.off = uint32_t(lo);
      sg.n = uint32_t(hi - lo);
      sg.w0 = uint32_t(a - lo);
      sg.w1 = uint32_t(z - lo);
      sg.ends = (lo == 0 ? kSegFirst : 0u) | (hi == n ? kSegLast : 0u);
      out.push_back(sg);
    }
  }

  // a rod of n elements that one piece holds
  static Seg whole_piece(uint32_t rod, uint32_t n) {
    Seg sg{};
    sg.rod = rod;
    sg.n = sg.w1 = n;
    sg.ends = kSegFirst | kSegLast;
    return sg;
  }

  // The halo of the pieces where the caller left their shape free: as wide as
  // leaves every piece a CU of its own (beside the whole rods' tiles), up to
  // 64, a launch taking as many steps.  Until then wider halos cost no time,
  // and longer launches save it (a launch costs 20 us beside its steps): 24
  // rods of 2,500 to 6,000 elements, us a step FP32-bulk 3.75 -> 2.31, FP64 7.7
  // -> 4.95; 3 rods of 1,200 to 1,500 2.2 -> 1.64 and 3.6 -> 2.90.  FP32-bulk's
  // runs stay `halo` / 2 steps, so results don't depend on it.
  static uint64_t wide_halo(const erod_batch* b, int main_shape, uint64_t pcap, uint64_t halo) {
    const uint64_t step = halo / 2, cap = uint64_t(fused_shape_lanes(main_shape));
    uint64_t wide = halo, whole = 0;
    for (uint64_t r = 0; r < b->n_rods; ++r)
      if (planned(b, r) && !cut_rod(b, b->n_active[r], main_shape)) whole += b->n_active[r];
    const uint64_t beside = (whole + cap - 1) / cap;
    for (uint64_t h = halo; h <= 64 && 4 * h <= pcap; h += step) {
      uint64_t pieces = beside;
      for (uint64_t r = 0; r < b->n_rods && pieces <= uint64_t(b->cus); ++r)
        if (planned(b, r) && cut_rod(b, b->n_active[r], main_shape)) pieces += n_pieces(b->n_active[r], pcap, h);
      if (pieces > uint64_t(b->cus)) break;
      wide = h;
    }
    return wide;
  }

  // Device copy of one group.  The arrays grow to the largest plan seen and
  // are reused when the rod set changes.
  template <typename T>
  static int grow(T*& p, uint64_t& cap, uint64_t need, hipStream_t stream) {
    if (cap >= need) return EROD_OK;
    EROD_HIP(hipStreamSynchronize(stream));
    if (p) EROD_HIP(hipFree(p));
    p = nullptr;
    cap = 0;
    EROD_HIP(hipMalloc(&p, need * sizeof(T)));
    cap = need;
    return EROD_OK;
  }

  static int upload_group(erod_batch* b, const Packed& pk, TileGroup& g) {
    const uint64_t need = std::max<uint64_t>({pk.tiles.size(), pk.trods.size(), 1});
    if (g.capacity < need) {
      uint64_t c1 = g.capacity, c2 = g.capacity, c3 = g.capacity;
      if (int rc = grow(g.d_tiles, c1, need, b->stream)) return rc;
      if (int rc = grow(g.d_tile_rods, c2, need, b->stream)) return rc;
      if (int rc = grow(g.d_tile_lane0, c3, need, b->stream)) return rc;
      g.capacity = need;
    }
    if (!pk.tiles.empty()) {
      EROD_HIP(hipMemcpyAsync(g.d_tiles, pk.tiles.data(), pk.tiles.size() * sizeof(Tile), hipMemcpyHostToDevice, b->stream));
      EROD_HIP(hipMemcpyAsync(g.d_tile_rods, pk.trods.data(), pk.trods.size() * sizeof(uint32_t), hipMemcpyHostToDevice,
                              b->stream));
      EROD_HIP(hipMemcpyAsync(g.d_tile_lane0, pk.tlane0.data(), pk.tlane0.size() * sizeof(uint32_t),
                              hipMemcpyHostToDevice, b->stream));
    }
    return EROD_OK;
  }

  // Few FP64 rods in 256 lanes: those that need no cut go in the pieces' group
  // too, each as one piece.  In a group of their own they would need a hardware
  // queue of their own: 61 rods of up to 301 elements take 3.5 us a step in two
  // groups on two queues and 6.2 where the batch's two streams share one, which
  // is the runtime's choice (whole in 512 lanes 4.6).  Not FP32-bulk's, which
  // rounds a piece by its halo.
  static bool one_group(const erod_batch* b, int si, int ps, int precision, bool free) {
    return free && si == kShape256 && ps == si && b->plan.split_lanes == 0 && few_in_256(b, extent(b), precision);
  }

  // free: the caller requested no shape
  static int plan_tiles(erod_batch* b, int si, int ps, int precision, bool free) {
    const uint64_t cap = uint64_t(fused_shape_lanes(si));
    if (ps == -2) {
      set_error("plan_tiles: no tile shape of the requested piece lanes and elements per thread");
      return EROD_ERR_INVALID;
    }
    const uint64_t pcap = uint64_t(fused_shape_lanes(ps));
    const uint64_t halo = uint64_t(b->plan.halo);
    if (halo < 2 || 2 * halo + 2 > pcap) {
      set_error("plan_tiles: the halo of rod pieces must be at least 2 and leave room in the pieces' tile");
      return EROD_ERR_INVALID;
    }
    // whole rods of the main (and second) group, and pieces of long rods
    std::vector<uint32_t> len(b->n_rods), whole;
    std::vector<uint32_t> seg_rods;
    std::vector<Seg> segs;
    const uint64_t wide = b->plan.seg_lanes == 0 && !b->plan.halo_set && free ? wide_halo(b, si, pcap, halo) : halo;
    const bool one = one_group(b, si, ps, precision, free);
    uint64_t uncut = 0;
    for (uint32_t i = 0; i < b->n_rods; ++i) {
      if (!planned(b, i)) continue;
      len[i] = static_cast<uint32_t>(b->n_active[i]);
      if (cut_rod(b, b->n_active[i], si)) {
        if (b->n_active[i] > (uint64_t(1) << 31)) {
          set_error("plan_tiles: a rod longer than 2^31 elements");
          return EROD_ERR_INVALID;
        }
        seg_rods.push_back(i);
        cut(i, b->n_active[i], pcap, wide, segs);
      } else if (one) {
        seg_rods.push_back(i);
        segs.push_back(whole_piece(i, len[i]));
        ++uncut;
      } else {
        whole.push_back(i);
      }
    }
    const int s2 = split_shape(b, precision);
    if (s2 == -2) {
      set_error("plan_tiles: no tile shape of the requested split lanes and elements per thread");
      return EROD_ERR_INVALID;
    }
    // a second group only of tiles smaller than the main ones (a requested
    // split at least as large as the main tile is ignored); it takes rods of
    // at most its lanes and at least its elements per thread
    uint64_t cap2 = s2 >= 0 ? uint64_t(fused_shape_lanes(s2)) : 0;
    if (cap2 >= cap) cap2 = 0;
    const uint64_t min2 = cap2 ? uint64_t(fused_shape_epl(s2)) : 0;
    // each entry takes a whole number of its group's threads: its length
    // rounded up to the elements per thread (the kernel puts the idle pad
    // lanes before the entry's elements, so that its last element is a
    // thread's last)
    auto padded = [](uint64_t n, uint64_t p) { return static_cast<uint32_t>((n + p - 1) / p * p); };
    std::vector<uint32_t> len1(len.size());
    for (const uint32_t i : whole) len1[i] = padded(len[i], uint64_t(fused_shape_epl(si)));
    Packed g1, g2, g3;
    pack(len1, cap, longest_first(len1, whole, cap), cap2, min2, g1);
    if (!g1.overflow.empty()) {
      std::vector<uint32_t> len2(len.size());
      for (const uint32_t i : g1.overflow) len2[i] = padded(len[i], uint64_t(fused_shape_epl(s2)));
      pack(len2, cap2, g1.overflow, 0, 0, g2);
    }
    std::vector<uint32_t> slen(segs.size()), sids(segs.size());
    for (uint32_t k = 0; k < segs.size(); ++k) {
      slen[k] = padded(segs[k].n, uint64_t(fused_shape_epl(ps)));
      sids[k] = k;
    }
    if (!segs.empty()) pack(slen, pcap, longest_first(slen, sids, pcap), 0, 0, g3);
    // the kernel stages a tile's entry table in NT entries of LDS (rods have
    // at least two elements, and at least P: a feasible shape never exceeds it)
    const int shapes[3] = {si, s2 >= 0 ? s2 : si, ps};
    const Packed* pks[3] = {&g1, &g2, &g3};
    for (int k = 0; k < 3; ++k)
      for (const Tile& t : pks[k]->tiles)
        if (t.count > uint32_t(fused::kShapes[shapes[k]].NT)) {
          set_error("plan_tiles: more rods in a tile than threads");
          return EROD_ERR_INVALID;
        }
    FusedPlan& pl = b->plan;
    for (int k = 0; k < 3; ++k)
      if (!pks[k]->tiles.empty())
        if (int rc = upload_group(b, *pks[k], pl.g[k])) return rc;
    TileGroup& gs = pl.g[2];
    if (!segs.empty()) {
      if (int rc = grow(gs.d_segs, gs.seg_capacity, segs.size(), b->stream)) return rc;
      if (int rc = grow(gs.d_seg_rods, gs.seg_rod_capacity, seg_rods.size(), b->stream)) return rc;
      if (!b->d_time_next) EROD_HIP(hipMalloc(&b->d_time_next, sizeof(double) * b->n_rods));
      const int shadow_fields[4] = {EROD_POSITION, EROD_VELOCITY, EROD_DIRECTOR, EROD_ANGULAR_VELOCITY};
      for (int k = 0; k < 4; ++k)
        if (!b->d_shadow[k])
          EROD_HIP(hipMalloc(&b->d_shadow[k], sizeof(double) * field_info(shadow_fields[k]).ncomp *
                                                  b->field_slots(shadow_fields[k])));
      EROD_HIP(hipMemcpyAsync(gs.d_segs, segs.data(), segs.size() * sizeof(Seg), hipMemcpyHostToDevice, b->stream));
      EROD_HIP(hipMemcpyAsync(gs.d_seg_rods, seg_rods.data(), seg_rods.size() * sizeof(uint32_t), hipMemcpyHostToDevice,
                              b->stream));
    }
    EROD_HIP(hipStreamSynchronize(b->stream));
    for (int k = 0; k < 3; ++k) {
      pl.g[k].n_tiles = pks[k]->tiles.size();
      pl.g[k].shape = pks[k]->tiles.empty() ? -1 : shapes[k];
      pl.g[k].max_steps = 0;
    }
    if (uncut) pl.g[0].shape = si;  // (their tiles are the pieces')
    gs.n_segs = segs.size() - uncut;
    gs.n_seg_rods = seg_rods.size();
    // FP32-bulk's merged half steps end every halo / 2 steps, wherever launches
    // end; a launch holds two such runs (three for a halo of 3, more in a wide
    // one).  13 launches per 100 steps (halo 16) became 7: 24 rods of 2,500 to
    // 6,000 elements 6.05 -> 5.08 us a step (FP32-bulk), 2,048 ragged rods 29.6
    // -> 28.0 (FP64, long rods in pieces)
    gs.run_steps = int(halo / 2);
    gs.max_steps = int(wide / (halo / 2)) * gs.run_steps;
    if (segs.empty()) gs.shape = -1;
    pl.precision = precision;
    pl.main_shape = si;
    pl.piece_shape = ps;
    pl.split_shape = s2;
    pl.one_group = one;
    pl.valid = true;
    b->graph_precision = -1;
    return EROD_OK;
  }

  int fused_prepare(erod_batch* b, int precision, uint64_t launch) {
    const OnDevice here(b->device);
    int rc = sync_rods(b);
    if (rc) return rc;
    FusedPlan& pl = b->plan;
    if (!pl.valid) pl.kept.valid = false;  // the rods changed: so did its
    // (the calls' lengths decide on free shapes only)
    const bool brief = precision == EROD_FP64 && shapes_free(b) && launch < uint64_t(std::max(pl.halo, 16));
    if (!pl.valid || pl.precision != precision || pl.brief != brief) {
      const int si = default_shape(b, precision, brief);
      if (si < 0) {
        set_error("no fused tile shape holds this batch (a requested shape with more elements per thread than "
                  "a rod has)");
        return EROD_ERR_UNSUPPORTED;
      }
      const bool free = unrequested(b);
      const int ps = piece_shape(b, si, precision, free);
      const int s2 = split_shape(b, precision);
      const bool one = one_group(b, si, ps, precision, free);
      const auto same = [&](const auto& p) {
        return p.main_shape == si && p.piece_shape == ps && p.split_shape == s2 && p.one_group == one;
      };
      if (pl.valid && !same(pl)) {
        // other shapes than this plan's: the kept one comes in, this one is kept
        for (int k = 0; k < 3; ++k) std::swap(pl.g[k], pl.kept.g[k]);
        std::swap(pl.main_shape, pl.kept.main_shape);
        std::swap(pl.piece_shape, pl.kept.piece_shape);
        std::swap(pl.split_shape, pl.kept.split_shape);
        std::swap(pl.one_group, pl.kept.one_group);
        std::swap(pl.valid, pl.kept.valid);
        pl.valid = pl.valid && same(pl);
      }
      if (!pl.valid && (rc = plan_tiles(b, si, ps, precision, free))) return rc;
      pl.precision = precision;
      pl.brief = brief;
    }
    if (precision == EROD_FP32_BULK && b->const32_dirty) {
      const uint64_t total = const32_offset(b, kNConst32);
      if (!b->d_const32 || b->const32_floats != total) {
        if (b->d_const32) EROD_HIP(hipFree(b->d_const32));
        b->d_const32 = nullptr;
        EROD_HIP(hipMalloc(&b->d_const32, sizeof(float) * total));
        b->const32_floats = total;
      }
      for (int i = 0; i < kNConst32; ++i) {
        const int f = kConst32Fields[i];
        const uint64_t n = uint64_t(field_info(f).ncomp) * b->field_slots(f);
        hipLaunchKernelGGL(k_to_f32, dim3(grid_for(n)), dim3(kThreads), 0, b->stream, b->d_const32 + const32_offset(b, i),
                           b->d_field[f], n);
      }
      EROD_HIP(hipGetLastError());
      b->const32_dirty = false;
    }
    return EROD_OK;
  }

  template <typename R>
  static Consts<R> make_consts(erod_batch* b);

  template <>
  Consts<double> make_consts<double>(erod_batch* b) {
    Consts<double> C;
    C.m = b->d_field[EROD_MASS];
    C.invm = b->d_field[EROD_INV_MASS];
    C.l0 = b->d_field[EROD_REFERENCE_ELEMENT_LENGTH];
    C.sig0 = b->d_field[EROD_REFERENCE_SHEAR_STRETCH_STRAIN];
    C.S = b->d_field[EROD_SHEAR_STRETCH_RIGIDITY];
    C.J = b->d_field[EROD_MASS_SECOND_MOMENT_OF_INERTIA];
    C.iJ = b->d_field[EROD_INV_MASS_SECOND_MOMENT_OF_INERTIA];
    C.D0 = b->d_field[EROD_REFERENCE_VORONOI_LENGTH];
    C.kap0 = b->d_field[EROD_REFERENCE_CURVATURE];
    C.B = b->d_field[EROD_BENDING_TWIST_RIGIDITY];
    C.gf = b->d_field[EROD_FORCE_DAMPING_RATE];
    C.gt = b->d_field[EROD_TORQUE_DAMPING_RATE];
    return C;
  }

  template <>
  Consts<float> make_consts<float>(erod_batch* b) {
    const float* p = b->d_const32;
    Consts<float> C;
    C.m = p + const32_offset(b, 0);
    C.invm = p + const32_offset(b, 1);
    C.l0 = p + const32_offset(b, 2);
    C.sig0 = p + const32_offset(b, 3);
    C.S = p + const32_offset(b, 4);
    C.J = p + const32_offset(b, 5);
    C.iJ = p + const32_offset(b, 6);
    C.D0 = p + const32_offset(b, 7);
    C.kap0 = p + const32_offset(b, 8);
    C.B = p + const32_offset(b, 9);
    C.gf = p + const32_offset(b, 10);
    C.gt = p + const32_offset(b, 11);
    return C;
  }

  // Measured choice of the tile shape: every feasible shape advances the
  // batch `trial_steps` steps from the same snapshot of x, v, Q, w and the rod
  // clocks (restored afterwards), timed with HIP events; the fastest is kept.
  // Unless the caller set a second group, each smaller shape is then tried as
  // one for the rods that find no room beside longer ones, and kept if faster.
  int fused_autotune(erod_batch* b, int precision, int trial_steps, double* best_ms) {
    const OnDevice here(b->device);
    int rc = fused_prepare(b, precision, uint64_t(trial_steps));
    if (rc) return rc;
    const int snap_fields[4] = {EROD_POSITION, EROD_VELOCITY, EROD_DIRECTOR, EROD_ANGULAR_VELOCITY};
    // snapshot buffers and the plan settings the trials change, released and
    // restored on every return
    struct Guard {
      erod_batch* b;
      double* snap[5] = {};
      int lanes, epl, split_lanes, split_epl;
      bool budgets;
      bool keep_split = false;  // a second group chosen by the trials stays
      ~Guard() {
        for (double* p : snap)
          if (p) (void)hipFree(p);
        b->plan.lanes_per_tile = lanes;
        b->plan.elements_per_thread = epl;
        if (!keep_split) {
          b->plan.split_lanes = split_lanes;
          b->plan.split_epl = split_epl;
        }
        b->budgets = budgets;
        b->last_launches = 0;  // the trial launches are not a fused call's timing
      }
    } g{b, {}, b->plan.lanes_per_tile, b->plan.elements_per_thread, b->plan.split_lanes, b->plan.split_epl, b->budgets};
    size_t bytes[5];
    for (int i = 0; i < 4; ++i) bytes[i] = sizeof(double) * field_info(snap_fields[i]).ncomp * b->field_slots(snap_fields[i]);
    bytes[4] = sizeof(double) * b->n_rods;
    auto dev = [&](int i) { return i < 4 ? b->d_field[snap_fields[i]] : b->d_time; };
    for (int i = 0; i < 5; ++i) {
      EROD_HIP(hipMalloc(&g.snap[i], bytes[i]));
      EROD_HIP(hipMemcpyAsync(g.snap[i], dev(i), bytes[i], hipMemcpyDeviceToDevice, b->stream));
    }
    auto restore = [&]() -> int {
      for (int i = 0; i < 5; ++i) EROD_HIP(hipMemcpyAsync(dev(i), g.snap[i], bytes[i], hipMemcpyDeviceToDevice, b->stream));
      return EROD_OK;
    };
    b->plan.lanes_per_tile = 0;
    b->plan.elements_per_thread = 0;
    b->budgets = false;  // trial launches leave the step budgets alone
    // each trial's plan is the one that its shape would get once chosen, pieces
    // and halos included (for 24 rods of 2,500 to 6,000 elements that is the
    // untuned plan or a faster one, not launches of 16 steps over pieces of the
    // main shape)
    const bool free = g.lanes == 0 && g.epl == 0;
    auto plan = [&](int si) { return plan_tiles(b, si, piece_shape(b, si, precision, free), precision, free); };
    b->plan.kept.valid = false;
    // FP64 has no registers for two elements per thread in one wave (see
    // default_shape).  FP32-bulk rounds a rod that is cut by its halo: where 512
    // lanes hold every rod, shapes that cut some are not tried, so that a tuned
    // batch returns what an untuned one does, and not what the trials' times
    // happen to decide.  (Pieces with wide halos would be faster for few rods,
    // ms a pass: 21 of 76 to 355 elements 1.40 against 2.02, 15 of 80 to 349 1.01
    // and 1.43, 11 of 105 to 258 1.11 and 1.23; slower for many, 476 of 17 to 287
    // 3.68 and 3.42.  With longer rods, beside which whole ones run in 1024
    // lanes, 2.9 against 4.3 for 70 of 44 to 718, they are tried.)
    const uint64_t longest = extent(b).longest;
    const bool keep_whole = precision != EROD_FP64 && b->plan.seg_lanes == 0 && longest <= 512;
    auto has_registers = [&](int si) { return si != kShape128x2 || precision != EROD_FP64; };
    auto candidate = [&](int si) { return has_registers(si) && (!keep_whole || uint64_t(fused_shape_lanes(si)) >= longest); };
    int best = -1;
    double best_t = 0.0;
    for (int si = 0; si < fused::kNShapes && rc == EROD_OK; ++si) {
      if (!shape_feasible(b, si) || !candidate(si)) continue;
      if ((rc = plan(si))) break;
      if ((rc = fused_launch(b, precision, trial_steps, false))) break;  // warm
      if ((rc = fused_launch(b, precision, trial_steps, true))) break;
      float ms = 0.0f;
      if ((rc = hip_check(hipEventSynchronize(b->ev1), "autotune sync"))) break;
      if ((rc = hip_check(hipEventElapsedTime(&ms, b->ev0, b->ev1), "autotune time"))) break;
      if (best < 0 || ms < best_t) {
        best = si;
        best_t = ms;
      }
      if ((rc = restore())) break;
    }
    // a second group of smaller tiles, when the caller has not set one
    int best_split = -1;
    if (rc == EROD_OK && best >= 0 && g.split_lanes == 0) {
      const int cap = fused_shape_lanes(best);
      for (int s2 = 0; s2 < fused::kNShapes && rc == EROD_OK; ++s2) {
        if (fused_shape_lanes(s2) >= cap || !has_registers(s2)) continue;
        b->plan.split_lanes = fused_shape_lanes(s2);
        b->plan.split_epl = fused_shape_epl(s2);
        const int prc = plan(best);
        if (prc == EROD_ERR_HIP) {  // a device failure ends the search; an infeasible shape does not
          rc = prc;
          break;
        }
        // infeasible here, or no second group, or every rod in it (a plan of
        // that shape alone, which the first trials timed)
        if (prc != EROD_OK || b->plan.g[1].shape < 0 || b->plan.g[0].shape < 0) continue;
        if ((rc = fused_launch(b, precision, trial_steps, false))) break;  // warm
        if ((rc = fused_launch(b, precision, trial_steps, true))) break;
        float ms = 0.0f;
        if ((rc = hip_check(hipEventSynchronize(b->ev1), "autotune sync"))) break;
        if ((rc = hip_check(hipEventElapsedTime(&ms, b->ev0, b->ev1), "autotune time"))) break;
        if (ms < best_t) {
          best_split = s2;
          best_t = ms;
        }
        if ((rc = restore())) break;
      }
    }
    // the chosen plan is made with the caller's settings and budgets; the
    // chosen main shape is kept for later replans while it stays feasible
    b->plan.tuned_shape = best;
    b->plan.lanes_per_tile = g.lanes;
    b->plan.elements_per_thread = g.epl;
    b->plan.split_lanes = best_split >= 0 ? fused_shape_lanes(best_split) : g.split_lanes;
    b->plan.split_epl = best_split >= 0 ? fused_shape_epl(best_split) : g.split_epl;
    b->plan.split_tuned |= best_split >= 0;
    g.keep_split = true;
    b->budgets = g.budgets;
    if (rc == EROD_OK && best >= 0) rc = plan(best);
    if (rc == EROD_OK) rc = restore();
    if (rc == EROD_OK) rc = hip_check(hipStreamSynchronize(b->stream), "autotune");
    if (rc == EROD_OK && best < 0) {
      set_error("no feasible fused tile shape");
      rc = EROD_ERR_UNSUPPORTED;
    }
    if (best_ms) *best_ms = best_t / trial_steps;
    return rc;
  }

  int fused_launch(erod_batch* b, int precision, int steps, bool timed) {
    if (timed) EROD_HIP(hipEventRecord(b->ev0, b->stream));
    const int rc = precision == EROD_FP64 ? fused_launch_fp64(b, make_consts<double>(b), steps)
                                          : fused_launch_fp32(b, make_consts<float>(b), steps);
    if (rc) return rc;
    if (timed) EROD_HIP(hipEventRecord(b->ev1, b->stream));
    return EROD_OK;
  }

  int fused_reorthonormalize(erod_batch* b) {
    hipLaunchKernelGGL(k_reortho, dim3(grid_for(b->E)), dim3(kThreads), 0, b->stream, b->d_field[EROD_DIRECTOR], b->E);
    return hip_check(hipGetLastError(), "reorthonormalize");
  }

  int fused_reorthonormalize_live(erod_batch* b) {
    const unsigned g = static_cast<unsigned>(b->n_rods < 65535 ? b->n_rods : 65535);
    hipLaunchKernelGGL(k_reortho_live, dim3(g), dim3(256), 0, b->stream, b->d_field[EROD_DIRECTOR], b->E, b->d_rods,
                       b->n_rods, static_cast<const uint32_t*>(b->d_steps_left));
    return hip_check(hipGetLastError(), "scheduled reorthonormalization");
  }

  int fused_check_finite(erod_batch* b, uint8_t* flags) {
    int rc = sync_rods(b);
    if (rc) return rc;
    EROD_HIP(hipMemsetAsync(b->d_flags, 0, sizeof(int) * b->n_rods, b->stream));
    const unsigned g = static_cast<unsigned>(b->n_rods < 65535 ? b->n_rods : 65535);
    hipLaunchKernelGGL(k_check_finite<int>, dim3(g), dim3(256), 0, b->stream, b->d_field[EROD_POSITION],
                       b->d_field[EROD_VELOCITY], b->d_field[EROD_DIRECTOR], b->d_field[EROD_ANGULAR_VELOCITY], b->d_rods,
                       b->n_rods, b->E, b->d_flags);
    EROD_HIP(hipGetLastError());
    std::vector<int> h(b->n_rods);
    EROD_HIP(hipMemcpyAsync(h.data(), b->d_flags, sizeof(int) * b->n_rods, hipMemcpyDeviceToHost, b->stream));
    EROD_HIP(hipStreamSynchronize(b->stream));
    for (uint64_t i = 0; i < b->n_rods; ++i) flags[i] = static_cast<uint8_t>(h[i] != 0);
    return EROD_OK;
  }

  // ---- finiteness check that allocates nothing -----------------------------------
  //
  // The per-rod flags live in `scratch`, a file-scope device array of
  // kScratchRods bytes that every GPU the library runs on holds until the
  // process ends (each GPU its own copy).  Its device address is looked up
  // once per device and kept; the array's name is never used as an address
  // in host code.  The flags the kernel needs cleared are cleared by a small
  // kernel before each check (no memset node), and the result is copied
  // straight into the caller's array.  Calls that overlap on one GPU share
  // the array and race.

  constexpr uint64_t kScratchRods = uint64_t(1) << 20;  // 1 MiB: one byte per rod
  static __device__ __align__(256) uint8_t scratch[kScratchRods];

  namespace {
    constexpr int kMaxDevices = 64;
    std::mutex g_scratch_mutex;
    uint8_t* g_scratch_ptr[kMaxDevices] = {};

    // the address of `scratch` on `device`, looked up on the first call there
    int scratch_on(int device, uint8_t** out) {
      if (device < 0 || device >= kMaxDevices) {
        set_error("check_finite_noalloc: device ordinal out of range");
        return EROD_ERR_INVALID;
      }
      std::lock_guard<std::mutex> lock(g_scratch_mutex);
      if (!g_scratch_ptr[device]) {
        int current = 0;
        EROD_HIP(hipGetDevice(&current));
        if (current != device) EROD_HIP(hipSetDevice(device));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (current != device) EROD_HIP(hipSetDevice(current));
        EROD_HIP(e);
        g_scratch_ptr[device] = static_cast<uint8_t*>(p);
      }
      *out = g_scratch_ptr[device];
      return EROD_OK;
    }
  }  // namespace

  int fused_check_finite_noalloc(erod_batch* b, uint8_t* flags) {
    if (b->n_rods > kScratchRods) {
      set_error("erod_check_finite_noalloc: at most 1,048,576 rods (the size of its device scratch array)");
      return EROD_ERR_INVALID;
    }
    uint8_t* d = nullptr;
    if (int rc = scratch_on(b->device, &d)) return rc;
    // rod records changed on the host go up whole (the staged upload of a
    // few records would allocate its staging buffer)
    if (b->rods_dirty || !b->dirty_rods.empty()) {
      EROD_HIP(hipMemcpyAsync(b->d_rods, b->rods.data(), sizeof(RodInfo) * b->n_rods, hipMemcpyHostToDevice, b->stream));
      b->rods_dirty = false;
      b->dirty_rods.clear();
    }
    hipLaunchKernelGGL(k_zero_u8, dim3(grid_for(b->n_rods)), dim3(kThreads), 0, b->stream, d, b->n_rods);
    const unsigned g = static_cast<unsigned>(b->n_rods < 65535 ? b->n_rods : 65535);
    hipLaunchKernelGGL(k_check_finite<uint8_t>, dim3(g), dim3(256), 0, b->stream, b->d_field[EROD_POSITION],
                       b->d_field[EROD_VELOCITY], b->d_field[EROD_DIRECTOR], b->d_field[EROD_ANGULAR_VELOCITY], b->d_rods,
                       b->n_rods, b->E, d);
    EROD_HIP(hipGetLastError());
    EROD_HIP(hipMemcpyAsync(flags, d, b->n_rods, hipMemcpyDeviceToHost, b->stream));
    EROD_HIP(hipStreamSynchronize(b->stream));
    return EROD_OK;
  }

}  // namespace erod
