// k_nlist.hip -- Verlet neighbor-list build over the cell-sorted atoms.
//
// Pair set (H/src/NeighborList.cu:327-420, all-pairs build of the adaptive
// engine; U/src/NeighborList_interface.cu:361-491 for the uniform one):
//     j in L(i)  <=>  j != i  and  |d_ij|^2 < (rc_i + skin)^2
// with the per-atom radius rc_i + skin of atom i (the list is asymmetric).
//
// Candidates: a wavefront takes kBuildAtoms consecutive sorted atoms.  Atoms
// of one cell column share one window: the (x, y) cell columns that meet the
// union of their spheres, and in each the z cells covering the union of the
// chords, which are one or two contiguous runs of cell-sorted atoms.  The
// runs, column after column, form one flat candidate sequence, taken 64 at a
// time, one candidate per lane.  Every atom is tested against the 64
// candidates at once, the accepted lanes form a scalar 64-bit mask, and a
// candidate's place in the atom's list is the atom's count plus the accepted
// lanes below it: the list order is the candidate order (column by column,
// ascending within a run), whatever the window was.  Entries go to the
// wave-tiled column-major layout the force kernel reads (list_slot()).
// Writes beyond the capacity are dropped but still counted; the host regrows
// and rebuilds.  (Large dilute systems and batches of small boxes: a window
// per atom, the same lists.)
//
// The distance test is |x_i|^2 - rl_i^2 - 2 x_i.x_j + |x_j|^2 < 0 on
// coordinates relative to the tile's centre, a contraction over (x, y, z, 1)
// that the matrix cores do in FP32: v_mfma_f32_4x4x1_16b holds four atoms
// against the wavefront's 64 candidates, candidate = lane.  It decides every
// pair whose value lies outside a band around 0 that bounds its rounding;
// the rare pair inside the band is decided by the exact predicate, so the
// pair set is the exact predicate's.
#include <algorithm>

#include "sre_internal.h"

namespace sre {

constexpr int kBuildBlock = 256;
constexpr int kBuildTile = 16;    // atoms per entry of part[]
constexpr int kTileAtoms = 80000; // atoms from which a tile has eight (launch_build_list)
constexpr int kBuildWaves = kBuildBlock / kWave;

typedef float sre_f32x4 __attribute__((ext_vector_type(4)));

// minimum / maximum over a wave's M atoms (atom lane % M), as a scalar: quad
// partners, then mirrored halves and rows of lanes
template <int M>
__device__ __forceinline__ uint32_t tile_min(uint32_t v) {
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false));
  if (M > 4) v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xF, 0xF, false));
  if (M > 8) v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xF, 0xF, false));
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
template <int M>
__device__ __forceinline__ uint32_t tile_max(uint32_t v) {
  return ~tile_min<M>(~v);
}
__device__ __forceinline__ uint64_t ballot64(bool v) { return __builtin_amdgcn_ballot_w64(v); }
__device__ __forceinline__ int lane_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// What bounds it: VALU issue (79 % busy at 2 million atoms, 145 instructions
// per atom; a form with one atom per 4 lanes and a divergent cursor over its
// own windows took 240), and below ~100 000 atoms the length of the heaviest
// wavefronts.  Per 64 candidates, 12 instructions form the local coordinates
// for all M atoms, and each atom takes a compare of the matrix result and,
// when lanes were accepted, the mask count (2), the slot (3) and the store.
// Measured, M as chosen below, before -> now: 4 000 atoms (uniform cutoff)
// 31 -> 16 us, 16 000 atoms with lists of 1 350 (IMG) 228 -> 125 us, 62 500
// (slab) 53 -> 39.4 us, 2 048 000 (rc 2.5 to 6, 140 million entries, 0.56 GB
// written) 1 004 -> 615 us; boxes little wider than twice the list radius,
// where chunks take the exact predicate, are faster too while few atoms fill the
// chip (a rebuild of 3 000 atoms in a cube of 16, rc 7.5: 166 -> 113 us).  Large
// dilute systems and batches of small boxes are not, and keep a window per atom
// (k_build_list_sparse).
// M = 16 (fewer, longer wavefronts) was slower at
// every size.  Register budgets: seven (M = 4), six (M = 8) and four (IMG)
// wavefronts per SIMD; eight spill scalar registers into vector lanes.
template <int M, int TF, bool IMG>
__global__ __launch_bounds__(kBuildBlock) __attribute__((amdgpu_waves_per_eu(IMG ? 4 : (M == 4 ? 7 : 6)))) void
k_build_list(int n, const uint4 *__restrict__ pos4, const float *__restrict__ rcut,
             const RepInfo *__restrict__ reps, const int *__restrict__ start, float skin,
             int cap, int *__restrict__ list, size_t list_len, int *__restrict__ nnb,
             int2 *__restrict__ part) {
  constexpr int G = M / 4;   // groups of four atoms
  __shared__ int2 s_part[kBuildWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int wib = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int s0 = ((int)blockIdx.x * kBuildWaves + wib) * M;
  int cnt[M];   // list lengths, the same on every lane
#pragma unroll
  for (int r = 0; r < M; ++r) cnt[r] = 0;
  int longest = 0;
  if (s0 < n) {   // wave-uniform
    const int na = min(M, n - s0);
    const __amdgpu_buffer_rsrc_t prs = pos_rsrc_idx(pos4, n);
    // lane l holds atom l % M, and as matrix operands atoms 4 g + l % 4
    const uint4 pi = pos4[min(s0 + (lane & (M - 1)), n - 1)];
    const float rl = rcut[min(s0 + (lane & (M - 1)), n - 1)] + skin;
    uint4 pg[G];
#pragma unroll
    for (int g = 0; g < G; ++g) pg[g] = pos4[min(s0 + 4 * g + (lane & 3), n - 1)];
    // list slots in the force kernel's layout (T = TF lanes per atom): entry k
    // of atom r lies (k / TF) * 64 + k % TF ints after the atom's first,
    // addressed through a resource based at the first atom's tile
    constexpr int AF = kWave / TF;
    const size_t tile0 = (size_t)(s0 / AF) * ((size_t)cap * AF);
    const size_t lrem = list_len > tile0 ? list_len - tile0 : 0;
    const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc(
        list + tile0, (short)0, (int)min(lrem * 4, (size_t)0x7fffffff), 0x00020000);
    const int off0 = (s0 % AF) * TF * 4;
    unsigned todo = (1u << na) - 1u;
    while (todo) {   // one pass per cell column the wave's atoms lie in
      const int lead = __builtin_ctz(todo);
      const uint32_t lw = (uint32_t)lane_i((int)pi.w, lead);
      const RepInfo &R = reps[lw >> 8];
      const float qx = R.q[0], qy = R.q[1], qz = R.q[2];
      const int ncx = R.nc[0], ncy = R.nc[1], ncz = R.nc[2];
      const float hx = R.h[0], hy = R.h[1], hz = R.h[2];
      const float rm = rl * 1.0001f + 1e-4f;   // conservative window radius
      // atoms sharing the leader's replica, column and kinds of window form
      // the tile (a direction whose window takes in every cell is traversed
      // from cell 0, so its order differs from a proper window's)
      const int cxi = cell_of(pi.x, ncx), cyi = cell_of(pi.y, ncy);
      const float ihz = __builtin_amdgcn_rcpf(hz);
      // (the radius carries a margin of 1e-4, far above the rounding of these)
      const int kxi = (int)ceilf(rm * __builtin_amdgcn_rcpf(hx));
      const int kyi = (int)ceilf(rm * __builtin_amdgcn_rcpf(hy));
      const int ki = (2 * kxi + 1 >= ncx ? 1 : 0) | (2 * kyi + 1 >= ncy ? 2 : 0) |
                     (2 * (int)ceilf(rm * ihz) + 1 >= ncz ? 4 : 0);
      const int cx = lane_i(cxi, lead), cy = lane_i(cyi, lead), kd = lane_i(ki, lead);
      unsigned tile = (unsigned)ballot64((pi.w >> 8) == (lw >> 8) && cxi == cx && cyi == cy &&
                                         ki == kd) & todo;
      const bool fullx = kd & 1, fully = kd & 2, fullz = kd & 4;
      const uint32_t lz = (uint32_t)lane_i((int)pi.z, lead);
      const float rml = lane_f(rm, lead);
      float rlm;                         // the tile's largest window radius
      uint32_t z0, z1;                   // lattice bounds of the tile's atoms
      int czl, czh;
      float fzl, fzh;
      for (;;) {
        const bool in = (tile >> (lane & (M - 1))) & 1u;
        z0 = tile_min<M>(in ? pi.z : lz);
        z1 = tile_max<M>(in ? pi.z : lz);
        // (positive floats order as their bit patterns)
        rlm = __uint_as_float(tile_max<M>(__float_as_uint(in ? rm : rml)));
        czl = cell_of(z0, ncz);
        czh = cell_of(z1, ncz);
        // position inside a cell from the low 32 bits of u * nc
        fzl = (float)(uint32_t)((uint64_t)z0 * (uint64_t)ncz) * (hz * 0x1p-32f);
        fzh = (float)(uint32_t)((uint64_t)z1 * (uint64_t)ncz) * (hz * 0x1p-32f);
        // a union window around the whole column has no order that is every
        // atom's own: such atoms are taken one at a time
        if (fullz || (tile & (tile - 1u)) == 0u) break;
        const int lo = czl + (int)floorf((fzl - rlm) * ihz);
        const int hi = czh + (int)floorf((fzh + rlm) * ihz);
        if (hi - lo + 1 < ncz) break;
        tile = 1u << lead;
      }
      todo &= ~tile;
      const bool in = (tile >> (lane & (M - 1))) & 1u;
      const int kx = (int)tile_max<M>((uint32_t)(in ? kxi : 0));
      const int ky = (int)tile_max<M>((uint32_t)(in ? kyi : 0));
      const float rlm2 = rlm * rlm;
      const int ox0 = fullx ? -cx : -kx, ox1 = fullx ? ncx - 1 - cx : kx;
      const int oy0 = fully ? -cy : -ky, oy1 = fully ? ncy - 1 - cy : ky;
      const int noy = oy1 - oy0 + 1;
      const int ncol = (ox1 - ox0 + 1) * noy;
      // a wide window makes a long wave: it goes first, or it would still be
      // running when the others are done
      if (ncol > 16) __builtin_amdgcn_s_setprio(3);
      else if (ncol > 9) __builtin_amdgcn_s_setprio(1);
      // local coordinates about the centre of the tile's column.  A candidate's nearest
      // image about the centre is its nearest image about every atom, or
      // neither is within reach, while no atom lies farther than L/2 - rl from
      // the centre.  Wider tiles (cells of a large part of the box) test the
      // next image along x and y too (at most one of them is within reach);
      // along z, where cells are flat, they take the exact predicate.
      const uint32_t ux = (2u * cx + 1u) * R.half_cell[0], uy = (2u * cy + 1u) * R.half_cell[1],
                     uz = z0 + ((z1 - z0) >> 1);
      const float wx = 0.5001f * hx, wy = 0.5001f * hy, wz = (float)(z1 - z0) * (0.5f * qz);
      const float Lx = R.L[0], Ly = R.L[1];
      const bool images = !(wx < 0.5f * Lx - rlm && wy < 0.5f * Ly - rlm);
      const bool local = wz < 0.5f * R.L[2] - rlm && (IMG || !images);
      // rounding of the matrix form: coordinates (2^-23 relative) and a sum
      // of five terms of at most (rl + 2 w)^2; twice the bound of 2^-20
      const float wsum = rlm + 2.f * (wx + wy + wz);
      const float band = wsum * wsum * 0x1p-19f;
      auto loc = [&](uint32_t u, uint32_t o, float q) { return (float)(int32_t)(u - o) * q; };
      float ax[G], ay[G], az[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        ax[g] = -2.f * loc(pg[g].x, ux, qx);
        ay[g] = -2.f * loc(pg[g].y, uy, qy);
        az[g] = -2.f * loc(pg[g].z, uz, qz);
      }
      // |x_i|^2 - rl_i^2; atoms outside the tile accept nothing
      const float xl = loc(pi.x, ux, qx), yl = loc(pi.y, uy, qy), zl = loc(pi.z, uz, qz);
      const float ci = in ? __builtin_fmaf(zl, zl, __builtin_fmaf(yl, yl, xl * xl)) - rl * rl : 1e30f;
      sre_f32x4 cg[G];
#pragma unroll
      for (int r = 0; r < M; ++r) cg[r / 4][r & 3] = __shfl(ci, r, kWave);
      // appends the candidates of mask (scalar) to atom r's list
      auto emit = [&](int r, uint64_t mask, int j, bool full) {
        const uint32_t k = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)cnt[r]));
        cnt[r] += __builtin_popcountll(mask);
        if (full) mask &= ballot64((int)k < cap);
        const uint32_t off = (k << 2) + __umul24(k / TF, 256 - 4 * TF);
        if (__builtin_amdgcn_inverse_ballot_w64(mask))
          __builtin_amdgcn_raw_buffer_store_b32(
              (uint32_t)j, lrs, (int)off,
              off0 + (r % AF) * (TF * 4) + (r / AF) * (cap * AF * 4), 0);
      };
      // may some list pass its capacity with `more` further candidates?  longest
      // is an upper bound of the lists' lengths, made exact only when it is
      // near the capacity (so it takes in every chunk, whichever way it is tested)
      auto near_cap = [&](int more) {
        if (longest + more > cap) {
          longest = cnt[0];
#pragma unroll
          for (int r = 1; r < M; ++r) longest = max(longest, cnt[r]);
          longest = __builtin_amdgcn_readfirstlane(longest);
        }
        longest += more;
        return longest > cap;
      };

      for (int cbase = 0; cbase < ncol; cbase += kWave / 2) {
        // lane = (column, run): the run's first atom and length
        int rp = 0, rn = 0;
        {
          const int c = cbase + (lane >> 1);
          const bool second = lane & 1;
          // c / noy for small integers
          const int co = (int)(((float)c + 0.5f) * __builtin_amdgcn_rcpf((float)noy));
          const int ox = ox0 + co, oy = oy0 + (c - co * noy);
          if (c < ncol) {
            float gx = 0.f, gy = 0.f;
            if (!fullx) gx = (float)(abs(ox) - 1) * hx;
            if (!fully) gy = (float)(abs(oy) - 1) * hy;
            gx = fmaxf(gx, 0.f);
            gy = fmaxf(gy, 0.f);
            const float gxy2 = gx * gx + gy * gy;
            if (gxy2 < rlm2) {
              int cxw = cx + ox;
              cxw += cxw < 0 ? ncx : 0;
              cxw -= cxw >= ncx ? ncx : 0;
              int cyw = cy + oy;
              cyw += cyw < 0 ? ncy : 0;
              cyw -= cyw >= ncy ? ncy : 0;
              const int colbase = R.cell_off + (cxw * ncy + cyw) * ncz;
              int r0 = 0, r1 = second ? -1 : ncz - 1;  // whole column unless the chord is shorter
              if (!fullz) {
                // (the window radius carries a 1e-4 margin, far above the
                // rounding of the square root and of 1/hz)
                const float dz = __builtin_amdgcn_sqrtf(fmaxf(rlm2 - gxy2, 0.f));
                const int lo = czl + (int)floorf((fzl - dz) * ihz);
                const int hi = czh + (int)floorf((fzh + dz) * ihz);
                if (hi - lo + 1 < ncz) {
                  // lo .. hi, the part beyond an end of the column wrapped
                  const bool wl = lo < 0, wh = hi >= ncz;
                  r0 = second ? ((wl || wh) ? 0 : 1) : (wl ? lo + ncz : lo);
                  r1 = second ? (wl ? hi : (wh ? hi - ncz : 0)) : ((wl || wh) ? ncz - 1 : hi);
                }
              }
              if (r1 >= r0) {
                // runs lie inside [0, n) by construction; the clamps keep every
                // gather in bounds whatever the cell offsets hold
                rp = min(max(start[colbase + r0], 0), n);
                rn = max(min(start[colbase + r1 + 1], n) - rp, 0);
              }
            }
          }
        }
        uint64_t runs = ballot64(rn > 0);
        int cp = 0, cl = 0;      // rest of the current run (scalar); cl = 0: no more
        auto run = [&]() {
          if (runs) {
            const int r = __builtin_ctzll(runs);
            runs &= runs - 1;
            cp = lane_i(rp, r);
            cl = lane_i(rn, r);
          }
        };
        run();
        // the next (up to) 64 candidates of the flat sequence
        struct Chunk {
          int j, filled;
          uint4 c;
        };
        auto next = [&]() {
          Chunk q;
          q.filled = 0;
          int d = 0;             // candidate - lane
          while (cl > 0 && q.filled < kWave) {
            d = __builtin_amdgcn_inverse_ballot_w64(~0ull << q.filled) ? cp - q.filled : d;
            const int take = min(kWave - q.filled, cl);
            cp += take;
            cl -= take;
            q.filled += take;
            if (cl == 0) run();
          }
          // (a lane past the sequence may hold an atom past its run: any atom
          // inside the array will do, its test is masked)
          q.j = lane + d;
          q.c = gather_pos_idx<false>(prs, min(q.j, n - 1));
          return q;
        };
        auto test = [&](const Chunk &q) {
          const uint64_t valid = q.filled == kWave ? ~0ull : (1ull << q.filled) - 1ull;
          if (local) {
            const float bx = loc(q.c.x, ux, qx), by = loc(q.c.y, uy, qy), bz = loc(q.c.z, uz, qz);
            float b2 = __builtin_fmaf(bz, bz, __builtin_fmaf(by, by, bx * bx));
            b2 = __builtin_amdgcn_inverse_ballot_w64(valid) ? b2 : 1e30f;
            auto dist = [&](sre_f32x4 *dg, float x, float y, float n2) {
#pragma unroll
              for (int g = 0; g < G; ++g)
                dg[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(ax[g], x, cg[g], 0, 0, 0);
#pragma unroll
              for (int g = 0; g < G; ++g)
                dg[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(ay[g], y, dg[g], 0, 0, 0);
#pragma unroll
              for (int g = 0; g < G; ++g)
                dg[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(az[g], bz, dg[g], 0, 0, 0);
#pragma unroll
              for (int g = 0; g < G; ++g)
                dg[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(1.f, n2, dg[g], 0, 0, 0);
            };
            sre_f32x4 dg[G];
            dist(dg, bx, by, b2);
            if (IMG && images) {
              const float cx2 = bx - copysignf(Lx, bx), cy2 = by - copysignf(Ly, by);
              const float ix = __builtin_fmaf(cx2, cx2, -bx * bx);   // change of |x_j|^2
              const float iy = __builtin_fmaf(cy2, cy2, -by * by);
              sre_f32x4 d1[G], d2[G], d3[G];
              dist(d1, cx2, by, b2 + ix);
              dist(d2, bx, cy2, b2 + iy);
              dist(d3, cx2, cy2, b2 + (ix + iy));
#pragma unroll
              for (int r = 0; r < M; ++r)
                dg[r / 4][r & 3] = fminf(fminf(dg[r / 4][r & 3], d1[r / 4][r & 3]),
                                         fminf(d2[r / 4][r & 3], d3[r / 4][r & 3]));
            }
            float near = fabsf(dg[0][0]);
#pragma unroll
            for (int r = 1; r < M; ++r) near = fminf(near, fabsf(dg[r / 4][r & 3]));
            const bool full = near_cap(q.filled);
            if (!full && !ballot64(near < band)) {
              if (ballot64((unsigned)(q.j - s0) < (unsigned)M)) {   // the wave's own atoms
#pragma unroll
                for (int r = 0; r < M; ++r)
                  emit(r, ballot64(dg[r / 4][r & 3] < 0.f && q.j != s0 + r), q.j, false);
              } else {
#pragma unroll
                for (int r = 0; r < M; ++r)
                  emit(r, ballot64(dg[r / 4][r & 3] < 0.f), q.j, false);
              }
              return;
            }
          }
          // the exact predicate: a pair inside the band, a box too small for
          // one image per tile, or a list near its capacity
          for (unsigned m = tile; m; m &= m - 1u) {
            const int r = __builtin_ctz(m);
            const uint4 p = pos4[s0 + r];        // (scalar loads)
            const float rli = rcut[s0 + r] + skin;
            const float dx = disp(q.c.x, p.x, qx);
            const float dy = disp(q.c.y, p.y, qy);
            const float dz = disp(q.c.z, p.z, qz);
            const uint64_t ok = ballot64(dist2(dx, dy, dz) < rli * rli) & valid &
                                ~ballot64(q.j == s0 + r);
#pragma unroll
            for (int t = 0; t < M; ++t)
              if (t == r) emit(t, ok, q.j, true);
          }
        };
        // the gathers of the next chunk are in flight while one is tested
        Chunk cur = next();
        while (cur.filled > 0) {
          const Chunk nx = next();
          asm volatile("" ::: "memory");
          test(cur);
          cur = nx;
        }
      }
    }
    // an overflowing list keeps its first cap entries (the partials below
    // carry the full count, from which the host regrows), so no reader of the
    // list ever runs past its rows
    int c = cnt[0];
#pragma unroll
    for (int r = 1; r < M; ++r) c = lane == r ? cnt[r] : c;
    if (lane < na) nnb[s0 + lane] = min(c, cap);
  }
  // longest list and total list length per kBuildTile atoms
  int mx = 0, tot = 0;
#pragma unroll
  for (int r = 0; r < M; ++r) {
    mx = max(mx, cnt[r]);
    tot += cnt[r];
  }
  if (lane == 0) s_part[wib] = make_int2(mx, tot);
  __syncthreads();
  constexpr int W = kBuildTile / M;   // wavefronts per entry
  static_assert(W >= 1 && kBuildWaves % W == 0, "whole part[] entries per block");
  if ((int)threadIdx.x < kBuildWaves / W) {
    int2 v = s_part[threadIdx.x * W];
    for (int w = 1; w < W; ++w) {
      const int2 u = s_part[threadIdx.x * W + w];
      v.x = max(v.x, u.x);
      v.y += u.y;
    }
    part[blockIdx.x * (kBuildWaves / W) + threadIdx.x] = v;
  }
}

// ---------------------------------------------------------- sparse build --
//
// The same lists, entry for entry, with a group of four lanes per atom and a
// window of each atom's own: in a dilute gas the atoms of a tile lie far apart
// along their column, and the window of all of them holds many times the
// candidates of each; and in boxes of two to three list radii tiles have much
// to test or fall apart (build_form: where the lines lie).  Lane l of a group sets
// up kSparseCols of the (x, y) columns that meet the sphere at a time: one or
// two runs each, whose bounds are loaded together; a prefix sum over the group
// turns the runs into one flat candidate sequence in LDS, of which the group
// takes kSparseUnroll candidates per lane and round, the next round's gathers
// in flight.  What bounds it: VALU issue, 74 instructions per atom where the
// tiles take 108 (250 000 atoms, 0.02 per unit volume, cutoff 2.5).
constexpr int kSparseLanes = 4;
constexpr int kSparseCols = 4;     // columns per lane per chunk
constexpr int kSparseUnroll = 6;   // candidates per lane per round

__device__ __forceinline__ int sparse_max(int v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, kWave));
  return v;
}

__global__ __launch_bounds__(kBuildBlock) void k_build_list_sparse(
    int n, int n_parts, int TF, const uint4 *__restrict__ pos4,
    const float *__restrict__ rcut, const RepInfo *__restrict__ reps,
    const int *__restrict__ start, float skin, int cap, int *__restrict__ list,
    int *__restrict__ nnb, int2 *__restrict__ part) {
  constexpr int TB = kSparseLanes, A = kWave / TB;
  constexpr int CC = kSparseCols * TB;   // columns per chunk
  constexpr int NS = 2 * CC;            // runs per chunk
  constexpr int U = kSparseUnroll;
  __shared__ int s_p0[kBuildBlock / TB][NS];    // first sorted atom of each run
  __shared__ int s_end[kBuildBlock / TB][NS];   // inclusive prefix of run lengths
  const int lane = threadIdx.x & (kWave - 1);
  const int g = lane / TB, l = lane % TB;
  const int gb = threadIdx.x / TB;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int s = wave * A + g;
  const bool act = s < n;
  const int si = act ? s : n - 1;

  const uint4 pi = pos4[si];
  const __amdgpu_buffer_rsrc_t prs = pos_rsrc_idx(pos4, n);
  const RepInfo &R = reps[pi.w >> 8];
  const float qx = R.q[0], qy = R.q[1], qz = R.q[2];
  const int ncx = R.nc[0], ncy = R.nc[1], ncz = R.nc[2];
  const float hx = R.h[0], hy = R.h[1], hz = R.h[2];
  const float ihz = 1.f / hz;
  const float rl = rcut[si] + skin;
  const float rl2 = rl * rl;
  const float rlm = rl * 1.0001f + 1e-4f;  // conservative window radius
  const float rlm2 = rlm * rlm;
  const int cx = cell_of(pi.x, ncx), cy = cell_of(pi.y, ncy),
            cz = cell_of(pi.z, ncz);
  // position inside the own cell from the low 32 bits of u * nc
  const float fx = (float)(uint32_t)((uint64_t)pi.x * (uint64_t)ncx) * (hx * 0x1p-32f);
  const float fy = (float)(uint32_t)((uint64_t)pi.y * (uint64_t)ncy) * (hy * 0x1p-32f);
  const float fz = (float)(uint32_t)((uint64_t)pi.z * (uint64_t)ncz) * (hz * 0x1p-32f);
  const int kx = (int)ceilf(rlm / hx), ky = (int)ceilf(rlm / hy),
            kz = (int)ceilf(rlm / hz);
  const bool fullx = 2 * kx + 1 >= ncx, fully = 2 * ky + 1 >= ncy,
             fullz = 2 * kz + 1 >= ncz;
  const int ox0 = fullx ? -cx : -kx, ox1 = fullx ? ncx - 1 - cx : kx;
  const int oy0 = fully ? -cy : -ky, oy1 = fully ? ncy - 1 - cy : ky;
  const int noy = oy1 - oy0 + 1;
  const int ncol = act ? (ox1 - ox0 + 1) * noy : 0;
  const int ncol_w = __builtin_amdgcn_readfirstlane(sparse_max(ncol));

  // list slots of this atom in the force kernel's layout (T = TF lanes):
  // slot(k) = sbase + (k / TF) * 64 + k % TF, TF a power of two
  const int AF = kWave / TF;
  const int lt = __builtin_ctz((unsigned)TF);
  const size_t sbase =
      (size_t)(si / AF) * (size_t)cap * (size_t)AF + (size_t)((si % AF) * TF);
  int *const lrow = list + sbase;
  int *const sp0 = s_p0[gb];
  int *const send = s_end[gb];
  int count = 0;
  for (int cbase = 0; cbase < ncol_w; cbase += CC) {
    // runs of this lane's kSparseCols columns -> (first atom, length) in LDS
    const int slot0 = l * 2 * kSparseCols;
    int tot = 0;
    // this lane's first column; the following ones step oy, then ox
    int c = cbase + l * kSparseCols;
    int ox = ox0 + c / noy, oy = oy0 + c % noy;
#pragma unroll 2
    for (int m = 0; m < kSparseCols; ++m, ++c) {
      int ra0 = 0, rb0 = -1, ra1 = 0, rb1 = -1, colbase = 0;
      if (c < ncol) {
        float gx = 0.f, gy = 0.f;
        if (!fullx) gx = ox > 0 ? ox * hx - fx : (ox < 0 ? fx + (-ox - 1) * hx : 0.f);
        if (!fully) gy = oy > 0 ? oy * hy - fy : (oy < 0 ? fy + (-oy - 1) * hy : 0.f);
        gx = fmaxf(gx, 0.f);
        gy = fmaxf(gy, 0.f);
        const float gxy2 = gx * gx + gy * gy;
        if (gxy2 < rlm2) {
          int cxw = cx + ox;
          cxw += cxw < 0 ? ncx : 0;
          cxw -= cxw >= ncx ? ncx : 0;
          int cyw = cy + oy;
          cyw += cyw < 0 ? ncy : 0;
          cyw -= cyw >= ncy ? ncy : 0;
          colbase = R.cell_off + (cxw * ncy + cyw) * ncz;
          rb0 = ncz - 1;  // whole column unless the chord is shorter
          if (!fullz) {
            // (the window radius carries a 1e-4 margin, far above the
            // rounding of a multiplication by 1/hz)
            const float dz = sqrtf(fmaxf(rlm2 - gxy2, 0.f));
            const int lo = cz + (int)floorf((fz - dz) * ihz);
            const int hi = cz + (int)floorf((fz + dz) * ihz);
            if (hi - lo + 1 < ncz) {
              if (lo < 0) {
                ra0 = lo + ncz; rb0 = ncz - 1; ra1 = 0; rb1 = hi;
              } else if (hi >= ncz) {
                ra0 = lo; rb0 = ncz - 1; ra1 = 0; rb1 = hi - ncz;
              } else {
                ra0 = lo; rb0 = hi;
              }
            }
          }
        }
      }
      const int b0 = rb0 >= ra0 ? start[colbase + ra0] : 0;
      const int e0 = rb0 >= ra0 ? start[colbase + rb0 + 1] : 0;
      const int b1 = rb1 >= ra1 ? start[colbase + ra1] : 0;
      const int e1 = rb1 >= ra1 ? start[colbase + rb1 + 1] : 0;
      // runs lie inside [0, n) by construction; the clamps keep every gather
      // in bounds whatever the cell offsets hold
      const int q0 = min(max(b0, 0), n), q1 = min(max(b1, 0), n);
      const int n0 = max(min(e0, n) - q0, 0), n1 = max(min(e1, n) - q1, 0);
      sp0[slot0 + 2 * m] = q0;
      send[slot0 + 2 * m] = n0;       // length for now, prefix below
      sp0[slot0 + 2 * m + 1] = q1;
      send[slot0 + 2 * m + 1] = n1;
      if (++oy > oy1) {
        oy = oy0;
        ++ox;
      }
      tot += n0 + n1;
    }
    // flat sequence: prefix over the group (lane-major slot order)
    int incl = tot;
#pragma unroll
    for (int o = 1; o < TB; o <<= 1) {
      const int t = __shfl_up(incl, o, TB);
      if (l >= o) incl += t;
    }
    const int T = __shfl(incl, TB - 1, TB);
    int run = incl - tot;
    for (int r = 0; r < 2 * kSparseCols; ++r) {
      run += send[slot0 + r];
      send[slot0 + r] = run;
    }
    __builtin_amdgcn_wave_barrier();
    // stream the flat sequence: in round k0 lane l takes the U consecutive
    // candidates v = (k0 TB + l) U + u
    const int rounds = __builtin_amdgcn_readfirstlane(sparse_max((T + TB * U - 1) / (TB * U)));
    // cursor over the runs: run cur covers flat indices [send[cur-1],
    // end) and candidate v of it is sorted atom off + v (kept in registers;
    // LDS is read only when the cursor moves to the next run)
    int cur = 0, end = send[0], off = sp0[0];
    // candidates of round k0 and their gathers (a lane past the sequence
    // takes its own atom si, which the self test below rejects)
    auto load = [&](int k0, int *jj, uint4 *cj) {
      const int v0 = (k0 * TB + l) * U;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = v0 + u;
        int j = si;
        if (v < T) {
          while (v >= end) {
            ++cur;
            const int b = end;
            end = send[cur];
            off = sp0[cur] - b;
          }
          j = off + v;
        }
        jj[u] = j;
        cj[u] = gather_pos_idx<false>(prs, j);
      }
      asm volatile("" ::: "memory");
    };
    // the accepted candidates of a round, placed in flat-sequence order
    // (lane by lane, each lane's U candidates in turn: an exclusive prefix
    // of the lanes' accepted counts over the group), so that consecutive
    // list entries are consecutive candidates -- neighbouring atoms of one
    // cell column -- and the force kernel's lanes of one atom gather from
    // the same few cache lines
    auto accept = [&](const int *jj, const uint4 *cj) {
      bool ok[U];
      int c = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dx = disp(cj[u].x, pi.x, qx);
        const float dy = disp(cj[u].y, pi.y, qy);
        const float dz2 = disp(cj[u].z, pi.z, qz);
        // (an inactive group, s >= n, has no candidates: all its lanes
        // hold j = si)
        ok[u] = (jj[u] != si) & (dist2(dx, dy, dz2) < rl2);
        c += ok[u] ? 1 : 0;
      }
      int incl = c;
#pragma unroll
      for (int o = 1; o < TB; o <<= 1) {
        const int t = __shfl_up(incl, o, TB);
        if (l >= o) incl += t;
      }
      int k = count + incl - c;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (ok[u] && k < cap) lrow[(unsigned)(((k >> lt) << 6) + (k & (TF - 1)))] = jj[u];
        k += ok[u] ? 1 : 0;
      }
      count += __shfl(incl, TB - 1, TB);
    };
    // software pipeline: the gathers of round k0 + 1 are in flight while
    // round k0 is tested; whole pairs of rounds in the loop (no branch in its
    // body, so each gather is waited for only where it is used), the odd
    // last round after it (every branch is wave-uniform)
    int ja[U], jb[U];
    uint4 ca[U], cb[U];
    load(0, ja, ca);
    int k0 = 0;
    for (; k0 + 1 < rounds; k0 += 2) {
      load(k0 + 1, jb, cb);
      accept(ja, ca);
      load(k0 + 2, ja, ca);
      accept(jb, cb);
    }
    if (k0 < rounds) accept(ja, ca);
    __builtin_amdgcn_wave_barrier();  // LDS reuse by the next chunk
  }
  // an overflowing list keeps its first cap entries (the partials below carry
  // the full count, from which the host regrows), so no reader of the list
  // ever runs past its rows
  if (act && l == 0) nnb[s] = min(count, cap);
  // this wave's longest list and total list length
  int m = act ? count : 0;
  int t = (act && l == 0) ? count : 0;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    m = max(m, __shfl_xor(m, o, kWave));
    t += __shfl_xor(t, o, kWave);
  }
  if (lane == 0 && wave < n_parts) part[wave] = make_int2(m, t);
}

int build_part_count(int mode, int n, int n_cols) {
  if (n <= 0) return 0;
  if (mode == 1) return (n + kWave - 1) / kWave + n_cols;  // tile grid
  // whole blocks of the launch with the most atoms per wavefront
  constexpr int per_block = kBuildWaves * 8;
  return (n + per_block - 1) / per_block * (per_block / kBuildTile);
}

static bool needs_images(const RepInfo &R, float skin) {
  const float rlm = (R.rc_max + skin) * 1.0001f + 1e-4f;
  for (int d = 0; d < 2; ++d)
    if (!(0.5001f * R.h[d] < 0.5f * R.L[d] - rlm)) return true;
  return false;
}

// Windows per atom where a rebuild is faster with them for the batch as a whole.
// x = list entries per atom at the mean density and the replica's largest cutoff;
// rebuild with tiles / with windows per atom, us.
// (a) Dilute: x < 16 and 40 000 atoms (uniform and graded cutoffs of 2.5 to 5).
//   16 000 atoms   x = 3.3  70.5 / 71.6    x = 12.5   71.3 / 76.2   x = 23   48.5 / 56.0
//   40 000         x = 3.3  74.0 / 69.8    x = 12.5   85.3 / 82.6   x = 23   76.0 / 75.4
//   120 000        x = 3.3 107.6 / 97.3    x = 12.5  140.8 / 125.3  x = 23  122.1 / 120.0
//   600 000        x = 3.3 276.8 / 246.5   x = 12.5  392.5 / 347.7  x = 23  344.1 / 354.9
//   1 500 000      x = 3.3 544.9 / 468.6   x = 12.5  822.4 / 715.2  x = 23  690.3 / 731.1
// (at x = 18.4 within 5 % at every size).  A drop or a film in a large box has a
// low mean too, but its lists are a liquid's, more than 60 entries: once such
// lists have been met, tiles (a gas of 16 entries hardly has one of 40).
// (b) Boxes so short along z that a tile's window takes in the whole column
// where its atoms' own do not, which has the tile done atom by atom (2.8 to 3.15
// list radii along z at the default cells; liquids, tiles over windows):
//                        5 000   11 000   16 000   60 000  100 000  200 000  400 000 atoms
//   cube of 2.9  x = 69    1.15     1.21     1.23     1.59     2.71     2.82     3.02
//   (second      x = 250   1.01     1.12     1.13     1.27     1.93     1.86     1.84
//   images too)  x = 468   1.00     1.09     1.13     1.14     1.75     1.53     1.46
//                x = 785                     1.08     1.09     1.54     1.31     1.21
//                x = 1491                    1.00     0.93     1.35     1.13     1.01
//   plate 6 x 6 x 2.9
//                x = 69    0.99     1.05     1.10     1.48     2.09     2.09     2.24
//                x = 113   0.93     0.97     1.01     1.17     1.70     1.66     1.70
//                x = 172   0.90     0.90     0.94     1.02     1.52     1.51     1.48
//                x = 250   0.92     0.91     0.97     0.93     1.42     1.29     1.25
//                x = 347                     0.87     0.81     1.31     1.02     0.97
//                x = 468   0.97     0.97     0.96     0.79     1.13     0.94     0.83
// (4 x 4 x 3: 1.14 at x = 172 and 60 000, 1.23 at x = 468 and 100 000; cubes of
// 3.1 lie near the plates).  With eight atoms a tile spans more of its cell
// than with four, so more tiles are done atom by atom.  A batch of 80 000 atoms
// in which such boxes hold a part only, the rest in cubes of 5:
//   cube of 2.9, x = 69   100 000 atoms: a quarter 1.11, 45 % 1.37   300 000: 1.14, 1.39
//   4 x 4 x 3,   x = 250  100 000        a quarter 1.11, 45 % 1.26   300 000: 0.94, 1.08
// (60 000 atoms: 0.83 to 1.13); so from a quarter of the atoms on, else a half.
// (c) Boxes whose atoms see second images (x < 200), or so short along z that a
// tile's pairs take the exact predicate (x < 500): 40 000 atoms.
//   cube of 2.1 list radii, x = 69   24 000  50.2 / 46.7   65 000  72.9 / 61.7   400 000  259 / 208
//   2.6 x 8 x 8 list radii, x = 69   24 000  56.3 / 61.1   65 000  85.8 / 77.0   400 000  314 / 279
//   cube of 2.6, x = 113            400 000  357 / 297     x = 172   439 / 394   x = 260  514 / 510
//   plate of 2.05, x = 69           400 000  328 / 305     x = 260   752 / 696   x = 470  1195 / 1050
//   (plate of 2.35, x = 69          400 000  330 / 321     x = 260   583 / 746)
BuildForm build_form(const RepInfo *reps, int n_rep, float skin, bool dense) {
  double atoms = 0.0, dilute = 0.0, whole = 0.0, small = 0.0;
  bool images = false;
  for (int r = 0; r < n_rep; ++r) atoms += reps[r].n_atoms;
  for (int r = 0; r < n_rep; ++r) {
    const RepInfo &R = reps[r];
    const double rl = (double)R.rc_max + skin;
    const double rho = R.n_atoms / ((double)R.L[0] * R.L[1] * R.L[2]);
    const double x = 4.18879 * rl * rl * rl * rho;
    const bool second = needs_images(R, skin);
    // a tile's length along its column: 4 or 8 atoms, or a cell, inside which
    // they are in caller order
    const double len = std::max((double)R.h[2], (atoms < kTileAtoms ? 4 : 8) /
                                                    (rho * R.h[0] * R.h[1]));
    const bool column = 2 * (int)ceil(rl / R.h[2]) + 1 < R.nc[2] &&
                        (len + 2.0 * rl) / R.h[2] + 2.0 > R.nc[2];
    const bool flat = 0.3 * R.h[2] > 0.5 * R.L[2] - rl;
    const double most_x = second ? (atoms < 6000.0       ? 0.0
                                    : atoms < kTileAtoms ? 1000.0
                                                         : 1500.0)
                                 : (atoms < 10000.0      ? 0.0
                                    : atoms < 20000.0    ? 100.0
                                    : atoms < 40000.0    ? 128.0
                                    : atoms < kTileAtoms ? 200.0
                                    : atoms < 150000.0   ? 500.0
                                                         : 400.0);
    const bool own = column && x < most_x;
    if (x < 16.0 && !dense) dilute += R.n_atoms;
    if (own) whole += R.n_atoms;
    if ((second && x < 200.0) || own || (flat && x < 500.0)) small += R.n_atoms;
    images |= second;
  }
  const double most = 0.5 * atoms;
  if (atoms >= 40000.0 && (dilute > most || small > most)) return BuildForm::kSparse;
  if (whole > (atoms < kTileAtoms ? most : 0.25 * atoms)) return BuildForm::kSparse;
  return images ? BuildForm::kImages : BuildForm::kTiles;
}

template <int M, int TF>
static void launch_build_m(BuildForm form, int n, const uint4 *pos4, const float *rcut,
                           const RepInfo *reps, const int *start, float skin, int cap,
                           int *list, size_t list_len, int *nnb, int2 *part, hipStream_t st) {
  constexpr int most = kBuildWaves * 8;   // every part[] entry is written
  const dim3 g((n + most - 1) / most * (8 / M)), b(kBuildBlock);
  if (form == BuildForm::kImages)
    hipLaunchKernelGGL((k_build_list<M, TF, true>), g, b, 0, st, n, pos4, rcut, reps, start,
                       skin, cap, list, list_len, nnb, part);
  else
    hipLaunchKernelGGL((k_build_list<M, TF, false>), g, b, 0, st, n, pos4, rcut, reps, start,
                       skin, cap, list, list_len, nnb, part);
}

void launch_build_list(int force_lanes, BuildForm form, int n, const uint4 *pos4,
                       const float *rcut, const RepInfo *reps, const int *start,
                       float skin, int cap, int *list, size_t list_len, int *nnb,
                       int2 *part, hipStream_t st) {
  if (n <= 0) return;
  if (form == BuildForm::kSparse) {
    constexpr int per_block = kBuildBlock / kSparseLanes;
    hipLaunchKernelGGL(k_build_list_sparse, dim3((n + per_block - 1) / per_block),
                       dim3(kBuildBlock), 0, st, n, build_part_count(0, n, 0), force_lanes,
                       pos4, rcut, reps, start, skin, cap, list, nnb, part);
    return;
  }
  // Four atoms per wavefront while eight leave the chip short of wavefronts
  // to even out the heavy ones (interface atoms): the list build alone takes
  // 15.4 against 19.0 us at 4 000 atoms (uniform cutoff) and 39.7 against
  // 42.8 us at 62 500 (slab); at 90 000 a rebuild takes 127.0 against 124.3,
  // at 1 000 000 582 against 501 us, since eight share the candidates' local
  // coordinates and half as many tiles set up windows.
  const bool few = n < kTileAtoms;
#define SRE_BUILD(TF)                                                                       \
  do {                                                                                      \
    if (few)                                                                                \
      launch_build_m<4, TF>(form, n, pos4, rcut, reps, start, skin, cap, list, list_len,  \
                            nnb, part, st);                                                 \
    else                                                                                    \
      launch_build_m<8, TF>(form, n, pos4, rcut, reps, start, skin, cap, list, list_len,  \
                            nnb, part, st);                                                 \
  } while (0)
  switch (force_lanes) {
    case 1: SRE_BUILD(1); break;
    case 2: SRE_BUILD(2); break;
    case 4: SRE_BUILD(4); break;
    case 8: SRE_BUILD(8); break;
    default: SRE_BUILD(16); break;
  }
#undef SRE_BUILD
}

// ------------------------------------------------------------ tile build --
//
// One wave per tile: up to 64 consecutive cell-sorted atoms of one (x, y)
// cell column.  The tile's candidate region is the union of its atoms'
// spheres: the columns within (rl_max + margin) of the tile's column and, in
// each, the z cells from the tile's lowest cell - kz to its highest + kz --
// one or two contiguous runs of sorted atoms.  Runs are staged 64 atoms at a
// time in LDS and every lane tests its own atom against each staged candidate
// (a broadcast LDS read), so all loops are wave-uniform and the only
// divergence is the list write of an accepted pair.  The predicate is the
// same exact one as above; entries are written in candidate order.

__device__ __forceinline__ int find_replica_by_col(const RepInfo *reps, int n_rep,
                                                   int c) {
  int lo = 0, hi = n_rep - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (reps[mid].col_off <= c) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ __launch_bounds__(256) void k_col_tiles(int n_cols, int n_rep,
                                                   const RepInfo *reps,
                                                   const int *start, int tile,
                                                   uint32_t *tiles_per_col) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cols) return;
  const RepInfo &R = reps[find_replica_by_col(reps, n_rep, c)];
  const int base = R.cell_off + (c - R.col_off) * R.nc[2];
  const int cnt = start[base + R.nc[2]] - start[base];
  tiles_per_col[c] = (uint32_t)((cnt + tile - 1) / tile);
}

__global__ __launch_bounds__(kWave) void k_build_tiles(
    int n_cols, int n_rep, int TF, const uint32_t *__restrict__ tile_off,
    const uint32_t *__restrict__ tiles_per_col, const uint4 *__restrict__ pos4,
    const float *__restrict__ rcut, const RepInfo *__restrict__ reps,
    const int *__restrict__ start, float skin, int cap, int *__restrict__ list,
    int *__restrict__ nnb, int2 *__restrict__ part) {
  __shared__ uint4 cand[kWave];
  const int t = blockIdx.x;
  const int n_tiles = (int)(tile_off[n_cols - 1] + tiles_per_col[n_cols - 1]);
  if (t >= n_tiles) {  // the grid is an upper bound of the tile count
    if (threadIdx.x == 0) part[t] = make_int2(0, 0);
    return;
  }
  // column of this tile: last c with tile_off[c] <= t
  int lo = 0, hi = n_cols - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int)tile_off[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  const int c = lo;
  const RepInfo &R = reps[find_replica_by_col(reps, n_rep, c)];
  const int ncx = R.nc[0], ncy = R.nc[1], ncz = R.nc[2];
  const float hx = R.h[0], hy = R.h[1], hz = R.h[2];
  const float qx = R.q[0], qy = R.q[1], qz = R.q[2];
  const int col = c - R.col_off;
  const int cx = col / ncy, cy = col - cx * ncy;
  const int cbase = R.cell_off + col * ncz;
  const int a0 = start[cbase] + (t - (int)tile_off[c]) * kWave;
  const int a1 = min(start[cbase + ncz], a0 + kWave);
  const int lane = threadIdx.x;
  const int s = a0 + lane;
  const bool act = s < a1;
  const uint4 pi = pos4[act ? s : a0];
  const float rl = rcut[act ? s : a0] + skin;
  const float rl2 = rl * rl;
  float rlmax = act ? rl : 0.f;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1)
    rlmax = fmaxf(rlmax, __shfl_xor(rlmax, o, kWave));
  const float rlm = rlmax * 1.0001f + 1e-4f;
  const float rlm2 = rlm * rlm;
  const int cz_lo = cell_of(pos4[a0].z, ncz), cz_hi = cell_of(pos4[a1 - 1].z, ncz);
  const int kx = (int)ceilf(rlm / hx), ky = (int)ceilf(rlm / hy),
            kz = (int)ceilf(rlm / hz);
  const bool fullx = 2 * kx + 1 >= ncx, fully = 2 * ky + 1 >= ncy;
  const int ox0 = fullx ? -cx : -kx, ox1 = fullx ? ncx - 1 - cx : kx;
  const int oy0 = fully ? -cy : -ky, oy1 = fully ? ncy - 1 - cy : ky;
  // list slots of this lane's atom (layout of the force kernel, T = TF)
  const int A = kWave / TF;
  const int lt = __builtin_ctz((unsigned)TF);
  const size_t sbase = act ? (size_t)(s / A) * (size_t)cap * A + (size_t)((s % A) * TF) : 0;
  int count = 0;
  for (int ox = ox0; ox <= ox1; ++ox) {
    const float gx = fullx ? 0.f : fmaxf(0.f, (float)(abs(ox) - 1) * hx);
    if (gx * gx >= rlm2) continue;
    int cxw = cx + ox;
    cxw += cxw < 0 ? ncx : 0;
    cxw -= cxw >= ncx ? ncx : 0;
    for (int oy = oy0; oy <= oy1; ++oy) {
      const float gy = fully ? 0.f : fmaxf(0.f, (float)(abs(oy) - 1) * hy);
      if (gx * gx + gy * gy >= rlm2) continue;
      int cyw = cy + oy;
      cyw += cyw < 0 ? ncy : 0;
      cyw -= cyw >= ncy ? ncy : 0;
      const int colbase = R.cell_off + (cxw * ncy + cyw) * ncz;
      int ra0 = 0, rb0 = ncz - 1, ra1 = 0, rb1 = -1;
      const int zl = cz_lo - kz, zh = cz_hi + kz;
      if (zh - zl + 1 < ncz) {
        if (zl < 0) {
          ra0 = zl + ncz; rb0 = ncz - 1; ra1 = 0; rb1 = zh;
        } else if (zh >= ncz) {
          ra0 = zl; rb0 = ncz - 1; ra1 = 0; rb1 = zh - ncz;
        } else {
          ra0 = zl; rb0 = zh;
        }
      }
      for (int run = 0; run < 2; ++run) {
        const int ca = run ? ra1 : ra0, cb = run ? rb1 : rb0;
        if (cb < ca) continue;
        const int p0 = start[colbase + ca], p1 = start[colbase + cb + 1];
        for (int p = p0; p < p1; p += kWave) {
          const int q = p + lane;
          cand[lane] = pos4[q < p1 ? q : p0];
          __syncthreads();
          const int m = min(kWave, p1 - p);
          for (int k = 0; k < m; ++k) {
            const uint4 cj = cand[k];
            const float d2 = dist2(disp(cj.x, pi.x, qx), disp(cj.y, pi.y, qy),
                                   disp(cj.z, pi.z, qz));
            const int j = p + k;
            if (act && j != s && d2 < rl2) {
              if (count < cap)
                list[sbase + ((size_t)(count >> lt) << 6) + (count & (TF - 1))] = j;
              ++count;
            }
          }
          __syncthreads();
        }
      }
    }
  }
  if (act) nnb[s] = min(count, cap);   // as in k_build_list
  int mx = count, tot = count;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    mx = max(mx, __shfl_xor(mx, o, kWave));
    tot += __shfl_xor(tot, o, kWave);
  }
  if (lane == 0) part[t] = make_int2(mx, tot);
}

void launch_tile_map(int n_cols, int n_rep, const RepInfo *reps, const int *start,
                     int tile, uint32_t *tiles_per_col, uint32_t *tile_off,
                     uint32_t *scan_tmp, hipStream_t st) {
  if (n_cols <= 0) return;
  hipLaunchKernelGGL(k_col_tiles, dim3((n_cols + 255) / 256), dim3(256), 0, st,
                     n_cols, n_rep, reps, start, tile, tiles_per_col);
  device_exscan_u32((size_t)n_cols, tiles_per_col, tile_off, scan_tmp, st);
}

void launch_build_tiles(int n, int n_cols, int n_rep, int force_lanes,
                        const uint4 *pos4, const float *rcut,
                        const RepInfo *reps, const int *start, float skin,
                        int cap, int *list, int *nnb, int2 *part,
                        uint32_t *tiles_per_col, uint32_t *tile_off,
                        uint32_t *scan_tmp, hipStream_t st) {
  if (n <= 0 || n_cols <= 0) return;
  launch_tile_map(n_cols, n_rep, reps, start, kWave, tiles_per_col, tile_off, scan_tmp,
                  st);
  // every column adds at most one partial tile
  const int max_tiles = (n + kWave - 1) / kWave + n_cols;
  hipLaunchKernelGGL(k_build_tiles, dim3(max_tiles), dim3(kWave), 0, st, n_cols,
                     n_rep, force_lanes, tile_off, tiles_per_col, pos4, rcut,
                     reps, start, skin, cap, list, nnb, part);
}

}  // namespace sre
