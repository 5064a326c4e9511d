// BiCGStab runs that stay on the chip: one launch iterates to the end, each
// block holding one stencil tile of every vector in registers (gfx950).
//
// The launch-per-phase iteration (pb_krylov2d.hip) is bound by the fixed
// chain of a launch (dispatch, state and partial records, then the tile's
// loads) and by re-reading ten vectors per iteration: 29 us per iteration at
// 1025x513 and 12-14 us at 161x81, where the vectors' own traffic would take
// 11 us and 0.3 us.  A grid whose tiles are all resident at once (64 x 4 RY
// nodes per 256-thread block, up to ~770 blocks) needs neither: r, p, v, t,
// r~, x, diag_inv and the cell weights fit the register file (38 of its 128
// MB at 1025x513), and what blocks exchange is one ring of edge values and a
// few sums per stencil.  FP64 at 4-row tiles, us per iteration, launches ->
// resident: two phases 14.0 -> 6.7 (161x81), 13.6 -> 9.8 (513x257), 24.7 ->
// 15.3 (1025x513); the exact variant's three 18.7 -> 9.1, 18.5 -> 13.5, 28.5 ->
// 19.3.  What is left is latency: per phase at 161x81 about 1.5 us for the
// hand-over and 1.9 us for the chain combine, stencil, sums, scalars of one
// tile.  (x updated in the chain instead of behind the hand-over: 7.3; eight
// waves per tile instead of four: 6.8; waves that sleep between polls: 7.3.)
//
// Exchange.  Every word that crosses blocks carries its own tag: 8-byte
// relaxed agent-scope atomics holding 32 bits of a value and the 32-bit
// number of the phase it belongs to.  A reader polls the data itself, so one
// trip through memory is both the hand-over and the synchronisation; no
// counter, fence or cache flush.  Measured for an all-reduce of one value:
// 2.0 / 2.2 / 2.3 us at 32 / 64 / 256 blocks, against 4.5 / 17 us at 64 / 256
// for an atomic-counter barrier alone.  Up to kDirect = 96 blocks each block
// sums all records itself; above, one wave per value, record class and copy
// (up to eight copies, for a share of the readers each) sums them and every
// block reads 4 class sums.  Per iteration of two phases, all reading all
// against class sums: 11.9 against 10.2 us at 153 tiles (513x257), 8.3 against
// 8.9 us at 95.
//
// Buffers are reused without a handshake: a block writes the words of a phase
// only after it has the sums of the phase before, to which every block
// contributed after its last read of what is being overwritten.
//
// The arithmetic, the tile numbering and every summation order are those of
// the launches, so the iterates are bitwise theirs.
//
// Every wait is bounded (kWaitTicks).  When one runs out, because the blocks
// are not all resident next to other work, the launch ends without a result
// and the caller runs the launches.  Room is accounted for per device, so that
// runs of several streams or threads of a process are not resident in part; for
// what the account does not see, as another process on the device, the wait is
// short and a context that has given up kMaxGiveUps times stops trying.
#include <atomic>
#include <type_traits>
#include <vector>

#include "pb_resident2d.hpp"

using namespace pb2d;

// The launches' products that feed a sum are contracted; here, where the flux
// products meet their sums in registers instead of through LDS, each fused
// operation is written out and nothing else is contracted.
#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// the next lane's value (lane 63 receives zero)
__device__ __forceinline__ float next_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double next_lane(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// lane k's value in every lane
__device__ __forceinline__ float from_lane(float v, int k) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}
__device__ __forceinline__ double from_lane(double v, int k) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, k), hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

typedef unsigned long long u64;
typedef unsigned int u32;

constexpr int kRecValues = 8;        // records per tile: A 1, B 5, C 2
constexpr int kDirect = 96;          // tiles up to which every block sums the records itself
constexpr int kMaxPerLane = 3;       // records of a class sum's lane: up to 768 tiles
constexpr int kCopies = 8;           // copies of the class sums
constexpr int kSumWords = 64;        // words of one copy's class sums (<= 40 used)
constexpr long long kWaitTicks = 20000000LL;   // 0.2 s of the 100 MHz clock; a phase takes ~10 us
constexpr int kSkipAfterAbort = 64;  // solves of a context that go by launches after a wait ran out
constexpr int kMaxGiveUps = 3;       // and after so many, all of them

template <typename T>
struct RMember {
  OpDev<T> op;
  const T* b;
  const T* r0;
  const double* x0;
  double* x;
  ResOut* out;
  u64* halo_v;
  u64* halo_t;
  u64* rec;
  u64* sums;
  KState init;
  u32 epoch;
  int begin, nbx, nby;
};

// Pointers out of the member table are generic; as global ones their accesses
// are not flat ones, which would also hold up the LDS counter.
template <typename P>
__device__ __forceinline__ __attribute__((address_space(1))) P* glob(P* p) {
  return (__attribute__((address_space(1))) P*)p;
}

__device__ __forceinline__ void put_word(u64* p, u64 v) {
  __hip_atomic_store(glob(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get_word(const u64* p) {
  return __hip_atomic_load(glob(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A tagged value: two words for a double, one for a float.
template <typename T>
struct Tagged;
template <>
struct Tagged<double> {
  static constexpr int W = 2;
  u64 a, b;
  __device__ static void put(u64* p, double v, u32 tag) {
    const u64 w = (u64)__double_as_longlong(v);
    put_word(p, (w << 32) | tag);
    put_word(p + 1, (w & 0xffffffff00000000ull) | tag);
  }
  __device__ void load(const u64* p) {
    a = get_word(p);
    b = get_word(p + 1);
  }
  __device__ bool ready(u32 tag) const { return (u32)a == tag && (u32)b == tag; }
  __device__ double value() const { return __longlong_as_double((long long)((a >> 32) | (b & 0xffffffff00000000ull))); }
};
template <>
struct Tagged<float> {
  static constexpr int W = 1;
  u64 a;
  __device__ static void put(u64* p, float v, u32 tag) { put_word(p, ((u64)__float_as_uint(v) << 32) | tag); }
  __device__ void load(const u64* p) { a = get_word(p); }
  __device__ bool ready(u32 tag) const { return (u32)a == tag; }
  __device__ float value() const { return __uint_as_float((u32)(a >> 32)); }
};

// Poll until attempt() holds; false when the time is up or the member has
// been given up by another block.
template <class F>
__device__ __forceinline__ bool poll(const int* abort, F&& attempt) {
  long long t0 = 0;
  for (int n = 1;; ++n) {
    if (attempt()) return true;
    if ((n & 63) == 0) {
      const long long now = wall_clock64();
      if (t0 == 0) t0 = now;
      if (now - t0 > kWaitTicks) return false;
      if (__hip_atomic_load(glob(abort), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    }
  }
}

__global__ void k_clear_words(long n, u64* w) {
  for (long g = blockIdx.x * (long)blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x) w[g] = 0;
}

// One tile of one member for a whole run.  All blocks of a launch are resident
// at once (run_jobs), so any tile order is right; each takes its tile from the
// ticket counter in the order the blocks start.  Tiles by block index instead,
// us per iteration, exact / fast: 161x81 (18 tiles) 8.9 / 6.7 -> 9.5 / 7.2,
// 257x129 (45) 9.9 / 7.4 -> 10.5 / 7.7; above 96 tiles, where a few blocks form
// the class sums for all, the index is the better order (513x257, 153 tiles:
// 13.9 / 10.0 -> 11.8 / 9.0).
template <typename T, bool CROSS, bool CENTER, int RY, bool EXACT, int MINB>
__global__ __launch_bounds__(NTHR, MINB) void k_resident(const RMember<T>* __restrict__ tab, int nmem, u32* ticket,
                                                   u32 ticket0) {
  constexpr int TY = TYT * RY;
  constexpr int NW = NTHR / kWave;
  constexpr int W = Tagged<T>::W;
  constexpr bool LATE = MINB == 2 && RY <= 4;   // registers to update x in while the words travel
  // the stencil's input with its ring, and spare rows that take the stores of
  // threads past the grid
  __shared__ T sp[(TY + 2 + RY) * (TX + 2)];
  __shared__ T so[TY * TX];               // its output
  __shared__ double sred[5 * NW], ssum[5 * NW];
  // used once per phase by the thread they belong to, so kept off the registers
  __shared__ T Lrt[TY * TX], Ldv[RY][NTHR];
  __shared__ double Lx[RY][NTHR];
  __shared__ KState sst;
  __shared__ int sdead, sid;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + TX * ty;
  const int lane = tid & (kWave - 1), wid = tid / kWave;
  if (tid == 0) {
    sdead = 0;
    sid = (int)(atomicAdd(ticket, 1u) - ticket0);
  }
  for (int k = tid; k < (TY + 2 + RY) * (TX + 2); k += NTHR) sp[k] = T(0);
  // A class of records no tile belongs to adds zero.  Cleared here, before the
  // barrier, and not in the exchanges: which classes are written depends on the
  // tile count alone, and from 65 to 96 tiles other waves write theirs with no
  // barrier in between.
  if (tid < 5 * NW) ssum[tid] = 0.0;
  __syncthreads();
  const int blk = __builtin_amdgcn_readfirstlane(sid);
  int m = 0;
  for (int lo = 0, hi = nmem - 1;;) {
    if (lo >= hi) {
      m = lo;
      break;
    }
    const int mid = (lo + hi + 1) >> 1;
    if (tab[mid].begin <= blk) lo = mid;
    else hi = mid - 1;
  }
  const RMember<T>& M = tab[m];
  if (tid == 0) sst = M.init;   // read first after the first exchange's barrier
  const int local = blk - M.begin, nbx = M.nbx, nby = M.nby, nb = nbx * nby;
  const int bx = local % nbx, by = local / nbx;
  const int nx = M.op.nx, ny = M.op.ny;
  const int i0 = bx * TX, j0 = by * TY;
  const int H = min(TY, ny - j0), Wd = min(TX, nx - i0);   // the tile's own nodes
  int* const abort = &M.out->abort;

  // own nodes: rows ty RY + q of column tx (a wave's rows are consecutive, so
  // its cells' fluxes serve two rows).  The sums take rows ty + TYT q, the
  // launches' order, from LDS.
  T r[RY], p[RY], v[RY], t[RY], hv[RY];
  double vals[5];
  int okm = 0, oks = 0;
#pragma unroll
  for (int q = 0; q < RY; ++q) {
    const int j = j0 + ty * RY + q, i = i0 + tx;
    const bool ok = j < ny && i < nx;
    okm |= (int)ok << q;
    oks |= (int)(j0 + ty + TYT * q < ny && i < nx) << q;
    const long g = ok ? (long)j * nx + i : 0;
    r[q] = ok ? glob(M.r0)[g] : T(0);
    Lrt[(ty * RY + q) * TX + tx] = r[q];
    Ldv[q][tid] = ok ? glob(M.op.dinv)[g] : T(0);
    hv[q] = (CENTER && ok) ? glob(M.op.hc)[g] : T(0);
    Lx[q][tid] = (M.x0 && ok) ? glob(M.x0)[g] : 0.0;
    p[q] = v[q] = t[q] = T(0);
  }
  // weights of the cells left of the own nodes, RY + 1 cell rows, and, in lane
  // c <= RY, of cell row c right of the tile's last column
  T wa[RY + 1], wb[RY + 1], wc[RY + 1], wd[RY + 1], ea, eb, ec, ed;
  auto weights = [&](int cy, int cx, T& a, T& b, T& c, T& d) {
    const int j = j0 + cy, i = i0 + cx;
    const bool cok = j <= ny && i <= nx;
    const long cc = cok ? (long)j * (nx + 1) + i : 0;
    a = cok ? glob(M.op.wxx)[cc] : T(0);
    b = cok ? glob(M.op.wyy)[cc] : T(0);
    c = (CROSS && cok) ? glob(M.op.wyx)[cc] : T(0);
    d = (CROSS && cok) ? glob(M.op.wxy)[cc] : T(0);
  };
#pragma unroll
  for (int c = 0; c <= RY; ++c) weights(ty * RY + c, tx, wa[c], wb[c], wc[c], wd[c]);
  const int erow = ty * RY + min(lane, RY);
  weights(erow, TX, ea, eb, ec, ed);
  // The ring of nodes around the tile, one per thread: rows -1 and H over
  // columns -1..Wd, then columns -1 and Wd over rows 0..H-1, with the
  // operator's wrap (-1 -> n - 2, n -> 1).  Row values are exchanged by row
  // class (first and last row of every tile row, then rows 1 and ny - 2 for
  // the wrap), column values by column class likewise.
  const int nring = 2 * (Wd + 2) + 2 * H;
  const bool ring = tid < nring;
  int rpos = 0;
  int rsrc = 0, rnode = 0;
  const int colbase = (2 * nby + 2) * nx;
  if (ring) {
    int lr, lc;
    if (tid < 2 * (Wd + 2)) {
      lr = tid < Wd + 2 ? -1 : H;
      lc = (tid < Wd + 2 ? tid : tid - (Wd + 2)) - 1;
    } else {
      const int k = tid - 2 * (Wd + 2);
      lr = k < H ? k : k - H;
      lc = k < H ? -1 : Wd;
    }
    int j = j0 + lr, i = i0 + lc;
    const int jw = j < 0 ? ny - 2 : (j == ny ? 1 : j), iw = i < 0 ? nx - 2 : (i == nx ? 1 : i);
    if (tid < 2 * (Wd + 2)) {
      const int cls = j < 0 ? 2 * nby + 1 : (j == ny ? 2 * nby : (lr < 0 ? 2 * by - 1 : 2 * by + 2));
      rsrc = cls * nx + iw;
    } else {
      const int cls = i < 0 ? 2 * nbx + 1 : (i == nx ? 2 * nbx : (lc < 0 ? 2 * bx - 1 : 2 * bx + 2));
      rsrc = colbase + cls * ny + jw;
    }
    rpos = (lr + 1) * (TX + 2) + lc + 1;
    rnode = jw * nx + iw;
    if (nb == 1) rsrc = jw * TX + iw;   // the only tile: its own value, in so
  }
  T hr = ring ? glob(M.r0)[rnode] : T(0), hp = T(0), hvv = T(0), ht = T(0);

  // The tile's values that others read, out of so: its first and last row
  // and column, and rows 1 and ny - 2, columns 1 and nx - 2 for the wrap.
  auto len_other = [&](bool row) { return row ? H : Wd; };
  const int wr0 = 1 - j0, wr1 = ny - 2 - j0, wc0 = 1 - i0, wc1 = nx - 2 - i0;   // their tile rows and columns
  auto publish = [&](u64* buf, u32 tag) {
    const int n = 4 * Wd + 4 * H;
    for (int e = tid; e < n; e += NTHR - kWave) {
      const bool row = e < 4 * Wd;
      const int len = row ? Wd : H, k = row ? e : e - 4 * Wd;
      const int which = k >= 2 * len ? (k >= 3 * len ? 3 : 2) : (k >= len ? 1 : 0), at = k - which * len;
      // the tile row or column of this list, and its class
      const int line = which == 0 ? 0 : which == 1 ? len_other(row) - 1 : which == 2 ? (row ? wr0 : wc0) : (row ? wr1 : wc1);
      if (line < 0 || line >= len_other(row)) continue;
      const int cls = which < 2 ? 2 * (row ? by : bx) + which : 2 * (row ? nby : nbx) + which - 2;
      const int ly = row ? line : at, lx = row ? at : line;
      const int dst = row ? cls * nx + i0 + at : colbase + cls * ny + j0 + at;
      Tagged<T>::put(buf + (u32)dst * W, so[ly * TX + lx], tag);
    }
  };

  // y = diag_inv (A in) on the own nodes, also left in so; ``in`` = own values
  // c and the ring's value h.  A thread forms the fluxes of the cells left of
  // its nodes, the right ones come from the next lane; stencil_tile2's
  // operations in its order, with 5 LDS words per node instead of 15.
  auto flux = [](T tl, T tr, T bl, T br, T a, T b, T c, T d, T& fx, T& fy) {
    const T gx = (tr - tl) + (br - bl);
    const T gy = (bl - tl) + (br - tr);
    fx = CROSS ? fma_(a, gx, c * gy) : a * gx;
    fy = CROSS ? fma_(b, gy, d * gx) : b * gy;
  };
  auto stencil = [&](const T(&c)[RY], T h, T(&y)[RY]) {
    T* const row0 = sp + (ty * RY) * (TX + 2) + tx;   // left of the row above the own ones
    T* const spare = sp + (TY + 2) * (TX + 2) + tx;
    T* const own = tx < Wd ? row0 + (TX + 2) + 1 : spare;
#pragma unroll
    for (int q = 0; q < RY; ++q) (ty * RY + q < H ? own : spare)[q * (TX + 2)] = c[q];
    if (ring) sp[rpos] = h;
    __syncthreads();
    T left[RY + 2], mid[RY + 2], fx[RY + 1], fy[RY + 1], ex, ey;
#pragma unroll
    for (int k = 0; k < RY + 2; ++k) left[k] = row0[k * (TX + 2)];
    // the own column from LDS too: a tile's ring row or column may lie inside it
#pragma unroll
    for (int k = 0; k < RY + 2; ++k) mid[k] = row0[k * (TX + 2) + 1];
    {
      const T* e = sp + erow * (TX + 2) + TX;
      const T e0 = e[0], e1 = e[1], e2 = e[TX + 2], e3 = e[TX + 3];
      flux(e0, e1, e2, e3, ea, eb, ec, ed, ex, ey);
    }
#pragma unroll
    for (int k = 0; k <= RY; ++k)
      flux(left[k], mid[k], left[k + 1], mid[k + 1], wa[k], wb[k], wc[k], wd[k], fx[k], fy[k]);
    T fxr[RY + 1], fyr[RY + 1];
#pragma unroll
    for (int k = 0; k <= RY; ++k) {
      fxr[k] = next_lane(fx[k]);
      fyr[k] = next_lane(fy[k]);
      const T ox = from_lane(ex, k), oy = from_lane(ey, k);
      if (lane == kWave - 1) {
        fxr[k] = ox;
        fyr[k] = oy;
      }
    }
#pragma unroll
    for (int q = 0; q < RY; ++q) {
      T acc = ((fxr[q] + fxr[q + 1]) - (fx[q] + fx[q + 1])) + ((fy[q + 1] + fyr[q + 1]) - (fy[q] + fyr[q]));
      if (CENTER) acc = fma_(hv[q], c[q], acc);
      y[q] = Ldv[q][tid] * acc;   // past the grid: unused
      so[(ty * RY + q) * TX + tx] = y[q];
    }
    __syncthreads();
  };

  // One phase's hand-over: the tile's edges out (from so) and the ring's
  // values in, if ``buf``; ``vals`` summed over every tile and given to
  // ``scalars``, which advances the run's state sst.  ``meanwhile`` runs once
  // the tile's words are out.  REC: the phase's first record value.  False: a
  // wait ran out.
  auto exchange = [&](auto nv_, auto rec_, u64* buf, T* h, u32 tag, auto&& meanwhile, auto&& scalars) -> bool {
    constexpr int NV = decltype(nv_)::value, REC = decltype(rec_)::value;
    constexpr int LAST = NW - 1;
    wave_sum_n<NV>(reinterpret_cast<double(&)[NV]>(vals));
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < NV; ++k) sred[k * NW + wid] = vals[k];
    }
    __syncthreads();
    bool good = true;
    u64* const rec = M.rec + (u32)(REC * nb * 2);
    if (wid == LAST) {
      double own = 0.0;
      if (lane < NV) {
#pragma unroll
        for (int w = 0; w < NW; ++w) own += sred[lane * NW + w];
      }
      // Classes no tile belongs to are zero already (prologue).  Written again in
      // the three-block kinds, whose registers spill, the loop's assignment is the
      // better one: 1025x513 20.2 / 16.0 -> 19.3 / 15.3 us per exact / fast
      // iteration; the two-block kinds lose 1 % by it.
      if (MINB == 3 && lane < NV * NW && (lane % NW) * kWave >= nb) ssum[lane] = 0.0;
      if (nb == 1) {
        if (lane < NV) ssum[lane * NW] = own;
      } else if (lane < NV) {
        Tagged<double>::put(rec + (u32)(lane * nb + local) * 2, own, tag);
      }
    } else if (buf && nb > 1) {
      publish(buf, tag);
    }
    meanwhile();
    // The order of sum_partials: class w adds records 64 w + lane + 256 h,
    // then its lanes; the class sums are added in order of w.
    if (nb > kDirect) {
      if (wid == LAST) {
        const int ncopy = min(kCopies, nb / (NW * NV));
        u64* const sums = M.sums + REC * kCopies * kSumWords;
        if (local < ncopy * NW * NV) {   // this block sums one value of one class for one copy
          const int copy = local / (NW * NV), kw = local % (NW * NV);
          const u64* const src = rec + (u32)((kw / NW) * nb) * 2;
          Tagged<double> w[kMaxPerLane];
          const int b = (kw % NW) * kWave + lane;
          good = poll(abort, [&] {
            bool all = true;
#pragma unroll
            for (int h = 0; h < kMaxPerLane; ++h) w[h].load(src + (u32)min(b + h * NTHR, nb - 1) * 2);
#pragma unroll
            for (int h = 0; h < kMaxPerLane; ++h) all = all && w[h].ready(tag);
            return all;
          });
          double s[1] = {0.0};
#pragma unroll
          for (int h = 0; h < kMaxPerLane; ++h)
            if (b + h * NTHR < nb) s[0] += w[h].value();
          wave_sum_n<1>(s);
          if (lane == 0) Tagged<double>::put(sums + (u32)(copy * kSumWords + kw * 2), s[0], tag);
        }
        if (lane < NV * NW) {
          Tagged<double> w;
          const u64* src = sums + (u32)((local % ncopy) * kSumWords + lane * 2);
          good = poll(abort, [&] {
            w.load(src);
            return w.ready(tag);
          }) && good;
          ssum[lane] = w.value();
        }
      }
    } else if (nb > 1) {
      const int cls = LAST - wid;   // the last wave, which has no edges to publish, takes class 0
      if (cls * kWave < nb) {
        const int b = min(cls * kWave + lane, nb - 1);
        Tagged<double> w[NV];
        good = poll(abort, [&] {
          bool all = true;
#pragma unroll
          for (int k = 0; k < NV; ++k) w[k].load(rec + (u32)(k * nb + b) * 2);
#pragma unroll
          for (int k = 0; k < NV; ++k) all = all && w[k].ready(tag);
          return all;
        });
        double s[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) s[k] = cls * kWave + lane < nb ? w[k].value() : 0.0;
        wave_sum_n<NV>(s);
        if (lane == 0) {
#pragma unroll
          for (int k = 0; k < NV; ++k) ssum[k * NW + cls] = s[k];
        }
      }
    }
    if (buf && ring) {
      if (nb == 1) {
        *h = so[rsrc];
      } else {
        Tagged<T> w;
        const u64* src = buf + (u32)rsrc * W;
        good = poll(abort, [&] {
          w.load(src);
          return w.ready(tag);
        }) && good;
        *h = w.value();
      }
    }
    if (!good) sdead = 1;
    if (nb > kWave && nb <= kDirect) __syncthreads();   // several waves wrote class sums
    if (wid == LAST) {
      __builtin_amdgcn_wave_barrier();
      double tot[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        tot[k] = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) tot[k] += ssum[k * NW + w];
      }
      KState st = sst;
      scalars(st, tot);
      if (lane == 0) sst = st;
    }
    __syncthreads();
    return sdead == 0;
  };
  using std::integral_constant;
  const integral_constant<int, 0> recA{};
  const integral_constant<int, 1> recB{}, one{};
  const integral_constant<int, 2> two{};
  const integral_constant<int, 5> five{};
  const integral_constant<int, 6> recC{};

  u32 tag = M.epoch;
  auto give_up = [&] {
    if (tid == 0) __hip_atomic_store(glob(abort), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  // r0.r0 and b.b
  vals[0] = vals[1] = 0.0;
#pragma unroll
  for (int q = 0; q < RY; ++q) {
    if (oks >> q & 1) {
      const long g = (long)(j0 + ty + TYT * q) * nx + i0 + tx;
      const double rd = (double)glob(M.r0)[g], bd = (double)glob(M.b)[g];
      vals[0] = fma_(rd, rd, vals[0]);
      vals[1] = fma_(bd, bd, vals[1]);
    }
  }
  if (!exchange(two, recC, nullptr, nullptr, ++tag, [] {}, [](KState& st, const double(&tot)[2]) {
        st = scalars_after_init(st, tot[0], tot[1]);
        st.phase = PH_A;
      }))
    return give_up();
  for (;;) {
    if (sst.status != ST_RUN) {
      if (sst.status >= ST_P_CONV) {   // final x update of a finished run (fast variant)
        const bool half = sst.status == ST_P_HALF;
        const T alpha = (T)sst.alpha;
#pragma unroll
        for (int q = 0; q < RY; ++q) {
          const double xg = fma_(sst.alpha, (double)p[q], Lx[q][tid]);
          const T s = fma_(-alpha, v[q], r[q]);
          Lx[q][tid] = half ? xg : fma_(sst.omega, (double)s, xg);
        }
      }
      break;
    }
    // A: p and v = A p
    T xp[RY], xs[RY];   // the last iteration's p and s, for x
    const double alpha_x = sst.alpha, omega_x = sst.omega;
    const int xupd = !EXACT && sst.x_upd;
    {
      const double alpha_d = alpha_x, omega_d = omega_x;
      const T alpha = (T)alpha_d, omega = (T)omega_d, beta = (T)sst.beta;
      if (EXACT) {
#pragma unroll
        for (int q = 0; q < RY; ++q) p[q] = fma_(beta, fma_(-omega, v[q], p[q]), r[q]);
        hp = fma_(beta, fma_(-omega, hvv, hp), hr);
      } else {
#pragma unroll
        for (int q = 0; q < RY; ++q) {
          const T s = fma_(-alpha, v[q], r[q]);
          const T rn = fma_(-omega, t[q], s);
          if (LATE) {
            xp[q] = p[q];
            xs[q] = s;
          } else if (xupd) {
            Lx[q][tid] = fma_(omega_d, (double)s, fma_(alpha_d, (double)p[q], Lx[q][tid]));
          }
          p[q] = fma_(beta, fma_(-omega, v[q], p[q]), rn);
          r[q] = rn;
        }
        const T rn = fma_(-omega, ht, fma_(-alpha, hvv, hr));
        hp = fma_(beta, fma_(-omega, hvv, hp), rn);
        hr = rn;
      }
    }
    stencil(p, hp, v);
    ++tag;
    vals[0] = 0.0;
#pragma unroll
    for (int q = 0; q < RY; ++q) {
      const int k = (ty + TYT * q) * TX + tx;
      if (oks >> q & 1) vals[0] = fma_((double)Lrt[k], (double)so[k], vals[0]);
    }
    auto update_x = [&] {
      if (LATE && xupd) {
#pragma unroll
        for (int q = 0; q < RY; ++q)
          Lx[q][tid] = fma_(omega_x, (double)xs[q], fma_(alpha_x, (double)xp[q], Lx[q][tid]));
      }
    };
    if (!exchange(one, recA, M.halo_v, &hvv, tag, update_x, [](KState& st, const double(&tot)[1]) {
          const double alpha = st.rho / tot[0];
          st.phase = PH_B;
          if (tot[0] == 0.0 || !isfinite(alpha)) st.status = ST_BRK_OMEGA;
          else st.alpha = alpha;
        }))
      return give_up();
    if (sst.status != ST_RUN) break;
    const double alpha_d = sst.alpha;
    const T alpha = (T)alpha_d;
    // B: s and t = A s
    T sv[RY];
#pragma unroll
    for (int q = 0; q < RY; ++q) sv[q] = fma_(-alpha, v[q], r[q]);
    stencil(sv, fma_(-alpha, hvv, hr), t);
    ++tag;
#pragma unroll
    for (int k = 0; k < 5; ++k) vals[k] = 0.0;
#pragma unroll
    for (int q = 0; q < RY; ++q) {
      const int ly = ty + TYT * q, k = ly * TX + tx;
      if (oks >> q & 1) {
        const double sd = (double)sp[(ly + 1) * (TX + 2) + tx + 1], yd = (double)so[k], rd = (double)Lrt[k];
        vals[0] = fma_(sd, sd, vals[0]);
        vals[1] = fma_(yd, sd, vals[1]);
        vals[2] = fma_(yd, yd, vals[2]);
        vals[3] = fma_(rd, sd, vals[3]);
        vals[4] = fma_(rd, yd, vals[4]);
      }
    }
    if (!exchange(five, recB, M.halo_t, &ht, tag, [] {}, [](KState& st, const double(&tot)[5]) {
          if (!EXACT) {
            st = scalars_after_b(st, tot);
            st.phase = PH_A;
            return;
          }
          // the exact variant's ||s|| test and omega
          const double snrm = sqrt(tot[0]);
          const double om = tot[1] / tot[2];
          if (snrm <= st.atol) {
            st.phase = PH_L3;
            st.resid = snrm;
            st.half = 1;
            st.status = ST_P_HALF;
          } else if (!isfinite(om) || !isfinite(snrm)) {
            st.status = ST_BRK_OMEGA;
          } else {
            st.phase = PH_L3;
            st.omega = om;
          }
        }))
      return give_up();
    if (!EXACT) continue;
    // the exact variant's update of x and r
    if (sst.status != ST_RUN && sst.status != ST_P_HALF) break;
    const bool half = sst.status == ST_P_HALF;
    const double omega_d = sst.omega;
    const T omega = (T)omega_d;
    T sn[RY];
#pragma unroll
    for (int q = 0; q < RY; ++q) {
      sn[q] = fma_(-alpha, v[q], r[q]);
      if (half) {
        Lx[q][tid] = fma_(alpha_d, (double)p[q], Lx[q][tid]);
      } else {
        r[q] = fma_(-omega, t[q], sn[q]);
        so[(ty * RY + q) * TX + tx] = r[q];
      }
    }
    if (half) break;
    __syncthreads();
    hr = fma_(-omega, ht, fma_(-alpha, hvv, hr));
    vals[0] = vals[1] = 0.0;
#pragma unroll
    for (int q = 0; q < RY; ++q) {
      const int k = (ty + TYT * q) * TX + tx;
      if (oks >> q & 1) {
        const double rn = (double)so[k];
        vals[0] = fma_((double)Lrt[k], rn, vals[0]);
        vals[1] = fma_(rn, rn, vals[1]);
      }
    }
    auto update_x_exact = [&] {
#pragma unroll
      for (int q = 0; q < RY; ++q)
        Lx[q][tid] = fma_(omega_d, (double)sn[q], fma_(alpha_d, (double)p[q], Lx[q][tid]));
    };
    if (!exchange(two, recC, nullptr, nullptr, ++tag, update_x_exact, [](KState& st, const double(&tot)[2]) {
          st = scalars_after_l3(st, tot[0], tot[1]);
          st.phase = PH_A;
        }))
      return give_up();
  }
#pragma unroll
  for (int q = 0; q < RY; ++q)
    if (okm >> q & 1) glob(M.x)[(long)(j0 + ty * RY + q) * nx + i0 + tx] = Lx[q][tid];
  if (local == 0 && tid == 0) {
    KState st = sst;
    if (st.status == ST_P_HALF) st.half = 1;
    st.status = finalize(st.status);
    M.out->st = st;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Compute units (CUs) taken by resident launches, per device.  A launch of at
// most a block per CU is charged a CU per block, rounded up to the same number on
// every XCD: blocks go to the XCDs in turn and spread over their CUs, and a CU
// that holds blocks of one kind may have no registers or LDS left for another.
// So on every XCD each run finds as many CUs without foreign blocks as it has
// blocks there.  A larger launch, several blocks to a CU, is charged the device
// and runs alone; a run that finds no room goes by launches.
constexpr int kXcds = 8;
int units_of(int tiles, int n_cu) { return std::min(n_cu, ceil_div(tiles, kXcds) * kXcds); }

constexpr int kMaxDev = 64;
std::atomic<int> g_cus_taken[kMaxDev];

struct Room {
  std::atomic<int>* taken = nullptr;
  int cus = 0;
  bool acquire(int device, int n, int have) {
    if (device < 0 || device >= kMaxDev) return false;
    std::atomic<int>& a = g_cus_taken[device];
    int cur = a.load();
    while (cur + n <= have) {
      if (a.compare_exchange_weak(cur, cur + n)) {
        taken = &a;
        cus = n;
        return true;
      }
    }
    return false;
  }
  ~Room() {
    if (taken) taken->fetch_sub(cus);
  }
};

template <typename T>
using ResKernel = void (*)(const RMember<T>*, int, u32*, u32);

template <typename T, int RY, bool EXACT, int MINB>
ResKernel<T> pick_kind(bool cross, bool center) {
  if (cross) return center ? k_resident<T, true, true, RY, EXACT, MINB> : k_resident<T, true, false, RY, EXACT, MINB>;
  return center ? k_resident<T, false, true, RY, EXACT, MINB> : k_resident<T, false, false, RY, EXACT, MINB>;
}
// The kernel of a tile height for grids of ``nb`` tiles.  Blocks per CU that
// the registers are to leave room for: two; three up to 3-row tiles, and for
// 4-row tiles on grids with more than two tiles per CU (1025x513: 561).  Spilled
// VGPRs of the FP64 kinds: 2 rows 0-6, 3 rows 4-36, 4 rows 27-80 with three
// blocks and none with two, 5 rows 0-25, 6 rows 3-59, 8 rows (one block) none;
// no FP32 kind spills.
template <typename T, bool EXACT>
ResKernel<T> pick(int ry, bool cross, bool center, bool many) {
  switch (ry) {
    case 2: return pick_kind<T, 2, EXACT, 3>(cross, center);
    case 3: return pick_kind<T, 3, EXACT, 3>(cross, center);
    case 5: return pick_kind<T, 5, EXACT, 2>(cross, center);
    case 6: return pick_kind<T, 6, EXACT, 2>(cross, center);
    case 8: return pick_kind<T, 8, EXACT, 2>(cross, center);
    default:
      return many ? pick_kind<T, 4, EXACT, 3>(cross, center) : pick_kind<T, 4, EXACT, 2>(cross, center);
  }
}
template <typename T>
ResKernel<T> pick(int ry, bool cross, bool center, bool exact, bool many) {
  // the mixed mode's FP32 runs use the fast variant only
  if constexpr (std::is_same<T, double>::value) {
    if (exact) return pick<T, true>(ry, cross, center, many);
  }
  return pick<T, false>(ry, cross, center, many);
}

constexpr long kSumsAll = (long)kRecValues * kCopies * kSumWords;

// Memory of the resident runs, taken once a run is known to fit.  Without it the
// runs go by launches, which need none of it: false, and no error left behind.
bool take(hipError_t e) {
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess;
}

bool ensure_records(ResRecords& rec, size_t bytes, hipStream_t s) {
  if (!rec.ticket) {
    void* p = nullptr;
    if (!take(hipMalloc(&p, 256))) return false;
    rec.ticket = (unsigned*)p;
    rec.ticket_next = 0;
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(64), 0, s, 32L, (u64*)p);
  }
  if (rec.bytes >= bytes) return true;
  if (rec.dev) (void)hipFree(rec.dev);
  if (rec.host) (void)hipHostFree(rec.host);
  rec.dev = rec.host = nullptr;
  rec.bytes = 0;
  if (!take(hipMalloc(&rec.dev, bytes)) || !take(hipHostMalloc(&rec.host, bytes, hipHostMallocDefault))) return false;
  rec.bytes = bytes;
  return true;
}

bool ensure_words(pb_op2d* op) {
  Resident* R = resident_of(op);
  if (R->words) return true;
  // sized for the finest tiling, so every tile height uses the same buffers
  const dim3 g = stencil_grid(op, 2);
  R->halo_words = 2 * ((2L * g.y + 2) * op->g.nx + (2L * g.x + 2) * op->g.ny);
  R->rec_words = 2L * kRecValues * g.x * g.y;
  void* p = nullptr;
  if (!take(hipMalloc(&p, sizeof(u64) * (2 * R->halo_words + R->rec_words + kSumsAll)))) return false;
  R->words = (u64*)p;
  return true;
}

}  // namespace

void pb2d::ResRecords::release() {
  if (dev) (void)hipFree(dev);
  if (host) (void)hipHostFree(host);
  if (ticket) (void)hipFree(ticket);
  *this = ResRecords{};
}

Resident* pb2d::resident_of(pb_op2d* op) {
  if (!op->res) op->res = new Resident();
  return op->res;
}

void pb2d::resident_free(pb_op2d* op) {
  if (!op->res) return;
  op->res->records.release();
  if (op->res->words) (void)hipFree(op->res->words);
  delete op->res;
  op->res = nullptr;
}

namespace {
// resident_run without its switch and counts; kGaveUp when a wait ran out
constexpr int kGaveUp = 2;
template <typename T>
int run_jobs(pb_ctx* ctx, ResRecords& rec, const ResJob<T>* jobs, int count, bool exact, hipStream_t s, KState* out,
             const std::function<void()>& prepare) {
  for (int m = 0; m < count; ++m)   // tags of a run: three per iteration, far from wrapping
    if (jobs[m].maxiter > (1 << 28)) return 0;
  // Launches of one kind of kernel each, the members with the most tiles first,
  // and never more tiles in one launch than are resident at once: blocks go to
  // the XCDs in turn, so a member that had to wait for slots of another could
  // get all of them on some XCDs and too few on others, and wait for good.
  std::vector<int> order(count);
  for (int m = 0; m < count; ++m) order[m] = m;
  auto kind = [&](int m) {
    const pb_op2d* op = jobs[m].op;
    return op->ry * 4 + (op->cross ? 2 : 0) + (op->center ? 1 : 0);
  };
  auto tiles = [&](int m) {
    const dim3 g = stencil_grid(jobs[m].op, jobs[m].op->ry);
    return (int)(g.x * g.y);
  };
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return kind(a) != kind(b) ? kind(a) < kind(b) : tiles(a) > tiles(b);
  });
  // check the room of every launch before the first one
  int need = 0;
  struct Span {
    int f, e;
    ResKernel<T> fn;
  };
  std::vector<Span> spans;
  for (int f = 0; f < count;) {
    const pb_op2d* op = jobs[order[f]].op;
    const ResKernel<T> fn = pick<T>(op->ry, op->cross, op->center, exact, tiles(order[f]) > 2 * ctx->n_cu);
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void*)fn, NTHR, 0) != hipSuccess || occ < 1) return 0;
    const int slots = occ * ctx->n_cu;
    if (tiles(order[f]) > std::min(slots, kMaxPerLane * NTHR)) return 0;
    int e = f, total = 0;
    while (e < count && kind(order[e]) == kind(order[f]) && total + tiles(order[e]) <= slots) total += tiles(order[e++]);
    need = std::max(need, units_of(total, ctx->n_cu));
    spans.push_back(Span{f, e, fn});
    f = e;
  }
  Room room;
  if (!room.acquire(ctx->device, need, ctx->n_cu)) return 0;
  const size_t tab_bytes = (sizeof(RMember<T>) * count + 255) / 256 * 256, out_bytes = sizeof(ResOut) * count;
  if (!ensure_records(rec, tab_bytes + out_bytes, s)) return 0;
  for (int m = 0; m < count; ++m)
    if (!ensure_words(jobs[m].op)) return 0;
  if (prepare) prepare();
  RMember<T>* const tab = (RMember<T>*)rec.host;
  ResOut* const res = (ResOut*)((char*)rec.host + tab_bytes);
  RMember<T>* const dtab = (RMember<T>*)rec.dev;
  ResOut* const dres = (ResOut*)((char*)rec.dev + tab_bytes);
  const int give_up = ctx->resident_mode.load() == PB_RESIDENT_GIVE_UP;   // as if a wait had run out
  std::vector<int> total;
  for (int k = 0; k < count; ++k) {
    if (total.size() < spans.size() && k == spans[total.size()].f) total.push_back(0);
    const ResJob<T>& J = jobs[order[k]];
    pb_op2d* op = J.op;
    Resident* R = op->res;
    const u32 span = 3u * (u32)J.maxiter + 8u;
    if (!R->cleared || R->epoch > 0xffffffffu - span) {
      const long words = 2 * R->halo_words + R->rec_words + kSumsAll;
      hipLaunchKernelGGL(k_clear_words, dim3(elem_blocks(words)), dim3(256), 0, s, words, R->words);
      R->cleared = true;
      R->epoch = 0;
    }
    const dim3 g = stencil_grid(op, op->ry);
    RMember<T>& M = tab[k];
    M.op = opdev<T>(op);
    M.b = J.b;
    M.r0 = J.r0;
    M.x0 = J.x0;
    M.x = J.x;
    M.out = dres + k;
    res[k].abort = give_up;
    M.halo_v = R->words;
    M.halo_t = R->words + R->halo_words;
    M.rec = R->words + 2 * R->halo_words;
    M.sums = M.rec + R->rec_words;
    M.init = KState{};
    M.init.tol = J.tol;
    M.init.maxiter = J.maxiter;
    M.init.legacy = J.legacy;
    M.init.status = ST_RUN;
    M.init.phase = PH_INIT;
    M.epoch = R->epoch;
    M.begin = total.back();
    M.nbx = (int)g.x;
    M.nby = (int)g.y;
    total.back() += (int)(g.x * g.y);
    R->epoch += span;
  }
  PB_HIP(ctx, hipMemcpyAsync(rec.dev, rec.host, tab_bytes + out_bytes, hipMemcpyHostToDevice, s));
  for (size_t l = 0; l < spans.size(); ++l) {
    hipLaunchKernelGGL(spans[l].fn, dim3((unsigned)total[l]), dim3(TX, TYT), 0, s, (const RMember<T>*)(dtab + spans[l].f),
                       spans[l].e - spans[l].f, rec.ticket, rec.ticket_next);
    PB_LAUNCH_CHECK(ctx);
    rec.ticket_next += (unsigned)total[l];
  }
  PB_HIP(ctx, hipMemcpyAsync(res, dres, out_bytes, hipMemcpyDeviceToHost, s));
  PB_HIP(ctx, hipStreamSynchronize(s));
  for (int k = 0; k < count; ++k) {
    if (res[k].abort) return kGaveUp;
  }
  for (int k = 0; k < count; ++k) out[order[k]] = res[k].st;
  ctx->resident_count[PB_RESIDENT_LAUNCHES] += (long long)spans.size();
  return 1;
}
}  // namespace

template <typename T>
int pb2d::resident_run(pb_ctx* ctx, ResRecords& rec, const ResJob<T>* jobs, int count, bool exact, hipStream_t s,
                       KState* out, const std::function<void()>& prepare) {
  int rc = 0;
  const bool on = ctx->resident_mode.load() != PB_RESIDENT_OFF && ctx->resident_give_ups.load() < kMaxGiveUps;
  if (on && ctx->resident_skip.load() > 0) ctx->resident_skip.fetch_sub(1);
  else if (on) rc = run_jobs<T>(ctx, rec, jobs, count, exact, s, out, prepare);
  if (rc < 0) return rc;
  ctx->resident_count[rc == 1 ? PB_RESIDENT_RUNS : rc == kGaveUp ? PB_RESIDENT_GIVEN_UP : PB_RESIDENT_DECLINED] += count;
  if (rc == kGaveUp) {
    ctx->resident_give_ups.fetch_add(1);
    ctx->resident_skip.store(kSkipAfterAbort);
  }
  return rc == 1;
}

extern "C" int pb_resident_units(int tiles, int n_cu) { return tiles < 1 || n_cu < 1 ? PB_ERR_ARG : units_of(tiles, n_cu); }

template int pb2d::resident_run<double>(pb_ctx*, ResRecords&, const ResJob<double>*, int, bool, hipStream_t, KState*,
                                        const std::function<void()>&);
template int pb2d::resident_run<float>(pb_ctx*, ResRecords&, const ResJob<float>*, int, bool, hipStream_t, KState*,
                                       const std::function<void()>&);
