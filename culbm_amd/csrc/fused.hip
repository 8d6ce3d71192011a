// Two steps per launch with the intermediate populations kept in LDS (the
// mixed L1/L2 blocking of the reference, HALO_BLOCKING_L1L2,
// kernel.cu:138-329, redesigned for the 160 KB LDS of a gfx950 CU).
//
// A workgroup owns a TX x TY tile of cells and marches along z over a chunk
// of planes.  For each plane it computes the first step on the tile plus a
// one-cell xy halo ("A" cells, pulled from src in HBM) into one LDS plane, then
// the second step of the tile ("B" cells) into dst.  The second step of plane z
// pulls the c_z = +1 populations of plane z-1, the c_z = 0 ones of plane z and
// the c_z = -1 ones of plane z+1: a B cell reads each group from the LDS plane
// while that plane is there (c_z = +1 a plane later) and carries 18 values in
// registers until its own plane is complete, so the LDS holds 36 values per A
// cell and a tile can take all 1024 threads.
// HBM sees the first step's reads (tile + halo) and the second step's writes
// only.
//
// What bounds it, at 288x272x280 with 60 spheres on 96x8 tiles: FP32 the bytes,
// 128 per update counted (74 read of an ideal 54, 54 written) at 5.5 TB/s, above
// the 5.25 TB/s the population pattern streams at; 16-bit the VALU, 90 % busy
// (97 % with stochastic rounding; 76 and 71 bytes per update).  A ring of all
// three planes in LDS (54 values per A cell, 32x16 FP32 tiles, EQU inputs loaded
// on demand, every direction base held in scalar registers that spilled to vector
// lanes) ran 35.3k MLUPS in FP32, 53.4k in FP16, 45.3k with stochastic rounding;
// this march 42.6k, 62.5k and 54.3k (FP32 43.2k with non-temporal stores).  Of
// that, FP32: the wide tile and its waits +20 %; FP16: the same +4 %, computing in
// units of the storage scale +8 %, one barrier per plane +6 %.  Measured and left
// out: gathers two planes ahead (fewer waves or spills: FP32 64x8 34.5k), two
// workgroups of 32x12 per CU (29.5k), releasing the LDS before the second step's
// arithmetic (spills, 35.8k), non-temporal loads (30.3k; of the rows no other
// tile reads only, equal).
//
// The intermediate is kept in the storage format, exactly as a plain
// step would have stored it, so two fused steps equal two plain steps bit for
// bit.  A cell without STORE keeps its populations in both buffers (see
// culbm_set_state), so its intermediate value is its src value.
// Included by capi.hip after lbm_kernels.hip.

#include <type_traits>

namespace culbm {

// Limits of a workgroup's tile: (TX+2)(TY+2) A cells (the tile and a one-cell xy
// halo), one thread per A cell; the first TX*TY threads also hold one B cell
// each.  The sizes are chosen per domain (fused_plan).
constexpr int kFusedBlock = 1024, kFusedRows = 64;

struct FusedArgs {
  StepArgs a;
  int32_t tx, ty;            // tile (B cells)
  int32_t tiles_x, tiles_y;  // tile columns and rows
  int32_t zchunk;            // B planes per workgroup
  int32_t nchunk;
};

// LDS of one workgroup.  16-bit storage keeps two planes (three of c_z = +1),
// so a plane's first step writes while slower waves still read the one before
// and one barrier per plane is enough; FP32 has room for one (two).
template <class T>
struct FusedPlane {
  static constexpr bool kDouble = sizeof(T) == 2;
  static constexpr int kLo = kDouble ? 2 : 1, kUp = kLo + 1, kFl = 3;
  T lo[kLo][18][kFusedBlock];          // first-step populations of the latest plane(s), c_z = -1 and 0, slot = plane % kLo
  T up[kUp][9][kFusedBlock];           // c_z = +1, slot = plane % kUp
  uint8_t fl[kFl][kFusedBlock];        // step bits of the A cells (the B step's flags)
  float eq[kFl][2][kFusedRows][4];     // EQU inputs of the A cells on the low / high x face, by row
};

// Raw storage bits of one population, zero-extended.
template <class T>
__device__ __forceinline__ uint32_t to_raw(T v) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(uint32_t, v);
  else
    return __builtin_bit_cast(uint16_t, v);
}

template <class T>
__device__ __forceinline__ T from_raw(uint32_t r) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, r);
  else
    return __builtin_bit_cast(T, uint16_t(r));
}

// Pulled (not yet updated) populations of one A cell, gathered ahead so the
// HBM latency overlaps the second step of a plane before.
struct FusedPending {
  uint32_t r[27];
  uint32_t fl;
  EquIn eq;
};

// A lane's A cell (clamped into the domain).  The faces are lane masks (scalar
// registers); the offsets they select are formed anew for every plane, since
// vector registers held across the march would spill.
struct FusedLane {
  uint32_t c;           // cell index within the plane
  bool x0, x1, y0, y1;  // on the low / high face of x, of y
  bool face;            // on an x face and part of this tile
  int32_t row;          // A row within the tile
};

// Byte offsets within a plane of the sources of one A cell.
struct FusedOffsets {
  uint32_t row[3];  // clamped source row y - cy, [cy + 1], at the cell's x
  uint32_t xm, xp;  // to x-1 / x+1 (0 when clamped on that face)
};

template <int B>
__device__ __forceinline__ FusedOffsets fused_offsets(const StepArgs& a, const FusedLane& k) {
  uint32_t o = k.c * uint32_t(B), row = uint32_t(a.nx) * uint32_t(B), one = B;
  asm volatile("" : "+v"(o), "+s"(row), "+s"(one));  // not held across planes
  FusedOffsets l;
  l.row[0] = o + (k.y1 ? 0u : row);
  l.row[1] = o;
  l.row[2] = o - (k.y0 ? 0u : row);
  l.xm = k.x0 ? 0u : 0u - one;
  l.xp = k.x1 ? 0u : one;
  return l;
}

// Bounce-back register with register (v_swap_b32 under the lane mask): a swap
// through copies costs every wave 39 moves and selects whether it holds a solid
// cell or not.  (The one-step kernels keep the copies: there the tied registers
// cost occupancy, 69 -> 95 VGPRs in place.)
__device__ __forceinline__ void fused_bounce_back(float* f) {
#pragma unroll
  for (int i = 0; i < 13; ++i) asm volatile("v_swap_b32 %0, %1" : "+v"(f[i]), "+v"(f[26 - i]));
}

// update_cell on populations in units of the storage scale, for tiles about as
// wide as the domain, where most waves hold an x-face cell.
//
// An EQU cell that neither collides nor bounces (every inlet and outlet cell of
// the reference convention) takes its equilibrium from the relaxation of the
// wave's other cells: its rho/u replace the moments, and with weights 1 and -0
// on cleared populations the relaxation returns feq itself, every bit of it
// (x + -0 = x, a NaN or infinity among the pulled values cleared away), so a
// wave that meets an x face runs one equilibrium (95 instructions), not two.
template <class S>
__device__ __forceinline__ void fused_update(uint32_t fl, const StepArgs& a, uint32_t c, const EquIn& q,
                                             float* f) {
  const float one = S::kBytes == 4 ? 1.0f : a.scale;
  const bool equ = (fl & (kEqu | kBounceBack | kCollide)) == kEqu;
  float rho = q.rho, vx = q.vx, vy = q.vy, vz = q.vz;
  if ((fl & kEqu) || !(fl & kLoad)) {
    if ((fl & kEqu) && !q.ok) {  // an EQU cell off the x faces
      rho = a.rho[c];
      vx = a.vx[c];
      vy = a.vy[c];
      vz = a.vz[c];
    }
    if (S::kBytes == 2) rho *= one;
    clear(f);
    if ((fl & kEqu) && !equ) {
      EqTerms e;
      eq_terms(rho, vx, vy, vz, e, one);
      equ_one<0>(e, f);
    }
  }
  if (fl & kBounceBack) fused_bounce_back(f);
  if (equ || (fl & kCollide)) {
    Moments m = moments(f, one);
    float it = a.inv_tau, omt = a.omt;
    if (equ) {
      m = {rho, vx, vy, vz};
      it = 1.0f;
      omt = -0.0f;
    }
    EqTerms e;
    eq_terms(m.rho, m.ux, m.uy, m.uz, e, one);
    relax_one<0>(e, it, omt, f);
  }
}

// Storage bits to populations in units of the storage scale, and back.  The
// march computes on the scaled values: the host takes this kernel only where a
// power-of-two factor changes no rounding (see fused_scale_ok).
template <class S>
__device__ __forceinline__ float fused_dec(uint32_t r) {
  if constexpr (S::kBytes == 4)
    return __builtin_bit_cast(float, r);
  else if constexpr (std::is_same_v<S, StoreF16>)
    return float(from_raw<_Float16>(r));
  else
    return __builtin_bit_cast(float, r << 16);
}

template <class S, bool SR, int I>
__device__ __forceinline__ void fused_enc(const float* f, typename S::T* v, const SrHash& h) {
  if constexpr (SR)
    v[I] = S::enc_sr(f[I], 1.0f, h.template byte<I>());
  else
    v[I] = S::enc(f[I], 1.0f);
  if constexpr (I < 26) fused_enc<S, SR, I + 1>(f, v, h);
}

template <class S, int I>
__device__ __forceinline__ void fused_gather_dir(const char* const* zp, int64_t dsb, const FusedOffsets& k, uint32_t* r) {
  constexpr int cx = cx_of(I), cy = cy_of(I), cz = cz_of(I);
  const uint32_t ox = cx == 1 ? k.xm : (cx == -1 ? k.xp : 0u);
  r[I] = to_raw(ld_at<typename S::T>(zp[cz + 1] + I * dsb, k.row[cy + 1] + ox));
  if constexpr (I < 26) fused_gather_dir<S, I + 1>(zp, dsb, k, r);
}

// Every lane gathers, at a position clamped into the domain (the caller clamps
// the plane): loads issued on every path let the compiler wait for exactly one
// gather while later memory operations are still in flight.
template <class S>
__device__ __forceinline__ void fused_gather(const StepArgs& a, const FusedLane& k, int32_t p, FusedPending& q) {
  constexpr int64_t B = sizeof(typename S::T);
  const int64_t pc = int64_t(a.nx) * a.ny;
  const uint64_t zc = uint64_t(p) * uint64_t(pc);
  q.eq.ok = k.face;
  if (k.face) {
    q.eq.rho = (a.rho + zc)[k.c];
    q.eq.vx = (a.vx + zc)[k.c];
    q.eq.vy = (a.vy + zc)[k.c];
    q.eq.vz = (a.vz + zc)[k.c];
  }
  q.fl = (a.sflag + zc)[k.c];
  // one direction base at a time: without the barrier the compiler keeps all 27
  // (and the 27 of the stores) in scalar registers across the march and spills
  int64_t dsb = a.dstride * B;
  asm volatile("" : "+s"(dsb));
  const char* s = static_cast<const char*>(a.src) + zc * B;
  const char* zp[3] = {s + (p == a.nz - 1 ? 0 : pc * B), s, s - (p == 0 ? 0 : pc * B)};  // source plane p - cz
  fused_gather_dir<S, 0>(zp, dsb, fused_offsets<B>(a, k), q.r);
}

// The cell's own populations in src, one after the other (a cell without
// STORE: rare, so a rolled loop that holds no registers across the march).
template <class S, class W>
__device__ __forceinline__ void fused_keep(const StepArgs& a, uint64_t zc, uint32_t c, W&& write) {
  const typename S::T* src = static_cast<const typename S::T*>(a.src) + zc + c;
#pragma unroll 1
  for (int i = 0; i < 27; ++i) write(i, src[i * a.dstride]);
}

// First step of a gathered A cell into the LDS plane: a plain pull update (the
// state numbered a.state), or the cell's own populations when it has no STORE.
template <class S, bool SR>
__device__ __forceinline__ void fused_first(const StepArgs& a, int ac, const FusedLane& k, int32_t p,
                                            const FusedPending& q, bool ok, FusedPlane<typename S::T>& r) {
  using T = typename S::T;
  const uint64_t zc = uint64_t(p) * (uint64_t(a.nx) * uint64_t(a.ny));
  const uint32_t c = uint32_t(zc) + k.c;
  float f[27];
#pragma unroll
  for (int i = 0; i < 27; ++i) f[i] = fused_dec<S>(q.r[i]);
  fused_update<S>(q.fl, a, c, q.eq, f);
  T v[27];
  SrHash h;
  if constexpr (SR) h.make(c, a.state);
  fused_enc<S, SR, 0>(f, v, h);
  if (!ok) return;
  using P = FusedPlane<T>;
  const int sl = p % P::kUp, ll = p % P::kLo, sf = p % P::kFl;
  r.fl[sf][ac] = uint8_t(q.fl);
  if (k.face) {  // EQU inputs of the x-face cells, for the second step
    float* d = r.eq[sf][k.x0 ? 0 : 1][k.row];
    d[0] = q.eq.rho;
    d[1] = q.eq.vx;
    d[2] = q.eq.vy;
    d[3] = q.eq.vz;
  }
#pragma unroll
  for (int i = 0; i < 18; ++i) r.lo[ll][i][ac] = v[i];
#pragma unroll
  for (int j = 0; j < 9; ++j) r.up[sl][j][ac] = v[18 + j];
  if (!(q.fl & kStore)) fused_keep<S>(a, zc, k.c, [&](int i, T x) { (i < 18 ? r.lo[ll][i] : r.up[sl][i - 18])[ac] = x; });
}

template <class S, bool NT, int I>
__device__ __forceinline__ void fused_store_dir(char* base, int64_t dsb, uint32_t lb, const typename S::T* v) {
  using T = typename S::T;
  if constexpr (NT)
    __builtin_nontemporal_store(v[I], reinterpret_cast<T*>(base + I * dsb + lb));
  else
    st_at<T>(base + I * dsb, lb, v[I]);
  if constexpr (I < 26) fused_store_dir<S, NT, I + 1>(base, dsb, lb, v);
}

// NT: non-temporal stores of the second step (fused_plan says where).
template <class S, bool SR, bool NT>
__global__ __launch_bounds__(kFusedBlock) void k_fused2(const FusedArgs fa) {
  using T = typename S::T;
  using P = FusedPlane<T>;
  __shared__ P r;
  const StepArgs& a = fa.a;
  const uint32_t ntile = uint32_t(fa.tiles_x) * fa.tiles_y * fa.nchunk;
  const uint32_t w = xcd_group(blockIdx.x, ntile);
  const int32_t tx = int32_t(w % uint32_t(fa.tiles_x));
  const int32_t ty = int32_t((w / uint32_t(fa.tiles_x)) % uint32_t(fa.tiles_y));
  const int32_t zch = int32_t(w / (uint32_t(fa.tiles_x) * fa.tiles_y));
  const int32_t TX = fa.tx, TY = fa.ty, AX = TX + 2;
  const int32_t x0 = tx * TX, y0 = ty * TY;
  const int32_t nx = a.nx, ny = a.ny, nz = a.nz;
  const int32_t zs = zch * fa.zchunk, ze = min(nz, zs + fa.zchunk);
  const int t = threadIdx.x;

  // this lane's A cell, clamped into the domain
  const int32_t ax = x0 - 1 + t % AX, ay = y0 - 1 + t / AX;
  const bool a_ok = t < AX * (TY + 2) && ax >= 0 && ax < nx && ay >= 0 && ay < ny;
  FusedLane k;
  {
    const int32_t x = min(max(ax, 0), nx - 1), y = min(max(ay, 0), ny - 1);
    k.c = uint32_t(y) * uint32_t(nx) + uint32_t(x);
    k.x0 = x == 0;
    k.x1 = x == nx - 1;
    k.y0 = y == 0;
    k.y1 = y == ny - 1;
    k.face = a_ok && (k.x0 || k.x1);
    k.row = t / AX;
  }

  // One march for the waves that hold B cells and one for those that do not
  // (the last A cells, rows beyond the domain): in each, every path through the
  // loop issues the same memory operations, so a wait for a gather leaves the
  // operations issued after it in flight.
  auto march = [&](auto has_b) {
    constexpr bool HB = decltype(has_b)::value;
    // the B cell, clamped into the tile and the domain: a lane beyond them
    // repeats the last cell of its row or column and stores the same bits
    const int32_t gx = min(x0 + t % TX, nx - 1), gy = min(y0 + min(t / TX, TY - 1), ny - 1);
    const int bx = gx - x0, by = gy - y0;
    const uint32_t cxy = uint32_t(gy) * uint32_t(nx) + uint32_t(gx);
    const int bc = (by + 1) * AX + bx + 1;  // the B cell among the A cells
    const bool bx0 = gx == 0, bx1 = gx == nx - 1, by0 = gy == 0, by1 = gy == ny - 1;
    // A indices of the (clamped) source cells x - c, [cx + 1][cy + 1]
    struct Near {
      int o[3][3];
    };
    auto near = [&]() {
      int c = bc, one = 1, ax = AX;
      asm volatile("" : "+v"(c), "+s"(one), "+s"(ax));  // not held across planes
      const int rows[3] = {c + (by1 ? 0 : ax), c, c - (by0 ? 0 : ax)};
      const int xp = bx1 ? 0 : one, xm = bx0 ? 0 : one;
      Near n;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        n.o[0][j] = rows[j] + xp;
        n.o[1][j] = rows[j];
        n.o[2][j] = rows[j] - xm;
      }
      return n;
    };
    auto at = [&](const Near& n, int i) { return n.o[cx_of(i) + 1][cy_of(i) + 1]; };
    // groups carried for the next B plane: its own c_z = 0 and the c_z = +1 of
    // the plane below (of itself for z = 0)
    uint32_t mid[9], upz[9];
    auto carry = [&](int32_t z) {
      const Near n = near();
      const int su = (z == 0 ? z : z - 1) % P::kUp, sl = z % P::kLo;
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        mid[j] = to_raw(r.lo[sl][9 + j][at(n, 9 + j)]);
        upz[j] = to_raw(r.up[su][j][at(n, 18 + j)]);
      }
    };
    FusedPending q;
    int32_t p = max(zs - 1, 0);
    fused_gather<S>(a, k, p, q);
    // A plane p into LDS, and the gather of the next.  Every lane updates what
    // it gathered (no path leaves a load unwaited for), the lanes of the
    // domain's A cells write it.
    auto first = [&]() {
      fused_first<S, SR>(a, t, k, min(p, nz - 1), q, a_ok && p < nz, r);
      __builtin_amdgcn_sched_barrier(0);
      fused_gather<S>(a, k, min(p + 1, nz - 1), q);
      __syncthreads();
    };
    first();
    if constexpr (HB) carry(p);  // used where the chunk starts at z = 0
    if (zs > 0) {
      p = zs;
      __syncthreads();
      first();
      if constexpr (HB) carry(p);
    }
    // B plane z from A plane z + 1 and the carried groups.  (p = nz is not
    // written: the last plane pulls c_z = -1 from itself, the LDS still holds it.)
    auto plane = [&](int32_t z) {
      if constexpr (!P::kDouble) __syncthreads();
      p = z + 1;
      first();
      if constexpr (HB) {
        const Near n = near();
        const int sl = min(p, nz - 1) % P::kLo, sz = z % P::kFl;
        float f[27];
#pragma unroll
        for (int j = 0; j < 9; ++j) {
          f[j] = fused_dec<S>(to_raw(r.lo[sl][j][at(n, j)]));
          f[9 + j] = fused_dec<S>(mid[j]);
          f[18 + j] = fused_dec<S>(upz[j]);
        }
        const uint64_t zc = uint64_t(z) * (uint64_t(nx) * uint64_t(ny));
        const uint32_t c = uint32_t(zc) + cxy;
        const uint32_t fl = r.fl[sz][bc];
        EquIn e;
        e.ok = bx0 || bx1;
        const float* q4 = r.eq[sz][bx0 ? 0 : 1][by + 1];
        e.rho = q4[0];
        e.vx = q4[1];
        e.vy = q4[2];
        e.vz = q4[3];
        fused_update<S>(fl, a, c, e, f);
        T v[27];
        SrHash h;
        if constexpr (SR) h.make(c, a.state + 1);  // the state after the first step's
        fused_enc<S, SR, 0>(f, v, h);
        int64_t dsb = a.dstride * int64_t(sizeof(T));
        asm volatile("" : "+s"(dsb));
        uint32_t lb = cxy * uint32_t(sizeof(T));
        asm volatile("" : "+v"(lb));
        char* dst = static_cast<char*>(a.dst) + zc * sizeof(T);
        fused_store_dir<S, NT, 0>(dst, dsb, lb, v);
        if (!(fl & kStore)) {  // dst keeps its bits
          T* own = static_cast<T*>(a.dst) + zc + cxy;
          fused_keep<S>(a, zc, cxy, [&](int i, T x) { own[i * a.dstride] = x; });
        }
        __builtin_amdgcn_sched_barrier(0);
        carry(p);
      }
    };
    // The first plane outside the loop: on entry to it, as on every trip, the
    // stores of a B plane follow the gather in flight.
    plane(zs);
    for (int32_t z = zs + 1; z < ze; ++z) plane(z);
  };
  const int t0 = __builtin_amdgcn_readfirstlane(t);
  if (t0 < TX * TY && y0 + t0 / TX < ny)
    march(std::true_type{});
  else if (y0 - 1 + t0 / AX < ny)
    march(std::false_type{});
  else  // rows beyond the domain (ny not a multiple of TY): the barriers only
    for (int n = 1 + (zs > 0 ? 2 : 0) + (ze - zs) * (P::kDouble ? 1 : 2); n > 0; --n) __syncthreads();
}

}  // namespace culbm
