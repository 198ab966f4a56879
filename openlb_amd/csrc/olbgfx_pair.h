// olbgfx_pair.h -- two steps of a lattice in one pass over its populations.
// Included by olbgfx.hip after the single-step cell update; everything here
// lives in its anonymous namespace.
//
// A step moves every population through HBM once in each direction and does
// little arithmetic with it, so a run of steps is bound by that traffic.  The
// kernel below reads the state of time t and writes that of time t + 2: a
// workgroup owns a tile of y and z and sweeps along x.  At plane x it collides
// the cells of the tile and its rim of one cell (the first step, straight from
// memory) and hands the populations that leave their column to its neighbours
// through LDS; the cells inside the rim then collide plane x - 1 again (the
// second step) and store it.  The first step of a rim cell is done by up to
// four workgroups; nothing is exchanged between them, so the populations go to
// a second buffer.  Every value is rounded to the storage type between the
// steps and every collision is that of the single step, so the two paths agree
// bit for bit (in FP16 too: see pack_here).
//
// LDS holds 20 values a cell (80 KiB for 1024 threads in FP32): the four
// populations that move against the sweep and across columns for one plane,
// the eight that move within the plane for one plane (they are read before the
// next plane overwrites them), the four that move with the sweep for two
// planes.  The three that stay in their column stay in registers.
//
// The passes of one run other than its first and last use a flat layout of
// their own: a population is stored at the cell that collided it, and the next
// pass loads it from the neighbour.  Its addresses are one scalar base and one
// of nine column offsets for each population, without the ring arithmetic (3
// VALU instructions a load and 3 a store), and, on periodic lattices, the rows of all 19
// populations of one (x, y) lie side by side with the row pitch a multiple of
// a cache line.
//
// Measured on 512^3 BGK, us a step, against the single step: FP32 2765 / 4378,
// FP16 1752 / 2220, BF16 1705 / 2249.  In FP32 a pass reads 1.21 times and
// writes 1.01 times the populations at 4.1 TB/s, the VALU 43 % busy; the copy of the same card
// reaches 6.6, the single step in place 5.1.  The rest is the tiles' rims (1.33 x 1.13) and
// their ragged cache lines.  Rows side by side gained 2.5 % in FP32 and 5 % in
// FP16 over 19 separate rings; loading the next plane one turn of the sweep
// earlier gained 1.5 % in FP32 and lost 2 % in FP16, and more waves in flight
// (6 or 8 per SIMD by launch bounds) lost 10-15 %, so neither is done.

template <typename A>
struct PairArgs {
  StepArgs<A> a;        // a.pop: the source; a.shift: its offsets if it holds rings
  void* dst;            // destination, of the same size
  uint32_t dshift[Q];   // its offsets during the second step if it holds rings
  int32_t dx, dy, dz;   // cells updated: the core (periodic) or the padded block (closed)
  uint32_t plane;       // cells of a plane of the padded block
  uint32_t fx, fy, fq;  // flat layout: elements from one x, y and population to the next
  uint32_t tz, ty;      // tile along z and y, the rim included
  uint32_t ntz, nty;    // tiles along z and y
  uint32_t xlen;        // planes of one segment of the sweep
  uint32_t nwork;       // workgroups that carry a tile
  uint32_t per_xcd;     // ceil(nwork / 8)
};

// does population i leave its column (y, z)
__host__ __device__ constexpr bool crosses(int i) { return CY(i) != 0 || CZ(i) != 0; }

// LDS row of population i among those that leave their column: 0-3 against the
// sweep, 4-11 within the plane, 12-15 (and 16-19 for the other plane) with it
__host__ __device__ constexpr int pair_row(int i)
{
  int k = 0;
  for (int j = 1; j < i; ++j) {
    k += CX(j) == CX(i) && crosses(j) ? 1 : 0;
  }
  return CX(i) < 0 ? k : (CX(i) == 0 ? 4 + k : 12 + k);
}

// calls fn(k) for every dynamics id k that the active lanes hold, with the
// lanes that hold it and k in a scalar register
template <typename F>
__device__ __forceinline__ void by_id(int id, F&& fn)
{
  bool todo = true;
  while (todo) {
    const int k = __builtin_amdgcn_readfirstlane(id);
    if (k == id) {
      fn(k);
      todo = false;
    }
  }
}

// MODE k: every cell that collides has the dynamics kind k of slot uniform_id;
// kWithWalls + k: the ids of the mask have the kind k, BounceBack,
// BounceBackVelocity or NoDynamics; -1: any kind that step_cell takes there
constexpr int kWithWalls = 64;

template <int MODE, typename A>
__device__ __forceinline__ void pair_collide(A (&f)[Q], int id, bool collides, uint32_t n, const StepArgs<A>& a)
{
  A rho, usqr;
  if (collides) {
    if constexpr (MODE >= kWithWalls) {
      by_id(id, [&](int k) {
        const DynEntry<A>& e = a.table[k];
        if (e.kind == MODE - kWithWalls) {
          apply_kind<MODE - kWithWalls>(f, e, n, a, rho, usqr);
        } else if (e.kind == OLBGFX_BOUNCE_BACK) {
          apply_kind<OLBGFX_BOUNCE_BACK>(f, e, n, a, rho, usqr);
        } else if (e.kind == OLBGFX_BOUNCE_BACK_VELOCITY) {
          apply_kind<OLBGFX_BOUNCE_BACK_VELOCITY>(f, e, n, a, rho, usqr);
        }
      });
    } else if constexpr (MODE >= 0) {
      apply_kind<MODE>(f, a.table[a.uniform_id], n, a, rho, usqr);
    } else {
      const DynEntry<A> e = a.table[id];
      apply_any(f, e, n, a, rho, usqr);
    }
  }
}

// a value the compiler takes as new at this point, so that sums with it are
// formed here and not kept in registers across the sweep
__device__ __forceinline__ uint32_t opaque(uint32_t v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// the kernel's arguments, read again from the argument segment: scalar loads
// in every turn of the sweep instead of scalar registers spilled across it
template <typename P>
using ArgSegment = const __attribute__((address_space(4))) P*;
template <typename P>
__device__ __forceinline__ ArgSegment<P> arguments_again()
{
  auto k = (ArgSegment<P>)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return k;
}

// A population rounded to storage in the block that formed it.  The conversion
// to FP16 fuses with the FMA that ends a collision, and rounds once, only where
// both are in one block; the compiler moves a conversion whose result only the
// second step reads into that step's branch, where it rounds twice.
template <typename S>
__device__ __forceinline__ S pack_here(typename Storage<S>::A v)
{
  S s = Storage<S>::pack(v);
  if constexpr (std::is_same_v<S, f16_t>) {
    asm volatile("" : "+v"(s.v));
  }
  return s;
}

// scalar base and 32-bit vector offset
template <typename S>
__device__ __forceinline__ S* flat_at(uint64_t base, uint32_t offset)
{
  return (S*)((global_char*)base + offset);
}

// NT threads, one cell of the tile each.  PERIODIC: every axis is periodic,
// the core is updated and a rim cell outside it is computed as its image.
// Otherwise every axis is closed and the whole padded block is updated, its
// padding cells moving their populations as the rings do: along the linear
// cell index, modulo the block.
template <typename S, uint32_t NT, int MODE, bool PERIODIC, bool SRC_RING, bool DST_RING>
__global__ void __launch_bounds__(NT) pair_kernel(const PairArgs<typename Storage<S>::A> p)
{
  using A = typename Storage<S>::A;
  using St = Storage<S>;
  using Args = PairArgs<A>;
  __shared__ S lds[20][NT];
  constexpr uint32_t es = sizeof(S);
  const StepArgs<A>& a = p.a;
  // consecutive tiles, neighbours along z and then y, go to one XCD
  const uint32_t w = (blockIdx.x & 7u) * p.per_xcd + (blockIdx.x >> 3);
  if (w >= p.nwork) {
    return;  // uniform over the workgroup
  }
  const uint32_t zi = w % p.ntz, yi = w / p.ntz % p.nty, xi = w / p.ntz / p.nty;
  const uint32_t ly = threadIdx.x / p.tz, lz = threadIdx.x - ly * p.tz;
  // lanes beyond the tile or the block repeat the rim cell after its end, so
  // that every lane loads without a branch
  const int y = min((int)(yi * (p.ty - 2) + min(ly, p.ty - 1)) - 1, p.dy);
  const int z = min((int)(zi * (p.tz - 2) + lz) - 1, p.dz);
  const bool inside = ly > 0 && ly + 1 < p.ty && lz > 0 && lz + 1 < p.tz && y < p.dy && z < p.dz;
  const int x0 = (int)(xi * p.xlen), x1 = min(x0 + (int)p.xlen, p.dx);

  uint32_t column;      // this lane's cell in plane 0 of the padded block (modulo 2^32)
  uint32_t from[3][3];  // PERIODIC: byte offset of the column (y - cy, z - cz) in the flat layout
  bool core_column = true;
  if constexpr (PERIODIC) {
    auto wrap = [](int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); };
    const int yw = wrap(y, p.dy), zw = wrap(z, p.dz);
    column = (uint32_t)a.pad * p.plane + (uint32_t)(yw + a.pad) * a.pz + (uint32_t)(zw + a.pad);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      from[k / 3][k % 3] =
          ((uint32_t)wrap(yw - (k / 3 - 1), p.dy) * p.fy + (uint32_t)wrap(zw - (k % 3 - 1), p.dz)) * es;
    }
  } else {
    column = (uint32_t)(y * (int)a.pz + z);
    core_column = y >= a.pad && y < a.pad + a.ny && z >= a.pad && z < a.pad + a.nz;
  }
  // index modulo the block; blocks have fewer than 2^30 cells where they are
  // updated whole (a ring of 4-byte populations stays below 4 GiB)
  auto modulo = [&](uint32_t n) { return n < a.count ? n : ((int)n < 0 ? n + a.count : n - a.count); };
  auto cell = [&](int x) -> uint32_t {
    if constexpr (PERIODIC) {
      return column + (uint32_t)(x < 0 ? x + p.dx : (x >= p.dx ? x - p.dx : x)) * p.plane;
    } else {
      return modulo(column + (uint32_t)x * p.plane);
    }
  };
  auto core = [&](int x) { return PERIODIC || (core_column && x >= a.pad && x < a.pad + a.nx); };

  auto load = [&](int x, A (&f)[Q], int& id) {
    const uint32_t n = cell(x);
    const auto k = arguments_again<Args>();
    uint64_t base = (uint64_t)k->a.pop;
    if constexpr (MODE < 0 || MODE >= kWithWalls) {
      id = (int)a.mask[n];
    }
    if constexpr (SRC_RING) {
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        f[i] = St::load(flat_at<S>(base, ring_slot(n, k->a.shift[i], a.count) * es));
        base += a.stride * es;
      }
    } else if constexpr (PERIODIC) {
      const int xw = x < 0 ? x + p.dx : (x >= p.dx ? x - p.dx : x);
      const uint64_t here = (uint64_t)(uint32_t)xw * p.fx * es;
      const uint64_t before = (uint64_t)(uint32_t)(xw == 0 ? p.dx - 1 : xw - 1) * p.fx * es;
      const uint64_t after = (uint64_t)(uint32_t)(xw == p.dx - 1 ? 0 : xw + 1) * p.fx * es;
      uint32_t off[3][3];
#pragma unroll
      for (int c = 0; c < 9; ++c) off[c / 3][c % 3] = opaque(from[c / 3][c % 3]);
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        f[i] = St::load(flat_at<S>(base + (CX(i) == 0 ? here : (CX(i) > 0 ? before : after)),
                                   off[CY(i) + 1][CZ(i) + 1]));
        base += (uint64_t)p.fq * es;
      }
    } else if (x <= 1 || x >= p.dx - 2) {
      // the neighbours of these planes may wrap around the block
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int d = CX(i) * (int)k->plane + CY(i) * (int)a.pz + CZ(i);
        f[i] = St::load(flat_at<S>(base, modulo((uint32_t)((int)n - d)) * es));
        base += a.stride * es;
      }
    } else {
      const uint32_t off = opaque(n * es);
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int d = CX(i) * (int)k->plane + CY(i) * (int)a.pz + CZ(i);
        f[i] = St::load(flat_at<S>(base - (uint64_t)((int64_t)d * es), off));
        base += a.stride * es;
      }
    }
  };

  auto neighbour = [&](int i) { return threadIdx.x - (uint32_t)(CY(i) * (int)p.tz + CZ(i)); };
  A rest = A(0), ahead0 = A(0), ahead1 = A(0);  // the populations that stay in their column
  int id_before = 0;
  // One turn of the sweep: f holds plane x, and plane x + 1 afterwards.  A
  // lambda with f as its argument, like load: with f captured the compiler
  // keeps copies of it (128 VGPRs against 87 in the masked kernel, which then
  // takes 165 us a step against 149 on the porous channel in FP32).
  auto turn = [&](int x, A (&f)[Q], int& id) {
    const bool second = inside && x > x0;  // plane x - 1 belongs to this tile
    A g[Q];
    S (*const with)[NT] = &lds[12 + 4 * (x & 1)];
    if (second) {
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        if (CX(i) >= 0 && crosses(i)) {
          g[i] = St::unpack(CX(i) == 0 ? lds[pair_row(i)][neighbour(i)] : with[pair_row(i) - 12][neighbour(i)]);
        }
      }
    }
    pair_collide<MODE>(f, id, core(x), cell(x), a);
    __syncthreads();  // every lane has read what the next lines overwrite
#pragma unroll
    for (int i = 1; i < Q; ++i) {
      if (crosses(i)) {
        (CX(i) <= 0 ? lds[pair_row(i)] : with[pair_row(i) - 12])[threadIdx.x] = St::pack(f[i]);
      }
    }
    g[0] = rest;
    g[10] = ahead0;
    g[1] = St::unpack(pack_here<S>(f[1]));
    rest = St::unpack(pack_here<S>(f[0]));
    ahead0 = ahead1;
    ahead1 = St::unpack(pack_here<S>(f[10]));
    const int id2 = id_before;
    id_before = id;
    __syncthreads();
    if (x < x1) {
      load(x + 1, f, id);  // in flight during the second step
    }
    if (second) {
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        if (CX(i) < 0 && crosses(i)) {
          g[i] = St::unpack(lds[pair_row(i)][neighbour(i)]);
        }
      }
      const uint32_t n = cell(x - 1);
      pair_collide<MODE>(g, id2, core(x - 1), n, a);
      const auto k = arguments_again<Args>();
      uint64_t base = (uint64_t)k->dst;
      if constexpr (DST_RING) {
#pragma unroll
        for (int i = 0; i < Q; ++i) {
          *flat_at<S>(base, ring_slot(n, k->dshift[i], a.count) * es) = St::pack(g[i]);
          base += a.stride * es;
        }
        if constexpr (PERIODIC) {
          const bool lo[3] = {x - 1 == 0, y == 0, z == 0};
          const bool hi[3] = {x == a.nx, y == a.ny - 1, z == a.nz - 1};
          if (lo[0] | lo[1] | lo[2] | hi[0] | hi[1] | hi[2]) {
            uint32_t sh[Q];
#pragma unroll
            for (int i = 0; i < Q; ++i) sh[i] = k->dshift[i];
            const int64_t off[3] = {(int64_t)a.nx * a.py * a.pz, (int64_t)a.ny * a.pz, (int64_t)a.nz};
            ghost_all<S>((void*)k->dst, a.stride, a.count, sh, (int64_t)n, lo, hi, off, g,
                         std::make_integer_sequence<int, Q - 1>{});
          }
        }
      } else {
        base += (uint64_t)(uint32_t)(x - 1) * p.fx * es;
        const uint32_t own = opaque(PERIODIC ? from[1][1] : column * es);
#pragma unroll
        for (int i = 0; i < Q; ++i) {
          *flat_at<S>(base, own) = St::pack(g[i]);
          base += (uint64_t)p.fq * es;
        }
      }
    }
  };
  A f[Q];
  int id = 0;
  load(x0 - 1, f, id);
  for (int x = x0 - 1; x <= x1; ++x) {
    turn(x, f, id);
  }
}
