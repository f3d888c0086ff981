// The viscous velocity block (M + dt E^T W E) u = rhs of one dynamic viscosity on the full-cell strain rows
// of the pressure cells (AssembleFullCellMacStrain3D, native/src/viscosity.cc:762-946;
// SolveMacViscousVelocityBlock3D, :1331-1650), without forming the rows: the substep's case.
//
// With one viscosity every normal row carries the same weighted coefficient and every shear row another,
// and which faces a row holds follows from the lattice. The face vectors are stored in owned-slot order
// (192 per 4^3 block, zero off the links), so a face's neighbours are arithmetic on its slot and a table of
// the block's 26 neighbours; seven bits per face say whether it is open and which of its six rows exist.
// A row's strain and a face's sum over its rows are formed with the packed operator's terms, in its
// order (viscosity.hip), so an apply gives the same bits; only the dots add in another fixed order.
//
// One PCG iteration is two launches. k_uniform_apply forms the direction d' = z + beta d on the block and a
// one-cell halo in LDS, applies the operator, and its last workgroup reduces d'.q and sets the step;
// k_uniform_step advances v, r and z, and its last workgroup reduces max |r| and r.z, sets beta and
// decides whether the iteration stops (converged to the recursive residual, out of budget, or failed).
// After a stop the remaining launches of a batch return at once, so the host looks only once per batch
// and the iterates and their number are those of a look after every iteration.
//
// Bound by HBM: an iteration moves 41 + 72 bytes per face, against about 330 through packed rows and
// incidences. On the stirred 128^3 scene (0.79M links) an iteration fell from 88 us of kernels and 158 us with its
// launches and host reads to 41 and 44 us.
#include <cmath>
#include <new>

#include "context.h"

namespace fl {

// Scalars of one solve on the device, reset by k_uniform_start.
struct UniformScalars {
  double rz, max_r, step, beta;
  uint32_t status, stop, iterations, nonfinite;
};
constexpr int kCounters = 64;  // first level of the running reduction's arrival counters, one more on top

struct UniformBuffers {
  double *inertia = nullptr, *rhs = nullptr, *v = nullptr, *r = nullptr, *z = nullptr, *d[2] = {nullptr, nullptr},
         *q = nullptr, *diag = nullptr, *uwall = nullptr;
  uint8_t* mask = nullptr;
  int32_t* near = nullptr;          // 27 per block: ordinals of the block and its neighbours, -1 inactive
  unsigned long long* cells = nullptr;  // pressure cells of each block
  uint64_t* count = nullptr;        // shear rows
  double* partial = nullptr;
  uint32_t* arrived = nullptr;      // kCounters + 1
  UniformScalars* scal = nullptr;
  UniformScalars* host = nullptr;   // pinned
  uint64_t cap_blocks = 0;
  double cn = 0, cs = 0;            // weighted coefficients of the normal and shear rows
  void release() {
    void* ptrs[] = {inertia, rhs, v, r, z, d[0], d[1], q, diag, uwall, mask, near, cells, count, partial, arrived, scal};
    for (void* p : ptrs)
      if (p) (void)hipFree(p);
    if (host) (void)hipHostFree(host);
    *this = UniformBuffers{};
  }
};

namespace {

constexpr int kBlockFaces = 192;
constexpr unsigned kUniformGroups = 2048;  // eight workgroups of three waves on every CU
constexpr int kBatch = 8;                  // iterations queued between two looks at the scalars

template <typename T>
int take(T** p, uint64_t n) {
  if (hipMalloc(reinterpret_cast<void**>(p), std::max<uint64_t>(n, 1) * sizeof(T)) != hipSuccess) {
    *p = nullptr;
    return FL_RESOURCE_EXHAUSTED;
  }
  return FL_OK;
}

int allocate(UniformBuffers* B, uint64_t nb) {
  B->release();
  const uint64_t n = nb * kBlockFaces;
  double** fv[] = {&B->inertia, &B->rhs, &B->v, &B->r, &B->z, &B->d[0], &B->d[1], &B->q, &B->diag, &B->uwall};
  for (double** p : fv) FL_TRY(take(p, n));
  FL_TRY(take(&B->mask, n));
  FL_TRY(take(&B->near, 27 * nb));
  FL_TRY(take(&B->cells, nb));
  FL_TRY(take(&B->count, 1));
  FL_TRY(take(&B->partial, 2 * kUniformGroups));
  FL_TRY(take(&B->arrived, kCounters + 1));
  FL_TRY(take(&B->scal, 1));
  if (hipHostMalloc(reinterpret_cast<void**>(&B->host), sizeof(UniformScalars)) != hipSuccess) {
    B->host = nullptr;
    return FL_RESOURCE_EXHAUSTED;
  }
  B->cap_blocks = nb;
  return FL_OK;
}

// Room for nb blocks: what is there, or what fl_reserve took for the context's capacity; else a quarter more
// than asked for (within the capacity), so that a spreading liquid does not free and allocate in every substep.
int ensure(fl_ctx* ctx, uint64_t nb, UniformBuffers** out) {
  if (!ctx->uniform) ctx->uniform = new (std::nothrow) UniformBuffers();
  auto* B = static_cast<UniformBuffers*>(ctx->uniform);
  if (!B) return FL_RESOURCE_EXHAUSTED;
  *out = B;
  if (nb <= B->cap_blocks && B->host) return FL_OK;
  const uint64_t more = std::min(nb + nb / 4, ctx->cap.blocks);
  if (more > nb) {
    if (allocate(B, more) == FL_OK) return FL_OK;
    (void)hipGetLastError();  // the smaller try stands by itself
  }
  return allocate(B, nb);
}

// Weighted coefficient sqrt(dt) sqrt(w) c and strain weight mu h^3 2^k by exponent-separated products, as
// the packed rows form them (viscosity.hip).
double scaled_product(double a, double b, double c) {
  if (a == 0.0 || b == 0.0 || c == 0.0) return 0.0;
  int ea, eb, ec, ed;
  const double fa = std::frexp(a, &ea), fb = std::frexp(b, &eb), fc = std::frexp(c, &ec), fd = std::frexp(1.0, &ed);
  return std::scalbn((fa * (fb * fc)) / fd, ea + eb + ec - ed);
}
double weight(double mu, double h, int k) {
  int eh, em, ed;
  const double fh = std::frexp(h, &eh), fm = std::frexp(mu, &em), fd = std::frexp(1.0, &ed);
  return std::scalbn(((fm * (fh * fh)) / fd) * fh, em + eh + eh - ed + eh + k);
}

__device__ inline bool finite_d(double v) { return isfinite(v); }

// Bits of a face's mask: open, then its rows in the packed operator's row order. The row's low cell is
// given for the face at lattice l normal to a, with the other axes b1 < b2.
constexpr int kOpen = 0;
constexpr int kTail = 1;    // normal row of cell l - a
constexpr int kHead = 2;    // normal row of cell l
constexpr int kLowB2 = 3;   // shear row (a, b2) of low cell l - a - b2
constexpr int kLowB1 = 4;   // shear row (a, b1) of low cell l - a - b1
constexpr int kHighB1 = 5;  // shear row (a, b1) of low cell l - a
constexpr int kHighB2 = 6;  // shear row (a, b2) of low cell l - a

// Position in the 3 x 3 x 3 block table of a lattice position relative to a block, each in [-4, 7].
__device__ inline int near_index(int x, int y, int z) { return (((z >> 2) + 1) * 3 + (y >> 2) + 1) * 3 + (x >> 2) + 1; }
__device__ inline int local_index(int x, int y, int z) { return (z & 3) * 16 + (y & 3) * 4 + (x & 3); }

__global__ void k_uniform_near(GridView g, int32_t* near) {
  const uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (i >= 27 * g.nb) return;
  const uint64_t b = i / 27;
  const int k = static_cast<int>(i % 27);
  near[i] = g.ordinal(g.blocks[3 * b] + k % 3 - 1, g.blocks[3 * b + 1] + (k / 3) % 3 - 1, g.blocks[3 * b + 2] + k / 9 - 1);
}

__global__ void k_uniform_clear(uint64_t nb, double* inertia, double* rhs, double* diag, double* uwall, uint8_t* mask,
                                unsigned long long* cells, uint64_t* count) {
  const uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (i < nb) cells[i] = 0;
  if (i == 0) *count = 0;
  if (i >= nb * kBlockFaces) return;
  inertia[i] = rhs[i] = diag[i] = uwall[i] = 0.0;
  mask[i] = 0;
}

__device__ inline int32_t floor4(int32_t v) { return v >= 0 ? v / 4 : -1 - (-(v + 1)) / 4; }

__global__ void k_uniform_cells(GridView g, const fl_pressure_cell* cells, uint64_t n, unsigned long long* bits) {
  const uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  const fl_int3 c = cells[i].cell_index;
  const int32_t b = g.ordinal(floor4(c.x), floor4(c.y), floor4(c.z));
  if (b >= 0) atomicOr(bits + b, 1ull << local_index(c.x & 3, c.y & 3, c.z & 3));
}

__device__ inline bool has_cell(const int32_t* near, const unsigned long long* cells, int x, int y, int z) {
  const int32_t b = near[near_index(x, y, z)];
  return b >= 0 && ((cells[b] >> local_index(x, y, z)) & 1) != 0;
}

// Interior shear rows of a block's cells (the cell, its two neighbours and the diagonal one present).
__global__ void k_uniform_count(uint64_t nb, const int32_t* near_all, const unsigned long long* cells, uint64_t* count) {
  const uint64_t b = blockIdx.x;
  const int c = static_cast<int>(threadIdx.x), x = c & 3, y = (c >> 2) & 3, z = c >> 4;
  const int32_t* near = near_all + 27 * b;
  int rows = 0;
  if ((cells[b] >> c) & 1) {
    const bool hx = has_cell(near, cells, x + 1, y, z), hy = has_cell(near, cells, x, y + 1, z),
               hz = has_cell(near, cells, x, y, z + 1);
    rows = (hx && hy && has_cell(near, cells, x + 1, y + 1, z)) + (hx && hz && has_cell(near, cells, x + 1, y, z + 1)) +
           (hy && hz && has_cell(near, cells, x, y + 1, z + 1));
  }
  for (int o = 32; o > 0; o >>= 1) rows += __shfl_xor(rows, o);
  if (threadIdx.x == 0 && rows) atomicAdd(reinterpret_cast<unsigned long long*>(count), static_cast<unsigned long long>(rows));
}

// Per link: its mask, the Jacobi diagonal (inertia plus the squared coefficients, in row order) and the
// wall velocity at its slot. A diagonal that is not finite is OutOfRange.
__global__ void k_uniform_links(const uint64_t* slot, uint64_t nf, const int32_t* near_all,
                                const unsigned long long* cells, const double* inertia, const double* uwall_links,
                                double cn, double cs, uint8_t* mask, double* diag, double* uwall, uint64_t* err) {
  const uint64_t f = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (f >= nf) return;
  const uint64_t s = slot[f], b = s / kBlockFaces;
  const int within = static_cast<int>(s % kBlockFaces), a = within / 64, c = within % 64;
  const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
  const int l[3] = {c & 3, (c >> 2) & 3, c >> 4};
  const int32_t* near = near_all + 27 * b;
  const auto has = [&](int da, int d1, int d2) {
    int q[3] = {l[0], l[1], l[2]};
    q[a] += da;
    q[b1] += d1;
    q[b2] += d2;
    return has_cell(near, cells, q[0], q[1], q[2]);
  };
  const bool tail = has(-1, 0, 0), head = has(0, 0, 0), both = tail && head;
  uint32_t m = 0;
  const double in = inertia[s];
  if (in > 0.0) m |= 1u << kOpen;
  if (tail) m |= 1u << kTail;
  if (head) m |= 1u << kHead;
  if (both && has(-1, 0, -1) && has(0, 0, -1)) m |= 1u << kLowB2;
  if (both && has(-1, -1, 0) && has(0, -1, 0)) m |= 1u << kLowB1;
  if (both && has(-1, 1, 0) && has(0, 1, 0)) m |= 1u << kHighB1;
  if (both && has(-1, 0, 1) && has(0, 0, 1)) m |= 1u << kHighB2;
  mask[s] = static_cast<uint8_t>(m);
  uwall[s] = uwall_links[f];
  double d = in;
  if (in > 0.0) {
    for (int k = kTail; k <= kHead; ++k)
      if ((m >> k) & 1) d += cn * cn;
    for (int k = kLowB2; k <= kHighB2; ++k)
      if ((m >> k) & 1) d += cs * cs;
  }
  if (!finite_d(d)) atomicMin(reinterpret_cast<unsigned long long*>(err), (static_cast<unsigned long long>(f) << 8) | FL_OUT_OF_RANGE);
  diag[s] = d;
}

// The six rows of face (l, a) with the neighbour values from at(axis, da, d1, d2) (offsets along a, b1 and
// b2): calls row(sign, shear, t0, t1, t2, t3) for each row that exists, in row order, where sign is the
// sign of the face's own coefficient and the row's terms are -t0 + t1 (- t2 + t3 for shear rows).
template <class At, class Row>
__device__ __forceinline__ void face_rows(uint32_t m, int a, At at, Row row) {
  const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
  if ((m >> kTail) & 1) row(1.0, false, at(a, -1, 0, 0), at(a, 0, 0, 0), 0.0, 0.0);
  if ((m >> kHead) & 1) row(-1.0, false, at(a, 0, 0, 0), at(a, 1, 0, 0), 0.0, 0.0);
  // Terms of a shear row (p, q), p < q, of low cell c: p at c + p and c + p + q, q at c + q and c + p + q.
  const auto shear = [&](double sign, bool first, double a0, double a1, double o0, double o1) {
    if (first) row(sign, true, a0, a1, o0, o1);
    else row(sign, true, o0, o1, a0, a1);
  };
  if ((m >> kLowB2) & 1) shear(1.0, a < b2, at(a, 0, 0, -1), at(a, 0, 0, 0), at(b2, -1, 0, 0), at(b2, 0, 0, 0));
  if ((m >> kLowB1) & 1) shear(1.0, a < b1, at(a, 0, -1, 0), at(a, 0, 0, 0), at(b1, -1, 0, 0), at(b1, 0, 0, 0));
  if ((m >> kHighB1) & 1) shear(-1.0, a < b1, at(a, 0, 0, 0), at(a, 0, 1, 0), at(b1, -1, 1, 0), at(b1, 0, 1, 0));
  if ((m >> kHighB2) & 1) shear(-1.0, a < b2, at(a, 0, 0, 0), at(a, 0, 0, 1), at(b2, -1, 0, 1), at(b2, 0, 0, 1));
}

// Prescribed strain of the rows' eliminated faces moved to the right-hand side of each open link
// (mac_viscous_pressure_3d.cc:226-246), its rows in order.
__global__ void k_uniform_eliminate(const uint64_t* slot, uint64_t nf, const int32_t* near_all, const uint8_t* mask,
                                    const double* inertia, const double* uwall, double dt, double wn, double ws,
                                    double normal, double shear, double* base) {
  const uint64_t f = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (f >= nf) return;
  const uint64_t s = slot[f], b = s / kBlockFaces;
  const uint32_t m = mask[s];
  if (!(m & 1)) return;
  const int within = static_cast<int>(s % kBlockFaces), a = within / 64, c = within % 64;
  const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
  const int l[3] = {c & 3, (c >> 2) & 3, c >> 4};
  const int32_t* near = near_all + 27 * b;
  // The wall velocity of an eliminated face; an open one (whose own value is never zero inertia) adds zero.
  const auto at = [&](int axis, int da, int d1, int d2) -> double {
    int q[3] = {l[0], l[1], l[2]};
    q[a] += da;
    q[b1] += d1;
    q[b2] += d2;
    const int32_t n = near[near_index(q[0], q[1], q[2])];
    if (n < 0) return 0.0;
    const uint64_t t = uint64_t(n) * kBlockFaces + axis * 64 + local_index(q[0], q[1], q[2]);
    return inertia[t] == 0.0 ? uwall[t] : 0.0;
  };
  double sum = base[f];
  face_rows(m, a, at, [&](double sign, bool sh, double t0, double t1, double t2, double t3) {
    const double k = sh ? shear : normal, w = sh ? ws : wn;
    double prescribed = 0.0;
    prescribed += -k * t0;
    prescribed += k * t1;
    if (sh) {
      prescribed += -k * t2;
      prescribed += k * t3;
    }
    if (prescribed != 0.0) sum += -(dt * w * prescribed * (sign * k));
  });
  base[f] = sum;
}

// Sum and maximum of the workgroups' partials: every workgroup stores its two, the last one to arrive folds
// them in a fixed order and returns true with the totals (on every lane). Partials, counters and the
// non-finite flag are relaxed device-scope atomics, and each wave waits for its own before its workgroup
// arrives: an acquire or release here would write back and invalidate the XCD's L2 once per workgroup
// (on 0.79M links an iteration took 123 us with it, 41 us without). Arrivals count in two levels, so that no
// counter takes more than kCounters of them in a row.
template <int kWaves>
__device__ inline bool grid_reduce(double sum, double mx, double* partial, uint32_t* arrived, double& total_sum,
                                   double& total_max) {
  __shared__ double red[2][kWaves];
  __shared__ bool last;
  const auto fold = [&](double& s, double& m) {
    for (int o = 32; o > 0; o >>= 1) {
      s += __shfl_xor(s, o);
      m = fmax(m, __shfl_xor(m, o));
    }
    if ((threadIdx.x & 63) == 0) {
      red[0][threadIdx.x >> 6] = s;
      red[1][threadIdx.x >> 6] = m;
    }
    __syncthreads();
    s = red[0][0];
    m = red[1][0];
    for (int w = 1; w < kWaves; ++w) {
      s += red[0][w];
      m = fmax(m, red[1][w]);
    }
    __syncthreads();
  };
  const auto settle = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  settle();
  fold(sum, mx);
  if (threadIdx.x == 0) {
    __hip_atomic_store(partial + 2 * blockIdx.x, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(partial + 2 * blockIdx.x + 1, mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    settle();
    const uint32_t groups = gridDim.x, k = blockIdx.x % kCounters;
    const uint32_t members = groups / kCounters + (k < groups % kCounters ? 1 : 0);
    last = false;
    if (__hip_atomic_fetch_add(arrived + k, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == members - 1) {
      const uint32_t counters = groups < kCounters ? groups : kCounters;
      last = __hip_atomic_fetch_add(arrived + kCounters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == counters - 1;
    }
  }
  __syncthreads();
  if (!last) return false;
  for (unsigned k = threadIdx.x; k <= kCounters; k += blockDim.x) arrived[k] = 0;
  sum = 0.0;
  mx = 0.0;
  for (unsigned g = threadIdx.x; g < gridDim.x; g += blockDim.x) {
    sum += __hip_atomic_load(partial + 2 * g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    mx = fmax(mx, __hip_atomic_load(partial + 2 * g + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  fold(sum, mx);
  total_sum = sum;
  total_max = mx;
  return true;
}

// r = rhs, z = r / diag on open faces, v = 0; r.z and the solve's scalars.
__global__ __launch_bounds__(kThreads) void k_uniform_start(uint64_t n, const uint8_t* mask, const double* rhs,
                                                            const double* diag, double* v, double* r, double* z,
                                                            double* partial, uint32_t* arrived,
                                                            UniformScalars* scal) {
  double rz = 0.0;
  for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
    const bool open = (mask[i] & 1) != 0;
    const double ri = open ? rhs[i] : 0.0, zi = open ? ri / diag[i] : 0.0;
    v[i] = 0.0;
    r[i] = ri;
    z[i] = zi;
    rz += ri * zi;
  }
  double sum, mx;
  if (!grid_reduce<kThreads / 64>(rz, 0.0, partial, arrived, sum, mx)) return;
  if (threadIdx.x != 0) return;
  scal->rz = sum;
  scal->max_r = scal->step = scal->beta = 0.0;
  scal->status = scal->stop = scal->iterations = scal->nonfinite = 0;
}

// kDirection: d' = z + beta d in LDS over the block and its halo, q = H d', d'.q and the step. Otherwise the
// check of an iterate: q = H v, the true residual r = rhs - q, z, max |r| and r.z; a converged check stays
// stopped, one that is not goes on from a fresh direction (beta 0).
// One workgroup of three waves per 4^3 block, a wave per face axis; each XCD takes a run of blocks, so that
// the halos of neighbouring blocks meet in its L2.
constexpr int kSide = 6, kHalo = kSide * kSide * kSide;
template <bool kDirection>
__global__ __launch_bounds__(kBlockFaces) void k_uniform_apply(uint64_t nb, const int32_t* near_all,
                                                               const uint8_t* mask, const double* inertia, double cn,
                                                               double cs, const double* z, const double* d,
                                                               double* d_next, double* q, const double* rhs,
                                                               const double* diag, double* r, double* z_next,
                                                               double tolerance, double* partial, uint32_t* arrived,
                                                               UniformScalars* scal) {
  if (kDirection && scal->stop) return;
  __shared__ double xs[3][kHalo];
  __shared__ int32_t near[27];
  const double beta = kDirection ? scal->beta : 0.0;
  const int tid = static_cast<int>(threadIdx.x), a = tid >> 6, c = tid & 63;
  const int l[3] = {c & 3, (c >> 2) & 3, c >> 4};
  const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
  // Strides of a step along a, b1 and b2 in the staged cube.
  const auto pitch = [](int axis) { return axis == 0 ? 1 : (axis == 1 ? kSide : kSide * kSide); };
  const int pa = pitch(a), p1 = pitch(b1), p2 = pitch(b2);
  const int own = ((l[2] + 1) * kSide + l[1] + 1) * kSide + l[0] + 1;
  double sum = 0.0, mx = 0.0;
  const uint32_t xcd = blockIdx.x & 7, lane = blockIdx.x >> 3, step = gridDim.x >> 3;
  const uint64_t lo = nb * xcd / 8, hi = nb * (xcd + 1) / 8;
  for (uint64_t b = lo + lane; b < hi; b += step) {
    const uint64_t s = b * kBlockFaces + tid;
    const uint32_t m = mask[s];
    __syncthreads();  // the previous block's values are read
    if (tid < 27) near[tid] = near_all[27 * b + tid];
    const bool any = __syncthreads_or(m != 0) != 0;
    if (!any) {  // no link in the block: its vectors stay zero and no open face of another block reads more
      if (kDirection) d_next[s] = 0.0;
      continue;
    }
    for (int e = tid; e < 3 * kHalo; e += kBlockFaces) {
      const int axis = e / kHalo, i = e % kHalo;
      const int x = i % kSide - 1, y = (i / kSide) % kSide - 1, zz = i / (kSide * kSide) - 1;
      const int32_t n = near[near_index(x, y, zz)];
      double value = 0.0;
      if (n >= 0) {
        const uint64_t t = uint64_t(n) * kBlockFaces + axis * 64 + local_index(x, y, zz);
        value = z[t];
        if (kDirection && beta != 0.0) value += beta * d[t];
      }
      xs[axis][i] = value;
    }
    __syncthreads();
    const double x = xs[a][own];
    double y = 0.0;
    if (m & 1) {
      y = inertia[s] * x;
      const auto at = [&](int axis, int da, int d1, int d2) { return xs[axis][own + da * pa + d1 * p1 + d2 * p2]; };
      face_rows(m, a, at, [&](double sign, bool sh, double t0, double t1, double t2, double t3) {
        const double k = sh ? cs : cn;
        double e = 0.0;
        e += -k * t0;
        e += k * t1;
        if (sh) {
          e += -k * t2;
          e += k * t3;
        }
        y += sign * k * e;
      });
    }
    if (kDirection) {
      d_next[s] = x;
      q[s] = y;
      if (!finite_d(y)) atomicOr(&scal->nonfinite, 1u);
      sum += x * y;
    } else {
      double rf = 0.0, zf = 0.0;
      if (m & 1) {
        rf = rhs[s] - y;
        zf = rf / diag[s];
        if (!finite_d(rf)) atomicOr(&scal->nonfinite, 1u);
      }
      r[s] = rf;
      z_next[s] = zf;
      mx = fmax(mx, fabs(rf));
      sum += rf * zf;
    }
  }
  double total, most;
  if (!grid_reduce<kBlockFaces / 64>(sum, mx, partial, arrived, total, most)) return;
  if (tid != 0) return;
  const uint32_t bad = __hip_atomic_load(&scal->nonfinite, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (kDirection) {
    // r.z positive and finite with a finite apply, else OutOfRange; a positive finite curvature, else
    // Aborted; a normal step, else OutOfRange.
    const double rz = scal->rz, s = rz / total;
    uint32_t status = 0;
    if (!finite_d(rz) || rz <= 0.0 || bad) status = FL_OUT_OF_RANGE;
    else if (!finite_d(total) || total <= 0.0) status = FL_ABORTED;
    else if (!__builtin_isnormal(s)) status = FL_OUT_OF_RANGE;
    scal->step = status ? 0.0 : s;
    if (status) {
      scal->status = status;
      scal->stop = 1;
    }
  } else {
    scal->max_r = most;
    scal->rz = total;
    scal->beta = 0.0;
    scal->stop = most <= tolerance ? 1 : 0;
  }
}

// v += step d, r -= step q, z = r / diag on open faces; max |r|, r.z, beta and the stop.
__global__ __launch_bounds__(kThreads) void k_uniform_step(uint64_t n, const uint8_t* mask, const double* d,
                                                           const double* q, const double* diag, double* v, double* r,
                                                           double* z, double tolerance, uint32_t max_iterations,
                                                           double* partial, uint32_t* arrived,
                                                            UniformScalars* scal) {
  if (scal->stop) return;
  const double step = scal->step;
  double rz = 0.0, mx = 0.0;
  for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
    if (!(mask[i] & 1)) continue;
    const double vi = v[i] + step * d[i];
    const double ri = r[i] - step * q[i];
    v[i] = vi;
    r[i] = ri;
    if (!finite_d(vi) || !finite_d(ri)) atomicOr(&scal->nonfinite, 1u);
    mx = fmax(mx, fabs(ri));
    const double zi = ri / diag[i];
    z[i] = zi;
    rz += ri * zi;
  }
  double sum, most;
  if (!grid_reduce<kThreads / 64>(rz, mx, partial, arrived, sum, most)) return;
  if (threadIdx.x != 0) return;
  scal->max_r = most;
  scal->beta = sum / scal->rz;
  scal->rz = sum;
  const uint32_t it = scal->iterations + 1;
  scal->iterations = it;
  const uint32_t bad = __hip_atomic_load(&scal->nonfinite, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (bad) scal->status = FL_OUT_OF_RANGE;
  if (bad || most <= tolerance || it >= max_iterations) scal->stop = 1;
}

__global__ void k_uniform_zero(uint64_t n, double* v, uint32_t* arrived) {
  const uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x;
  if (i < n) v[i] = 0.0;
  if (i <= kCounters) arrived[i] = 0;
}

}  // namespace

int uniform_reserve(fl_ctx* ctx) {
  UniformBuffers* B = nullptr;
  return ensure(ctx, std::max<uint64_t>(ctx->cap.blocks, 1), &B);
}

int uniform_prepare(fl_ctx* ctx, UniformBlock* out) {
  UniformBuffers* B = nullptr;
  FL_TRY(ensure(ctx, ctx->nb, &B));
  const uint64_t n = ctx->nb * kBlockFaces;
  hipStream_t s = ctx->stream;
  if (n) {
    k_uniform_near<<<grid_for(27 * ctx->nb), kThreads, 0, s>>>(grid_view(ctx), B->near);
    k_uniform_clear<<<grid_for(n), kThreads, 0, s>>>(ctx->nb, B->inertia, B->rhs, B->diag, B->uwall, B->mask, B->cells,
                                                     B->count);
  }
  k_uniform_zero<<<grid_for(n), kThreads, 0, s>>>(n, B->v, B->arrived);
  FL_HIP(hipGetLastError());
  *out = UniformBlock{B->inertia, B->rhs, B->v, B->diag};
  return FL_OK;
}

int uniform_rows(fl_ctx* ctx, const CoupledSystem& S, const fl_pressure_cell* cells, double mu, double h, double dt,
                 double* base, uint64_t* err, uint64_t* rows) {
  auto& B = *static_cast<UniformBuffers*>(ctx->uniform);
  hipStream_t s = ctx->stream;
  const double normal = 1.0 / h, shear = 0.5 * normal;
  if (!std::isnormal(normal)) return FL_OUT_OF_RANGE;
  const double wn = weight(mu, h, 1), ws = weight(mu, h, 2);
  if (!std::isnormal(wn)) return FL_OUT_OF_RANGE;
  B.cn = scaled_product(std::sqrt(dt), std::sqrt(wn), normal);
  B.cs = scaled_product(std::sqrt(dt), std::sqrt(ws), shear);
  if (!std::isnormal(B.cn)) return FL_OUT_OF_RANGE;
  if (S.nc) k_uniform_cells<<<grid_for(S.nc), kThreads, 0, s>>>(grid_view(ctx), cells, S.nc, B.cells);
  if (ctx->nb) k_uniform_count<<<static_cast<unsigned>(ctx->nb), 64, 0, s>>>(ctx->nb, B.near, B.cells, B.count);
  FL_HIP(hipGetLastError());
  FL_HIP(hipMemcpyAsync(ctx->host_words, B.count, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
  FL_HIP(hipStreamSynchronize(s));
  const uint64_t shear_rows = ctx->host_words[0];
  *rows = 3 * S.nc + shear_rows;
  if (shear_rows && !(std::isnormal(shear) && std::isnormal(ws) && std::isnormal(B.cs))) return FL_OUT_OF_RANGE;
  if (S.nf) {
    k_uniform_links<<<grid_for(S.nf), kThreads, 0, s>>>(S.slot, S.nf, B.near, B.cells, B.inertia, S.uwall, B.cn, B.cs,
                                                        B.mask, B.diag, B.uwall, err);
    k_uniform_eliminate<<<grid_for(S.nf), kThreads, 0, s>>>(S.slot, S.nf, B.near, B.mask, B.inertia, B.uwall, dt, wn,
                                                            ws, normal, shear, base);
  }
  FL_HIP(hipGetLastError());
  return FL_OK;
}

int uniform_solve(fl_ctx* ctx, double max_rhs, uint64_t max_iterations, double relative_tolerance,
                  uint64_t* iterations, double* max_residual) {
  auto& B = *static_cast<UniformBuffers*>(ctx->uniform);
  hipStream_t s = ctx->stream;
  const uint64_t nb = ctx->nb, n = nb * kBlockFaces;
  *iterations = 0;
  *max_residual = 0.0;
  if (max_rhs == 0.0) {
    k_uniform_zero<<<grid_for(n), kThreads, 0, s>>>(n, B.v, B.arrived);
    FL_HIP(hipGetLastError());
    return FL_OK;
  }
  const double tolerance = relative_tolerance * max_rhs;
  const uint32_t budget = static_cast<uint32_t>(std::min<uint64_t>(max_iterations, 0xffffffffu));
  // Eight faces a lane before more workgroups: the last of them waits for all the others' arrivals.
  const unsigned eg = std::min(kUniformGroups, grid_for((n + 7) / 8));
  const unsigned ag = static_cast<unsigned>(std::min<uint64_t>(kUniformGroups, (nb + 7) / 8 * 8));  // whole XCD rounds
  auto look = [&]() -> int {
    FL_HIP(hipMemcpyAsync(B.host, B.scal, sizeof(UniformScalars), hipMemcpyDeviceToHost, s));
    FL_HIP(hipStreamSynchronize(s));
    return FL_OK;
  };
  k_uniform_start<<<eg, kThreads, 0, s>>>(n, B.mask, B.rhs, B.diag, B.v, B.r, B.z, B.partial, B.arrived, B.scal);
  FL_HIP(hipGetLastError());
  int flip = 0;
  while (*iterations < max_iterations) {
    for (int k = 0; k < kBatch; ++k, flip ^= 1) {
      k_uniform_apply<true><<<ag, kBlockFaces, 0, s>>>(nb, B.near, B.mask, B.inertia, B.cn, B.cs, B.z, B.d[flip],
                                                       B.d[flip ^ 1], B.q, B.rhs, B.diag, B.r, B.z, tolerance,
                                                       B.partial, B.arrived, B.scal);
      k_uniform_step<<<eg, kThreads, 0, s>>>(n, B.mask, B.d[flip ^ 1], B.q, B.diag, B.v, B.r, B.z, tolerance, budget,
                                             B.partial, B.arrived, B.scal);
    }
    FL_HIP(hipGetLastError());
    FL_TRY(look());
    *iterations = B.host->iterations;
    if (B.host->status) return static_cast<int>(B.host->status);
    if (!B.host->stop) continue;
    // The recursive residual meets the tolerance or the budget is spent: the true residual decides.
    k_uniform_apply<false><<<ag, kBlockFaces, 0, s>>>(nb, B.near, B.mask, B.inertia, B.cn, B.cs, B.v, B.v, B.q, B.q,
                                                      B.rhs, B.diag, B.r, B.z, tolerance, B.partial, B.arrived, B.scal);
    FL_HIP(hipGetLastError());
    FL_TRY(look());
    if (B.host->nonfinite) return FL_OUT_OF_RANGE;
    if (B.host->max_r <= tolerance) {
      *max_residual = B.host->max_r;
      return FL_OK;
    }
  }
  return FL_ABORTED;
}

void release_uniform(fl_ctx* ctx) {
  auto* B = static_cast<UniformBuffers*>(ctx->uniform);
  if (!B) return;
  B->release();
  delete B;
  ctx->uniform = nullptr;
}

}  // namespace fl
