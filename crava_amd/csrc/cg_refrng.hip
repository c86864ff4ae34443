// cg_refrng.hip -- the reference's own noise stream, generated in parallel on the GPU.
//
// FFTGrid::fillInComplexNoise (fftgrid.cpp:997-1045) draws, in linear cell order, one or two
// normals per cell (none where it copies the conjugate of an earlier partner) from
// RandomGen::rnorm01 (random.cpp:38-111: Marsaglia-Bray), which consumes a variable number of
// uniforms u = seed * 2^-32 of the LCG seed <- 69069 seed + 1 (random.h:11-14,
// random.cpp:113-118).  Sequential as written; parallel here because the number of uniforms a
// normal consumes is a function of its starting offset in the uniform stream alone:
//   1. the stream is cut into chunks of kChunk offsets, one wavefront each: the uniforms consumed
//      by a normal starting at every offset go to LDS (97.45% of the offsets are decided by one
//      comparison; the rest are listed and their rejection loops run on consecutive lanes), then
//      each of 64 lanes follows one entry offset through the chunk: exit offset (into the next
//      chunk) and normals started inside it (k_chunk_maps);
//   2. groups of kGroup chunks compose those maps in LDS, one lane per entry (k_group_maps);
//   3. one thread chains the groups from offset 0 (k_chain), one thread per group its chunks
//      (k_chunk_entries), both through LDS; an entry outside the maps (a normal that consumed 64
//      or more uniforms across a boundary) is walked exactly;
//   4. one wavefront per chunk lists its normals' starts and computes them into an array indexed
//      by normal number, common and rare branches apart (k_emit), and one thread per cell picks
//      its normals (the number of normals drawn before a cell depends on indices only).
// What bounds it: the dependent chain of one LDS read per normal in 1 and 4 and their vector
// instructions, not memory.  Measured per fill of a 280 x 224 x 180 grid (11.4 M normals): maps
// 433 us, group maps 48, chain 19, entries 38, emission 365, cells 29 -- 0.93 ms, where chunks of
// 4096 with 8 tabulated entries, one thread per chunk and a group chain that walked every exit
// past the table took 9.0 ms (5.4 of them that chain).
// The state word advances as the reference's process-wide seed does (by the uniforms consumed).
// Arithmetic is the reference's: double uniforms, double exp/log/sqrt, float rounding of
// std * normal.
#include <cmath>
#include <vector>

#include "cg_internal.h"

// named (not anonymous) so that profilers show the kernels' names
namespace cgrng {

constexpr uint32_t kMul = 69069u;    // random.h:11
constexpr uint32_t kAdd = 1u;        // random.h:12
constexpr int kChunk = 2048;         // uniforms per chunk
constexpr int kEntries = 64;         // tabulated entry offsets per chunk: one per lane
constexpr int kGroup = 256;          // chunks per group (their maps fill 64 KB of LDS)
constexpr int kChain = 128;          // groups whose maps k_chain holds in LDS at a time (64 KB)
constexpr int kThreadsRng = 256;
constexpr unsigned kFar = 0xFFFFu;   // a step or exit that does not fit 16 bits (or a bad stream)
constexpr int kMaxDraw = 1 << 20;    // uniforms one normal may consume before the stream is declared bad

struct Affine {
  uint32_t a, c;  // x -> a x + c (mod 2^32)
};

__host__ __device__ inline Affine compose(Affine f, Affine g) { return Affine{f.a * g.a, f.a * g.c + f.c}; }

// LCG state after k steps from s.
__host__ __device__ inline uint32_t lcg_skip(uint32_t s, unsigned long long k)
{
  Affine r{1u, 0u}, p{kMul, kAdd};
  while (k) {
    if (k & 1ull) r = compose(p, r);
    p = compose(p, p);
    k >>= 1;
  }
  return r.a * s + r.c;
}

__host__ __device__ inline double unif01(uint32_t &st)
{
  st = kMul * st + kAdd;
  return (double)st * (1.0 / 4294967296.0);  // random.h:14: 2^-30 / 4
}

__host__ __device__ inline double mb_g(double x)  // random.cpp:96-111
{
  const double a = 17.49731196, b = 2.36785163, c = 2.15787544;
  const double absx = fabs(x);
  double result = a * exp(-x * x / 2.0);
  if (absx < 1.0)
    result -= 2.0 * b * (3.0 - x * x) + c * (1.5 - absx);
  else if (absx < 1.5)
    result -= b * (3.0 - absx) * (3.0 - absx) + c * (1.5 - absx);
  else
    result -= b * (3.0 - absx) * (3.0 - absx);
  return result;
}

// One Marsaglia-Bray normal from state st (advanced); returns the uniforms consumed, 0 if a
// rejection loop ran past kMaxDraw.
__host__ __device__ inline int rnorm01(uint32_t &st, double &x)
{
  int n = 1;
  const double u = unif01(st);
  if (u < 0.8638) {
    const double u1 = unif01(st), u2 = unif01(st), u3 = unif01(st);
    x = 2.0 * (u1 + u2 + u3) - 3.0;
    return n + 3;
  }
  if (u < 0.9745) {
    const double u1 = unif01(st), u2 = unif01(st);
    x = 1.5 * (u1 + u2 - 1.0);
    return n + 2;
  }
  if (u < 0.9973002039) {
    double u2;
    do {
      const double u1 = unif01(st);
      u2 = unif01(st);
      x = 6.0 * u1 - 3.0;
      n += 2;
      if (n > kMaxDraw) return 0;
    } while (0.358 * u2 > mb_g(x));
    return n;
  }
  double s, t;
  do {
    double v1, v2, w;
    do {
      const double u1 = unif01(st), u2 = unif01(st);
      v1 = 2.0 * u1 - 1.0;
      v2 = 2.0 * u2 - 1.0;
      w = v1 * v1 + v2 * v2;
      n += 2;
      if (n > kMaxDraw) return 0;
    } while (w >= 1.0);
    const double c = sqrt((9.0 - 2.0 * log(w)) / w);
    s = c * v1;
    t = c * v2;
  } while ((fabs(s) <= 3.0) && (fabs(t) <= 3.0));
  x = (fabs(s) > 3.0) ? s : t;
  return n;
}

struct Hop {
  int exit;   // entry offset into the next chunk (or group); < 0: bad stream
  int count;  // normals started inside
};

// Normals starting at offsets in [pos, end), the first at pos: exit offset past end and count.
__host__ __device__ inline Hop walk(uint32_t seed, unsigned long long pos, unsigned long long end)
{
  uint32_t st = lcg_skip(seed, pos);
  int cnt = 0;
  double x;
  while (pos < end) {
    const int n = rnorm01(st, x);
    if (!n) return Hop{-1, cnt};
    pos += (unsigned)n;
    ++cnt;
  }
  return Hop{(int)(pos - end), cnt};
}

// The thresholds of rnorm01's branches on the state word: u < t <=> word < t 2^32 (the product is
// exact), as integers.
__device__ __forceinline__ constexpr uint32_t below(double t)
{
  const double v = t * 4294967296.0;
  const uint32_t i = (uint32_t)v;
  return (double)i < v ? i + 1u : i;
}

// LCG constants of a jump by 64 uniforms (lanes take every 64th offset of a chunk).
constexpr Affine jump64()
{
  Affine p{kMul, kAdd};
  for (int i = 0; i < 6; ++i) p = Affine{p.a * p.a, p.a * p.c + p.c};
  return p;
}

// step[o] = uniforms consumed by a normal starting at offset o of the chunk whose first state is
// cs, for every o < kChunk (kFar: does not fit).  One wavefront; rare: LDS list of kChunk offsets.
__device__ __forceinline__ void chunk_steps(uint32_t cs, uint16_t *step, uint16_t *rare)
{
  constexpr Affine J = jump64();
  constexpr uint32_t t1 = below(0.8638), t2 = below(0.9745);
  const int lane = threadIdx.x;
  uint32_t st = lcg_skip(cs, (unsigned)lane);
  int nrare = 0;
  for (int o = lane; o < kChunk; o += 64) {
    const uint32_t w = kMul * st + kAdd;
    const bool hard = w >= t2;
    const unsigned long long m = __ballot(hard);
    if (hard) rare[nrare + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)o;
    else step[o] = w < t1 ? 4 : 3;
    nrare += __popcll(m);
    st = J.a * st + J.c;
  }
  __syncthreads();
  for (int i = lane; i < nrare; i += 64) {
    const int o = rare[i];
    uint32_t s = lcg_skip(cs, (unsigned)o);
    double x;
    const int n = rnorm01(s, x);
    step[o] = (uint16_t)(n > 0 && n < (int)kFar ? (unsigned)n : kFar);
  }
  __syncthreads();
}

// Chunk map entries: exit offset (low 16 bits, kFar: walk exactly) and normals (high 16 bits).
__global__ void __launch_bounds__(64) k_chunk_maps(uint32_t seed, uint32_t *__restrict__ maps)
{
  __shared__ uint16_t step[kChunk], rare[kChunk];
  const long c = blockIdx.x;
  const uint32_t cs = lcg_skip(seed, (unsigned long long)c * kChunk);
  chunk_steps(cs, step, rare);
  unsigned pos = threadIdx.x, cnt = 0;
  bool far = false;
  while (pos < (unsigned)kChunk) {
    const unsigned n = step[pos];
    if (n == kFar) {
      far = true;
      break;
    }
    pos += n;
    ++cnt;
  }
  const unsigned ex = pos - kChunk;
  maps[c * kEntries + threadIdx.x] = (far || ex >= kFar) ? kFar : (ex | (cnt << 16));
}

// Entry `cur` of chunk c: its exit and count from the chunk's map, or exactly.
__device__ __forceinline__ Hop hop_chunk(uint32_t seed, long c, const uint32_t *map, int cur)
{
  if (cur < kEntries) {
    const uint32_t v = map[cur];
    if ((v & 0xFFFFu) != kFar) return Hop{(int)(v & 0xFFFFu), (int)(v >> 16)};
  }
  const unsigned long long start = (unsigned long long)c * kChunk;
  return walk(seed, start + (unsigned)cur, start + kChunk);
}

// A group's chunk maps to LDS; returns its number of chunks.
__device__ __forceinline__ int load_group(long g, long nchunks, const uint32_t *__restrict__ maps, uint32_t *lds)
{
  const long c0 = g * kGroup;
  const int nc = (int)(nchunks - c0 < kGroup ? nchunks - c0 : kGroup);
  for (int i = threadIdx.x; i < nc * kEntries; i += blockDim.x) lds[i] = maps[c0 * kEntries + i];
  __syncthreads();
  return nc;
}

__global__ void __launch_bounds__(kThreadsRng) k_group_maps(uint32_t seed, long nchunks,
                                                            const uint32_t *__restrict__ maps, Hop *__restrict__ gmaps)
{
  __shared__ uint32_t lds[kGroup * kEntries];
  const long g = blockIdx.x;
  const int nc = load_group(g, nchunks, maps, lds);
  if (threadIdx.x >= kEntries) return;
  int cur = threadIdx.x, total = 0;
  for (int i = 0; i < nc; ++i) {
    const Hop h = hop_chunk(seed, g * kGroup + i, lds + i * kEntries, cur);
    if (h.exit < 0) {
      cur = -1;
      break;
    }
    total += h.count;
    cur = h.exit;
  }
  gmaps[g * kEntries + threadIdx.x] = Hop{cur, total};
}

// One workgroup: every group's entry offset and first normal number, from offset 0 until nnorm
// normals are placed (-1 and nnorm for the groups past them).  *status: 0, or 1 for a rejection
// loop past its bound, 2 for a stream too short.
__global__ void __launch_bounds__(kThreadsRng) k_chain(uint32_t seed, long nchunks, long ngroups,
                                                       const uint32_t *__restrict__ maps, const Hop *__restrict__ gmaps,
                                                       long long nnorm, int *__restrict__ gentry,
                                                       long long *__restrict__ gfirst, unsigned long long *status)
{
  __shared__ Hop lds[kChain * kEntries];
  int cur = 0;  // of thread 0
  long long first = 0;
  for (long g0 = 0; g0 < ngroups; g0 += kChain) {
    const int ng = (int)(ngroups - g0 < kChain ? ngroups - g0 : kChain);
    for (int i = threadIdx.x; i < ng * kEntries; i += blockDim.x) lds[i] = gmaps[g0 * kEntries + i];
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int i = 0; i < ng; ++i) {
        const bool live = cur >= 0 && first < nnorm;
        gentry[g0 + i] = live ? cur : -1;
        gfirst[g0 + i] = live ? first : nnorm;
        if (!live) continue;
        Hop h;
        if (cur < kEntries) {
          h = lds[i * kEntries + cur];
        } else {  // rare: through the group's chunks
          const long c0 = (g0 + i) * kGroup, c1 = c0 + kGroup < nchunks ? c0 + kGroup : nchunks;
          h = Hop{cur, 0};
          for (long c = c0; c < c1 && h.exit >= 0; ++c) {
            const Hop w = hop_chunk(seed, c, maps + c * kEntries, h.exit);
            h = Hop{w.exit, h.count + w.count};
          }
        }
        first += h.count;
        cur = h.exit;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *status = cur < 0 && first < nnorm ? 1ull : (first < nnorm ? 2ull : 0ull);
}

// One workgroup per group: entry offset and first normal number of its chunks.
__global__ void __launch_bounds__(kThreadsRng) k_chunk_entries(uint32_t seed, long nchunks,
                                                               const uint32_t *__restrict__ maps,
                                                               const int *__restrict__ gentry,
                                                               const long long *__restrict__ gfirst,
                                                               int *__restrict__ centry, long long *__restrict__ cfirst)
{
  __shared__ uint32_t lds[kGroup * kEntries];
  const long g = blockIdx.x;
  const int nc = load_group(g, nchunks, maps, lds);
  if (threadIdx.x != 0) return;
  int cur = gentry[g];
  long long first = gfirst[g];
  for (int i = 0; i < nc; ++i) {
    centry[g * kGroup + i] = cur;
    cfirst[g * kGroup + i] = first;
    if (cur < 0) continue;  // past the end of the requested normals
    const Hop h = hop_chunk(seed, g * kGroup + i, lds + i * kEntries, cur);
    cur = h.exit;  // negative: a bad stream; the chunks after it hold no normals
    first += h.count;
  }
}

// One wavefront per chunk: its normals, numbered from cfirst, while below nnorm; the offset after
// the last requested normal goes to *end_pos.  Lane 0 lists the starts (the dependent chain),
// then the lanes take the normals, the ones in rnorm01's rejection branches last and together.
__global__ void __launch_bounds__(64) k_emit(uint32_t seed, const int *__restrict__ centry,
                                             const long long *__restrict__ cfirst, long long nnorm,
                                             double *__restrict__ X, unsigned long long *__restrict__ end_pos)
{
  constexpr int kMost = kChunk / 3 + 1;  // a normal consumes at least three uniforms
  __shared__ uint16_t step[kChunk], rare[kChunk], start_at[kMost];
  __shared__ int listed;
  const long c = blockIdx.x;
  const int entry = centry[c];
  const long long first = cfirst[c];
  if (entry < 0 || entry >= kChunk || first >= nnorm) return;  // uniform over the workgroup
  const unsigned long long base = (unsigned long long)c * kChunk;
  const uint32_t cs = lcg_skip(seed, base);
  chunk_steps(cs, step, rare);
  const long long left = nnorm - first;
  const int lane = threadIdx.x;
  if (lane == 0) {
    unsigned pos = (unsigned)entry;
    int n = 0;
    while (pos < (unsigned)kChunk && n < left) {
      start_at[n++] = (uint16_t)pos;
      pos += step[pos];  // kFar ends the chunk, as the normal it stands for does
    }
    listed = n;
  }
  __syncthreads();
  const int n = listed;
  constexpr uint32_t t2 = below(0.9745);
  int nrare = 0;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int i = i0 + lane;
    bool hard = false;
    if (i < n) {
      uint32_t st = lcg_skip(cs, (unsigned)start_at[i]);
      hard = kMul * st + kAdd >= t2;
      if (!hard) {
        double x;
        (void)rnorm01(st, x);
        X[first + i] = x;
      }
    }
    const unsigned long long m = __ballot(hard);
    if (hard) rare[nrare + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)i;
    nrare += __popcll(m);
  }
  __syncthreads();
  for (int k = lane; k < nrare; k += 64) {
    const int i = rare[k];
    uint32_t st = lcg_skip(cs, (unsigned)start_at[i]);
    double x;
    if (rnorm01(st, x)) X[first + i] = x;
  }
  if (lane == 0 && first + n == nnorm && n > 0) {
    const unsigned at = start_at[n - 1];
    uint32_t st = lcg_skip(cs, at);
    double x;
    *end_pos = base + at + (unsigned)rnorm01(st, x);
  }
}

// Draws of a special cell (x = 0 column, or the x = cnxp-1 column at an odd linear index):
// 1 if it is its own conjugate, 2 if its partner comes later, 0 if it copies an earlier one.
__host__ __device__ inline int special_draws(long jk, int nyp, int nzp, long *jkcc_out)
{
  const long jind = jk % nyp, kind = jk / nyp;
  const long jcc = jind == 0 ? 0 : nyp - jind;
  const long kcc = kind == 0 ? 0 : nzp - kind;
  const long jkcc = jcc + kcc * nyp;
  *jkcc_out = jkcc;
  return jkcc == jk ? 1 : (jkcc > jk ? 2 : 0);
}

__host__ __device__ inline bool is_special(long i, int cnxp)
{
  const long xs = i % cnxp;
  return xs == 0 || (xs == cnxp - 1 && (i % 2) == 1);
}

// Normals drawn before cell i: rowbase[jk] + those of the cells before it in its row (the
// x = 0 cell, then ordinary cells with two each; the x = cnxp-1 cell is the row's last).
__device__ inline long long draws_before(long i, int cnxp, int nyp, int nzp, const long long *rowbase)
{
  const long jk = i / cnxp, xs = i % cnxp;
  if (xs == 0) return rowbase[jk];
  long jkcc;
  const int d0 = special_draws(jk, nyp, nzp, &jkcc);
  return rowbase[jk] + d0 + 2ll * (xs - 1);
}

// status as k_chain sets it: a stream that does not hold the normals leaves the grid alone.
__global__ void k_noise_cells(float2 *__restrict__ out, long csize, int cnxp, int nyp, int nzp,
                              const long long *__restrict__ rowbase, const double *__restrict__ X,
                              const unsigned long long *__restrict__ status)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= csize || *status != 0) return;
  const double sd = (double)(float)(1.0 / sqrt(2.0));  // fftgrid.cpp:1003, a float
  long src = i;
  bool conj = false, self = false;
  if (is_special(i, cnxp)) {
    const long jk = i / cnxp, xs = i % cnxp;
    long jkcc;
    const int d = special_draws(jk, nyp, nzp, &jkcc);
    if (d == 1) {
      self = true;
    } else if (d == 0) {
      src = jkcc * cnxp + xs;  // an earlier cell that drew two normals
      conj = true;
    }
  }
  const long long b = draws_before(src, cnxp, nyp, nzp, rowbase);
  float2 v;
  if (self) {
    v = make_float2((float)X[b], 0.f);
  } else {
    v = make_float2((float)(sd * X[b]), (float)(sd * X[b + 1]));
    if (conj) v.y = -v.y;
  }
  out[i] = v;
}

}  // namespace cgrng

namespace cg {

using namespace cgrng;

// Fills `out` (cnxp x nyp x nzp complex) as FFTGrid::fillInComplexNoise does from the state
// *seed and advances *seed past the uniforms consumed.  Synchronises the context stream.
int fill_noise_reference(cg_ctx *ctx, float2 *out, int nxp, int nyp, int nzp, uint32_t *seed)
{
  const int cnxp = nxp / 2 + 1;
  const long rows = (long)nyp * nzp, csize = rows * cnxp;
  // normals drawn before each row (index arithmetic only): the row's x = 0 cell draws d (as
  // special_draws: 1 where it is its own conjugate, 2 where the partner comes later, else 0), its
  // last cell d at an odd linear index and 2 otherwise, the cells between two each
  std::vector<long long> rowbase(rows + 1);
  long long acc = 0, jk = 0;
  const long long inner = 2ll * (cnxp > 2 ? cnxp - 2 : 0);
  for (long k = 0; k < nzp; ++k)
    for (long j = 0; j < nyp; ++j, ++jk) {
      rowbase[jk] = acc;
      const long kc = k == 0 ? 0 : nzp - k, jc = j == 0 ? 0 : nyp - j;
      const int d = kc != k ? (kc > k ? 2 : 0) : (jc == j ? 1 : (jc > j ? 2 : 0));
      acc += d + inner;
      if (cnxp > 1) acc += ((jk * cnxp + cnxp - 1) & 1) ? d : 2;
    }
  rowbase[rows] = acc;
  const long long nnorm = acc;
  // uniforms: about 3.93 per normal on average; the margin covers the spread many times over
  const unsigned long long ulen = (unsigned long long)nnorm * 4ull + (1ull << 20);
  const long nchunks = (long)((ulen + kChunk - 1) / kChunk);
  const long ngroups = (nchunks + kGroup - 1) / kGroup;
  const uint32_t s0 = *seed;
  // one device block: chunk and group maps, group and chunk entries and first normals, the rows'
  // bases, the normals, the end offset and status
  size_t size = 0;
  auto part = [&size](size_t bytes) {
    const size_t off = size;
    size += (bytes + 255) / 256 * 256;
    return off;
  };
  const size_t o_maps = part(sizeof(uint32_t) * nchunks * kEntries), o_gmaps = part(sizeof(Hop) * ngroups * kEntries),
               o_ge = part(sizeof(int) * ngroups), o_gf = part(sizeof(long long) * ngroups),
               o_ce = part(sizeof(int) * nchunks), o_cf = part(sizeof(long long) * nchunks),
               o_rows = part(sizeof(long long) * (rows + 1)), o_x = part(sizeof(double) * (nnorm + 2)),
               o_end = part(2 * sizeof(unsigned long long));
  char *dev = nullptr;
  hipError_t e = dev_alloc(ctx, (void **)&dev, size);
  if (e != hipSuccess) return fail(ctx, CG_ENOMEM, "reference noise: device memory");
  uint32_t *maps = reinterpret_cast<uint32_t *>(dev + o_maps);
  Hop *gmaps = reinterpret_cast<Hop *>(dev + o_gmaps);
  int *gentry = reinterpret_cast<int *>(dev + o_ge), *centry = reinterpret_cast<int *>(dev + o_ce);
  long long *gfirst = reinterpret_cast<long long *>(dev + o_gf), *cfirst = reinterpret_cast<long long *>(dev + o_cf),
            *rowbase_d = reinterpret_cast<long long *>(dev + o_rows);
  double *X = reinterpret_cast<double *>(dev + o_x);
  unsigned long long *end_pos = reinterpret_cast<unsigned long long *>(dev + o_end);
  e = hipMemcpyAsync(rowbase_d, rowbase.data(), sizeof(long long) * (rows + 1), hipMemcpyHostToDevice, ctx->stream);
  if (e != hipSuccess) {  // nothing may be launched on row bases that did not arrive
    dev_free(ctx, dev);
    return hip_fail(ctx, e, "reference noise: upload");
  }
  auto blocks = [](long n) { return (unsigned)((n + kThreads - 1) / kThreads); };
  hipEvent_t ev;
  launch_begin(ctx, CG_K_NOISE, &ev);
  k_chunk_maps<<<(unsigned)nchunks, 64, 0, ctx->stream>>>(s0, maps);
  k_group_maps<<<(unsigned)ngroups, kThreadsRng, 0, ctx->stream>>>(s0, nchunks, maps, gmaps);
  k_chain<<<1, kThreadsRng, 0, ctx->stream>>>(s0, nchunks, ngroups, maps, gmaps, nnorm, gentry, gfirst, end_pos + 1);
  k_chunk_entries<<<(unsigned)ngroups, kThreadsRng, 0, ctx->stream>>>(s0, nchunks, maps, gentry, gfirst, centry, cfirst);
  k_emit<<<(unsigned)nchunks, 64, 0, ctx->stream>>>(s0, centry, cfirst, nnorm, X, end_pos);
  k_noise_cells<<<blocks(csize), kThreads, 0, ctx->stream>>>(out, csize, cnxp, nyp, nzp, rowbase_d, X,
                                                                end_pos + 1);
  launch_end(ctx, CG_K_NOISE, ev);
  unsigned long long got[2] = {0, 0};  // end offset, status
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(got, end_pos, sizeof(got), hipMemcpyDeviceToHost, ctx->stream);
  const hipError_t es = hipStreamSynchronize(ctx->stream);
  dev_free(ctx, dev);
  if (e == hipSuccess) e = es;
  if (e != hipSuccess) return hip_fail(ctx, e, "reference noise");
  if (got[1] == 1) return fail(ctx, CG_EINVAL, "reference noise: a rejection loop exceeded its bound");
  if (got[1] == 2) return fail(ctx, CG_EINVAL, "reference noise: uniform stream shorter than the normals need");
  const unsigned long long endp = got[0];
  *seed = lcg_skip(s0, endp);
  return CG_OK;
}

}  // namespace cg
