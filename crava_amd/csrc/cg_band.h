// cg_band.h -- FFT passes of an inversion that computes the inverted wavenumbers only (templates;
// instantiated per length by cg_fft_fixed_part.hip, run by cg_invert's band-limited sequence).
//
// The posterior changes the wavenumbers of the planes k_z with invert[k_z] alone: elsewhere it keeps
// the prior mean, whose inverse transform is the prior mean itself.  So the z transform runs
// first, on the real cube, and only the band's frequencies go on through the x and y passes; the
// posterior's update (not the mean) comes back the same way, and the last pass adds it to the prior
// mean.  At a band of 40% of the planes (5-55 Hz of 125) a grid costs 1 + 6 x 0.4 grids of traffic
// on the way in instead of 6, and 2 + 6 x 0.4 on the way out.
//
// Band layout: B frequencies kb[0] < kb[1] < ... in 0..nzp/2 (k and nzp - k share one), a plane per
// frequency, [B][nyp][rnxp] complex with rnxp = 2 (nxp/2 + 1): the x axis is whole (the cube is
// real along z, not along x), W[b][y][x] = sum_z a(x, y, z) w^(z kb[b]).  A wavenumber (x, y, kb[b])
// of the reference's half spectrum is W[b][y][x]; (x, y, nzp - kb[b]) is conj W[b][-y][-x].  The
// columns past nxp hold a second copy of the columns 0 and (even nxp) nxp/2, which belong to both:
// forward a duplicate, on the way back the mirrored plane's own value, and the inverse x pass takes
// the mean of the two -- the Hermitian part, which is all that the reference's half-complex inverse
// keeps of those columns.
#pragma once

#include "cg_fft_fixed.h"

namespace cgfix {

// Stages of a z tile.  A length of two radices P1 <= P2 <= 2 P1 runs on TPS = P2 threads per column,
// the radix P1 on the side that touches memory (forward first, inverse last), so that every thread
// takes part in the loads or stores with P1 values each; other lengths take their plan.  The plans
// of the y and z passes hold 20 to 32 values a thread, which leaves few wavefronts per CU once the
// prior mean's pairs wait in registers too.  Microseconds per grid, plan / this, nzp 384 at 1152 x
// 576: forward 305 / 292, inverse 1014 / 516 (4.8 TB/s); nzp 360 at 405 x 375: 66.6 / 63.9, 128 / 130;
// unbalanced radices lose (nzp 243 = 9 x 27 at 280 x 270: 26.6 / 30.9, 44.6 / 47.0).
template <int N, int DIR, int ES, bool TWO = (row_split(N) > 1 && N <= 2 * row_split(N) * row_split(N))>
struct BandZ {
  static constexpr int TPS = Plan<N>::TPS, LAST = Plan<N>::LAST;
  using IO = typename Plan<N>::template IO<DIR, ES>;
};
template <int N, int DIR, int ES>
struct BandZ<N, DIR, ES, true> {
  static constexpr int P1 = row_split(N), P2 = N / P1, TPS = P2, LAST = DIR < 0 ? P2 : P1;
  using IO = StagesIO<N, DIR, TPS, ES, 1, DIR < 0 ? P1 : P2, DIR < 0 ? P2 : P1>;
};

// Columns (pairs of neighbouring x) per z tile: as the strided passes, with the table of the band's
// planes in the LDS too.
template <int N>
constexpr int band_tile()
{
  constexpr int ti = strided_tile0<N>();
  return ti > 8 && sizeof(float2) * N * (ti + 1) + sizeof(short) * (N / 2 + 1) > kLds ? ti / 2 : ti;
}
template <int N>
constexpr int band_threads()
{
  return band_tile<N>() * BandZ<N, -1, band_tile<N>()>::TPS;  // the same both ways
}

// Item of a list (items[i] owns blocks [block0_i, block0_{i+1})).
__device__ __forceinline__ unsigned band_item(const cg::BandArgs *items, int nitems, cg::BandArgs &a)
{
  const unsigned g = cg_xcd_remap(blockIdx.x, gridDim.x);
  a = items[nitems > 1 ? find_item(items, nitems, g) : 0];
  return g - a.block0;
}

// z forward.  A column of the grid's float pairs is z = a + i b of two neighbouring traces; after
// the complex transform A[k] = (Z[k] + conj Z[N-k]) / 2, B[k] = -i (Z[k] - conj Z[N-k]) / 2.  The
// strided pass's tile; the last stage's outputs stay in LDS and the band's frequencies leave as
// 16-byte pairs (TI of them: 256-byte segments).  4.4 TB/s at 576 x 576 x 320.
template <int N>
__global__ void __launch_bounds__(band_threads<N>())
k_bandz_fwd(const cg::BandArgs *__restrict__ items, int nitems, const float2 *__restrict__ twg)
{
  constexpr int TI = band_tile<N>(), TPS = BandZ<N, -1, TI>::TPS, NT = TI * TPS;
  using IO = typename BandZ<N, -1, TI>::IO;
  extern __shared__ float2 smem[];
  float2 *tw = smem, *buf = smem + N;
  __shared__ short at[N / 2 + 1];  // the band's plane of a frequency, or -1
  cg::BandArgs a;
  const unsigned blk = band_item(items, nitems, a);
  const int tid = threadIdx.x, c = tid % TI, t = tid / TI;
  const unsigned q = blk * TI + c, xp = q % a.cnxp;
  const bool live = q < a.ncols;
  const bool first = live && 2 * (int)xp < a.nxp, second = live && 2 * (int)xp + 1 < a.nxp;
  const float2 *col = reinterpret_cast<const float2 *>(a.real) + (live ? q : 0);
  load_tw(tw, twg, N, tid, NT);
  for (int k = tid; k <= N / 2; k += NT) at[k] = (short)cg::gld(a.at + k);
  float2 v[IO::BPT][IO::P_];
#pragma unroll
  for (int b = 0; b < IO::BPT; ++b) {
    const int j = t + b * TPS;
#pragma unroll
    for (int r = 0; r < IO::P_; ++r) {
      v[b][r] = (first && (IO::EVEN || j < IO::NB)) ? cg::gld(col + (long)(j + r * IO::NB) * a.ncols) : make_float2(0.f, 0.f);
      if (!second) v[b][r].y = 0.f;  // the row padding is no data
    }
  }
  lds_sync();
  float2 *mine = buf + c;
  auto sink = [&](int e, float2 x) { mine[e * TI] = x; };
  IO::step(v, mine, t, tw, sink);
  lds_sync();
  const float s = 0.5f * a.scale;
  typedef float fvec4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int i = 0; i < (N / 2 + TPS) / TPS; ++i) {  // every frequency 0..N/2, the band's stored
    const int k = t + i * TPS;
    const int p = k <= N / 2 ? at[k] : -1;
    if (p >= 0) {
      const float2 z = cscale(mine[k * TI], s), m = cscale(mine[(k ? N - k : 0) * TI], s);
      if (live)
        *(__attribute__((address_space(1))) fvec4 *)(a.band + 2 * ((size_t)p * a.ncols + q)) =
            fvec4{z.x + m.x, z.y - m.y, z.y + m.y, m.x - z.x};
    }
  }
}

// z inverse: the band's frequencies of two neighbouring columns make Z[k] = A + i B and
// Z[N-k] = conj A + i conj B (the imaginary parts of a self-conjugate frequency dropped), the rest is
// zero; the transform's pairs are the two real traces, scaled and added to the prior mean.  Every
// frequency is loaded once and placed in LDS at k and N - k (loading each input of the first stage
// from memory read the band twice and held 8 of them a thread: 289 -> 221 us per grid at 576 x 576 x
// 320, 4.6 TB/s).
template <int N>
__global__ void __launch_bounds__(band_threads<N>())
k_bandz_inv(const cg::BandArgs *__restrict__ items, int nitems, const float2 *__restrict__ twg)
{
  constexpr int TI = band_tile<N>(), TPS = BandZ<N, +1, TI>::TPS, NT = TI * TPS;
  using IO = typename BandZ<N, +1, TI>::IO;
  constexpr int LP = BandZ<N, +1, TI>::LAST, LNB = N / LP, LB = (LNB + TPS - 1) / TPS;  // the last stage's outputs
  extern __shared__ float2 smem[];
  float2 *tw = smem, *buf = smem + N;
  __shared__ short at[N / 2 + 1];  // the band's plane of a frequency, or -1
  cg::BandArgs a;
  const unsigned blk = band_item(items, nitems, a);
  const int tid = threadIdx.x, c = tid % TI, t = tid / TI;
  const unsigned q = blk * TI + c, xp = q % a.cnxp;
  const bool live = q < a.ncols;
  const bool first = live && 2 * (int)xp < a.nxp, second = live && 2 * (int)xp + 1 < a.nxp;
  load_tw(tw, twg, N, tid, NT);
  for (int k = tid; k <= N / 2; k += NT) at[k] = (short)cg::gld(a.at + k);
  lds_sync();
  typedef float fvec4 __attribute__((ext_vector_type(4)));
  const float2 *src = a.band + 2 * (size_t)(live ? q : 0);
  // every frequency 0..N/2 once (zero outside the band), all loads in flight
  constexpr int KPT = (N / 2 + TPS) / TPS;
  fvec4 f[KPT];
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    const int k = t + i * TPS;
    const int p = first && k <= N / 2 ? at[k] : -1;
    f[i] = p >= 0 ? *(const __attribute__((address_space(1))) fvec4 *)(src + 2 * (size_t)p * a.ncols) : fvec4{0.f, 0.f, 0.f, 0.f};
    if (!second) f[i].z = f[i].w = 0.f;  // the column past an odd row: the x pass leaves it as the work grid had it
  }
  // the prior mean's pairs of this thread's outputs (element j + r LNB of the column), in flight
  // during the transform
  const float2 *add = reinterpret_cast<const float2 *>(a.real) + (live ? q : 0);
  float2 m[LB][LP];
#pragma unroll
  for (int b = 0; b < LB; ++b) {
    const int j = t + b * TPS;
#pragma unroll
    for (int r = 0; r < LP; ++r)
      m[b][r] = (first && (LNB % TPS == 0 || j < LNB)) ? cg::gld(add + (long)(j + r * LNB) * a.ncols) : make_float2(0.f, 0.f);
  }
  float2 *mine = buf + c;
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    const int k = t + i * TPS;
    if (k > N / 2) continue;
    const bool self = k == 0 || 2 * k == N;
    mine[k * TI] = self ? make_float2(f[i].x, f[i].z) : make_float2(f[i].x - f[i].w, f[i].y + f[i].z);
    if (!self) mine[(N - k) * TI] = make_float2(f[i].x + f[i].w, f[i].z - f[i].y);
  }
  lds_sync();
  const float scale = a.scale;
  float2 *out = reinterpret_cast<float2 *>(a.out) + (live ? q : 0);
  auto sink = [&](int e, float2 x, int b, int r) {
    const float2 y = m[b][r];
    float2 o = make_float2(x.x * scale + y.x, x.y * scale + y.y);
    if (!first) o.x = 0.f;
    if (!second) o.y = 0.f;
    if (live) cg::gst(out + (long)e * a.ncols, o);
  };
  IO::from_lds(mine, t, tw, sink);
}

// x pass of the band's rows (complex, whole length N = nxp; pitch rnxp).  Lengths that split into
// two radices P1 P2 <= 32 run with a row on T = P2 lanes of one wavefront: the first stage's inputs
// come straight from memory, one exchange through the wavefront's own LDS (element q of lane t at
// q PITCH + t, read back at t PITCH + q, PITCH odd: no bank conflicts), the second stage's outputs
// go straight back, and no barrier but the one for the twiddles.  The others take the length's
// plan with a row on TPS threads.
template <int N>
struct BandRow {
  static constexpr int P1 = row_split(N);
  static constexpr bool WAVE = P1 > 0;
  static constexpr int P2 = WAVE ? N / (WAVE ? P1 : 1) : 1;
  static constexpr int TPS = WAVE ? P2 : Plan<N>::TPS;     // threads per row
  static constexpr int R = WAVE ? 64 / TPS : 0;            // rows per wavefront
  // workgroups of 4 wavefronts, 8 at the long lengths (fewer loads of the twiddles per row); plans:
  // about 256 threads.  Measured in place on 64 x 576 rows of 576: 71.6 us (4.76 TB/s; 75.5 with 4
  // wavefronts, 75.0 by the plan; a copy takes 60.2); 40 x 280 rows of 224: 8.3 us against 11.8 by
  // the plan; 77 x 1152 rows of 1152 (no split): 345 us, 4.75 TB/s.
  static constexpr int WAVES = N >= 512 ? 8 : 4;
  static constexpr int ROWS = WAVE ? WAVES * R : (TPS >= 128 ? 2 : 256 / TPS);
  static constexpr int THREADS = WAVE ? 64 * WAVES : ROWS * TPS;
  static constexpr int PITCH = P2 | 1;
  static constexpr int LDS = WAVE ? R * P1 * PITCH : 1;    // float2 per wavefront
};

// Element k of an inverse row: columns 0 and N/2 with the mirrored plane's copy past the row.
template <int N>
__device__ __forceinline__ float2 band_load(const float2 *in, int k, bool inverse)
{
  float2 x = cg::gld(in + k);
  if (inverse && (k == 0 || (N % 2 == 0 && k == N / 2))) {
    const float2 y = cg::gld(in + (k == 0 ? N : N + 1));
    x = make_float2(0.5f * (x.x + y.x), 0.5f * (x.y + y.y));
  }
  return x;
}
template <int N>
__device__ __forceinline__ void band_store(float2 *out, int k, float2 x, bool forward)
{
  cg::gst(out + k, x);
  if (forward && k == 0) cg::gst(out + N, x);
  if (forward && N % 2 == 0 && k == N / 2) cg::gst(out + N + 1, x);
}

template <int N, int DIR>
__global__ void __launch_bounds__(BandRow<N>::THREADS)
k_bandx(const cg::BandArgs *__restrict__ items, int nitems, const float2 *__restrict__ twg)
{
  using P = BandRow<N>;
  constexpr bool FWD = DIR < 0;
  constexpr int RP = 2 * (N / 2 + 1);
  __shared__ float2 tw[N];
  cg::BandArgs a;
  const unsigned blk = band_item(items, nitems, a);
  const int tid = threadIdx.x;
  if constexpr (P::WAVE) {
    constexpr int P1 = P::P1, P2 = P::P2;
    __shared__ float2 lds[P::WAVES][P::LDS];
    const int lane = tid & 63, r = lane / P2, t = lane - r * P2;
    const long row = (long)blk * P::ROWS + (tid >> 6) * P::R + r;
    const bool on = r < P::R && row < a.rows;
    const float2 *in = a.band + (on ? row * RP : 0);
    float2 *out = a.band_out + (on ? row * RP : 0);
    float2 v[P1], u[P2];
    if (on) {
#pragma unroll
      for (int q = 0; q < P1; ++q) v[q] = band_load<N>(in, t + q * P2, !FWD);
    }
    load_tw(tw, twg, N, tid, P::THREADS);
    lds_sync();
    float2 *buf = lds[tid >> 6] + (r < P::R ? r : 0) * P1 * P::PITCH;
    if (on) {
      dft<DIR, P1>(v);
#pragma unroll
      for (int q = 0; q < P1; ++q) buf[q * P::PITCH + t] = v[q];
    }
    wave_lds_order();
    if (on && t < P1) {
#pragma unroll
      for (int q = 0; q < P2; ++q) u[q] = buf[t * P::PITCH + q];
      if (P1 > 1) {
#pragma unroll
        for (int q = 1; q < P2; ++q) {
          float2 w = tw[q * t];
          if (DIR > 0) w.y = -w.y;
          u[q] = cmul(u[q], w);
        }
      }
      dft<DIR, P2>(u);
#pragma unroll
      for (int q = 0; q < P2; ++q) band_store<N>(out, t + q * P1, u[q], FWD);
    }
  } else {
    using IO = typename Plan<N>::template IO<DIR, 1>;
    constexpr int TPS = P::TPS;
    __shared__ float2 buf[P::ROWS * (N + 1)];
    const int r = tid / TPS, t = tid % TPS;
    const long row = (long)blk * P::ROWS + r;
    const bool on = row < a.rows;
    const float2 *in = a.band + (on ? row * RP : 0);
    float2 *out = a.band_out + (on ? row * RP : 0);
    float2 v[IO::BPT][IO::P_];
#pragma unroll
    for (int b = 0; b < IO::BPT; ++b) {
      const int j = t + b * TPS;
#pragma unroll
      for (int q = 0; q < IO::P_; ++q)
        v[b][q] = on && (IO::EVEN || j < IO::NB) ? band_load<N>(in, j + q * IO::NB, !FWD) : make_float2(0.f, 0.f);
    }
    load_tw(tw, twg, N, tid, P::THREADS);
    lds_sync();
    auto sink = [&](int e, float2 x) {
      if (on) band_store<N>(out, e, x, FWD);
    };
    IO::step(v, buf + r * (N + 1), t, tw, sink);
  }
}

// ---------------------------------------------------------------- host launchers
// dir < 0: z forward (real -> band), else z inverse (band -> out, added to real).
template <int N>
int bandz_launch(cg_ctx *ctx, int dir, const cg::BandArgs *items, int nitems, unsigned nblocks, const float2 *tw)
{
  constexpr int TI = band_tile<N>();
  const size_t lds = sizeof(float2) * (N + (size_t)N * TI);
  constexpr int NT = band_threads<N>();
  if (dir < 0) k_bandz_fwd<N><<<nblocks, NT, lds, ctx->stream>>>(items, nitems, tw);
  else k_bandz_inv<N><<<nblocks, NT, lds, ctx->stream>>>(items, nitems, tw);
  return cg::hip_fail(ctx, hipGetLastError(), "k_bandz");
}

template <int N>
int bandx_launch(cg_ctx *ctx, int dir, const cg::BandArgs *items, int nitems, unsigned nblocks, const float2 *tw)
{
  if (dir < 0) k_bandx<N, -1><<<nblocks, BandRow<N>::THREADS, 0, ctx->stream>>>(items, nitems, tw);
  else k_bandx<N, +1><<<nblocks, BandRow<N>::THREADS, 0, ctx->stream>>>(items, nitems, tw);
  return cg::hip_fail(ctx, hipGetLastError(), "k_bandx");
}

}  // namespace cgfix
