/*
 * FP64 plain solver: one path per lane, FP64 throughout, the arithmetic and
 * the random draws of the walk in htgx_device.h (track, stage_consume,
 * real_begin) realisation for realisation and bit for bit, in a persistent
 * kernel. It is the device counterpart of draw_pixel_xwave / draw_pixel_flux
 * (src/atmosphere/htrdr_atmosphere_draw_map.c:210-436) driven by the tile
 * loop of draw_map (src/core/htrdr_draw_map.c:324-491).
 *
 * What bounds it: instruction issue with partly filled wavefronts, and on
 * small maps the chain of dependent steps of the longest walk. As one loop
 * per thread -- query, segments, collisions, nested -- a wavefront ran every
 * lane's inner loops to the longest one's end, through 261 KB of code (a
 * Threefry-4x64 block inlined at each of some twenty draw sites) that did not
 * fit the 64 KB instruction cache, with 264 bytes of spills a lane. Here a
 * lane is a state machine, and in each iteration the wavefront runs a segment
 * step, a collision step and, once enough lanes need it, an event step, each
 * for the lanes in that state; a collision step holds one Threefry site and
 * an event step three. 128x128 pixels x 32 realisations, shortwave: 557 ->
 * 85 ms; longwave flux map, 128x128 x 16: 173 -> 27 ms.
 *
 * State the tracking steps use stays in registers (at most 256: 2 waves per
 * SIMD), the rest of the walk in LDS as arrays over the lanes (65 KB per
 * block, so two blocks per CU).
 */
#include "htgx_internal.h"
#include "htgx_queue.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>

using namespace htgx;

#define HIP_OK(expr) do {                                                     \
  hipError_t e_ = (expr);                                                    \
  if(e_ != hipSuccess) {                                                     \
    fprintf(stderr, "htgx: %s failed: %s (%s:%d)\n", #expr,                  \
      hipGetErrorString(e_), __FILE__, __LINE__);                            \
    return e_ == hipErrorOutOfMemory ? HTGX_MEM_ERR : HTGX_UNKNOWN_ERR;       \
  }                                                                           \
} while(0)

namespace {

constexpr int kBlock = 256;

struct Launch {
  uint32_t width, height, ntx;
  uint32_t K;         /* realisations per chunk (the last of a pixel may be shorter) */
  uint32_t nsub;      /* chunks per pixel */
  uint32_t planes;    /* 3 for the channels of a CIE XYZ image, else 1 */
  uint32_t plane_tiles, ntiles, xcd_tiles;
  uint32_t lanes;     /* lanes of each wavefront that take work */
  Gptr<unsigned int> counters;   /* [kXcds] next chunk of each XCD range */
  Gptr<htgx_mc_accum> partials;  /* [ntiles * nsub * 64] */
  Gptr<unsigned long long> stats;
};

struct KArgs {
  DevScene S;
  DevMap M;
  Launch P;
};

enum { LS_SEG = 0, LS_COLL = 1, LS_EVENT = 2, LS_DONE = 3 };
/* stages beside those of htgx::Stage */
enum { ST_BEGIN = 7, ST_FETCH = 8 };
enum { ITER_END = 0, ITER_SEGMENT = 1, ITER_AGAIN = 2 };

/* Per-lane state of the tracking steps */
struct Lane {
  uint32_t pixel, r;    /* the realisation, counted from the map's spp_offset */
  uint32_t draw;        /* next draw of its stream */
  uint64_t buf[4];      /* the Threefry block holding it, unless draw % 4 == 0 */
  uint32_t iband, kquad; /* band, k-point row */
  uint32_t channel;     /* of an image of several channels: 1 + the lane's, else 0 */
  uint32_t surface : 1, rayleigh : 1, gh_hit : 1, specular : 1, prev_edge : 1, gh_edge : 1;
  uint32_t pending : 1, nq : 1, nq_ground : 1;
  uint32_t done : 1, adv : 1, adv_g : 1, adv_c : 1, s_cloud : 1;
  uint32_t lstate : 2, mode : 2, prop : 2, ev : 2;
  uint32_t cstate : 3;  /* 0 before grid, 1 in leaf, 2 outside, 3 locate at t, 4 step out of leaf */
  uint32_t exit_axis : 2;
  double o[3], d[3], inv[3];
  double t, tmax, tnext; /* iterator; grid entry or leaf exit */
  double Ts, Tmin;
  uint32_t lo[3], hi[3]; /* leaf range in blocks */
  float lmn, lmx;
  int32_t j, s_layer;
  double s_t1, s_kmin, maj, tc; /* segment; next tentative collision */
  double c;             /* particle coefficient per LWC of the query's property */
  double ca, cs;        /* longwave: those of absorption and scattering */
  double g, gs;         /* gas coefficient of the segment: the property's; longwave: ka and ks */
  /* repeated clouds */
  double ow[2], shift[2];
  int64_t k[2], ntiles;
  /* counters */
  uint32_t n_leaf, n_seg, n_coll, n_cell, n_ev;
};

/* Per-lane state of the event step, in LDS */
struct LaneCold {
  double pdf[kBlock], g[kBlock], L_sun[kBlock], wlen[kBlock];
  double w[kBlock], ksi[kBlock], R[kBlock], refl[kBlock], gas_ratio[kBlock];
  double dir_next[3][kBlock];
  double sum[kBlock], sum_c[kBlock], sum2[kBlock], sum2_c[kBlock], tsum[kBlock], tsum2[kBlock];
  double org[3][kBlock], dir0[3][kBlock], cosN[kBlock], Ld[kBlock]; /* shortwave flux */
  uint32_t stage[kBlock], mask[kBlock], phase[kBlock], t0[kBlock];
  int32_t prev_prim[kBlock], gh_prim[kBlock];
  uint32_t n[kBlock], nfail[kBlock], chunk[kBlock], r_end[kBlock], plane[kBlock];
};
__shared__ LaneCold g_cold;
/* The arguments, one copy per wavefront, for the event step */
__shared__ KArgs g_args[kBlock / 64];
#define LC(f) (g_cold.f[threadIdx.x])
#define LCA(f, a) (g_cold.f[a][threadIdx.x])

__device__ __forceinline__ double canonical(uint64_t v) { return (double)(v >> 11) * 0x1.0p-53; }

/* Block b of the realisation's stream (Stream of htgx_rng.h) */
__device__ __forceinline__ void stream_block(const Lane& L, uint64_t seed, uint32_t spp_offset, uint32_t b,
                                             uint64_t out[4])
{
  const uint64_t ctr[4] = {b, 0, 0, 0};
  const uint64_t key[4] = {seed ^ ((uint64_t)L.channel << 56), L.pixel, (uint64_t)spp_offset + L.r, 0};
  threefry4x64_20(ctr, key, out);
}

/* The draws of one event, in stream order, and how many it takes before the
 * optical thickness of its next query, which is the draw `ts'. Every index is a
 * constant where it is used: an index that varies over the lanes would put the
 * array in scratch memory, a load of several hundred cycles each. */
constexpr int kMaxDraws = 10;
struct Draws {
  uint64_t w[kMaxDraws];
  uint64_t ts;
  uint32_t n;

  __device__ __forceinline__ double at(int i) const { return canonical(w[i]); }
  __device__ __forceinline__ void end(int i) { ts = w[i]; n = (uint32_t)i; }
};

/* Kernels without GEN: a plane ground or none, grey materials, no repetition,
 * pinhole camera, wavelength modes 0 and 1 */
template<bool GEN>
__device__ __forceinline__ GroundHit trace(const DevScene& S, const double o[3], const double d[3], double r1,
                                           int32_t prev_prim, bool prev_edge, bool any)
{
  if(GEN) return ground_trace(S, o, d, 0.0, r1, prev_prim, prev_edge, any);
  GroundHit h;
  h.hit = false;
  h.t = FLT_MAX;
  h.N[0] = h.N[1] = h.N[2] = 0;
  h.mtl = 0;
  h.prim = -1;
  h.edge = false;
  if(S.ground_type == HTGX_GROUND_PLANE && prev_prim != 0 && d[2] != 0) {
    const double t = (S.plane_z - o[2]) / d[2];
    if(t > 0.0 && t < r1) {
      h.hit = true;
      h.t = t;
      h.N[2] = 1;
      h.mtl = S.plane_mtl;
      h.prim = 0;
    }
  }
  return h;
}

/* Normal and material of ground primitive prim, as ground_trace gives them */
template<bool GEN>
__device__ __forceinline__ uint32_t ground_surface(const DevScene& S, int32_t prim, double N[3])
{
  if(GEN && S.ground_type == HTGX_GROUND_MESH) {
    const BvhTri& T = S.tris[prim];
    const float n0 = T.e1[1] * T.e2[2] - T.e1[2] * T.e2[1];
    const float n1 = T.e1[2] * T.e2[0] - T.e1[0] * T.e2[2];
    const float n2 = T.e1[0] * T.e2[1] - T.e1[1] * T.e2[0];
    N[0] = n0; N[1] = n1; N[2] = n2;
    normalize3(N);
    return S.tri_mtl[prim];
  }
  N[0] = N[1] = 0;
  N[2] = 1;
  return S.plane_mtl;
}

/*******************************************************************************
 * Segment iterator: SegIter of htgx_device.h, one pass at a time
 ******************************************************************************/
template<bool GEN>
__device__ __forceinline__ void iter_init(const DevScene& S, Lane& L)
{
  const bool repeat = GEN && S.repeat;
#pragma unroll
  for(int a = 0; a < 3; ++a) L.inv[a] = 1.0 / L.d[a];
  L.t = 0.0;
  L.done = false;
  L.adv = false;
  L.cstate = 2;
  if(GEN) {
    L.k[0] = L.k[1] = 0;
    L.shift[0] = L.shift[1] = 0.0;
    L.ow[0] = L.o[0];
    L.ow[1] = L.o[1];
    L.ntiles = 0;
  }
  if(S.has_clouds) {
    double tn = -INFINITY, tf = INFINITY;
    bool miss = false;
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      if(repeat && a < 2) continue;
      const double plo = S.lower[a] + 0.0 * S.bs[a], phi = S.lower[a] + (double)S.dims0[a] * S.bs[a];
      if(L.d[a] != 0) {
        const double ta = (plo - L.o[a]) * L.inv[a];
        const double tb = (phi - L.o[a]) * L.inv[a];
        const double n = ta < tb ? ta : tb;
        const double f = ta < tb ? tb : ta;
        if(n > tn) tn = n;
        if(f < tf) tf = f;
      } else if(L.o[a] < plo || L.o[a] > phi) {
        miss = true;
      }
    }
    if(!miss && fmax(tn, L.t) < fmin(tf, L.tmax)) {
      if(repeat) {
        const double te = fmax(tn, L.t);
#pragma unroll
        for(int a = 0; a < 2; ++a) {
          L.k[a] = (int64_t)floor((L.ow[a] + te * L.d[a] - S.lower[a]) / S.period[a]);
          L.shift[a] = (double)L.k[a] * S.period[a];
          L.o[a] = L.ow[a] - L.shift[a];
        }
      }
      if(tn > L.t) { L.cstate = 0; L.tnext = tn; }
      else L.cstate = 3;
    }
  }
  const double z = L.o[2] + L.t * L.d[2];
  const double fj = floor((z - S.zb) * S.inv_dzl);
  L.j = fj < -1.0 ? -1 : fj > (double)S.nlayers ? (int32_t)S.nlayers : (int32_t)fj;
}

/* The next leaf (cstate 3: the one holding the point at t; 4: the one across
 * the exit face of the current leaf) and its exit distance */
template<bool GEN, bool COUNT>
__device__ __forceinline__ void next_leaf(const DevScene& S, Lane& L)
{
  const bool step = L.cstate == 4;
  uint32_t c[3];
  bool out = false;
  int oa = 0;
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    const uint32_t n = S.dims0[a], lo = step ? L.lo[a] : 0u, hi = step ? L.hi[a] : n;
    const bool fwd = L.d[a] > 0;
    const bool across = step && a == (int)L.exit_axis;
    const bool out_a = across && (fwd ? hi >= n : lo == 0);
    const double p = L.o[a] + L.t * L.d[a];
    const double f = (p - S.lower[a]) * S.inv_bs[a];
    /* clamped whole numbers: the conversion's truncation is their floor */
    const uint32_t cl = (uint32_t)fmin(fmax(f, (double)lo), (double)(hi - 1));
    c[a] = across ? (fwd ? hi : lo - 1) : cl;
    out = out || out_a;
    oa = out_a ? a : oa;
  }
  if(out) {
    if(!GEN || !S.repeat || oa == 2 || ++L.ntiles > kMaxTiles) { L.cstate = 2; return; }
    /* into the next copy of the grid */
#pragma unroll
    for(int a = 0; a < 2; ++a)
      if(a == oa) {
        L.k[a] += L.d[a] > 0 ? 1 : -1;
        L.shift[a] = (double)L.k[a] * S.period[a];
        L.o[a] = L.ow[a] - L.shift[a];
        c[a] = L.d[a] > 0 ? 0u : S.dims0[a] - 1;
      }
  }
  const uint32_t word = S.lmap[((size_t)c[2] * S.dims0[1] + c[1]) * S.dims0[0] + c[0]];
  const uint32_t lvl = word >> kLeafIdBits;
  const float2 b = S.bounds[word & kLeafIdMask];
  L.lmn = b.x;
  L.lmx = b.y;
  double best = INFINITY;
  int ax = 0;
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    L.lo[a] = (c[a] >> lvl) << lvl;
    L.hi[a] = min(L.lo[a] + (1u << lvl), S.dims0[a]);
    const double plane = S.lower[a] + (double)(L.d[a] > 0 ? L.hi[a] : L.lo[a]) * S.bs[a];
    const double ta0 = (plane - L.o[a]) * L.inv[a];
    const double ta = L.d[a] != 0 ? ta0 : INFINITY;
    const bool better = ta < best;
    best = better ? ta : best;
    ax = better ? a : ax;
  }
  L.tnext = best;
  L.exit_axis = ax;
  L.cstate = 1;
  if(COUNT) L.n_leaf++;
}

template<bool GEN, bool COUNT, bool kLW>
__device__ __forceinline__ int iter_next(const DevScene& S, Lane& L, double* t0, double* kmax)
{
  {
    /* past the boundary of the last pass */
    const bool end = L.s_t1 >= L.tmax;
    const bool move = L.adv && !end;
    L.done = L.done || (L.adv && end);
    L.t = move ? L.s_t1 : L.t;
    const int32_t dj = L.d[2] > 0 ? 1 : -1;
    L.j += move && L.adv_g ? dj : 0;
    L.cstate += move && L.adv_c && L.cstate < 2 ? 3 : 0;
    L.adv = false;
  }
  if(L.done || !(L.t < L.tmax)) return ITER_END;
  const bool in_gas = L.j >= 0 && L.j < (int32_t)S.nlayers;
  double ga = 0.0, gs = 0.0;
  if(in_gas) {
    ga = S.gas_ka[(size_t)L.kquad * S.nlayers + (uint32_t)L.j];
    gs = S.gas_ks[(size_t)L.iband * S.nlayers + (uint32_t)L.j];
  }
  if(L.cstate >= 3) next_leaf<GEN, COUNT>(S, L);
  const double t = L.t;
  const double tc = L.cstate == 0 ? L.tnext : L.cstate == 1 ? fmax(L.tnext, t) : INFINITY;
  double tg = INFINITY;
  if(L.d[2] > 0 && L.j < (int32_t)S.nlayers) tg = (S.zb + (double)(L.j + 1) * S.dzl - L.o[2]) * L.inv[2];
  else if(L.d[2] < 0 && L.j >= 0) tg = (S.zb + (double)L.j * S.dzl - L.o[2]) * L.inv[2];
  tg = fmax(tg, t);
  const double t1 = fmin(fmin(tc, tg), L.tmax);
  const bool in_cloud = L.cstate == 1;
  L.s_t1 = t1;
  L.adv = true;
  L.adv_g = tg == t1;
  L.adv_c = tc == t1;
  if(!(t1 > t && (in_gas || in_cloud))) {
    /* both boundaries at infinity: the end, t1 being the range's */
    return ITER_AGAIN;
  }
  const double g = !in_gas ? 0.0 : kLW ? ga + gs : L.prop == HTGX_Ka ? ga : L.prop == HTGX_Ks ? gs : ga + gs;
  *t0 = t;
  L.s_kmin = in_cloud ? g + L.c * (double)L.lmn : g;
  *kmax = in_cloud ? g + L.c * (double)L.lmx : g;
  L.g = kLW ? ga : g;
  if(kLW) L.gs = gs;
  L.s_cloud = in_cloud;
  L.s_layer = in_gas ? L.j : -1;
  if(COUNT) L.n_seg++;
  return ITER_SEGMENT;
}

/* LWC of the cell holding x (world), clamped into the segment's leaf (seg_lwc) */
template<bool GEN, bool COUNT>
__device__ __forceinline__ float cell_lwc(const DevScene& S, Lane& L, const double x[3])
{
  uint32_t ci[3];
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    const double xa = GEN && a < 2 ? x[a] - L.shift[a] : x[a];
    const double f = (xa - S.lower[a]) * S.inv_cs[a];
    ci[a] = (uint32_t)fmin(fmax(f, (double)(L.lo[a] * S.B)), (double)(L.hi[a] * S.B - 1));
  }
  if(COUNT) L.n_cell++;
  return S.lwc[((size_t)ci[2] * S.def[1] + ci[1]) * S.def[0] + ci[0]];
}

/*******************************************************************************
 * Walk logic: the stages of htgx_device.h on the lane's state. Stage functions
 * only request the next query; it is set up once at the end of the event step.
 ******************************************************************************/
__device__ __forceinline__ void request(Lane& L, int mode, int prop, bool ground, double r1)
{
  L.mode = mode;
  L.prop = prop;
  L.tmax = r1;
  L.nq = true;
  L.nq_ground = ground;
}

__device__ __forceinline__ void request_scatter(Lane& L)
{
  LC(stage) = ST_SCATTER;
  request(L, MODE_SC, HTGX_Ks, true, 0.0);
}

template<bool GEN>
__device__ __forceinline__ void sw_begin(const DevScene& S, Lane& L, int mask, const double pos[3],
                                         const double dir[3])
{
  LC(mask) = (uint32_t)mask;
#pragma unroll
  for(int a = 0; a < 3; ++a) { L.o[a] = pos[a]; L.d[a] = dir[a]; }
  LC(ksi) = 1;
  LC(w) = 0;
  LC(prev_prim) = -1;
  L.prev_edge = false;
  if((mask & HTGX_RADIANCE_DIRECT) && in_solar_cone(S, L.d)) {
    const GroundHit h = trace<GEN>(S, L.o, L.d, FLT_MAX, -1, false, true);
    if(!h.hit) {
      LC(stage) = ST_DIRECT;
      request(L, MODE_TR, HTGX_Kext, false, (double)FLT_MAX);
      return;
    }
  }
  if(mask & HTGX_RADIANCE_DIFFUSE) request_scatter(L);
  else LC(stage) = ST_WALK_DONE;
}

/* Next-event estimate and Russian roulette (the draw `rr' of a surface event)
 * closing a SW event, ..._sw.c:494-504; the lane's origin is the event. False
 * if the walk ends. */
__device__ __forceinline__ bool sw_accumulate(const DevScene& S, Lane& L, double rr, double Tr)
{
  const double sun_pdf = L.specular ? 1.0 : 1.0 / S.sun_solid_angle;
  LC(w) += LC(ksi) * LC(L_sun) * Tr * LC(R) / sun_pdf;
  if(L.surface && rr >= LC(refl)) { LC(stage) = ST_WALK_DONE; return false; }
#pragma unroll
  for(int a = 0; a < 3; ++a) L.d[a] = LCA(dir_next, a);
  request_scatter(L);
  return true;
}

/* Draws the event of a lane takes at most, the optical thickness of the next
 * query included */
template<bool GEN, bool kLW>
__device__ __forceinline__ int event_draws(const DevScene& S, const DevMap& M, const Lane& L, int stage)
{
  if(stage == ST_BEGIN) return M.sensor == HTGX_SENSOR_RECTANGLE && !kLW ? 10 : 8;
  if(!L.pending) return 1;
  const int brdf = GEN && S.gmat ? 1 : 0;
  if(kLW) return L.ev == EV_SCA ? 3 : L.ev == EV_NONE && L.gh_hit ? 4 + brdf : 0;
  if(stage == ST_ABS) return L.surface ? 6 + brdf : 6;
  if(stage == ST_SUN) return L.surface ? 2 : 1;
  return 1;
}

template<bool GEN, bool kLW, bool COUNT>
__device__ __forceinline__ void consume(const DevScene& S, Lane& L, Draws& u)
{
  const int stage = (int)LC(stage);
  if(kLW) {
    if(stage != ST_LW) return;
    u.n = 0;
    if(!L.gh_hit && L.ev == EV_NONE) { LC(w) = 0; LC(stage) = ST_WALK_DONE; return; }
    if(COUNT) L.n_ev++;
    if(L.ev == EV_ABS) {
      LC(w) = planck_mono(LC(wlen) * 1e-9, layer_temperature(S, L.s_layer));
      LC(stage) = ST_WALK_DONE;
      return;
    }
    const double dst = L.ev != EV_NONE ? L.tc : L.tmax;
    double pn[3], dn[3];
#pragma unroll
    for(int a = 0; a < 3; ++a) pn[a] = (GEN && a < 2 ? L.ow[a] : L.o[a]) + L.d[a] * dst;
    if(L.ev == EV_SCA) {
      local_to_world(L.d, hg_cos_sample(LC(g), u.at(0)), 2.0 * kPi * u.at(1), dn);
      u.end(2);
      LC(prev_prim) = -1; /* ..._lw.c:236 */
      L.prev_edge = false;
    } else {
      double N[3], refl, T;
      bool specular = false;
      const uint32_t mtl = ground_surface<GEN>(S, LC(gh_prim), N);
      if(GEN && S.gmat) { /* ..._lw.c:249-252 */
        const int32_t m = interface_mtl(S.ifcs[mtl], S.mtls, dot3(N, L.d) > 0);
        const DevBrdf& b = brdf_fetch(S.mtls[m], S.brdfs, LC(wlen), u.at(0));
        refl = b.refl;
        specular = b.type == HTGX_BRDF_SPECULAR;
        T = S.mtls[m].T;
      } else {
        refl = S.mtl_albedo[mtl];
        T = S.mtl_T ? S.mtl_T[mtl] : 0.0;
      }
      if(-(L.d[0]*N[0] + L.d[1]*N[1] + L.d[2]*N[2]) < 0) {
        N[0] = -N[0]; N[1] = -N[1]; N[2] = -N[2];
      }
      /* the draws of the hemisphere and of the roulette follow the BRDF's */
      const bool brdf = GEN && S.gmat;
      if(specular) reflect3(L.d, N, dn);
      else cos_hemisphere(N, brdf ? u.at(1) : u.at(0), brdf ? u.at(2) : u.at(1), dn);
      double rr;
      if(specular) { rr = u.at(1); u.end(2); }
      else if(brdf) { rr = u.at(3); u.end(4); }
      else { rr = u.at(2); u.end(3); }
      if(rr >= refl) {
        LC(w) = T > 0 ? planck_mono(LC(wlen) * 1e-9, T) : 0;
        LC(stage) = ST_WALK_DONE;
        return;
      }
      LC(prev_prim) = LC(gh_prim); /* ..._lw.c:272 */
      L.prev_edge = L.gh_edge;
    }
#pragma unroll
    for(int a = 0; a < 3; ++a) { L.o[a] = pn[a]; L.d[a] = dn[a]; }
    request(L, MODE_LW, HTGX_Kext, true, 0.0);
    return;
  }

  u.end(0);
  if(GEN) { /* back from the copy of the grid the query ended in */
    L.o[0] = L.ow[0];
    L.o[1] = L.ow[1];
  }
  const double Tr = L.ev == EV_HIT ? 0.0 : (L.Tmin != 0 ? exp(-L.Tmin) : 1.0);
  switch(stage) {
    case ST_DIRECT:
      LC(w) = LC(L_sun) * Tr;
      if(LC(mask) & HTGX_RADIANCE_DIFFUSE) request_scatter(L);
      else LC(stage) = ST_WALK_DONE;
      break;

    case ST_SCATTER: {
      const bool hit = L.ev == EV_HIT;
      if(!L.gh_hit && !hit) { LC(stage) = ST_WALK_DONE; break; }
      if(COUNT) L.n_ev++;
      L.surface = !hit;
      const double dst = L.surface ? L.tmax : L.tc;
      /* ..._sw.c:392: the next traces leave this surface hit, if any */
      LC(prev_prim) = L.surface ? LC(gh_prim) : -1;
      L.prev_edge = L.surface && L.gh_edge;
      LC(stage) = ST_ABS;
      request(L, MODE_TR, HTGX_Ka, false, dst);
    } break;

    case ST_ABS: {
      if(Tr <= 0) { LC(stage) = ST_WALK_DONE; break; }
      LC(ksi) *= Tr;
      L.specular = false;
      double pn[3], dn[3], sun[3], R, N[3] = {0, 0, 1};
#pragma unroll
      for(int a = 0; a < 3; ++a) pn[a] = L.o[a] + L.d[a] * L.tmax;
      /* draws: a surface's BRDF or a volume's phase choice, directions, sun */
      double albedo = 1;
      const bool one = !L.surface || (GEN && S.gmat);
      if(L.surface) {
        const uint32_t mtl = ground_surface<GEN>(S, LC(gh_prim), N);
        if(GEN && S.gmat) {
          /* the hit side's material and its BRDF at the wavelength,
           * ..._sw.c:403-411 */
          const int32_t m = interface_mtl(S.ifcs[mtl], S.mtls, dot3(N, L.d) > 0);
          const DevBrdf& b = brdf_fetch(S.mtls[m], S.brdfs, LC(wlen), u.at(0));
          albedo = b.refl;
          L.specular = b.type == HTGX_BRDF_SPECULAR;
        } else {
          albedo = S.mtl_albedo[mtl];
        }
        if(-(L.d[0]*N[0] + L.d[1]*N[1] + L.d[2]*N[2]) < 0) {
          N[0] = -N[0]; N[1] = -N[1]; N[2] = -N[2];
        }
      } else {
        L.rayleigh = u.at(0) < LC(gas_ratio);
      }
      if(GEN && L.specular) {
        reflect3(L.d, N, dn);
        /* the mirror direction is the sun direction, ..._sw.c:446-455 */
        sun[0] = dn[0]; sun[1] = dn[1]; sun[2] = dn[2];
        R = !in_solar_cone(S, sun) || dot3(N, sun) < 0 ? 0 : albedo;
      } else {
        /* surface and volume scattering share the two direction sites */
        const double u0 = one ? u.at(1) : u.at(0), u1 = one ? u.at(2) : u.at(1);
        double axis[3], mu;
#pragma unroll
        for(int a = 0; a < 3; ++a) axis[a] = L.surface ? N[a] : L.d[a];
        if(L.surface) mu = sqrt(1.0 - u0);
        else mu = L.rayleigh ? rayleigh_cos_sample(u0) : hg_cos_sample(LC(g), u0);
        local_to_world(axis, mu, 2.0 * kPi * u1, dn);
        const double s0 = one ? u.at(3) : u.at(2), s1 = one ? u.at(4) : u.at(3);
        const double sd[3] = {S.sun_dir[0], S.sun_dir[1], S.sun_dir[2]};
        local_to_world(sd, 1.0 - s0 * (1.0 - S.sun_cos_half), 2.0 * kPi * s1, sun);
        if(L.surface) {
          const double c = dot3(N, sun);
          R = c < 0 ? 0 : albedo / kPi * c;
        } else {
          const double m = dot3(L.d, sun);
          R = L.rayleigh ? rayleigh_eval(m) : hg_eval(LC(g), m);
        }
      }
      LC(refl) = albedo;
      LC(R) = R;
#pragma unroll
      for(int a = 0; a < 3; ++a) { LCA(dir_next, a) = dn[a]; L.o[a] = pn[a]; }
      bool shadowed = R <= 0;
      if(!shadowed)
        shadowed = trace<GEN>(S, pn, sun, (double)FLT_MAX, LC(prev_prim), L.prev_edge, true).hit;
      const bool spec = GEN && L.specular;
      if(spec) u.end(1);
      else if(one) u.end(5);
      else u.end(4);
      if(shadowed) {
        const double rr = canonical(u.ts);
        if(sw_accumulate(S, L, rr, 0.0) && L.surface) {
          if(spec) u.end(2);
          else if(one) u.end(6);
          else u.end(5);
        }
        break;
      }
#pragma unroll
      for(int a = 0; a < 3; ++a) L.d[a] = sun[a];
      LC(stage) = ST_SUN;
      request(L, MODE_TR, HTGX_Kext, false, (double)FLT_MAX);
    } break;

    case ST_SUN:
      if(sw_accumulate(S, L, u.at(0), Tr) && L.surface) u.end(1);
      break;

    default: break;
  }
}

/* Start a realisation: sensor ray, wavelength, band, k-point, first walk */
template<bool GEN, bool kLW>
__device__ __forceinline__ void real_begin(const DevScene& S, const DevMap& M, Lane& L, Draws& u)
{
  const uint32_t px = L.pixel % M.width, py = L.pixel / M.width;
  const double psx = 1.0 / (double)M.width, psy = 1.0 / (double)M.height;
  double org[3], dir0[3];
  const double x = ((double)px + u.at(0)) * psx;
  const double y = ((double)py + u.at(1)) * psy;
  const double l0 = u.at(2), l1 = u.at(3);
  if(M.sensor == HTGX_SENSOR_CAMERA) {
    if(GEN) {
      camera_ray(M, x, y, l0, l1, org, dir0);
    } else {
      /* camera_ray's pinhole */
      const double sx = 2.0 * x - 1.0, sy = 1.0 - 2.0 * y;
#pragma unroll
      for(int a = 0; a < 3; ++a) {
        dir0[a] = M.z[a] + M.x[a] * (sx * M.tan_half * M.aspect) + M.y[a] * (sy * M.tan_half);
        org[a] = M.pos[a];
      }
      normalize3(dir0);
    }
  } else {
    /* sample_rectangle_ray, ..._draw_map.c:52-107 */
#pragma unroll
    for(int a = 0; a < 3; ++a)
      org[a] = M.pos[a] + M.axis_x[a] * (x * 2.0 - 1.0) + M.axis_y[a] * (y * 2.0 - 1.0);
    const double up[3] = {0, 0, 1};
    const GroundHit h = trace<GEN>(S, org, up, DBL_MAX, -1, false, false);
    const bool under = GEN ? sensor_under_ground(S, h) : h.N[2] >= 0;
    if(h.hit && under) {
      LC(nfail)++;
      LC(phase) = 3; /* rejected */
      LC(stage) = ST_REAL_DONE;
      return;
    }
    const double z[3] = {M.z[0], M.z[1], M.z[2]};
    cos_hemisphere(z, l0, l1, dir0);
  }
  const double r0 = u.at(4), r1 = u.at(5), r2 = u.at(6);
  u.end(7);
  double pdf;
  const double wlen = sample_wavelength<GEN, GEN>(M, r0, r1, &pdf, GEN ? LC(plane) : 0u);
  pdf *= 1e9;
  LC(pdf) = pdf;
  LC(wlen) = wlen;
  L.iband = find_band(S, wlen);
  L.kquad = S.quad_off[L.iband] + sample_quad(S, L.iband, r2);
  LC(g) = S.has_clouds ? S.hg_g[L.iband] : 0.0;
  LC(L_sun) = planck_mono(wlen * 1e-9, 5778.0);
  if(kLW) {
    LC(phase) = 0;
#pragma unroll
    for(int a = 0; a < 3; ++a) { L.o[a] = org[a]; L.d[a] = dir0[a]; }
    LC(w) = 0;
    LC(prev_prim) = -1;
    L.prev_edge = false;
    LC(stage) = ST_LW;
    request(L, MODE_LW, HTGX_Kext, true, 0.0);
    return;
  }
  int mask = HTGX_RADIANCE_ALL;
  double dir[3] = {dir0[0], dir0[1], dir0[2]};
  LC(phase) = 0;
  if(M.sensor != HTGX_SENSOR_CAMERA) {
    const double s0 = u.at(7), s1 = u.at(8);
    u.end(9);
    const double sd[3] = {S.sun_dir[0], S.sun_dir[1], S.sun_dir[2]};
    double sun[3];
    local_to_world(sd, 1.0 - s0 * (1.0 - S.sun_cos_half), 2.0 * kPi * s1, sun);
    const double cosN = M.z[0]*sun[0] + M.z[1]*sun[1] + M.z[2]*sun[2];
    LC(cosN) = cosN;
    LC(Ld) = 0;
    const bool direct = cosN > 0;
    LC(phase) = direct ? 1 : 2;
    mask = direct ? HTGX_RADIANCE_DIRECT : HTGX_RADIANCE_DIFFUSE;
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      LCA(org, a) = org[a];
      LCA(dir0, a) = dir0[a];
      dir[a] = direct ? sun[a] : dir0[a];
    }
  }
  sw_begin<GEN>(S, L, mask, org, dir);
}

/* A walk ended: weight of the realisation or start of the next walk */
template<bool GEN, bool kLW>
__device__ __forceinline__ void walk_done(const DevScene& S, const DevMap& M, Lane& L)
{
  LC(stage) = ST_REAL_DONE;
  if(M.sensor == HTGX_SENSOR_CAMERA) {
    LC(w) = LC(w) / LC(pdf);
  } else if(kLW) {
    LC(w) = LC(w) * kPi / LC(pdf);
  } else if(LC(phase) == 1) {
    LC(Ld) = LC(w);
    LC(phase) = 2;
    double o[3], d[3];
#pragma unroll
    for(int a = 0; a < 3; ++a) { o[a] = LCA(org, a); d[a] = LCA(dir0, a); }
    sw_begin<GEN>(S, L, HTGX_RADIANCE_DIFFUSE, o, d);
  } else {
    LC(w) = (LC(cosN) * S.sun_solid_angle * LC(Ld) + kPi * LC(w)) / LC(pdf);
  }
}

/* The event step runs once this many of a full wavefront's lanes wait for it
 * (fewer in proportion when lanes are out of work) and no other step has more;
 * the segment step once no fewer wait for it than for the collision step.
 * 256x256x16 image 118 -> 113 ms against fixed thresholds of 24 and 16. */
constexpr uint32_t kEventLanes = 24;

template<bool GEN, bool kLW, bool COUNT>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
plain_kernel(KArgs A)
{
  (void)A;
  const KPtr<KArgs> pK = (KPtr<KArgs>)__builtin_amdgcn_kernarg_segment_ptr();
  const DevScene S = kload(&pK->S);
  const uint64_t seed = kload(&pK->M.seed);
  const uint32_t spp_offset = kload(&pK->M.spp_offset), lanes = kload(&pK->P.lanes);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  copy_to_lds(pK, &g_args[wave]);
  Lane L;
  L.lstate = (threadIdx.x & 63u) < lanes ? LS_EVENT : LS_DONE;
  LC(stage) = ST_FETCH;
  L.pending = L.nq = false;
  L.pixel = L.r = L.draw = L.channel = 0;
  if(COUNT) L.n_leaf = L.n_seg = L.n_coll = L.n_cell = L.n_ev = 0;
  const uint32_t xcd = blockIdx.x % (uint32_t)kXcds;
  uint32_t tried = 0;

  for(;;) {
    const uint64_t want0 = __ballot(L.lstate == LS_EVENT);
    const uint64_t bs = __ballot(L.lstate == LS_SEG), bc = __ballot(L.lstate == LS_COLL);
    if(!(want0 | bs | bc)) break;
    const uint32_t alive = (uint32_t)__popcll(want0 | bs | bc);

    /* next segment of the query, and the first tentative collision in it */
    const uint32_t ne = (uint32_t)__popcll(want0), ns = (uint32_t)__popcll(bs), nc = (uint32_t)__popcll(bc);
    const bool run_seg = bs && (!bc || ns >= nc);
    const bool run_ev = !(bs | bc) || (ne >= (kEventLanes * alive >> 6) && ne >= ns && ne >= nc);
    if(run_seg && L.lstate == LS_SEG) {
      double t0, kmax;
      const int it = iter_next<GEN, COUNT, kLW>(S, L, &t0, &kmax);
      if(it == ITER_SEGMENT) {
        const double maj = !kLW && L.mode == MODE_TR ? kmax - L.s_kmin : kmax;
        if(!kLW && L.mode == MODE_TR) L.Tmin += (L.s_t1 - t0) * L.s_kmin;
        const double T = (L.s_t1 - t0) * maj;
        if(L.Ts > T || !(maj > 0)) {
          L.Ts -= T;
        } else {
          L.maj = maj;
          L.tc = t0 + L.Ts / maj;
          /* ..._sw.c:123: a scattering candidate beyond 1e9 m is dropped */
          if(kLW || L.mode != MODE_SC || !(L.tc > 1e9)) L.lstate = LS_COLL;
        }
      } else if(it == ITER_END) {
        L.ev = EV_NONE;
        L.pending = true;
        L.lstate = LS_EVENT;
      }
    }

    /* one tentative collision */
    if(L.lstate == LS_COLL) {
      double x[3];
#pragma unroll
      for(int a = 0; a < 3; ++a) x[a] = (GEN && a < 2 ? L.ow[a] : L.o[a]) + L.tc * L.d[a];
      if(COUNT) L.n_coll++;
      const float v = L.s_cloud ? cell_lwc<GEN, COUNT>(S, L, x) : 0.f;
      /* its two draws, the second unused if the collision is real: at most
       * one new block, whichever the phase of the stream */
      const uint32_t ph = L.draw & 3u;
      uint64_t w0 = ph == 1 ? L.buf[1] : ph == 2 ? L.buf[2] : L.buf[3];
      if(ph == 0 || ph == 3) {
        stream_block(L, seed, spp_offset, (L.draw >> 2) + (ph == 3 ? 1u : 0u), L.buf);
        w0 = ph == 0 ? L.buf[0] : w0;
      }
      const uint64_t w1 = ph == 0 ? L.buf[1] : ph == 1 ? L.buf[2] : ph == 2 ? L.buf[3] : L.buf[0];
      const double r = canonical(w0);
      int ev = EV_NONE;
      if(kLW) {
        const double ka = L.g + (L.s_cloud ? L.ca * (double)v : 0.0);
        const double ks = L.gs + (L.s_cloud ? L.cs * (double)v : 0.0);
        const double pa = ka / L.maj, ps = ks / L.maj;
        ev = r < pa ? EV_ABS : r < pa + ps ? EV_SCA : EV_NONE;
      } else {
        const double c = L.s_cloud ? L.c * (double)v : 0.0;
        const double k = L.g + c;
        const double proba = L.mode == MODE_TR ? (k - L.s_kmin) / L.maj : k / L.maj;
        if(r < proba) {
          ev = EV_HIT;
          /* gas vs particle scattering at the event, ..._sw.c:427-438 */
          if(L.mode == MODE_SC) LC(gas_ratio) = L.g / (c + L.g);
        }
      }
      if(ev != EV_NONE) {
        L.draw += 1;
        L.ev = ev;
        L.pending = true;
        L.lstate = LS_EVENT;
      } else {
        L.draw += 2;
        L.Ts = -log(1.0 - canonical(w1));
        const double T = (L.s_t1 - L.tc) * L.maj;
        if(L.Ts > T) {
          L.Ts -= T;
          L.lstate = LS_SEG;
        } else {
          L.tc += L.Ts / L.maj;
          if(!kLW && L.mode == MODE_SC && L.tc > 1e9) L.lstate = LS_SEG;
        }
      }
    }

    /* events, when enough lanes need them or nothing else is left */
    if(run_ev && __ballot(L.lstate == LS_EVENT)) {
      uint32_t wv = wave;
      asm volatile("" : "+s"(wv));
      const DevScene& SE = g_args[wv].S;
      const DevMap& M = g_args[wv].M;
      const Launch& P = g_args[wv].P;
      const bool fetch = L.lstate == LS_EVENT && LC(stage) == ST_FETCH;
      if(__ballot(fetch)) {
        uint32_t c = 0;
        const bool got = fetch_chunks(P, xcd, &tried, fetch, &c);
        if(fetch && !got) {
          L.lstate = LS_DONE;
        } else if(fetch) {
          uint32_t pixel, sub, plane;
          if(chunk_pixel(P, c, &pixel, &sub, &plane)) {
            LC(chunk) = c;
            if(GEN) {
              LC(plane) = plane;
              L.channel = P.planes > 1 ? plane + 1u : 0u;
            }
            L.pixel = pixel;
            L.r = sub * P.K;
            LC(r_end) = min(L.r + P.K, M.spp);
            LC(n) = LC(nfail) = 0;
            LC(sum) = LC(sum_c) = LC(sum2) = LC(sum2_c) = LC(tsum) = LC(tsum2) = 0.0;
            LC(stage) = ST_BEGIN;
          } /* else: outside the image, fetch again next time */
        }
      }
      if(L.lstate == LS_EVENT && LC(stage) != ST_FETCH) {
        const int stage = (int)LC(stage);
        const bool begin = stage == ST_BEGIN;
        if(begin) {
          L.draw = 0;
          LC(t0) = (uint32_t)wall_clock64();
        }
        /* the blocks of the event's draws: the one the stream is in, if the
         * lane has it, and those that follow as far as the event goes */
        Draws u;
        uint64_t W[12];
        const uint32_t ph = L.draw & 3u, b0 = L.draw >> 2;
        const int need = (int)ph + event_draws<GEN, kLW>(SE, M, L, stage);
        if(ph == 0 && need > 0) stream_block(L, seed, spp_offset, b0, L.buf);
#pragma unroll
        for(int i = 0; i < 4; ++i) { W[i] = L.buf[i]; W[4 + i] = W[8 + i] = 0; }
        if(need > 4) stream_block(L, seed, spp_offset, b0 + 1u, W + 4);
        if(need > 8) stream_block(L, seed, spp_offset, b0 + 2u, W + 8);
#pragma unroll
        for(int i = 0; i < kMaxDraws; ++i) {
          /* (a begin, the only event of more than 7 draws, has phase 0) */
          u.w[i] = i > 6 ? W[i] : ph == 0 ? W[i] : ph == 1 ? W[i + 1] : ph == 2 ? W[i + 2] : W[i + 3];
        }
        u.end(0);
        if(begin) {
          real_begin<GEN, kLW>(SE, M, L, u);
        } else if(L.pending) {
          L.pending = false;
          consume<GEN, kLW, COUNT>(SE, L, u);
        }
        while(LC(stage) == ST_WALK_DONE) walk_done<GEN, kLW>(SE, M, L);
        if(LC(stage) == ST_REAL_DONE) {
          const uint64_t t1 = wall_clock64();
          if(LC(phase) != 3) {
            const double us = (double)((uint32_t)t1 - LC(t0)) * M.us_per_tick, w = LC(w);
            double s = LC(sum), sc = LC(sum_c), s2 = LC(sum2), s2c = LC(sum2_c);
            neumaier(s, sc, w);
            neumaier(s2, s2c, w * w);
            LC(sum) = s; LC(sum_c) = sc; LC(sum2) = s2; LC(sum2_c) = s2c;
            LC(tsum) += us;
            LC(tsum2) += us * us;
            LC(n)++;
          }
          L.r++;
          if(L.r != LC(r_end)) {
            LC(stage) = ST_BEGIN;
          } else {
            htgx_mc_accum a;
            a.sum = LC(sum); a.sum_c = LC(sum_c); a.sum2 = LC(sum2); a.sum2_c = LC(sum2_c);
            a.tsum = LC(tsum); a.tsum2 = LC(tsum2); a.n = LC(n); a.nfail = LC(nfail);
            P.partials[LC(chunk)] = a;
            LC(stage) = ST_FETCH;
          }
        }
        /* set-up of the requested query (single site) */
        if(L.nq) {
          L.nq = false;
          if(L.nq_ground) {
            const GroundHit gh = trace<GEN>(SE, L.o, L.d, DBL_MAX, LC(prev_prim), L.prev_edge, false);
            L.gh_hit = gh.hit;
            L.gh_edge = gh.edge;
            LC(gh_prim) = gh.prim;
            L.tmax = gh.t;
          }
          L.Ts = -log(1.0 - canonical(u.ts));
          ++u.n;
          L.Tmin = 0.0;
          L.c = L.ca = L.cs = 0.0;
          if(S.has_clouds) {
            const double ce = SE.cext[L.iband], w = SE.ssa[L.iband];
            const double ca = ce * (1.0 - w), cs = ce * w;
            if(kLW) { L.c = ce; L.ca = ca; L.cs = cs; }
            else L.c = L.prop == HTGX_Ka ? ca : L.prop == HTGX_Ks ? cs : ce;
          }
          iter_init<GEN>(S, L);
          L.lstate = LS_SEG;
        }
        /* the block the stream is in now */
        const uint32_t db = (ph + u.n) >> 2;
#pragma unroll
        for(int i = 0; i < 4; ++i) L.buf[i] = db == 0 ? W[i] : db == 1 ? W[4 + i] : W[8 + i];
        L.draw += u.n;
      }
    }
  }

  if(COUNT) {
    const uint64_t a = wave_sum64(L.n_leaf), b = wave_sum64(L.n_seg), c = wave_sum64(L.n_coll),
                   d = wave_sum64(L.n_cell), e = wave_sum64(L.n_ev);
    if((threadIdx.x & 63u) == 0) {
      unsigned long long* stats = g_args[wave].P.stats;
      atomicAdd(stats + 1, (unsigned long long)a);
      atomicAdd(stats + 2, (unsigned long long)b);
      atomicAdd(stats + 3, (unsigned long long)c);
      atomicAdd(stats + 4, (unsigned long long)d);
      atomicAdd(stats + 5, (unsigned long long)e);
    }
  }
}

template<bool GEN, bool COUNT>
int launch(const KArgs& A, uint32_t grid, hipStream_t stream)
{
  if(A.M.spectral_type == HTGX_SPECTRAL_LW) plain_kernel<GEN, true, COUNT><<<grid, kBlock, 0, stream>>>(A);
  else plain_kernel<GEN, false, COUNT><<<grid, kBlock, 0, stream>>>(A);
  HIP_OK(hipGetLastError());
  return HTGX_OK;
}

} /* namespace */

int htgx_render_plain(htgx_ctx* ctx, const DevMap& M, uint32_t planes, htgx_mc_accum* accum,
                      hipStream_t stream)
{
  int res;
  if(!ctx->plain_grid) {
    int ncu = 0, per_cu = 0;
    HIP_OK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));
    HIP_OK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, plain_kernel<false, false, false>, kBlock, 0));
    HIP_OK(hipMalloc(&ctx->d_plain_queue, kXcds * sizeof(unsigned int)));
    ctx->plain_grid = (uint32_t)std::max(1, ncu * std::max(1, per_cu));
  }
  KArgs A;
  std::memset(&A.P, 0, sizeof(A.P));
  A.S = ctx->S;
  A.M = M;
  Launch& P = A.P;
  const uint64_t npix = (uint64_t)M.width * M.height * planes;
  set_queue_size(P, M.width, M.height, planes);
  /* chunks as large as leaves 4 to each resident lane. A lane runs its chunk's
   * realisations one after the other, so a large map ends with that many walks
   * in a row: limits of 8, 4 and 2 realisations take 666, 648 and 637 ms for the
   * 721 of 1024x1024 x 16, and 671, 646 and 641 for the 825 of 512x512 x 64 */
  const uint64_t items = (uint64_t)P.ntiles * 64u, lanes = (uint64_t)ctx->plain_grid * kBlock;
  P.K = (uint32_t)std::min<uint64_t>(M.spp, std::max<uint64_t>(1, items * M.spp / (4 * lanes)));
  P.nsub = (M.spp + P.K - 1) / P.K;
  const uint64_t nchunks = items * P.nsub;
  if(planes > 1 && nchunks * sizeof(htgx_mc_accum) > kMaxPlanePartials)
    return htgx_render_channels(ctx, M, planes, accum, stream, htgx_render_plain);
  if(nchunks > 0xFFFFFFFFull) return HTGX_BAD_ARG;
  /* fewer chunks than lanes: spread over all the wavefronts */
  const uint64_t nw = kBlock / 64;
  const uint32_t grid = (uint32_t)std::min<uint64_t>(ctx->plain_grid, (nchunks + nw - 1) / nw);
  P.lanes = (uint32_t)std::min<uint64_t>(64, (nchunks + nw * grid - 1) / (nw * grid));

  const size_t need = nchunks * sizeof(htgx_mc_accum);
  if(need > ctx->partials_cap) {
    if(ctx->d_partials) { HIP_OK(hipFree(ctx->d_partials)); ctx->d_partials = nullptr; ctx->partials_cap = 0; }
    HIP_OK(hipMalloc(&ctx->d_partials, need));
    ctx->partials_cap = need;
  }
  P.counters = ctx->d_plain_queue;
  P.partials = (htgx_mc_accum*)ctx->d_partials;
  P.stats = ctx->d_counters;
  zero_u32_kernel<<<1, 64, 0, stream>>>(P.counters, kXcds);
  HIP_OK(hipGetLastError());
  /* the lean kernels' conditions (trace, real_begin, iter_next) */
  const bool gen = A.S.repeat || A.S.ground_type == HTGX_GROUND_MESH || A.S.gmat || A.S.explicit_ifc ||
                   M.ortho || M.lens_radius > 0 || M.wmode > 1;
  if(ctx->counting) {
    zero_u64_kernel<<<1, 64, 0, stream>>>(ctx->d_counters, HTGX_NSTATS);
    HIP_OK(hipGetLastError());
    res = launch<true, true>(A, grid, stream);
  } else {
    res = gen ? launch<true, false>(A, grid, stream) : launch<false, false>(A, grid, stream);
  }
  if(res != HTGX_OK) return res;
  merge_chunks_kernel<<<(uint32_t)((npix + 255) / 256), 256, 0, stream>>>(P, accum);
  HIP_OK(hipGetLastError());
  ctx->last_nrealisations = npix * M.spp;
  return HTGX_OK;
}
