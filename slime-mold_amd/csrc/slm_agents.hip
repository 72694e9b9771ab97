// slm_agents.hip - the agent update (reference src/compute.wgsl:57-145) and the
// device-side agent initialisation / speed reassignment / resize scaling that
// replace the reference's host loops (src/main.rs:101-145, :262-282, :955-997).
//
// One lane per agent over structure-of-arrays state, launched over a pool of
// instances (a single simulation is a pool of one): each block walks the
// instances its 256 slots overlap, usually one, so instance geometry and
// parameters are block-uniform scalar loads.
//
// Sensing reads the trail as it was when the step began: a deposit does not
// write a value, it sets the sign bit of the target cell (trail values are
// never negative, so the bit is free); sensing reads |T|, and the trail pass
// that follows turns marked cells into clamp(|T| + deposit, 0, 1).  The mark is
// a plain load and store of that one cell, not an atomic: every agent landing
// in a cell stores the same bits (-|T|), and a sensor reading the cell
// meanwhile sees T or -T, whose |.| is the same, so the race is benign.  The
// result is therefore independent of the order agents run in.  (A global
// atomic OR per agent cost ~0.45 ms per 2^24 agents and serialised badly once
// agents are spatially sorted.)
//
// Arithmetic follows the reference shader operation by operation: this file is
// compiled with -ffp-contract=off, division is IEEE, '%' is a - b*trunc(a/b),
// and sin/cos come from slm_trig.h.  The f64-position variant keeps x and y in
// double: sensor offsets and the move step are still the shader's f32 products,
// added to the f64 position; the wrap, floor and deposit cell are taken in
// double; the bilinear weights and the jitter hash use the f32 roundings.
#include <type_traits>

#include "slm_internal.h"
#include "slm_trig.h"

namespace slm {
namespace {

constexpr float kTau = 6.28318530718f;  // compute.wgsl:4 and :121 (0x40c90fdb)
constexpr float kTimeStep = 0.016f;     // compute.wgsl:55

// ---- trail access by storage format -------------------------------------
// load_pair(t, i) returns |T[i]| and |T[i+1]| from one (4- or 2-byte aligned)
// load; gfx950 allows unaligned global loads, and the compiler only fuses the
// two cells into one instruction where the target permits it.
template <int S>
struct TrailRead;

template <>
struct TrailRead<SLM_STORAGE_F32> {
  using elem = uint32_t;
  static constexpr uint32_t kSign = 0x80000000u;
  __device__ static float value(uint32_t raw) { return __uint_as_float(raw); }
  __device__ static void load_pair(const void* t, uint32_t i, float& a, float& b) {
    uint2 v;
    __builtin_memcpy(&v, static_cast<const uint32_t*>(t) + i, sizeof v);
    a = __uint_as_float(v.x & 0x7fffffffu);
    b = __uint_as_float(v.y & 0x7fffffffu);
  }
  __device__ static void mark(void* t, uint32_t i) {
    uint32_t* p = static_cast<uint32_t*>(t) + i;
    const uint32_t v = *p;
    if (!(v >> 31)) *p = v | 0x80000000u;
  }
};

__device__ inline uint32_t load_u16_pair(const void* t, uint32_t i) {
  uint32_t w;
  __builtin_memcpy(&w, static_cast<const uint16_t*>(t) + i, sizeof w);
  return w;
}

// 16-bit cells are marked with a 2-byte store, which leaves the neighbour in
// the same 32-bit word untouched.  A cell that is marked already is not stored
// again: without a re-sort the agents of all XCDs store into all lines, and these
// stores, several to a cell where trails form, bound the pass (1365 x 767 f32, never
// re-sorted, 3 * 10^6 agents: 274 -> 167 us; re-sorted pools gain up to 2%).
__device__ inline void mark16(void* t, uint32_t i) {
  uint16_t* p = static_cast<uint16_t*>(t) + i;
  const uint32_t v = *p;
  if (!(v & 0x8000u)) *p = static_cast<uint16_t>(v | 0x8000u);
}

template <>
struct TrailRead<SLM_STORAGE_BF16> {
  using elem = uint16_t;
  static constexpr uint32_t kSign = 0x8000u;
  __device__ static float value(uint32_t raw) { return __uint_as_float(raw << 16); }
  __device__ static void load_pair(const void* t, uint32_t i, float& a, float& b) {
    uint32_t w = load_u16_pair(t, i);
    a = __uint_as_float((w & 0x7fffu) << 16);
    b = __uint_as_float(((w >> 16) & 0x7fffu) << 16);
  }
  // |T| of the two cells in a word.
  __device__ static void split(uint32_t w, float& a, float& b) {
    a = __builtin_fabsf(__uint_as_float(w << 16));
    b = __uint_as_float(w & 0x7fff0000u);
  }
  __device__ static void mark(void* t, uint32_t i) { mark16(t, i); }
};

template <>
struct TrailRead<SLM_STORAGE_F16> {
  using elem = uint16_t;
  static constexpr uint32_t kSign = 0x8000u;
  __device__ static float value(uint32_t raw) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(raw)));
  }
  __device__ static void load_pair(const void* t, uint32_t i, float& a, float& b) {
    split(load_u16_pair(t, i), a, b);
  }
  __device__ static void split(uint32_t w, float& a, float& b) {
    a = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w & 0x7fffu)));
    b = static_cast<float>(
        __builtin_bit_cast(_Float16, static_cast<uint16_t>((w >> 16) & 0x7fffu)));
  }
  __device__ static void mark(void* t, uint32_t i) { mark16(t, i); }
};

// ---- WGSL operations (S5) -------------------------------------------------
__device__ inline float wgsl_mix(float a, float b, float t) {
  float u = 1.0f - t;
  float l = a * u;
  float r = b * t;
  return l + r;
}
// WGSL '%' for b > 0.  When |a| < b, a/b truncates to +-0 and a - b*(+-0) is
// a itself (+0 for a = -0, which a + 0 gives), so the division is skipped;
// checked against the full formula for every float within 4b of 0 for 16
// moduli.
__device__ inline float wgsl_mod(float a, float b) {
  if (__builtin_fabsf(a) < b) return a + 0.0f;
  float q = a / b;
  float t = __builtin_truncf(q);
  float p = b * t;
  return a - p;
}
__device__ inline double mod64(double a, double b) {
  if (__builtin_fabs(a) < b) return a + 0.0;
  double q = a / b;
  double t = __builtin_trunc(q);
  double p = b * t;
  return a - p;
}
__device__ inline float wgsl_sign(float v) { return v > 0.0f ? 1.0f : (v < 0.0f ? -1.0f : 0.0f); }
__device__ inline float wgsl_min(float a, float b) { return a < b ? a : b; }
__device__ inline float wgsl_clamp(float e, float lo, float hi) {
  float m = e > lo ? e : lo;
  return m < hi ? m : hi;
}

// Bilinear trail sample, not toroidal (compute.wgsl:7-29), from the cell
// (x0, y0) and the weights (dx, dy).  Positions are kept finite and within
// [-2^24, 2^24] by the API, so the callers' i32 conversions are exact.
// Branch-free: an out-of-range sample loads cells 0 and 1 twice (every trail
// allocation is at least 256 bytes) and returns 0, so the six tap-pair loads
// of an agent's three sensors are all in flight at once instead of one
// sample's loads waiting behind the previous sample's branch.
template <int S>
__device__ inline float sample_at(const void* t, uint32_t w, uint32_t h, int x0, int y0, float dx,
                                  float dy) {
  bool in = x0 >= 0 && static_cast<uint32_t>(x0) < w - 1u && y0 >= 0 &&
            static_cast<uint32_t>(y0) < h - 1u;
  // grid sides are below 2^24, so the row offset is a full-rate 24-bit product
  uint32_t i00 = in ? __umul24(static_cast<uint32_t>(y0), w) + static_cast<uint32_t>(x0) : 0u;
  uint32_t down = in ? w : 0u;
  float v00, v10, v01, v11;
  TrailRead<S>::load_pair(t, i00, v00, v10);
  TrailRead<S>::load_pair(t, i00 + down, v01, v11);
  float v0 = wgsl_mix(v00, v10, dx);
  float v1 = wgsl_mix(v01, v11, dx);
  float v = wgsl_mix(v0, v1, dy);
  return in ? v : 0.0f;
}

// Taps straight from the trail in global memory.
template <int S>
struct GlobalTaps {
  void* t;
  uint32_t w, h;
  __device__ float sample(int x0, int y0, float dx, float dy) const {
    return sample_at<S>(t, w, h, x0, y0, dx, dy);
  }
  __device__ void mark(uint32_t x, uint32_t y) const { TrailRead<S>::mark(t, __umul24(y, w) + x); }
};

// Taps from a workgroup's window of the trail staged in LDS (windowed
// sensing, below): the raw elements of cells [wx0, wx0 + ww) x [wy0, wy0 + wh)
// at `pitch` cells per row (a whole number of 16-byte chunks; marks included,
// so values are read as |T|).  Taps outside it go to global memory, so the
// result does not depend on the window.
template <int S>
struct BoxTaps {
  using elem = typename TrailRead<S>::elem;
  void* t;
  uint32_t w, h;
  const uint32_t* win;  // LDS
  int wx0, wy0, ww, wh, pitch;
  // |T| of cells i and i + 1 of the window (element index i)
  __device__ void pair(int i, float& a, float& b) const {
    if constexpr (sizeof(elem) == 4) {
      a = __uint_as_float(win[i] & 0x7fffffffu);
      b = __uint_as_float(win[i + 1] & 0x7fffffffu);
    } else {
      // the two dwords around cells i, i + 1; the 32 bits starting at cell i
      const uint32_t lo = win[i >> 1], hi = win[(i >> 1) + 1];
      const uint32_t v = __builtin_amdgcn_alignbit(hi, lo, (i & 1) * 16);
      a = TrailRead<S>::value(v & 0x7fffu);
      b = TrailRead<S>::value((v >> 16) & 0x7fffu);
    }
  }
  __device__ float sample(int x0, int y0, float dx, float dy) const {
    bool in = x0 >= 0 && static_cast<uint32_t>(x0) < w - 1u && y0 >= 0 &&
              static_cast<uint32_t>(y0) < h - 1u;
    const int lx = x0 - wx0, ly = y0 - wy0;
    const bool inw = static_cast<uint32_t>(lx) < static_cast<uint32_t>(ww - 1) &&
                     static_cast<uint32_t>(ly) < static_cast<uint32_t>(wh - 1);
    float v00, v10, v01, v11;
    if (inw) {
      const int i = __mul24(ly, pitch) + lx;  // both below 2^16
      pair(i, v00, v10);
      pair(i + pitch, v01, v11);
    } else {
      // sides below 2^16 here, so the row offset is a 24-bit product
      uint32_t i00 = in ? __umul24(static_cast<uint32_t>(y0), w) + static_cast<uint32_t>(x0) : 0u;
      uint32_t down = in ? w : 0u;
      TrailRead<S>::load_pair(t, i00, v00, v10);
      TrailRead<S>::load_pair(t, i00 + down, v01, v11);
    }
    float v0 = wgsl_mix(v00, v10, dx);
    float v1 = wgsl_mix(v01, v11, dx);
    float v = wgsl_mix(v0, v1, dy);
    return in ? v : 0.0f;
  }
  // A cell inside the window: |T| (or -|T|) is known, so the mark is a store.
  __device__ void mark(uint32_t x, uint32_t y) const {
    const int lx = static_cast<int>(x) - wx0, ly = static_cast<int>(y) - wy0;
    if (static_cast<uint32_t>(lx) < static_cast<uint32_t>(ww) &&
        static_cast<uint32_t>(ly) < static_cast<uint32_t>(wh)) {
      const int i = __mul24(ly, pitch) + lx;
      uint32_t raw;
      if constexpr (sizeof(elem) == 4)
        raw = win[i];
      else
        raw = (win[i >> 1] >> ((i & 1) * 16)) & 0xffffu;
      static_cast<elem*>(t)[__umul24(y, w) + x] = static_cast<elem>(raw | TrailRead<S>::kSign);
    } else {
      TrailRead<S>::mark(t, __umul24(y, w) + x);
    }
  }
};

template <class Taps>
__device__ inline float sample(const Taps& taps, float px, float py) {
  int x0 = static_cast<int>(__builtin_floorf(px));
  int y0 = static_cast<int>(__builtin_floorf(py));
  float dx = px - static_cast<float>(x0);
  float dy = py - static_cast<float>(y0);
  return taps.sample(x0, y0, dx, dy);
}

template <class Taps>
__device__ inline float sample64(const Taps& taps, double px, double py) {
  double fx = __builtin_floor(px), fy = __builtin_floor(py);
  float dx = static_cast<float>(px - fx);
  float dy = static_cast<float>(py - fy);
  return taps.sample(static_cast<int>(fx), static_cast<int>(fy), dx, dy);
}

// compute.wgsl:98-112: turn towards the strongest of left/centre/right.
__device__ inline float turn(float angle, float lv, float rv, float cv, float turn_speed) {
  if (cv > lv && cv > rv) {
  } else if (lv > rv) {
    float target = angle - kTau;
    float diff = target - angle;
    angle += wgsl_min(turn_speed, __builtin_fabsf(diff)) * wgsl_sign(diff);
  } else if (rv > lv) {
    float target = angle + kTau;
    float diff = target - angle;
    angle += wgsl_min(turn_speed, __builtin_fabsf(diff)) * wgsl_sign(diff);
  }
  return angle;
}

// compute.wgsl:115-118 for the agent with original index `index` at (x, y).
__device__ inline float jitter_term(uint32_t index, float x, float y, float jitter) {
  float hx = static_cast<float>(static_cast<int32_t>(index)) * 12.9898f;
  hx = hx + x * 78.233f;
  hx = hx + y * 37.719f;
  float v = slm_sinf(hx) * 43758.5453f;
  float rnd = v - __builtin_floorf(v);
  return (rnd * 2.0f - 1.0f) * jitter;
}

// An agent's state as loaded at the start of its update.
template <bool P64>
struct AgentState {
  float angle, speed, x, y;
  double xd, yd;
};

template <bool P64>
__device__ inline AgentState<P64> load_agent(const AgentSoA& a, uint32_t j) {
  AgentState<P64> st;
  st.angle = a.th[j];
  st.speed = a.v[j];
  if (P64) {
    st.xd = a.x64[j];
    st.yd = a.y64[j];
    st.x = static_cast<float>(st.xd);
    st.y = static_cast<float>(st.yd);
  } else {
    st.xd = st.yd = 0.0;
    st.x = a.x[j];
    st.y = a.y[j];
  }
  return st;
}

// One agent (slot j of instance `in`, state st) for one step.
template <bool P64, class Taps>
__device__ inline void agent_update(const AgentSoA& a, uint32_t j, const AgentState<P64>& st,
                                    const Instance& in, const DevParams& p, const Taps& taps) {
  const uint32_t w = in.width, h = in.height;
  float angle = st.angle, speed = st.speed;
  float x = st.x, y = st.y;
  double xd = st.xd, yd = st.yd;

  float sp = wgsl_clamp(speed, p.speed_min, p.speed_max);  // :72
  if (sp != speed) a.v[j] = sp;
  speed = sp;

  float al = angle - p.sensor_angle, ar = angle + p.sensor_angle;  // :75-77
  float sl, cl, sr, cr, sc, cc;
  // every argument here is finite: positions, angles and parameters are
  slm_sincosf_finite(al, &sl, &cl);
  slm_sincosf_finite(ar, &sr, &cr);
  slm_sincosf_finite(angle, &sc, &cc);
  float sd = p.sensor_dist;
  float lv, rv, cv;
  // The wave senses at raised issue priority: its tap addresses and the six
  // tap-pair loads go out ahead of other waves' VALU work, so more gathers
  // are in flight on the vector memory path that bounds this kernel (C1,
  // 2^24 agents: 327 -> 296 us per pass while trails form, 237 -> 229 us
  // once formed; same bits).
  __builtin_amdgcn_s_setprio(2);
  if (P64) {
    lv = sample64(taps, xd + static_cast<double>(sd * cl), yd + static_cast<double>(sd * sl));
    rv = sample64(taps, xd + static_cast<double>(sd * cr), yd + static_cast<double>(sd * sr));
    cv = sample64(taps, xd + static_cast<double>(sd * cc), yd + static_cast<double>(sd * sc));
  } else {
    lv = sample(taps, x + sd * cl, y + sd * sl);  // :79-95, read order L, R, C
    rv = sample(taps, x + sd * cr, y + sd * sr);
    cv = sample(taps, x + sd * cc, y + sd * sc);
  }
  __builtin_amdgcn_s_setprio(0);
  angle = turn(angle, lv, rv, cv, p.turn);

  // With zero jitter the term is (finite) * 0 = +-0, which leaves the angle
  // unchanged, so the hash (and the original-index load) is skipped.
  if (p.jitter != 0.0f) {
    uint32_t index = a.id ? a.id[j] : j - in.agent_off;  // S6
    angle += jitter_term(index, x, y, p.jitter);
  }

  angle = wgsl_mod(angle, kTau);  // :121-122
  if (angle < 0.0f) angle = angle + kTau;

  float move = speed * kTimeStep;  // :125-127
  float ms, mc;
  slm_sincosf_finite(angle, &ms, &mc);
  int dx, dy;
  if (P64) {
    double fw = static_cast<double>(w), fh = static_cast<double>(h);
    xd = xd + static_cast<double>(move * mc);
    yd = yd + static_cast<double>(move * ms);
    xd = mod64(xd, fw);
    if (xd < 0.0) xd = xd + fw;
    yd = mod64(yd, fh);
    if (yd < 0.0) yd = yd + fh;
    dx = static_cast<int>(xd);
    dy = static_cast<int>(yd);
    a.x64[j] = xd;
    a.y64[j] = yd;
  } else {
    x = x + move * mc;
    y = y + move * ms;
    float fw = static_cast<float>(w), fh = static_cast<float>(h);  // :130-133
    x = wgsl_mod(x, fw);
    if (x < 0.0f) x = x + fw;
    y = wgsl_mod(y, fh);
    if (y < 0.0f) y = y + fh;
    dx = static_cast<int>(x);
    dy = static_cast<int>(y);
    a.x[j] = x;  // :144
    a.y[j] = y;
  }
  a.th[j] = angle;
  // the mark's load at raised priority too (290 / 226 us against 294 / 229)
  __builtin_amdgcn_s_setprio(2);
  if (dx >= 0 && static_cast<uint32_t>(dx) < w && dy >= 0 && static_cast<uint32_t>(dy) < h)
    taps.mark(static_cast<uint32_t>(dx), static_cast<uint32_t>(dy));  // :136-141
  __builtin_amdgcn_s_setprio(0);
}

// Agents begin + threadIdx.x, + block, ... below end, with the next agent's
// state loaded while the current one is computed.  begin and end are
// workgroup-uniform, so every thread runs the same number of rounds and each
// round starts at a barrier: the workgroup senses one round of neighbouring
// agents in step, and their shared tap lines stay in the vector L1 (C1,
// 1024 agents per workgroup: 400 -> 328 us per pass while trails form,
// 270 -> 239 us once formed).
template <bool P64, int kBlock, class Taps>
__device__ inline void agent_loop(const AgentSoA& a, uint32_t begin, uint32_t end,
                                  const Instance& in, const DevParams& p, const Taps& taps) {
  const uint32_t rounds = (end - begin + kBlock - 1u) / kBlock;
  uint32_t j = begin + threadIdx.x;
  AgentState<P64> cur{};
  if (j < end) cur = load_agent<P64>(a, j);
  for (uint32_t k = 0; k < rounds; k++) {
    const uint32_t nj = j + kBlock;
    AgentState<P64> nxt = cur;
    if (nj < end) nxt = load_agent<P64>(a, nj);
    __syncthreads();
    if (j < end) agent_update<P64>(a, j, cur, in, p, taps);
    j = nj;
    cur = nxt;
  }
}


struct AgentArgs {
  AgentSoA a;
  void* trail;
  const Instance* inst;
  const DevParams* params;
  const uint32_t* block_inst;  // per kAgentBlock slots
  uint32_t count, total;
  uint32_t group;  // agents per workgroup, a multiple of kAgentBlock
  int xcd_remap;
  uint32_t* claim;  // persistent launch: claim counters (nullptr: one workgroup per block)
  uint32_t blocks;  // logical workgroups of the pass
};

// ---- windowed sensing ----------------------------------------------------------
// After a Morton re-sort the 256 agents of a workgroup sit in a few
// neighbouring bins.  The workgroup takes the bounding box of their cells,
// widens it by the sensor reach (ceil|sensor distance| + 2 cells covers every
// bilinear tap) and stages that window of the trail in LDS with 16-byte row
// loads, then senses from LDS: one coalesced pass over the window instead of
// six divergent tap-pair loads per agent, which keep the texture addresser
// busy.  Taps outside the window still read global memory, so results do not
// depend on the window.  A window beyond the LDS budget (agents spread out,
// sensor distances in the hundreds) senses from global memory for the whole
// workgroup.
// 31 KiB (plus 16 bytes of padding for the 16-bit reads' second dword) keeps
// five workgroups resident per CU in gfx950's 160 KiB of LDS.
constexpr uint32_t kWinBytes = 31744;

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                                 __builtin_bit_cast(u16x2, b)));
}

// One workgroup of kAgentBlock slots [first, first + 256) inside instance
// `in` (whose sides are below 2^16 and whose rows are whole 16-byte chunks);
// thread j's agent when j <= last.
template <int S, bool P64>
__device__ inline void window_block(const AgentArgs& args, uint32_t j, uint32_t last,
                                    const Instance& in, const DevParams& p, uint32_t* s_win,
                                    uint32_t* s_box) {
  using elem = typename TrailRead<S>::elem;
  constexpr int V = static_cast<int>(16 / sizeof(elem));
  elem* trail = static_cast<elem*>(args.trail) + in.trail_off;
  const bool live = j <= last;
  AgentState<P64> st{};
  if (live) st = load_agent<P64>(args.a, j);
  // bounding box of the agents' cells: per-component u16 maxima of (x | y << 16)
  // and of its complement (the minima), over the wave, then the workgroup
  uint32_t cx = 0, cy = 0;
  if (live) {
    cx = static_cast<uint32_t>(P64 ? static_cast<int>(st.xd) : static_cast<int>(st.x));
    cy = static_cast<uint32_t>(P64 ? static_cast<int>(st.yd) : static_cast<int>(st.y));
  }
  // wave maxima by DPP row operations (no LDS round trips)
  const uint32_t mx = __ockl_wfred_max_u32(live ? cx : 0u);
  const uint32_t my = __ockl_wfred_max_u32(live ? cy : 0u);
  const uint32_t nx = __ockl_wfred_max_u32(live ? 0xffffu - cx : 0u);
  const uint32_t ny = __ockl_wfred_max_u32(live ? 0xffffu - cy : 0u);
  uint32_t hi = (my << 16) | mx;
  uint32_t lo = (ny << 16) | nx;
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = static_cast<int>(threadIdx.x) & 63;
  if (lane == 0) {
    s_box[2 * wave] = hi;
    s_box[2 * wave + 1] = lo;
  }
  __syncthreads();
  hi = pk_max_u16(pk_max_u16(s_box[0], s_box[2]), pk_max_u16(s_box[4], s_box[6]));
  lo = pk_max_u16(pk_max_u16(s_box[1], s_box[3]), pk_max_u16(s_box[5], s_box[7]));
  const int W = static_cast<int>(in.width), H = static_cast<int>(in.height);
  const int reach = static_cast<int>(__builtin_ceilf(__builtin_fabsf(p.sensor_dist))) + 2;
  const int minx = 0xffff - static_cast<int>(lo & 0xffffu), maxx = static_cast<int>(hi & 0xffffu);
  const int miny = 0xffff - static_cast<int>(lo >> 16), maxy = static_cast<int>(hi >> 16);
  const int wx0 = max(minx - reach, 0) & ~(V - 1);
  const int wy0 = max(miny - reach, 0);
  const int ww = min(maxx + reach + 1, W) - wx0;
  const int wh = min(maxy + reach + 1, H) - wy0;
  const int cpr = (ww + V - 1) / V;  // 16-byte chunks per window row
  const int pitch = cpr * V;
  const bool staged = cpr <= 64 && static_cast<uint32_t>(pitch) * static_cast<uint32_t>(wh) *
                                           sizeof(elem) <= kWinBytes;  // uniform
  if (!staged) {
    GlobalTaps<S> taps{trail, in.width, in.height};
    if (live) agent_update<P64>(args.a, j, st, in, p, taps);
    return;
  }
  // Stage: lane l takes chunk l % cw of sub-row l / cw (cw = the power of two
  // >= cpr), so a wave covers 64 / cw rows per pass; four loads in flight per
  // lane before their LDS stores.
  const int cw = cpr <= 1 ? 1 : 1 << (32 - __builtin_clz(static_cast<uint32_t>(cpr - 1)));
  const int per = 64 / cw;  // rows per wave pass
  const int c = lane & (cw - 1);
  const int step = 4 * per;  // rows per workgroup pass
  const elem* src = trail + static_cast<size_t>(wy0) * in.width + wx0 + c * V;
  unsigned char* dst = reinterpret_cast<unsigned char*>(s_win) + c * 16;
  const bool col_ok = c < cpr;
  auto load = [&](int r) {
    return *reinterpret_cast<const uint4*>(src + static_cast<size_t>(r) * in.width);
  };
  auto store = [&](int r, uint4 v) {
    *reinterpret_cast<uint4*>(dst + static_cast<size_t>(r) * pitch * sizeof(elem)) = v;
  };
  for (int r0 = wave * per + lane / cw; r0 < wh; r0 += 4 * step) {
    const int r1 = r0 + step, r2 = r0 + 2 * step, r3 = r0 + 3 * step;
    const uint4 z = make_uint4(0u, 0u, 0u, 0u);
    const uint4 v0 = col_ok ? load(r0) : z;
    const uint4 v1 = col_ok && r1 < wh ? load(r1) : z;
    const uint4 v2 = col_ok && r2 < wh ? load(r2) : z;
    const uint4 v3 = col_ok && r3 < wh ? load(r3) : z;
    if (col_ok) store(r0, v0);
    if (col_ok && r1 < wh) store(r1, v1);
    if (col_ok && r2 < wh) store(r2, v2);
    if (col_ok && r3 < wh) store(r3, v3);
  }
  __syncthreads();
  BoxTaps<S> taps{trail, in.width, in.height, s_win, wx0, wy0, ww, wh, pitch};
  if (live) agent_update<P64>(args.a, j, st, in, p, taps);
}

// One logical workgroup `blk` of the agent pass.  kWin: one-agent-per-thread
// workgroups that lie inside one instance sense through an LDS window
// (window_block).
template <int S, bool P64, bool kWin>
__device__ inline void agents_block(const AgentArgs& args, const Instance* __restrict__ insts,
                                    const DevParams* __restrict__ params,
                                    const uint32_t* __restrict__ block_inst, uint32_t blk,
                                    uint32_t* s_win, uint32_t* s_box) {
  using elem = typename TrailRead<S>::elem;
  if (args.group == kAgentBlock) {  // one agent per thread
    uint32_t first = blk * kAgentBlock;
    uint32_t last = min(first + kAgentBlock, args.total) - 1u;
    uint32_t j = first + threadIdx.x;
    if constexpr (kWin) {
      constexpr uint32_t V = 16 / sizeof(elem);
      const uint32_t ii = block_inst[blk];
      const Instance in = insts[ii];
      if (first >= in.agent_off && last < in.agent_off + in.agent_count && in.width < 65536u &&
          in.height < 65536u && in.width % V == 0u) {  // uniform
        window_block<S, P64>(args, j, last, in, params[ii], s_win, s_box);
        return;
      }
    }
    {
      // A block inside one instance: every thread loads its agent, then the
      // workgroup waits for all four waves before any senses.  The waves'
      // agents are neighbours after a re-sort and their sensor taps share
      // lines; sensing in step keeps those lines in the vector L1 for all
      // four (C1, 4096^2 f32, 2^24 agents: 363 -> 338 us per pass while
      // trails form).  (Written as its own path: folding it into the
      // instance walk below cost the kernel 24 VGPRs and two waves per SIMD.)
      const uint32_t ii = block_inst[blk];
      const Instance in = insts[ii];
      if (first >= in.agent_off && last < in.agent_off + in.agent_count) {  // uniform
        const bool live = j <= last;
        AgentState<P64> st{};
        if (live) st = load_agent<P64>(args.a, j);
        __syncthreads();
        const DevParams p = params[ii];
        GlobalTaps<S> taps{static_cast<elem*>(args.trail) + in.trail_off, in.width, in.height};
        if (live) agent_update<P64>(args.a, j, st, in, p, taps);
        return;
      }
    }
    // instances overlapping this block, one at a time (block-uniform)
    for (uint32_t ii = block_inst[blk];; ii++) {
      const Instance in = insts[ii];
      uint32_t end = in.agent_off + in.agent_count;
      if (j >= in.agent_off && j < end) {
        const DevParams p = params[ii];
        GlobalTaps<S> taps{static_cast<elem*>(args.trail) + in.trail_off, in.width, in.height};
        agent_update<P64>(args.a, j, load_agent<P64>(args.a, j), in, p, taps);
      }
      if (last < end || ii + 1u >= args.count) break;
    }
    return;
  }
  // `group` consecutive slots, each thread striding by the block size with the
  // next agent's state in flight
  uint32_t first = blk * args.group;
  uint32_t stop = min(first + args.group, args.total);
  for (uint32_t ii = block_inst[first / kAgentBlock];; ii++) {
    const Instance in = insts[ii];
    uint32_t end = in.agent_off + in.agent_count;
    uint32_t b = max(first, in.agent_off), e = min(stop, end);
    if (b < e) {
      const DevParams p = params[ii];
      GlobalTaps<S> taps{static_cast<elem*>(args.trail) + in.trail_off, in.width, in.height};
      agent_loop<P64, kAgentBlock>(args.a, b, e, in, p, taps);
    }
    if (stop <= end || ii + 1u >= args.count) break;
  }
}

// The tables are separate restrict-qualified arguments: nothing the kernel
// stores aliases them, so their block-uniform loads become scalar loads.
// With args.claim set the launch is persistent (persistent_blocks).
template <int S, bool P64, bool kWin>
__global__ __launch_bounds__(kAgentBlock) void agents_kernel(
    AgentArgs args, const Instance* __restrict__ insts, const DevParams* __restrict__ params,
    const uint32_t* __restrict__ block_inst) {
  __shared__ __align__(16) uint32_t s_win[kWin ? kWinBytes / 4 + 4 : 1];
  __shared__ uint32_t s_box[8];
  __shared__ uint32_t s_claim;
  if (!args.claim) {
    const uint32_t blk = args.xcd_remap ? xcd_logical_block(blockIdx.x, gridDim.x) : blockIdx.x;
    agents_block<S, P64, kWin>(args, insts, params, block_inst, blk, s_win, s_box);
    return;
  }
  persistent_blocks(args.claim, args.blocks, &s_claim, [&](uint32_t blk) {
    agents_block<S, P64, kWin>(args, insts, params, block_inst, blk, s_win, s_box);
  });
}

// ---- tile windows ------------------------------------------------------------
// After a re-sort the agents of each 2^k x 2^k-cell tile occupy consecutive
// slots (the tile is an aligned square of Morton bins).  One workgroup takes a
// work item (up to 1.5 * kItemAgents of a tile's slots) and stages the trail
// around the tile - the tile plus a margin of the sensor reach and the distance
// agents may have drifted since the re-sort - in LDS, as f32, and senses there.
//
// Why: the vector L1 serves a divergent gather one lane a cycle whatever lines
// the lanes share: a wave of 64 agents costs the global pass 525 accesses (384
// of them the six tap pairs, 128 the mark's load and store), which at 2.35 GHz
// are exactly its 229 us on 4096^2 with 2^24 agents once trails have formed.
// The LDS reads the same pairs at 64 banks a cycle, and the window comes in
// coalesced, 16 bytes a lane: 4.4 cells an agent at one agent a cell.  What it
// measured, us per pass with the global pass's in brackets: 4096^2 f32 with 2^24
// agents 175 (275) while trails form, 155 (205) once formed; 1600 x 900 with
// 10^7 agents 96 (137) and 78 (109); 8192^2 bf16 with f64 positions and 2^26
// agents 814 to 900 (1030 to 1200).
//
// Shape, all measured: 64-cell tiles and 1024 threads, two workgroups to a CU
// (80 KiB of LDS each, 64 VGPRs), so that one computes while the other stages;
// 32-cell tiles with 512 threads are 25% slower (they stage twice the cells),
// a persistent workgroup holding the next window in registers 15% slower (half
// the waves).  f64 positions need more registers: 512 threads.
//
// An agent's wave senses from the window when all its agents are where the
// margin covers them (a test per agent, so results never depend on the margin,
// the work list or the time since the re-sort) and angles and parameters are in
// the ordinary range, else it takes agent_update and reads global memory.
//
// The update itself is then mostly VALU issue: 557 instructions a wave of two agents a
// lane take 46 to 88% of the pass's cycles, the L1 36%, the LDS 29% (4096^2 f32, 2^24
// agents, trails formed).  On gfx950 f32 multiply, add
// and fma, and/xor/bitop3, right shifts and 32-bit adds issue in 2.3 cycles per
// wave when every operand is a vector register or a literal; with a scalar
// register operand, and for compares, selects, conversions, rounding, left
// shifts and 64-bit address adds, it is 4.4 (measured).  So tile_update keeps its
// uniform operands in vector registers (in_vgpr), replaces selects by bit
// operations and skips the range tests where the window is not clipped by the
// grid's edge: 239 instead of 325 VALU instructions per wave.  (The global pass
// keeps its own form: it gains nothing from fewer instructions.)
// A cell's mark in two halves, the load of the 16 bits that hold its sign and
// their store, so that a caller can have other stores between them.
// A mark from the window is noted there too (the upper half of the f32 cell, which
// the taps read as |T|), so that the tile's later agents skip the cell: 4096^2 f32
// with 2^24 agents 169 -> 164 us per pass, 8192^2 bf16 with f64 positions 826 -> 814.
struct Mark {
  uint16_t* p;
  uint32_t raw;
  uint16_t* win;   // in the window, or nullptr
  uint32_t upper;  // what `win` holds
  __device__ void store() const {
    if (!(raw & 0x8000u)) {
      *p = static_cast<uint16_t>(raw | 0x8000u);
      if (win) *win = static_cast<uint16_t>(upper | 0x8000u);
    }
  }
};

// Whether cells (x0, y0) .. (x0 + 1, y0 + 1) lie in the grid: a negative
// coordinate is a large unsigned one.
__device__ inline bool in_grid(int x0, int y0, uint32_t w, uint32_t h) {
  return static_cast<uint32_t>(x0) < w - 1u && static_cast<uint32_t>(y0) < h - 1u;
}

// The |T| values of the four cells around a sample's point (any values where the
// point is outside the grid: !in), and the bilinear weights.
struct Cells {
  float v00, v10, v01, v11;
  bool in;
};
struct Weights {
  float dx, dy;
};
__device__ inline float mix_cells(const Cells& c, const Weights& f) {
  const float v0 = wgsl_mix(c.v00, c.v10, f.dx);
  const float v1 = wgsl_mix(c.v01, c.v11, f.dx);
  return wgsl_mix(v0, v1, f.dy);
}

// Taps from a tile's window of the trail staged in LDS as f32 |T| (tile
// windows, below), for points whose cells the caller knows to lie in the window
// where they lie in the grid.  One 32-bit address serves a sample: the two cells
// of a row are neighbours and the row below is `pitch` bytes on.
template <int S>
struct TileTaps {
  using elem = typename TrailRead<S>::elem;
  void* t;
  uint32_t w, h;
  const char* win;   // LDS
  uint32_t pitch;    // bytes per window row
  uint32_t origin;   // byte offset of the map's cell (0, 0) (mod 2^32)
  __device__ Cells cells_inside(uint32_t x0, uint32_t y0) const {
    const char* p = win + (__umul24(y0, pitch) + (x0 * 4u + origin));
    const float* row = reinterpret_cast<const float*>(p);
    const float* below = reinterpret_cast<const float*>(p + pitch);
    return {fabsf(row[0]), fabsf(row[1]), fabsf(below[0]), fabsf(below[1]), true};
  }
  __device__ Cells cells(int x0, int y0) const {
    const bool in = in_grid(x0, y0, w, h);
    const uint32_t o = __umul24(static_cast<uint32_t>(y0), pitch) +
                       (static_cast<uint32_t>(x0) * 4u + origin);
    const char* p = win + (in ? o : 0u);
    const float* row = reinterpret_cast<const float*>(p);
    const float* below = reinterpret_cast<const float*>(p + pitch);
    return {fabsf(row[0]), fabsf(row[1]), fabsf(below[0]), fabsf(below[1]), in};
  }
  __device__ Mark mark(uint32_t x, uint32_t y) const {
    uint16_t* p = half_cell(x, y);
    return {p, *p, nullptr, 0u};
  }
  // The cell's |T| is in the window: the mark needs no load from the trail.
  // (Marking in the window and storing the marked cells a row per wave at the
  // workgroup's end measured 2% faster to 5% slower.)
  __device__ Mark mark_inside(uint32_t x, uint32_t y) const {
    const char* p = win + (__umul24(y, pitch) + (x * 4u + origin));
    uint32_t raw;
    if constexpr (S == SLM_STORAGE_F16)
      raw = __builtin_bit_cast(uint16_t,
                               static_cast<_Float16>(*reinterpret_cast<const float*>(p)));
    else
      raw = *reinterpret_cast<const uint16_t*>(p + 2);
    uint16_t* u = reinterpret_cast<uint16_t*>(const_cast<char*>(p) + 2);
    return {half_cell(x, y), raw, u, *u};
  }
  // The 16 bits that hold a cell's sign, in a trail below 2^32 bytes with rows
  // below 2^24 (tile_staged).
  __device__ uint16_t* half_cell(uint32_t x, uint32_t y) const {
    constexpr uint32_t kBytes = sizeof(elem);
    const uint32_t o = __umul24(y, w * kBytes) + (x * kBytes + (kBytes - 2u));
    return reinterpret_cast<uint16_t*>(static_cast<char*>(t) + o);
  }
};

// The cells around (px, py) and their weights.  kInside: the point is known to
// lie in the grid with its neighbour cells; truncation is the floor of a value
// >= 0, and v_fract is exact there.
template <bool kInside, class Taps>
__device__ inline Cells tap(const Taps& taps, float px, float py, Weights& f) {
  if constexpr (kInside) {
    f = {__builtin_amdgcn_fractf(px), __builtin_amdgcn_fractf(py)};
    return taps.cells_inside(static_cast<uint32_t>(static_cast<int>(px)),
                             static_cast<uint32_t>(static_cast<int>(py)));
  } else {
    const float fx = __builtin_floorf(px), fy = __builtin_floorf(py);
    f = {px - fx, py - fy};
    return taps.cells(static_cast<int>(fx), static_cast<int>(fy));
  }
}
template <bool kInside, class Taps>
__device__ inline Cells tap(const Taps& taps, double px, double py, Weights& f) {
  if constexpr (kInside) {
    f = {static_cast<float>(__builtin_amdgcn_fract(px)),
         static_cast<float>(__builtin_amdgcn_fract(py))};
    return taps.cells_inside(static_cast<uint32_t>(static_cast<int>(px)),
                             static_cast<uint32_t>(static_cast<int>(py)));
  } else {
    const double fx = __builtin_floor(px), fy = __builtin_floor(py);
    f = {static_cast<float>(px - fx), static_cast<float>(py - fy)};
    return taps.cells(static_cast<int>(fx), static_cast<int>(fy));
  }
}

// wgsl_mod with a second short case: when |a| < 2b, a/b truncates to +-1 (the
// quotient is at most pred(2), as pred(2b)/b is) and a - b*(+-1) is a -+ b.  The
// result is never -0.
__device__ inline float mod_near(float a, float b) {
  if (__builtin_fabsf(a) >= b && __builtin_fabsf(a) < b + b) return a - __builtin_copysignf(b, a);
  return wgsl_mod(a, b);
}
// r + (r < 0 ? b : 0) for a result r of mod_near: r is never -0, so its sign
// bit is the test, and adding +0 leaves the others.
__device__ inline float wrap_up(float r, float b) {
  uint32_t below;  // all ones below 0 (as asm: the compiler makes a compare and a select of it)
  asm("v_ashrrev_i32 %0, 31, %1" : "=v"(below) : "v"(r));
  return r + __uint_as_float(__float_as_uint(b) & below);
}
// `turn` for |angle| < kQuickAngle and turn_speed <= kQuickTurn: the distance to
// either target is then 2 pi to within 2.5e-4, above turn_speed, so the turn is
// -turn_speed or +turn_speed, the sign of rv - lv.  That is 0 only for equal values
// (f32 subtraction keeps denormals) and NaN only for values that compare neither way
// (two infinities, as f16 cells beyond 65504 are, or a NaN sample): |rv - lv| > 0 is
// lv < rv or lv > rv.
__device__ inline float turn_quick(float angle, float lv, float rv, float cv, float turn_speed,
                                   uint32_t sign) {
  const float d = rv - lv;
  const float turned =
      angle + __uint_as_float(__float_as_uint(turn_speed) ^ (__float_as_uint(d) & sign));
  const bool straight = !(__builtin_fabsf(d) > 0.0f) | ((cv > lv) & (cv > rv));
  return straight ? angle : turned;
}

// jitter_term with the middle range's shorter reduction.
__device__ inline float jitter_term_mid(uint32_t index, float x, float y, float jitter) {
  float hx = static_cast<float>(static_cast<int32_t>(index)) * 12.9898f;
  hx = hx + x * 78.233f;
  hx = hx + y * 37.719f;
  const float ax = __builtin_fabsf(hx);
  float s, c;
  // waves wholly inside the middle range, all but a few, take its shorter form
  if (__all(ax >= SLM_TRIG_SMALL_MAX && ax < SLM_TRIG_MID_MAX))
    s = slm_sinf_mid(hx);
  else
    slm_sincosf_finite(hx, &s, &c);  // finite: index, positions and products are bounded
  float v = s * 43758.5453f;
  float rnd = v - __builtin_floorf(v);
  return (rnd * 2.0f - 1.0f) * jitter;
}

// The agent arrays from slot `base` on (uniform), indexed by a lane's small
// offset: scalar bases and 32-bit lane offsets.
__device__ inline AgentSoA agents_from(const AgentSoA& a, uint32_t base, bool p64) {
  AgentSoA r = a;
  if (p64) {
    r.x64 += base;
    r.y64 += base;
  } else {
    r.x += base;
    r.y += base;
  }
  r.th += base;
  r.v += base;
  if (r.id) r.id += base;
  return r;
}

// Element j of an array at a uniform address: scalar base, 32-bit byte offset.
template <class T>
__device__ inline T& lane_at(T* base, uint32_t j) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + j * static_cast<uint32_t>(sizeof(T)));
}

template <bool P64>
__device__ inline AgentState<P64> load_lane(const AgentSoA& a, uint32_t j) {
  AgentState<P64> st;
  st.angle = lane_at(a.th, j);
  st.speed = lane_at(a.v, j);
  if (P64) {
    st.xd = lane_at(a.x64, j);
    st.yd = lane_at(a.y64, j);
    st.x = st.y = 0.0f;
  } else {
    st.xd = st.yd = 0.0;
    st.x = lane_at(a.x, j);
    st.y = lane_at(a.y, j);
  }
  return st;
}

constexpr float kQuickAngle = 2048.0f;
constexpr float kQuickSensorAngle = 1024.0f;  // angle +- it stays below SLM_TRIG_SMALL_MAX
constexpr float kQuickTurn = 6.25f;           // below 2 pi - 2.5e-4

__device__ inline float in_vgpr(float v) {
  asm("" : "+v"(v));
  return v;
}

// Uniform values of one instance's updates.
struct UpdateConsts {
  bool ordinary;          // parameters in the ordinary range
  float sa, sd, turn;
  float two_over_pi, pio2_c1;  // slm_sincosf_small_k's constants
  uint32_t sign;
  __device__ void sincos(float v, float* s, float* c) const {
    slm_sincosf_small_k(v, two_over_pi, pio2_c1, sign, s, c);
  }
};

__device__ inline UpdateConsts update_consts(const DevParams& p) {
  UpdateConsts k;
  k.ordinary = __builtin_fabsf(p.sensor_angle) <= kQuickSensorAngle && p.turn <= kQuickTurn &&
               p.speed_min <= p.speed_max;
  k.sa = in_vgpr(p.sensor_angle);
  k.sd = in_vgpr(p.sensor_dist);
  k.turn = in_vgpr(p.turn);
  k.two_over_pi = in_vgpr(SLM_TWO_OVER_PI_F);
  k.pio2_c1 = in_vgpr(SLM_PIO2_C1);
  k.sign = __float_as_uint(in_vgpr(-0.0f));
  return k;
}

// Has the loads of `st` counted as done here: they were issued before loads
// that have been waited for, and behind the stores that follow, a wait for
// them would be a wait for the stores.
template <bool P64>
__device__ inline void wait_state(AgentState<P64>& st) {
  asm volatile("" : "+v"(st.angle), "+v"(st.speed));
  if constexpr (P64)
    asm volatile("" : "+v"(st.xd), "+v"(st.yd));
  else
    asm volatile("" : "+v"(st.x), "+v"(st.y));
}

// One agent (lane offset j of `a`, state st, instance slot `slot`) for one
// step; nxt: the state in flight for the lane's next agent.
template <bool P64, bool kInside, class Taps>
__device__ inline void tile_update(const AgentSoA& a, uint32_t j, uint32_t slot,
                                   const AgentState<P64>& st, AgentState<P64>& nxt,
                                   const Instance& in, const DevParams& p, const Taps& taps,
                                   const UpdateConsts& k) {
  const uint32_t w = in.width, h = in.height;
  float angle = st.angle, speed = st.speed;
  double xd = st.xd, yd = st.yd;
  float x = P64 ? static_cast<float>(xd) : st.x, y = P64 ? static_cast<float>(yd) : st.y;

  // :72; the median is the clamp where speed_min <= speed_max
  float sp = __builtin_amdgcn_fmed3f(speed, p.speed_min, p.speed_max);
  if (sp != speed) lane_at(a.v, j) = sp;
  speed = sp;

  float al = angle - k.sa, ar = angle + k.sa;  // :75-77
  float sl, cl, sr, cr, sc, cc;
  k.sincos(al, &sl, &cl);
  k.sincos(ar, &sr, &cr);
  k.sincos(angle, &sc, &cc);
  const float sd = k.sd;
  Cells lc, rc, cc4;
  Weights lf, rf, cf;
  __builtin_amdgcn_s_setprio(2);
  if constexpr (P64) {
    lc = tap<kInside>(taps, xd + static_cast<double>(sd * cl), yd + static_cast<double>(sd * sl), lf);
    rc = tap<kInside>(taps, xd + static_cast<double>(sd * cr), yd + static_cast<double>(sd * sr), rf);
    cc4 = tap<kInside>(taps, xd + static_cast<double>(sd * cc), yd + static_cast<double>(sd * sc), cf);
  } else {
    lc = tap<kInside>(taps, x + sd * cl, y + sd * sl, lf);  // :79-95, read order L, R, C
    rc = tap<kInside>(taps, x + sd * cr, y + sd * sr, rf);
    cc4 = tap<kInside>(taps, x + sd * cc, y + sd * sc, cf);
  }
  const float lv = lc.in ? mix_cells(lc, lf) : 0.0f;
  const float rv = rc.in ? mix_cells(rc, rf) : 0.0f;
  const float cv = cc4.in ? mix_cells(cc4, cf) : 0.0f;
  __builtin_amdgcn_s_setprio(0);
  angle = turn_quick(angle, lv, rv, cv, k.turn, k.sign);

  // With zero jitter the term is (finite) * 0 = +-0, which leaves the angle
  // unchanged, so the hash (and the original-index load) is skipped.
  if (p.jitter != 0.0f) {
    uint32_t index = a.id ? lane_at(a.id, j) : slot;  // S6
    angle += jitter_term_mid(index, x, y, p.jitter);
  }

  angle = wrap_up(mod_near(angle, kTau), kTau);  // :121-122; now in [0, 2 pi]

  float move = speed * kTimeStep;  // :125-127
  float ms, mc;
  k.sincos(angle, &ms, &mc);
  int dx, dy;
  if (P64) {
    xd = xd + static_cast<double>(move * mc);
    yd = yd + static_cast<double>(move * ms);
    if (!kInside) {
      double fw = static_cast<double>(w), fh = static_cast<double>(h);
      xd = mod64(xd, fw);
      if (xd < 0.0) xd = xd + fw;
      yd = mod64(yd, fh);
      if (yd < 0.0) yd = yd + fh;
    }
    dx = static_cast<int>(xd);
    dy = static_cast<int>(yd);
  } else {
    x = x + move * mc;
    y = y + move * ms;
    if (!kInside) {
      float fw = static_cast<float>(w), fh = static_cast<float>(h);  // :130-133
      x = wrap_up(mod_near(x, fw), fw);
      y = wrap_up(mod_near(y, fh), fh);
    }
    dx = static_cast<int>(x);
    dy = static_cast<int>(y);
  }
  // The mark (:136-141): its load (clipped windows only), the state's stores, its store.
  __builtin_amdgcn_s_setprio(2);
  const uint32_t ux = static_cast<uint32_t>(dx), uy = static_cast<uint32_t>(dy);
  bool in_map = true;
  Mark mark{};
  if constexpr (kInside) {
    mark = taps.mark_inside(ux, uy);
  } else {
    in_map = ux < w && uy < h;  // wrapped positions are >= 0
    if (in_map) mark = taps.mark(ux, uy);
  }
  wait_state(nxt);
  if constexpr (P64) {
    lane_at(a.x64, j) = xd;  // :144
    lane_at(a.y64, j) = yd;
  } else {
    lane_at(a.x, j) = x;
    lane_at(a.y, j) = y;
  }
  lane_at(a.th, j) = angle;
  if (in_map) mark.store();
  __builtin_amdgcn_s_setprio(0);
}

constexpr uint32_t kMinStagedAgents = 256;  // sparser items read global memory

__device__ inline uint32_t compact_bits(uint32_t v) {  // even bits -> 16 bits
  v &= 0x55555555u;
  v = (v | (v >> 1)) & 0x33333333u;
  v = (v | (v >> 2)) & 0x0f0f0f0fu;
  v = (v | (v >> 4)) & 0x00ff00ffu;
  v = (v | (v >> 8)) & 0x0000ffffu;
  return v;
}

struct TiledArgs {
  AgentSoA a;
  void* trail;
  const WorkItem* items;
  uint32_t drift_steps;  // steps since the re-sort, this one included
};

// A work item's window: `rows` rows from y0 of `cpr` 16-byte chunks from x0,
// chunk q of the window being chunk q % cpr of row q / cpr, and in LDS 16-byte
// (f32) or 32-byte (16-bit formats, widened) entry q.
struct TileWindow {
  float cx, cy, half;       // agents with |x - cx| < half and |y - cy| < half sense inside it
  int x0, y0, cpr, rows;
  uint32_t inv_cpr;         // ceil(2^20 / cpr)
  bool staged, clipped;
};

template <int S>
__device__ inline TileWindow tile_window(const WorkItem& wi, const Instance& in,
                                         const DevParams& p, uint32_t drift_steps) {
  constexpr int V = static_cast<int>(16 / sizeof(typename TrailRead<S>::elem));
  const int tile = 1 << in.tile_log2;
  const int tx = static_cast<int>(compact_bits(wi.tile)) * tile;
  const int ty = static_cast<int>(compact_bits(wi.tile >> 1)) * tile;
  const TileReach r = tile_reach(p, drift_steps);
  // uniform, but computed in vector registers: back to a scalar one
  const int m = __builtin_amdgcn_readfirstlane(r.margin);
  const TileExtent e = tile_extent(in, tx, ty, m, V);
  TileWindow win;
  win.x0 = e.x0;
  win.y0 = e.y0;
  win.cpr = e.cpr;
  win.rows = e.rows;
  // q * inv_cpr stays below 2^32 (rows <= 1024), and it >> 20 is q / cpr while
  // q * cpr < 2^20
  win.inv_cpr = ((1u << 20) + static_cast<uint32_t>(e.cpr) - 1u) / static_cast<uint32_t>(e.cpr);
  win.clipped = tx - m < 0 || ty - m < 0 || tx + tile + m > static_cast<int>(in.width) ||
                ty + tile + m > static_cast<int>(in.height);
  win.staged = wi.end - wi.begin >= kMinStagedAgents && tile_staged(in, e, V);
  win.cx = static_cast<float>(tx) + 0.5f * static_cast<float>(tile);
  win.cy = static_cast<float>(ty) + 0.5f * static_cast<float>(tile);
  win.half = win.staged ? 0.5f * static_cast<float>(tile) + static_cast<float>(m) - r.reach : -1.0f;
  return win;
}

template <int S, bool P64, bool kOne>
__global__ __launch_bounds__(tile_block(P64))
    __attribute__((amdgpu_waves_per_eu(P64 ? 4 : 8))) void agents_tiled_kernel(
        TiledArgs args, const Instance* __restrict__ insts, const DevParams* __restrict__ params) {
  using elem = typename TrailRead<S>::elem;
  constexpr int V = static_cast<int>(16 / sizeof(elem));  // cells per 16-byte chunk
  constexpr int kTileBlock = tile_block(P64);
  constexpr int kDeep = (static_cast<int>(kTileLds) / (V * 4) + kTileBlock - 1) / kTileBlock;  // chunks per lane
  extern __shared__ __align__(16) char smem[];
  const uint32_t t = threadIdx.x;
  // kOne (a pool of one instance): the tables' loads do not wait for the item's
  WorkItem wi = args.items[blockIdx.x];
  Instance in = insts[kOne ? 0u : wi.inst];
  DevParams p = params[kOne ? 0u : wi.inst];
  if (wi.begin == wi.end) return;  // uniform: past the last item
  elem* trail = static_cast<elem*>(args.trail) + in.trail_off;

  AgentSoA here = agents_from(args.a, wi.begin, P64);
  AgentState<P64> cur{};
  if (t < wi.end - wi.begin) cur = load_lane<P64>(here, t);
  const TileWindow win =
      tile_window<S>(wi, in, p, args.drift_steps);
  if (win.staged) {
    const uint32_t n = static_cast<uint32_t>(win.cpr * win.rows);
    const char* src = reinterpret_cast<const char*>(
        trail + (static_cast<size_t>(win.y0) * in.width + static_cast<uint32_t>(win.x0)));
    uint4 raw[kDeep];  // every chunk in flight before the first is stored
#pragma unroll
    for (int k = 0; k < kDeep; k++) {
      const uint32_t q = min(t + k * kTileBlock, n - 1u);
      const uint32_t r = (q * win.inv_cpr) >> 20;
      const uint32_t c = q - __umul24(r, static_cast<uint32_t>(win.cpr));
      uint4 v;
      __builtin_memcpy(&v, src + (__umul24(r, in.width) + c * V) * static_cast<uint32_t>(sizeof(elem)),
                       sizeof v);
      raw[k] = v;
    }
#pragma unroll
    for (int k = 0; k < kDeep; k++) {
      const uint32_t q = t + k * kTileBlock;
      if (q < n) {
        const uint32_t u[4] = {raw[k].x, raw[k].y, raw[k].z, raw[k].w};
        if constexpr (V == 4) {  // marks included: the taps read |T|
          reinterpret_cast<uint4*>(smem)[q] = make_uint4(u[0], u[1], u[2], u[3]);
        } else {
          float f[8];
#pragma unroll
          for (int i = 0; i < 4; i++) TrailRead<S>::split(u[i], f[2 * i], f[2 * i + 1]);
          reinterpret_cast<float4*>(smem)[2 * q] = make_float4(f[0], f[1], f[2], f[3]);
          reinterpret_cast<float4*>(smem)[2 * q + 1] = make_float4(f[4], f[5], f[6], f[7]);
        }
      }
    }
  }
  __syncthreads();
  const uint32_t pitch = static_cast<uint32_t>(win.cpr) * (V * 4u);
  const TileTaps<S> taps{trail, in.width, in.height, smem, pitch,
                         0u - (static_cast<uint32_t>(win.y0) * pitch +
                               static_cast<uint32_t>(win.x0) * 4u)};
  const GlobalTaps<S> global{trail, in.width, in.height};
  const UpdateConsts k = update_consts(p);
  const float cx = in_vgpr(win.cx), cy = in_vgpr(win.cy);
  const uint32_t count = wi.end - wi.begin;
  const uint32_t first_slot = wi.begin - in.agent_off;
  for (uint32_t j = t;;) {
    const uint32_t nj = j + kTileBlock;
    AgentState<P64> nxt = cur;
    if (nj < count) nxt = load_lane<P64>(here, nj);
    if (j >= count) break;
    const float x = P64 ? static_cast<float>(cur.xd) : cur.x;
    const float y = P64 ? static_cast<float>(cur.yd) : cur.y;
    const bool ordinary = k.ordinary && __builtin_fabsf(cur.angle) < kQuickAngle;
    const uint32_t slot = first_slot + j;
    if (__all(ordinary && __builtin_fabsf(x - cx) < win.half &&
              __builtin_fabsf(y - cy) < win.half)) {
      if (!win.clipped)
        tile_update<P64, true>(here, j, slot, cur, nxt, in, p, taps, k);
      else
        tile_update<P64, false>(here, j, slot, cur, nxt, in, p, taps, k);
    } else {
      AgentState<P64> st = cur;
      if (P64) {
        st.x = x;
        st.y = y;
      }
      agent_update<P64>(args.a, wi.begin + j, st, in, p, global);
    }
    j = nj;
    cur = nxt;
  }
}

// ---- initialisation ------------------------------------------------------
// SplitMix64 (Steele, Lea & Flood 2014): output n of the generator seeded
// with `seed`; uniforms are its top 24 bits times 2^-24.
__device__ inline uint64_t splitmix64_at(uint64_t seed, uint64_t n) {
  uint64_t z = seed + (n + 1u) * 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
__device__ inline float uniform24(uint64_t seed, uint64_t n) {
  return static_cast<float>(static_cast<uint32_t>(splitmix64_at(seed, n) >> 40)) *
         (1.0f / 16777216.0f);
}

// src/main.rs:273-280, agent i (instance-local) drawing generator outputs 4i..4i+3.
__global__ void init_agents_kernel(AgentSoA a, uint32_t off, uint32_t n, int pos64, uint64_t seed,
                                   float fw, float fh, float smin, float range) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float pi = 3.14159265358979323846f;  // std::f32::consts::PI
  uint64_t k = 4ull * i;
  uint32_t j = off + i;
  float x = uniform24(seed, k) * fw;
  float y = uniform24(seed, k + 1) * fh;
  if (pos64) {
    a.x64[j] = x;
    a.y64[j] = y;
  } else {
    a.x[j] = x;
    a.y[j] = y;
  }
  a.th[j] = (uniform24(seed, k + 2) * 2.0f) * pi;
  a.v[j] = smin + uniform24(seed, k + 3) * range;
  if (a.id) a.id[j] = i;
}

// src/main.rs:132-137; the draw is keyed by the original index.
__global__ void reassign_speeds_kernel(AgentSoA a, uint32_t off, uint32_t n, uint64_t seed,
                                       float smin, float range) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint32_t j = off + s;
  uint32_t i = a.id ? a.id[j] : s;
  a.v[j] = smin + uniform24(seed, i) * range;
}

// src/main.rs:993-994
__global__ void scale_positions_kernel(AgentSoA a, uint32_t off, uint32_t n, int pos64, float sx,
                                       float sy) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint32_t j = off + s;
  if (pos64) {
    a.x64[j] *= static_cast<double>(sx);
    a.y64[j] *= static_cast<double>(sy);
  } else {
    a.x[j] *= sx;
    a.y[j] *= sy;
  }
}

__global__ void pack_agents_kernel(AgentSoA a, uint32_t off, uint32_t n, int pos64, float4* aos) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint32_t j = off + s;
  uint32_t i = a.id ? a.id[j] : s;
  float x = pos64 ? static_cast<float>(a.x64[j]) : a.x[j];
  float y = pos64 ? static_cast<float>(a.y64[j]) : a.y[j];
  aos[i] = make_float4(x, y, a.th[j], a.v[j]);
}

__global__ void unpack_agents_kernel(AgentSoA a, uint32_t off, uint32_t n, int pos64,
                                     const float4* aos) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t j = off + i;
  float4 r = aos[i];
  if (pos64) {
    a.x64[j] = r.x;
    a.y64[j] = r.y;
  } else {
    a.x[j] = r.x;
    a.y[j] = r.y;
  }
  a.th[j] = r.z;
  a.v[j] = r.w;
  if (a.id) a.id[j] = i;
}

// Snapshot helpers: (x64, y64) pairs in original order.
__global__ void pack_positions64_kernel(AgentSoA a, uint32_t off, uint32_t n, double2* xy) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint32_t j = off + s;
  uint32_t i = a.id ? a.id[j] : s;
  xy[i] = make_double2(a.x64[j], a.y64[j]);
}

__global__ void unpack_positions64_kernel(AgentSoA a, uint32_t off, uint32_t n,
                                          const double2* xy) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t j = off + i;  // after unpack_agents_kernel: slot j holds agent i
  double2 v = xy[i];
  a.x64[j] = v.x;
  a.y64[j] = v.y;
}

template <int S, bool P64, bool kWin>
void launch_agents_k(const AgentArgs& args, hipStream_t stream) {
  uint32_t grid = args.claim ? persistent_grid(agents_kernel<S, P64, kWin>, args.blocks,
                                               kAgentBlock)
                             : args.blocks;
  agents_kernel<S, P64, kWin><<<grid, kAgentBlock, 0, stream>>>(args, args.inst, args.params,
                                                               args.block_inst);
}

template <int S, bool kWin>
void launch_agents_w(const Pool& pool, const AgentArgs& args, hipStream_t stream) {
  if (pool.pos64)
    launch_agents_k<S, true, kWin>(args, stream);
  else
    launch_agents_k<S, false, kWin>(args, stream);
}

template <int S>
void launch_agents_t(const Pool& pool, const AgentArgs& args, hipStream_t stream) {
  if (pool.window_sensing && args.group == kAgentBlock)
    launch_agents_w<S, true>(pool, args, stream);
  else
    launch_agents_w<S, false>(pool, args, stream);
}

}  // namespace

void launch_agents(const Pool& pool, const AgentSoA& a, void* trail, hipStream_t stream) {
  if (pool.total_agents == 0) return;
  uint32_t group = pool.agents_per_group ? pool.agents_per_group : kAgentBlock;
  AgentArgs args{a,          trail,      pool.inst,         pool.params, pool.agent_block_inst,
                 pool.count, pool.total_agents, group, pool.xcd_remap, pool.claim_agents,
                 blocks_for(pool.total_agents, group)};
  switch (pool.storage) {
    case SLM_STORAGE_BF16:
      launch_agents_t<SLM_STORAGE_BF16>(pool, args, stream);
      break;
    case SLM_STORAGE_F16:
      launch_agents_t<SLM_STORAGE_F16>(pool, args, stream);
      break;
    default:
      launch_agents_t<SLM_STORAGE_F32>(pool, args, stream);
      break;
  }
}

void prime_persistent_agents() {
  auto each = [](auto s_tag) {
    constexpr int S = decltype(s_tag)::value;
    (void)persistent_grid(agents_kernel<S, false, false>, 8, kAgentBlock);
    (void)persistent_grid(agents_kernel<S, false, true>, 8, kAgentBlock);
    (void)persistent_grid(agents_kernel<S, true, false>, 8, kAgentBlock);
    (void)persistent_grid(agents_kernel<S, true, true>, 8, kAgentBlock);
  };
  each(std::integral_constant<int, SLM_STORAGE_F32>{});
  each(std::integral_constant<int, SLM_STORAGE_BF16>{});
  each(std::integral_constant<int, SLM_STORAGE_F16>{});
}

void launch_agents_tiled(const Pool& pool, const AgentSoA& a, void* trail, uint32_t drift_steps,
                         hipStream_t stream) {
  if (pool.total_agents == 0 || pool.max_items == 0) return;
  const int block = tile_block(pool.pos64 != 0);
  TiledArgs args{a, trail, pool.items, drift_steps};
  auto go = [&](auto* one, auto* many) {
    if (pool.count == 1)
      one<<<pool.max_items, block, kTileLds, stream>>>(args, pool.inst, pool.params);
    else
      many<<<pool.max_items, block, kTileLds, stream>>>(args, pool.inst, pool.params);
  };
  auto storage = [&](auto s_tag) {
    constexpr int S = decltype(s_tag)::value;
    if (pool.pos64)
      go(agents_tiled_kernel<S, true, true>, agents_tiled_kernel<S, true, false>);
    else
      go(agents_tiled_kernel<S, false, true>, agents_tiled_kernel<S, false, false>);
  };
  switch (pool.storage) {
    case SLM_STORAGE_BF16:
      storage(std::integral_constant<int, SLM_STORAGE_BF16>{});
      break;
    case SLM_STORAGE_F16:
      storage(std::integral_constant<int, SLM_STORAGE_F16>{});
      break;
    default:
      storage(std::integral_constant<int, SLM_STORAGE_F32>{});
      break;
  }
}

void launch_init_agents(const Instance& in, const AgentSoA& a, int pos64, uint64_t seed,
                        float speed_min, float speed_max, hipStream_t stream) {
  if (in.agent_count == 0) return;
  float range = speed_max - speed_min;
  init_agents_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, pos64, seed, static_cast<float>(in.width),
      static_cast<float>(in.height), speed_min, range);
}

void launch_reassign_speeds(const Instance& in, const AgentSoA& a, uint64_t stream_seed,
                            float speed_min, float speed_max, hipStream_t stream) {
  if (in.agent_count == 0) return;
  float range = speed_max - speed_min;
  reassign_speeds_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, stream_seed, speed_min, range);
}

void launch_scale_positions(const Instance& in, const AgentSoA& a, int pos64, float sx, float sy,
                            hipStream_t stream) {
  if (in.agent_count == 0) return;
  scale_positions_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, pos64, sx, sy);
}

void launch_pack_agents(const Instance& in, const AgentSoA& a, int pos64, float* aos,
                        hipStream_t stream) {
  if (in.agent_count == 0) return;
  pack_agents_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, pos64, reinterpret_cast<float4*>(aos));
}

void launch_unpack_agents(const Instance& in, const AgentSoA& a, int pos64, const float* aos,
                          hipStream_t stream) {
  if (in.agent_count == 0) return;
  unpack_agents_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, pos64, reinterpret_cast<const float4*>(aos));
}

void launch_pack_positions64(const Instance& in, const AgentSoA& a, double* xy,
                             hipStream_t stream) {
  if (in.agent_count == 0) return;
  pack_positions64_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, reinterpret_cast<double2*>(xy));
}

void launch_unpack_positions64(const Instance& in, const AgentSoA& a, const double* xy,
                               hipStream_t stream) {
  if (in.agent_count == 0) return;
  unpack_positions64_kernel<<<blocks_for(in.agent_count, 256), 256, 0, stream>>>(
      a, in.agent_off, in.agent_count, reinterpret_cast<const double2*>(xy));
}

}  // namespace slm
