// Many ticks of a small network in one launch (gfx950).
//
// A tick of a network of a thousand neurons is one launch of a few microseconds
// that the next tick waits for: as graph nodes, N=1024, M=16k, B=4 took 5.0 us per
// tick, plus 1.7 for a node that copied the new state into the caller's trace.
// Columns do not interact, and such a network's edges fit the registers of one
// compute unit.  So each column gets one 1024-lane workgroup for all the ticks: it
// decodes its edges into registers once (source offset in LDS, float32 weight),
// keeps s in LDS and d and a in registers, and needs only two workgroup barriers
// per tick, between the gathers and the update and between the update and the
// next tick's gathers.  The trace is written by the update.
//
// The row sums are those of the row-block tick, bit for bit: the host lays the
// rows out as tasks with the slices that kernel would use (ns_rollout), each
// lane adds its products to the same four running sums, and a row's lanes combine
// by the same xor butterfly.  That kernel feeds whole quads of a lane's edges to
// the four sums and the one to three edges left to the first; here the quads of a
// chunk come first and its lanes' leftovers share one last unit, so no lane
// selects.  (The sums start at +0 and so are never -0: adding a padding slot's
// zero changes nothing.)
//
// A tick is bound by the vector ALU of the one compute unit: a multiply and an add
// per slot (a fused one would round differently) and about 110 instructions per
// neuron, two tanhf among them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ns_common.h"
#include "ns_host.h"

namespace ns {

int check_step_head(const ns_step_args& a);

namespace {

constexpr int kRolloutWaves = 16;
constexpr int kRolloutThreads = kRolloutWaves * 64;
static_assert(NS_ROLLOUT_MAX_NEURONS <= 2 * kRolloutThreads, "at most two neurons per lane");

struct RolloutArgs {
  int64_t N;
  Plane s, d, a, u, v;
  int64_t u_tick, v_tick;
  Params p;
  const int32_t* col;
  const void* weight;
  const uint8_t* scales;
  const float* gscale;
  int64_t M;
  OutPlane os, od, oa, trace;
  int64_t trace_tick;
  const int32_t* tasks;
  const int32_t* rounds;
  int32_t n_rounds, ticks;
};

// A plane's element behind `at`, or its scalar.
__device__ __forceinline__ float blend(const Plane& p, const float* at) {
  const uint32_t x = __builtin_bit_cast(uint32_t, *at);
  return __builtin_bit_cast(float,
                            (x & p.mask) | (__builtin_bit_cast(uint32_t, p.scalar) & ~p.mask));
}

template <int kControl>
__device__ __forceinline__ float add_dpp(float x) {
  const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), kControl, 0xF, 0xF, true);
  return x + __builtin_bit_cast(float, y);
}

// The xor butterfly's sum over 2^log2 neighbouring lanes.  Below 16 lanes each
// step's partner sits in another half whose lanes all hold the same sum already, so
// a mirror within 8 or 16 lanes reads the same value as the xor would.
__device__ __forceinline__ float slice_sum(float x, int log2) {
  if (log2 > 0) x = add_dpp<0xB1>(x);    // quad_perm 1 0 3 2
  if (log2 > 1) x = add_dpp<0x4E>(x);    // quad_perm 2 3 0 1
  if (log2 > 2) x = add_dpp<0x141>(x);   // row_half_mirror
  if (log2 > 3) x = add_dpp<0x140>(x);   // row_mirror
  if (log2 > 4) x += __shfl_xor(x, 16, 64);
  if (log2 > 5) x += __shfl_xor(x, 32, 64);
  return x;
}

// kSlots edges per lane in registers, kOwn neurons per lane in the update (us per
// tick with staged drives and trace, this launch / graph nodes: N=256, 4k edges,
// B=1 0.8 / 5.6; N=1024, 16k, B=4 2.1 / 6.7, B=256 2.5 / 25; N=1024, 35k, B=2
// 3.6 / 6.9; N=2048, 16k, B=4 2.8 / 6.6).  At one
// neuron per lane d and a stay in registers too, and the parameters where 48 edges
// leave room (128 registers per lane at 16 wavefronts); else d and a are in LDS.
// LDS: s (N + 1 floats, the last one zero for padding slots), j, d and a (N floats
// each), and per round and lane the row whose sum the lane stores (negative: none).
template <int kSlots, int kOwn, int FMT>
__global__ __launch_bounds__(kRolloutThreads) void rollout_kernel(RolloutArgs A) {
#pragma clang fp contract(off)
  extern __shared__ float lds[];
  constexpr int kUnits = kSlots / 4;
  const int N = static_cast<int>(A.N);
  float* const s_lds = lds;
  float* const j_lds = lds + N + 1;
  float* const d_lds = lds + 2 * N + 1;
  float* const a_lds = lds + 3 * N + 1;
  int32_t* const meta = reinterpret_cast<int32_t*>(lds + 4 * N + 1);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t b = blockIdx.x;
  const float gscale = (FMT == NS_WEIGHT_E4M3 || FMT == NS_WEIGHT_NVFP4) ? *A.gscale : 1.0f;
  const int32_t* const rounds = A.rounds + wave * A.n_rounds;

  // The lane's edges: byte offsets into s (two per word at 48 slots) and weights.
  // Slots without an edge point at the zero behind s and weigh nothing.  A unit is
  // four slots: a quad of edges, or a chunk's leftovers (kTail, at most three).
  constexpr bool kPacked = kSlots == 48;
  const uint32_t zero = static_cast<uint32_t>(N) * 4u;
  uint32_t off[kPacked ? kSlots / 2 : kSlots];
  float w[kSlots];
#pragma unroll
  for (int k = 0; k < (kPacked ? kSlots / 2 : kSlots); ++k)
    off[k] = kPacked ? zero | (zero << 16) : zero;
#pragma unroll
  for (int k = 0; k < kSlots; ++k) w[k] = 0.0f;
  // Per wavefront: units in use, the units that end a round and those that are a
  // tail (a bit each), and log2 slices of each round (4 bits).
  int total = 0;
  uint32_t ends = 0, tails = 0, log2s = 0;
  {
    int r = -1, left = 0, at = 0, slices_log2 = 0, first = 0, count = 0;
    bool tail = false;
#pragma unroll
    for (int q = 0; q < kUnits; ++q) {
      if (left == 0 && r + 1 < A.n_rounds) {
        const uint32_t round = static_cast<uint32_t>(rounds[r + 1]);
        if ((round & 0xFFFFu) != 0) {
          ++r;
          left = static_cast<int>(round & 0xFFFFu);
          at = 0;
          tail = (round >> 31) != 0;
          slices_log2 = static_cast<int>((round >> 16) & 7u);
          log2s |= static_cast<uint32_t>(slices_log2) << (4 * r);
          const int32_t* const task = A.tasks + (static_cast<int64_t>(wave) * A.n_rounds + r) * 128 +
                                      lane * 2;
          first = task[0];
          const uint32_t word = static_cast<uint32_t>(task[1]);
          count = static_cast<int>(word & 0xFFFFu);
          const uint32_t row = word >> 16;
          const bool leads = row < static_cast<uint32_t>(N) &&
                             (lane & ((1 << slices_log2) - 1)) == 0;
          meta[r * kRolloutThreads + tid] = leads ? static_cast<int32_t>(row) : -1;
        }
      }
      if (left > 0) {
        const bool leftovers = tail && left == 1;
        // A quad takes the lane's edges 4 at .. 4 at + 3 if it has all four, the
        // tail those behind its whole quads.
        const int from = leftovers ? count & ~3 : 4 * at;
        const int until = leftovers ? count : (4 * at + 4 <= count ? 4 * at + 4 : 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int64_t e = first + (static_cast<int64_t>(from + k) << slices_log2);
          if (from + k < until && e >= 0 && e < A.M) {
            const uint32_t c = static_cast<uint32_t>(A.col[e]);
            const uint32_t o = (c < static_cast<uint32_t>(N) ? c : static_cast<uint32_t>(N)) * 4u;
            const int slot = 4 * q + k;
            if (!kPacked) off[slot] = o;
            else if (slot & 1) off[slot / 2] = (off[slot / 2] & 0xFFFFu) | (o << 16);
            else off[slot / 2] = (off[slot / 2] & 0xFFFF0000u) | o;
            w[slot] = csr_weight<FMT>(A.weight, A.scales, e, gscale);
          }
        }
        total = q + 1;
        if (leftovers) tails |= 1u << q;
        if (--left == 0) ends |= 1u << q;
        ++at;
      }
    }
  }

  // The lane's neurons: tid, tid + 1024.
  constexpr bool kStateRegs = kOwn == 1, kParamRegs = kOwn == 1 && kSlots < 48;
  float d_reg = 0.0f, a_reg = 0.0f;
  NeuronParams prm{};
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    const int n = tid + i * kRolloutThreads;
    if (n < N) {
      s_lds[n] = A.s.get(b, n);
      const float d = A.d.get(b, n), a = A.a.get(b, n);
      if (kStateRegs) {
        d_reg = d;
        a_reg = a;
      } else {
        d_lds[n] = d;
        a_lds[n] = a;
      }
    }
  }
  if (kParamRegs && tid < N) prm = load_params(A.p, tid);
  if (tid == 0) s_lds[N] = 0.0f;
  __syncthreads();

  const char* const s_bytes = reinterpret_cast<const char*>(s_lds);
  const auto read_unit = [&](int q, float out[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int slot = 4 * q + k;
      const uint32_t o = !kPacked ? off[slot]
                         : (slot & 1) ? off[slot / 2] >> 16 : off[slot / 2] & 0xFFFFu;
      out[k] = *reinterpret_cast<const float*>(s_bytes + o);
    }
  };
  // Walking pointers to the lane's first neuron (clamped into the planes).
  const int own = tid < N ? tid : 0;
  const float* u_at = A.u.data + b * A.u.sb + own * A.u.sn;
  const float* v_at = A.v.data + b * A.v.sb + own * A.v.sn;
  float* trace_at = A.trace.data ? A.trace.data + b * A.trace.sb + own * A.trace.sn : nullptr;
  for (int t = 0; t < A.ticks; ++t) {
    // The update's drives load while the sums are gathered.
    float u[kOwn], v[kOwn];
    u[0] = blend(A.u, u_at);
    v[0] = blend(A.v, v_at);
#pragma unroll
    for (int i = 1; i < kOwn; ++i) {
      u[i] = v[i] = 0.0f;
      if (tid + i * kRolloutThreads < N) {
        u[i] = blend(A.u, u_at + i * kRolloutThreads * A.u.sn);
        v[i] = blend(A.v, v_at + i * kRolloutThreads * A.v.sn);
      }
    }
    u_at += A.u_tick;
    v_at += A.v_tick;
    const int32_t* row_at = meta + tid;
    uint32_t log2_left = log2s;
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
    // The states of the next unit's sources are read while a unit is summed (at 48
    // slots the registers for that are not there).
    constexpr bool kAhead = !kPacked;
    float x[4], next[4];
    if (kAhead) read_unit(0, x);
#pragma unroll
    for (int q = 0; q < kUnits; ++q) {
      if (q < total) {
        if (!kAhead) read_unit(q, x);
        else if (q + 1 < kUnits) read_unit(q + 1, next);
        const float v0 = w[4 * q] * x[0], v1 = w[4 * q + 1] * x[1], v2 = w[4 * q + 2] * x[2];
        if ((tails >> q) & 1u) {
          a0 += v0;
          a0 += v1;
          a0 += v2;
        } else {
          const float v3 = w[4 * q + 3] * x[3];
          a0 += v0;
          a1 += v1;
          a2 += v2;
          a3 += v3;
        }
        if ((ends >> q) & 1u) {
          const float sum = slice_sum((a0 + a1) + (a2 + a3), static_cast<int>(log2_left & 7u));
          const int32_t row = *row_at;
          if (row >= 0) j_lds[row] = sum;
          a0 = a1 = a2 = a3 = 0.0f;
          row_at += kRolloutThreads;
          log2_left >>= 4;
        }
        if (kAhead && q + 1 < kUnits) {
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = next[k];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int n = tid + i * kRolloutThreads;
      if (n < N) {
        const NeuronParams p = kParamRegs ? prm : load_params(A.p, n);
        const NextState x = advance_loaded(p, j_lds[n], s_lds[n], kStateRegs ? d_reg : d_lds[n],
                                           kStateRegs ? a_reg : a_lds[n], u[i], v[i]);
        s_lds[n] = x.soma;
        if (kStateRegs) {
          d_reg = x.dendrite;
          a_reg = x.adaptation;
        } else {
          d_lds[n] = x.dendrite;
          a_lds[n] = x.adaptation;
        }
        if (trace_at) trace_at[i * kRolloutThreads * A.trace.sn] = x.soma;
      }
    }
    if (trace_at) trace_at += A.trace_tick;
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    const int n = tid + i * kRolloutThreads;
    if (n < N) {
      A.os.put(b, n, s_lds[n]);
      A.od.put(b, n, kStateRegs ? d_reg : d_lds[n]);
      A.oa.put(b, n, kStateRegs ? a_reg : a_lds[n]);
    }
  }
}

template <int kSlots, int kOwn>
hipError_t launch_format(const RolloutArgs& A, int fmt, unsigned batch, unsigned lds,
                         hipStream_t stream) {
  const dim3 grid(batch), block(kRolloutThreads);
  switch (fmt) {
    case NS_WEIGHT_F32:
      rollout_kernel<kSlots, kOwn, NS_WEIGHT_F32><<<grid, block, lds, stream>>>(A); break;
    case NS_WEIGHT_F16:
      rollout_kernel<kSlots, kOwn, NS_WEIGHT_F16><<<grid, block, lds, stream>>>(A); break;
    case NS_WEIGHT_E4M3:
      rollout_kernel<kSlots, kOwn, NS_WEIGHT_E4M3><<<grid, block, lds, stream>>>(A); break;
    default:
      rollout_kernel<kSlots, kOwn, NS_WEIGHT_NVFP4><<<grid, block, lds, stream>>>(A);
  }
  return hipGetLastError();
}

template <int kSlots>
hipError_t launch_own(const RolloutArgs& A, int fmt, unsigned batch, unsigned lds,
                      hipStream_t stream) {
  if (A.N <= kRolloutThreads) return launch_format<kSlots, 1>(A, fmt, batch, lds, stream);
  return launch_format<kSlots, 2>(A, fmt, batch, lds, stream);
}

bool same_plane(const ns_plane& in, const ns_out_plane& out) {
  return in.data == out.data && in.stride_b == out.stride_b && in.stride_n == out.stride_n;
}

}  // namespace

int rollout_step(const ns_step_args& a, hipStream_t stream) {
  const ns_rollout& r = *a.rollout;
  const int64_t n = a.n_neurons, batch = a.batch;
  if (a.panels) return fail("a rollout launch takes no panel layout");
  if (n > NS_ROLLOUT_MAX_NEURONS)
    return fail("a rollout launch takes at most %d neurons", NS_ROLLOUT_MAX_NEURONS);
  if (r.ticks <= 0) return fail("a rollout launch needs at least one tick");
  if (r.slots != 16 && r.slots != 32 && r.slots != 48)
    return fail("a rollout lane holds 16, 32 or 48 edges, not %d", r.slots);
  if (r.slots == 48 && n > kRolloutThreads)
    return fail("a rollout of more than %d neurons holds 16 or 32 edges per lane", kRolloutThreads);
  if (r.n_rounds < 1 || r.n_rounds > NS_ROLLOUT_MAX_ROUNDS)
    return fail("a rollout plan has 1 to %d rounds", NS_ROLLOUT_MAX_ROUNDS);
  if (!r.tasks || !r.rounds) return fail("a rollout plan needs tasks and rounds");
  if (batch == 0) return NS_OK;  // empty planes may carry null pointers
  if (batch > 0x7FFFFFFF) return fail("too many columns for one rollout launch");
  if (!a.state.data || !a.dendrite.data || !a.adaptation.data)
    return fail("state, dendrite and adaptation data are required");
  if (!a.out_state.data || !a.out_dendrite.data || !a.out_adaptation.data)
    return fail("three output planes are required");
  if (a.out_current.data) return fail("a rollout launch writes no current");
  const ns_plane ins[3] = {a.state, a.dendrite, a.adaptation};
  const ns_out_plane outs[4] = {a.out_state, a.out_dendrite, a.out_adaptation, r.trace};
  // The trace and the drives span every tick's plane.
  auto span = [&](const void* data, int64_t sb, int64_t sn, int64_t tick) {
    Extent x = extent_of(data, sb, sn, batch, n);
    if (x.hi != x.lo) x.hi += 4 * (r.ticks - 1) * (tick < 0 ? -tick : tick);
    return x;
  };
  const Extent drives[2] = {
      span(a.drive.data, a.drive.stride_b, a.drive.stride_n, r.drive_tick),
      span(a.dendritic_drive.data, a.dendritic_drive.stride_b, a.dendritic_drive.stride_n,
           r.dendritic_tick)};
  if (r.drive_tick < 0 || r.dendritic_tick < 0 || r.trace_tick < 0)
    return fail("a rollout's tick strides must not be negative");
  for (int o = 0; o < 4; ++o) {
    if (!outs[o].data) continue;
    if (!distinct_elements(outs[o].stride_b, outs[o].stride_n, batch, n))
      return fail("a rollout's output planes must not overlap themselves");
    const Extent out = span(outs[o].data, outs[o].stride_b, outs[o].stride_n,
                            o == 3 ? r.trace_tick : 0);
    for (int i = 0; i < 3; ++i)
      if (!(i == o && same_plane(ins[i], outs[o])) && overlaps(out, extent(ins[i], batch, n)))
        return fail("output planes must not overlap inputs");
    for (const Extent& drive : drives)
      if (overlaps(out, drive)) return fail("output planes must not overlap inputs");
    for (int p = o + 1; p < 4; ++p)
      if (overlaps(out, span(outs[p].data, outs[p].stride_b, outs[p].stride_n,
                             p == 3 ? r.trace_tick : 0)))
        return fail("output planes must not overlap each other");
  }

  RolloutArgs A{};
  A.N = n; A.M = a.matrix.n_edges;
  A.s = plane(a.state, a.state.data); A.d = plane(a.dendrite, a.state.data);
  A.a = plane(a.adaptation, a.state.data);
  A.u = plane(a.drive, a.state.data); A.v = plane(a.dendritic_drive, a.state.data);
  A.u_tick = a.drive.data ? r.drive_tick : 0;
  A.v_tick = a.dendritic_drive.data ? r.dendritic_tick : 0;
  for (int i = 0; i < 6; ++i) A.p.v[i] = Vec{a.params[i].data, a.params[i].stride};
  A.col = a.matrix.col; A.weight = a.matrix.weight;
  A.scales = a.matrix.block_scales; A.gscale = a.matrix.global_scale;
  A.os = out_plane(a.out_state); A.od = out_plane(a.out_dendrite);
  A.oa = out_plane(a.out_adaptation); A.trace = out_plane(r.trace);
  A.trace_tick = r.trace_tick;
  A.tasks = r.tasks; A.rounds = r.rounds;
  A.n_rounds = r.n_rounds; A.ticks = r.ticks;
  const unsigned lds = static_cast<unsigned>(4 * (4 * n + 1) + 4 * kRolloutThreads * r.n_rounds);
  hipError_t err;
  switch (r.slots) {
    case 16: err = launch_own<16>(A, a.matrix.format, static_cast<unsigned>(batch), lds, stream); break;
    case 32: err = launch_own<32>(A, a.matrix.format, static_cast<unsigned>(batch), lds, stream); break;
    default: err = launch_format<48, 1>(A, a.matrix.format, static_cast<unsigned>(batch), lds, stream);
  }
  return err == hipSuccess ? NS_OK : fail_launch("rollout", err);
}

}  // namespace ns
