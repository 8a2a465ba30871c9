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
// by the same xor butterfly.
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

__device__ __forceinline__ float plane_at(const Plane& p, int64_t at) {
  const uint32_t x = __builtin_bit_cast(uint32_t, p.data[at]);
  return __builtin_bit_cast(float,
                            (x & p.mask) | (__builtin_bit_cast(uint32_t, p.scalar) & ~p.mask));
}

// kSlots edges per lane in registers, kOwn neurons per lane in the update.  At one
// neuron per lane d and a stay in registers too, and the parameters where 48 edges
// leave room (128 registers per lane at 16 wavefronts); else d and a are in LDS.
// LDS: s (N + 1 floats, the last one zero for padding slots), j, d and a (N floats
// each), and per round and lane a word: row (low 16 bits), full quads (bits
// 16-30), bit 31 set on the lane that stores the row's sum.
template <int kSlots, int kOwn, int FMT>
__global__ __launch_bounds__(kRolloutThreads) void rollout_kernel(RolloutArgs A) {
#pragma clang fp contract(off)
  extern __shared__ float lds[];
  constexpr int kQuads = kSlots / 4;
  const int N = static_cast<int>(A.N);
  float* const s_lds = lds;
  float* const j_lds = lds + N + 1;
  float* const d_lds = lds + 2 * N + 1;
  float* const a_lds = lds + 3 * N + 1;
  uint32_t* const meta = reinterpret_cast<uint32_t*>(lds + 4 * N + 1);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t b = blockIdx.x;
  const float gscale = (FMT == NS_WEIGHT_E4M3 || FMT == NS_WEIGHT_NVFP4) ? *A.gscale : 1.0f;
  const int32_t* const rounds = A.rounds + wave * A.n_rounds;

  // The lane's edges: byte offsets into s (two per word) and weights.  Slots
  // without an edge point at the zero behind s and weigh nothing.
  const uint32_t zero = static_cast<uint32_t>(N) * 4u;
  uint32_t off[kSlots / 2];
  float w[kSlots];
#pragma unroll
  for (int k = 0; k < kSlots / 2; ++k) off[k] = zero | (zero << 16);
#pragma unroll
  for (int k = 0; k < kSlots; ++k) w[k] = 0.0f;
  int total = 0;
  {
    int r = -1, left = 0, at = 0, slices_log2 = 0, first = 0, count = 0;
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      if (left == 0 && r + 1 < A.n_rounds) {
        const int32_t round = rounds[r + 1];
        if ((round & 0xFFFF) != 0) {
          ++r;
          left = round & 0xFFFF;
          at = 0;
          slices_log2 = round >> 16;
          const int32_t* const task = A.tasks + (static_cast<int64_t>(wave) * A.n_rounds + r) * 128 +
                                      lane * 2;
          first = task[0];
          const uint32_t word = static_cast<uint32_t>(task[1]);
          count = static_cast<int>(word & 0xFFFFu);
          const uint32_t row = word >> 16;
          const bool leads = row < static_cast<uint32_t>(N) &&
                             (lane & ((1 << slices_log2) - 1)) == 0;
          meta[r * kRolloutThreads + tid] =
              (leads ? row | 0x80000000u : 0u) | (static_cast<uint32_t>(count >> 2) << 16);
        }
      }
      if (left > 0) {
        ++total;
        --left;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int64_t e = first + (static_cast<int64_t>(4 * at + k) << slices_log2);
          if (4 * at + k < count && e >= 0 && e < A.M) {
            const uint32_t c = static_cast<uint32_t>(A.col[e]);
            const uint32_t o = (c < static_cast<uint32_t>(N) ? c : static_cast<uint32_t>(N)) * 4u;
            const int slot = 4 * q + k;
            off[slot / 2] = (slot & 1) ? (off[slot / 2] & 0xFFFFu) | (o << 16)
                                       : (off[slot / 2] & 0xFFFF0000u) | o;
            w[slot] = csr_weight<FMT>(A.weight, A.scales, e, gscale);
          }
        }
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
  for (int t = 0; t < A.ticks; ++t) {
    // The update's drives load while the sums are gathered.
    float u[kOwn], v[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int n = tid + i * kRolloutThreads;
      u[i] = v[i] = 0.0f;
      if (n < N) {
        u[i] = plane_at(A.u, b * A.u.sb + n * A.u.sn + t * A.u_tick);
        v[i] = plane_at(A.v, b * A.v.sb + n * A.v.sn + t * A.v_tick);
      }
    }
    int r = 0, left = rounds[0] & 0xFFFF, at = 0;
    uint32_t word = total > 0 ? meta[tid] : 0u;
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      if (q < total) {
        const uint32_t o01 = off[2 * q], o23 = off[2 * q + 1];
        const float v0 = w[4 * q] * *reinterpret_cast<const float*>(s_bytes + (o01 & 0xFFFFu));
        const float v1 = w[4 * q + 1] * *reinterpret_cast<const float*>(s_bytes + (o01 >> 16));
        const float v2 = w[4 * q + 2] * *reinterpret_cast<const float*>(s_bytes + (o23 & 0xFFFFu));
        const float v3 = w[4 * q + 3] * *reinterpret_cast<const float*>(s_bytes + (o23 >> 16));
        // A full quad feeds the four running sums, the tail the first one (the
        // sums start at +0 and so are never -0: adding a padding slot's zero
        // changes nothing).
        const bool full = at < static_cast<int>((word >> 16) & 0x7FFFu);
        a0 += v0;
        a0 += full ? 0.0f : v1;
        a0 += full ? 0.0f : v2;
        a1 += full ? v1 : 0.0f;
        a2 += full ? v2 : 0.0f;
        a3 += full ? v3 : 0.0f;
        ++at;
        if (--left == 0) {
          const int lanes = 1 << (rounds[r] >> 16);
          float acc = (a0 + a1) + (a2 + a3);
          for (int x = 1; x < lanes; x <<= 1) acc += __shfl_xor(acc, x, 64);
          if (word >> 31) j_lds[word & 0xFFFFu] = acc;
          a0 = a1 = a2 = a3 = 0.0f;
          at = 0;
          ++r;
          if (q + 1 < total) {
            left = rounds[r] & 0xFFFF;
            word = meta[r * kRolloutThreads + tid];
          }
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
        if (A.trace.data)
          A.trace.data[t * A.trace_tick + b * A.trace.sb + n * A.trace.sn] = x.soma;
      }
    }
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
    default: err = launch_own<48>(A, a.matrix.format, static_cast<unsigned>(batch), lds, stream);
  }
  return err == hipSuccess ? NS_OK : fail_launch("rollout", err);
}

}  // namespace ns
