// Fused cyclic convolution at N = 32768 in one launch (gfx950).
//
// The reference runs a single-block conv up to N = 4096 and goes four-step
// beyond (run_large, bench_fufft.cu:357-492: 56 bytes per point over HBM).  A
// CU of MI355X holds 512 KiB of VGPRs, so one workgroup of 1024 lanes keeps a
// whole 32768-point transform in registers, 32 values per lane, and the conv
// becomes the radix-16 plan of the single-launch kernels, LEAD 8 then three
// radix-16 passes (the plan fufft_pipeline_v16 would run at this N,
// fufft.cuh:722-800), with each lane doing the work of two radix-16 lanes:
// groups L and L + T of every radix-16 pass (T = 1024 lanes), four groups of
// the radix-8 lead pass.  The arithmetic per group is the radix-16 kernels'
// own (compute_pass, the reference's butterflies and twiddle chains), so the
// result is bit for bit that plan's and the filter is the radix-16 plan's: in
// digit order, lane-major pairs or bperm, as fufft_plan_filter_f32 writes them
// for (32768, FUFFT_V16).  The signal crosses HBM twice (16 bytes per point),
// the filter once per launch when shared.
//
// The exchanges.  A complex exchange of 32768 points needs 256 KiB, beyond
// the CU's 160 KiB of LDS.  After a pass, though, every group of the next one
// lies in the lower or the upper half of the positions, so each exchange runs
// in two rounds of whole complex values, one half of the positions each, through
// one buffer of N/2 + N/32 slots (136 KiB), and a half's butterflies run while
// the LDS serves the other half (half_exchange).  One workgroup fills a CU, so
// nothing else hides those accesses.  Before, the rounds were the real and the
// imaginary parts, with no arithmetic between them.  (The halves' twiddle chains are
// the same values, and the compiler computes them once.)  us, parts -> halves, three states in turn:
// N = 32768, 1000 signals: lane-major 178 -> 170, digit order 192 -> 179, one filter per
// signal 186 -> 178 / 202 -> 184, four-step 191 -> 174, 1 signal 33.6 -> 30.8; N = 16384
// lane-major, 1 17.6 -> 16.8, 2000 137 -> 133.
//
// Races.  A lane's groups of the two halves use the same slots, so the last read
// of one exchange and the first write of the next, both of one pass, touch the
// lane's own slots and need no barrier between them; a pass inside each wavefront
// may switch layouts but stays in its wavefront's own slot range (the layouts
// below), and a wavefront fence keeps its accesses in order.  The three barriers of
// an exchange separate write from read within a round and the two rounds from
// each other.  Every wavefront of the workgroup reaches every barrier (one
// transform per workgroup, the whole group leaves together).
//
// Resources: 128 VGPRs with no scratch (16 wavefronts of 1024 lanes, 4 per
// SIMD), 136 KiB of LDS: one workgroup per CU.
//
// The four-step chain at N = 32768 (CHAIN: radix 16 with the single twiddle
// chain, then LEAD 8 and two radix-16 passes) is the same kernel with its passes
// in that order, for a filter in the chain order: one read and one write of the
// data where fufft_conv_large_f32's three launches make three of each.  1000
// transforms 244 us in three launches, 174 here; which batches take it is
// chain_batch's choice (fufft_internal.hpp).
//
// N = 16384 runs the same code with 512 lanes (LEAD 4, eight groups per lane
// in the lead pass): 68 KiB of LDS, so two workgroups share a CU and one's
// loads overlap the other's passes.  fufft_conv_f32 takes it for a shared
// lane-major filter (+2.8% over the workgroup kernel, bit-identical).
#include "fufft_device.hpp"
#include "fufft_plan.hpp"
#include "fufft_internal.hpp"

namespace fufft {

namespace {

template<int N, bool CHAIN = false>
using WPlan = Plan<N, 32, 16, CHAIN>;

// Slot layouts of one half's positions, 8-byte slots.  gfx950 serves ds_read_b64 32
// lanes at a time over 32 slot residues, ds_write_b64 and each access of the
// paired forms 16 lanes over 16.
//  - Pad16, i + i/16: 17 slots per lane at M = 1 and 272 per 16 lanes at
//    M = 16, both conflict free; a run of 32 consecutive positions (the
//    M >= 64 passes) spans 33 slots, and a ds_read_b64 of it costs 2 cycles.
//  - Pad256, i + 16*(i/256): 32-runs stay contiguous, and the M = 16 pass's
//    two 16-runs per half-wavefront land 16 residues apart: conflict free for
//    the passes at M >= 16, not at M = 1.
// Each exchange takes the layout its two passes need (Pad256 for the ones
// between the M >= 16 passes, Pad16 for the private one into M = 1).  Both put
// the 1024-aligned block c of positions inside slots [1088c, 1088c + 1088),
// so a private pass that reads one layout and writes the other stays inside
// its wavefront's own slot range; both are additive over every pass's taps
// (base + k*M).
struct Pad16 {
   __device__ __forceinline__ static int phys(int i) { return i + (i >> 4); }
   static constexpr int cphys(int i) { return i + (i >> 4); }
   static constexpr int size(int n) { return n + n / 16; }
};
struct Pad256 {
   __device__ __forceinline__ static int phys(int i) { return i + ((i >> 8) << 4); }
   static constexpr int cphys(int i) { return i + ((i >> 8) << 4); }
   static constexpr int size(int n) { return n + n / 16; }
};
static_assert(Pad16::size(CONV_WIDE_N / 2) == Pad256::size(CONV_WIDE_N / 2) && Pad16::size(8192) == Pad256::size(8192),
              "one buffer for both layouts");

// An exchange between passes P and P + 1 stays inside each wavefront when
// both run at M <= 64 with the same radix R: for every group g, wavefront w's
// 64 lanes then own positions [(64w + g*T)*R, (64w + g*T + 64)*R) on both
// sides, and the slots of those positions (a monotonic map) no other
// wavefront's.  Here: the exchange between the last two radix-16 passes (M =
// 16 and 1).  It takes wavefront fences instead of workgroup barriers, 6 of
// the 18 barriers of a transform.
template<class PL, int P>
constexpr bool exchange_private()
{
   return PL::stride(P) <= 64 && PL::stride(P + 1) <= 64 && PL::radix(P) == PL::radix(P + 1);
}

template<bool PRIVATE>
__device__ __forceinline__ void exchange_fence()
{
   if constexpr(PRIVATE) pass_barrier<64>();
   else                  __syncthreads();
}

// Half h of a pass is an array of V / 2 values: tap k of group g at g + k * groups,
// groups = V / (2 R), except pass 0, whose groups have their taps in both halves:
// tap k of group g at g + k * V / R, the lower taps first.  A position of the upper
// half uses the slot of the one N / 2 below it: a lane's upper groups (pass 0: taps)
// have the slots of its lower ones, so both halves are addressed alike.
template<class PL, int P, bool OUT, class FL>
__device__ __forceinline__ void half_io(float2 (&r)[PL::V / 2], float2* A, int L)
{
   constexpr int R = PL::radix(P), M = PL::stride(P);
   constexpr int G = P == 0 ? PL::V / R : PL::V / R / 2, K = P == 0 ? R / 2 : R;
   static_assert(P == 0 ? R / 2 * M == PL::N / 2 : PL::T * (PL::V / R / 2) % M == 0, "halves share slots");
#pragma unroll
   for(int g = 0; g < G; g++) {
      const int bp = FL::phys(tap_pos<PL, P>(L, g, 0));
#pragma unroll
      for(int k = 0; k < K; k++) {
         if constexpr(OUT) A[bp + FL::cphys(k * M)] = r[g + k * G];
         else              r[g + k * G] = A[bp + FL::cphys(k * M)];
      }
   }
}

// butterflies and twiddles of a half's groups (P > 0): compute_pass on V / (2 R)
// groups, which share one W^j
template<class PL, int P, int SIGN, bool DIT>
__device__ __forceinline__ void half_pass(float2 (&r)[PL::V / 2], const Twiddles<PL>& tw)
{
   constexpr int R = PL::radix(P), M = PL::stride(P), G = PL::V / R / 2;
   static_assert(P > 0 && Twiddles<PL>::distinct(P) == 1, "one base twiddle");
   float2 w1{};
   if constexpr(M > 1) {
      const float2 b = tw.w[Twiddles<PL>::slots_before(P)];
      w1 = SIGN < 0 ? make_float2(b.x, -b.y) : b;
   }
   if constexpr(DIT && M > 1) twiddle_group<R, CHAIN_EVENODD, 0, G, G>(r, w1);
   static_for<G>([&](auto gi) { dftR<R, SIGN, decltype(gi)::value, G>(r); });
   if constexpr(!DIT && M > 1) twiddle_group<R, CHAIN_EVENODD, 0, G, G>(r, w1);
}

// From pass PS, lower half computed (pass 0: both), to pass PG, its lower half
// computed (pass 0: neither).  The reads are issued before a half's butterflies and
// awaited after them.
template<class PL, int PS, int PG, int SIGN, bool DIT>
__device__ __forceinline__ void half_exchange(float2 (&lo)[PL::V / 2], float2 (&hi)[PL::V / 2], float2* A, int L,
                                              const Twiddles<PL>& tw)
{
   constexpr bool PRIVATE = exchange_private<PL, (PS < PG ? PS : PG)>();
   using FL = typename std::conditional<PRIVATE, Pad16, Pad256>::type;
   if constexpr(PL::stride(PS) <= 64) exchange_fence<true>();
   half_io<PL, PS, true, FL>(lo, A, L);
   exchange_fence<PRIVATE>();
   half_io<PL, PG, false, FL>(lo, A, L);
   if constexpr(PS > 0) half_pass<PL, PS, SIGN, DIT>(hi, tw);
   exchange_fence<PRIVATE>();
   half_io<PL, PS, true, FL>(hi, A, L);
   exchange_fence<PRIVATE>();
   half_io<PL, PG, false, FL>(hi, A, L);
   if constexpr(PG > 0) half_pass<PL, PG, SIGN, DIT>(lo, tw);
}

// The mid operation of half H.  After the forward DIF value k of half H of lane L
// is digit-order slot (L + H*T)*16 + k, i.e. slot 16*L' + k of radix-16 lane
// L' = L + H*T (of T16 = N/16), so the filter is read where the radix-16
// plan's lane L' reads it: 16 contiguous slots in digit order, pairs at
// 2(L' + m*T16) lane-major, slot 16L' + k at L' + k*T16 in bperm.  The layout
// is a template parameter: a run-time branch kept both sides' registers live
// and spilled.  FLY: the slots whose loads are in flight (the empty asm orders each
// step after the last); all 16 at once pushed the kernel past 128 VGPRs into scratch.
template<class PL, int MID, int FLT, int H>
__device__ __forceinline__ void half_mid(float2 (&r)[PL::V / 2], const Buf& fb, uint32_t fb0, int L)
{
   using Op = MidOf<MID>;
   constexpr int T16 = PL::N / 16;
   constexpr int FLY = PL::N != 16384 ? (FLT == FLT_DR ? 8 : 4) : FLT == FLT_LANE ? 4 : FLT == FLT_BPERM ? 8 : 2;
   const uint32_t l16 = (uint32_t)(L + H * PL::T);
   if constexpr(FLT == FLT_BPERM) {
#pragma unroll
      for(int h = 0; h < 16; h += FLY) {
         float2 f[FLY];
#pragma unroll
         for(int k = 0; k < FLY; k++) f[k] = fb.ld2((fb0 + l16) * 8u, (h + k) * T16 * 8);
#pragma unroll
         for(int k = 0; k < FLY; k++) {
            r[h + k] = Op::apply(r[h + k], f[k]);
            asm volatile("" :: "v"(r[h + k].x));
         }
      }
   } else {
      constexpr bool lane = FLT == FLT_LANE;
      const uint32_t so = lane ? fb0 * 8u + l16 * 16u : (fb0 + l16 * 16u) * 8u;
      constexpr uint32_t ms = lane ? (uint32_t)T16 * 16u : 16u;
#pragma unroll
      for(int h = 0; h < 8; h += FLY / 2) {
         float4 q[FLY / 2];
#pragma unroll
         for(int m = 0; m < FLY / 2; m++) q[m] = fb.ld4(so, (h + m) * ms);
#pragma unroll
         for(int m = 0; m < FLY / 2; m++) {
            float2 &x = r[2 * (h + m)], &y = r[2 * (h + m) + 1];
            x = Op::apply(x, make_float2(q[m].x, q[m].y));
            y = Op::apply(y, make_float2(q[m].z, q[m].w));
            asm volatile("" :: "v"(x.x), "v"(y.x));
         }
      }
   }
}

template<int N_, int MID, int FLT, bool CHAIN>
__global__ void __launch_bounds__(WPlan<N_>::T, 4)
conv_wide_kernel(const Conv1dParams p)
{
   using PL = WPlan<N_, CHAIN>;
   constexpr int N = PL::N, T = PL::T, V = PL::V;
   extern __shared__ float2 lds[];
   const int L = threadIdx.x;
   const uint32_t t = blockIdx.x;            // one transform per workgroup
   Twiddles<PL> tw;
   tw.load(p.tw, L);
   // the base twiddles held from here (an empty asm that may change them):
   // left free, the scheduler's placement of their loads and uses cost 28-72
   // bytes of scratch per lane; held, the kernel fits 128 VGPRs with none
#pragma unroll
   for(int i = 0; i < Twiddles<PL>::COUNT; i++) asm volatile("" : "+v"(tw.w[i].x), "+v"(tw.w[i].y));
   KeptChain<PL> kc;                         // not kept: two groups per lane
   float2 r[V];
   // the signal read and the result written once: streamed past the caches
   const Buf xb(static_cast<const char*>(p.in0) + (size_t)t * N * 8, N * 8);
#pragma unroll
   for(int q = 0; q < V; q++) r[q] = xb.ld2<POL_NT>((uint32_t)L * 8u, q * T * 8);
   constexpr int LAST = PL::NP - 1;
   compute_pass<PL, 0, -1, false, KEEP_NONE>(r, tw, kc);
   float2 lo[V / 2], hi[V / 2];
#pragma unroll
   for(int i = 0; i < V / 2; i++) { lo[i] = r[i]; hi[i] = r[V / 2 + i]; }
   static_for<LAST>([&](auto pi) {
      half_exchange<PL, decltype(pi)::value, decltype(pi)::value + 1, -1, false>(lo, hi, lds, L, tw);
   });
   const Buf fb(p.filt, p.fcount * (uint32_t)N * 8u);
   const uint32_t fb0 = mid_reads_filter<MID> ? modulo_count(t, p.fcount) * N : 0u;
   // The forward's arithmetic comes first and the filter loads stay together (the
   // scheduling barriers at N = 32768): a lane's digit-order slots are one 128-byte
   // line read in 8 pieces, and spread among the arithmetic of the last passes
   // the later pieces fetch the line again.  Digit order, 1000 signals, us: spread /
   // together 196 / 182, one filter per signal 224 / 187.  At N = 16384 the bperm
   // filter fits 128 VGPRs only with the lower half's product in front.
   constexpr bool MID_FIRST = N == 16384 && FLT == FLT_BPERM;
   if constexpr(!MID_FIRST) half_pass<PL, LAST, -1, false>(hi, tw);
   if constexpr(N != 16384 && !CHAIN) __builtin_amdgcn_sched_barrier(0);
   if constexpr(mid_reads_filter<MID>) half_mid<PL, MID, FLT, 0>(lo, fb, fb0, L);
   if constexpr(MID_FIRST) half_pass<PL, LAST, -1, false>(hi, tw);
   if constexpr(mid_reads_filter<MID>) half_mid<PL, MID, FLT, 1>(hi, fb, fb0, L);
   if constexpr(N != 16384 && !CHAIN) __builtin_amdgcn_sched_barrier(0);
   // At N = 16384 the lead pass holds eight groups' base twiddles per lane;
   // read again for the inverse's lead pass (from the cache), they are free
   // in between, and the kernel fits 128 VGPRs with no scratch (48-68 bytes
   // per lane when held throughout).
   constexpr bool RELOAD_LEAD = Twiddles<PL>::distinct(0) > 4;
   // (at N = 32768 the inverse of these two computes its LDS addresses anew: kept from
   // the forward they cost 12 bytes of scratch)
   int Li = L;
   if constexpr(N != 16384 && !CHAIN && (FLT == FLT_BPERM || !mid_reads_filter<MID>)) asm volatile("" : "+v"(Li));
   half_pass<PL, LAST, +1, true>(lo, tw);
   static_for<LAST>([&](auto qi) {
      constexpr int P = LAST - decltype(qi)::value;
      half_exchange<PL, P, P - 1, +1, true>(lo, hi, lds, Li, tw);
   });
   if constexpr(RELOAD_LEAD) {
      tw.template load_pass<0>(Buf(p.tw, FUFFT_TW_ENTRIES * 8u), L);
#pragma unroll
      for(int i = 0; i < Twiddles<PL>::distinct(0); i++) asm volatile("" : "+v"(tw.w[i].x), "+v"(tw.w[i].y));
   }
#pragma unroll
   for(int i = 0; i < V / 2; i++) { r[i] = lo[i]; r[V / 2 + i] = hi[i]; }
   compute_pass<PL, 0, +1, true, KEEP_NONE>(r, tw, kc);
   const Buf ob(static_cast<char*>(p.out0) + (size_t)t * N * 8, N * 8);
#pragma unroll
   for(int q = 0; q < V; q++) ob.st2<POL_NT>(r[q], (uint32_t)L * 8u, q * T * 8);
}

template<int N, int MID, int FLT, bool CHAIN>
hipError_t launch_wide_mid(const Conv1dParams& p, hipStream_t s)
{
   const void* k = reinterpret_cast<const void*>(&conv_wide_kernel<N, MID, FLT, CHAIN>);
   constexpr size_t shm = (size_t)Pad16::size(N / 2) * sizeof(float2);
   static std::atomic<uint64_t> lds_ok{};
   if(const hipError_t e = ensure_dynamic_lds(k, shm, lds_ok); e != hipSuccess) return e;
   Conv1dParams arg = p;
   void* argv[] = { &arg };
   return hipLaunchKernel(k, dim3(p.ntrans), dim3(WPlan<N>::T), argv, shm, s);
}

}  // namespace

// Per-signal filters address with 32-bit byte offsets: beyond 4 GiB of them
// the launch is split into chunks of transforms (signal, result and filter
// advance together).
template<int N, bool CHAIN>
hipError_t launch_conv_wide_n(const Conv1dParams& p, hipStream_t s)
{
   if(p.ntrans == 0) return hipSuccess;
   if(!modulo_count_ok(p.fcount, p.ntrans)) return hipErrorInvalidValue;
   if(p.fl != FLT_DR && p.fl != FLT_LANE && p.fl != FLT_BPERM) return hipErrorInvalidValue;
   auto one = [&](const Conv1dParams& q) {
      return with_mid(q.mid, [&](auto m) {
         constexpr int MID = decltype(m)::value;
         if constexpr(CHAIN || !mid_reads_filter<MID>) {
            return !mid_reads_filter<MID> || q.fl == FLT_DR ? launch_wide_mid<N, MID, FLT_DR, CHAIN>(q, s)
                                                            : hipErrorInvalidValue;
         } else {
            return q.fl == FLT_LANE  ? launch_wide_mid<N, MID, FLT_LANE, false>(q, s)
                 : q.fl == FLT_BPERM ? launch_wide_mid<N, MID, FLT_BPERM, false>(q, s)
                                     : launch_wide_mid<N, MID, FLT_DR, false>(q, s);
         }
      });
   };
   constexpr uint64_t bytes = (uint64_t)N * 8;
   if((uint64_t)p.fcount * bytes <= 0xffffffffull) return one(p);
   if(p.fcount != p.ntrans) return hipErrorInvalidValue;
   const uint32_t step = (uint32_t)(0xffffffffull / bytes) & ~255u;
   for(uint32_t t0 = 0; t0 < p.ntrans; t0 += step) {
      Conv1dParams q = p;
      q.ntrans = p.ntrans - t0 < step ? p.ntrans - t0 : step;
      q.fcount = q.ntrans;
      q.in0  = static_cast<const char*>(p.in0) + (size_t)t0 * bytes;
      q.out0 = static_cast<char*>(p.out0) + (size_t)t0 * bytes;
      q.filt = static_cast<const char*>(p.filt) + (size_t)t0 * bytes;
      if(const hipError_t e = one(q); e != hipSuccess) return e;
   }
   return hipSuccess;
}

hipError_t launch_conv_wide(const Conv1dParams& p, int n, hipStream_t s)
{
   if(n == CONV_WIDE_N) return launch_conv_wide_n<CONV_WIDE_N, false>(p, s);
   if(n == 16384)       return launch_conv_wide_n<16384, false>(p, s);
   return hipErrorInvalidValue;
}

hipError_t launch_conv_wide_chain(const Conv1dParams& p, int n, hipStream_t s)
{
   return n == CONV_WIDE_N ? launch_conv_wide_n<CONV_WIDE_N, true>(p, s) : hipErrorInvalidValue;
}

}  // namespace fufft
