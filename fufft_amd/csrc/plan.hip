// Filter planning on the GPU: the digit-order gather of natural-order spectra.
//
// The reference plans filters on the host: the digit-order permutation and the
// 1/N fold (mixedrev_host, bench_fufft.cu:63-82, 156-170), the four-step chain
// order (bench_fufft.cu:410-428) and the 2D order (verify_kernel.cpp:738-748).
// This kernel does the permutation for spectra already in device memory:
// output position (r, c) of an h x w item (h = 1 in 1D) receives bin
// (rev_h(r), rev_w(c')) times scale, each rev a bit-group reversal over the
// plan's radix widths in pass order, c' = c or, lane-major, the digit-order
// slot that position c holds (lane_slot).  (Taps are planned by the conv
// kernels' own forward half, K_PLAN_TAPS.)
//
// All of these maps only move the bits of an index, so planning is one
// bit-permuting transpose, whatever the layout: source bit s[b] is output bit
// b.  It is bound by HBM, 16 bytes per point, if both sides move whole cache
// lines.  A workgroup therefore takes a tile of 2^11 points that is closed
// under 11 of the bits: the lowest four of the output and the four that
// become the lowest of the source (128-byte runs on both sides), filled up
// from either side in turn.  It reads the tile in source order, turns it
// through 16 KiB of LDS and writes it in output order.  One thread per output
// point, each reading 8 bytes of a line of its own, had the same lines fetched
// by several XCDs: N = 4096, 3001 spectra, digit order 112 us; the tiles 34 us, 5.8 TB/s.
// The filters are written through (POL_WT): the conv reads them next (planning and
// conv of 8 M points 61.8 -> 59.3 us, 67 M 499 -> 491).
#include "fufft_device.hpp"
#include "fufft_internal.hpp"

namespace fufft {

// digit 0 (the first pass's radix) is the most significant bit group of idx
// and becomes the least significant group of the result
static uint32_t group_reverse(uint32_t idx, const GatherDigits& d)
{
   uint32_t out = 0;
   int pos = d.bits, op = 0;
   for(int i = 0; i < d.np; i++) {
      pos -= d.w[i];
      out |= ((idx >> pos) & ((1u << d.w[i]) - 1u)) << op;
      op += d.w[i];
   }
   return out;
}

// source bin of output position o of one item
static uint32_t source_of(uint32_t o, const GatherParams& p)
{
   const uint32_t r = o >> p.dw.bits;
   uint32_t c = o & ((1u << p.dw.bits) - 1u);
   if(p.lane_v) {
      // lane-major along the row (1D filters, 2D columns): the digit-order
      // slot that position c holds -- pairs, or the reference's bperm
      const uint32_t vlog = 31u - (uint32_t)__builtin_clz((uint32_t)p.lane_v);
      const uint32_t tlog = p.dw.bits - vlog;
      c = p.bperm ? ((c & ((1u << tlog) - 1u)) << vlog) | (c >> tlog) : lane_slot(c, tlog, vlog);
   }
   return (group_reverse(r, p.dh) << p.dw.bits) | group_reverse(c, p.dw);
}

constexpr int kTileBits = 11, kTile = 1 << kTileBits, kPer = kTile / 256;
constexpr int kItemBits = 30;

struct TileParams {
   const float2* in;
   float2*       out;
   uint64_t      total;               // points over all items
   float         scale;
   int32_t       bits;                // log2 of the points per item
   int32_t       nrest;               // output bits of an item outside the tile
   uint8_t       tile_out[kTileBits]; // tile index bit -> output bit, ascending
   uint8_t       load_src[kTileBits]; // load index bit -> source bit, ascending
   uint8_t       load_tile[kTileBits];// load index bit -> tile index bit
   uint8_t       rest_out[kItemBits]; // tile number bit -> output bit, ascending
   uint8_t       rest_src[kItemBits]; // tile number bit -> source bit
};

// LDS slot of tile index e: 16 lanes that differ in four neighbouring bits of
// e (consecutive outputs, or consecutive source points, which a radix-16 digit
// spreads over four neighbouring bits) fall on 16 residues modulo 16
__device__ __forceinline__ uint32_t tile_slot(uint32_t e) { return e ^ ((e >> 4) & 15u) ^ ((e >> 8) & 7u); }

// bits [b0, b0 + COUNT) of x moved to the positions map[b0 ..]
template<int B0, int COUNT>
__device__ __forceinline__ uint32_t spread(uint32_t x, const uint8_t (&map)[kTileBits])
{
   uint32_t y = 0;
#pragma unroll
   for(int b = B0; b < B0 + COUNT; b++) y |= ((x >> b) & 1u) << map[b];
   return y;
}

__global__ void __launch_bounds__(256) plan_tile_kernel(const TileParams p)
{
   __shared__ float2 lds[kTile];
   // items of at least a tile: the tile's item, and its place in it; smaller
   // ones: a tile of whole items (the maps are the identity above an item)
   uint64_t base;
   uint32_t points, out0 = 0, src0 = 0;
   if(p.bits >= kTileBits) {
      base = (uint64_t)(blockIdx.x >> p.nrest) << p.bits;
      points = 1u << p.bits;
      for(int b = 0; b < p.nrest; b++) {
         out0 |= ((blockIdx.x >> b) & 1u) << p.rest_out[b];
         src0 |= ((blockIdx.x >> b) & 1u) << p.rest_src[b];
      }
   } else {
      base = (uint64_t)blockIdx.x << kTileBits;
      points = p.total - base < kTile ? (uint32_t)(p.total - base) : (uint32_t)kTile;
   }
   // points past the last item read as zero and are not written
   const Buf ib(p.in + base, points * 8u), ob(p.out + base, points * 8u);
   const uint32_t ls = src0 | spread<0, 8>(threadIdx.x, p.load_src);
   const uint32_t lt = spread<0, 8>(threadIdx.x, p.load_tile);
   float2 v[kPer];
#pragma unroll
   for(int q = 0; q < kPer; q++) v[q] = ib.ld2<POL_NT>((ls | spread<8, kTileBits - 8>(q << 8, p.load_src)) * 8u, 0);
#pragma unroll
   for(int q = 0; q < kPer; q++) lds[tile_slot(lt | spread<8, kTileBits - 8>(q << 8, p.load_tile))] = v[q];
   __syncthreads();
   const uint32_t so = out0 | spread<0, 8>(threadIdx.x, p.tile_out);
#pragma unroll
   for(int q = 0; q < kPer; q++) {
      const float2 x = lds[tile_slot(threadIdx.x | (q << 8))];
      ob.st2<POL_WT>(make_float2(x.x * p.scale, x.y * p.scale), (so | spread<8, kTileBits - 8>(q << 8, p.tile_out)) * 8u, 0);
   }
}

hipError_t launch_gather(const GatherParams& p, hipStream_t s)
{
   if(p.total == 0) return hipSuccess;
   const int bits = p.dh.bits + p.dw.bits;
   if(bits < 1 || bits > 28 || p.dh.np > 32 || p.dw.np > 32) return hipErrorInvalidValue;
   // source bit of every output bit and the inverse; above an item both are the
   // item's number.  (Each planning call pays for these maps: looked up instead of
   // searched for, and no further than the tile and the item reach, 0.16 to 0.28 us
   // for items of 2^8 to 2^20 points, 0.38 to 0.55 before.)
   const int top = bits > kTileBits ? bits : kTileBits;
   uint8_t src[kItemBits], out_of[kItemBits];
   for(int b = 0; b < top; b++) {
      src[b] = (uint8_t)(b < bits ? 31 - __builtin_clz(source_of(1u << b, p)) : b);
      out_of[src[b]] = (uint8_t)b;
   }
   uint32_t tile = 0;                          // the tile's output bits
   for(int b = 0; b < 4; b++) tile |= (1u << b) | (1u << out_of[b]);
   for(bool from_out = true; __builtin_popcount(tile) < kTileBits; from_out = !from_out) {
      int b = 0;
      if(from_out) while(tile & (1u << b)) b++;
      else         while(tile & (1u << out_of[b])) b++;
      tile |= 1u << (from_out ? b : out_of[b]);
   }
   TileParams q{};
   q.in = p.in; q.out = p.out; q.total = p.total; q.scale = p.scale; q.bits = bits;
   int n = 0;
   for(int b = 0; b < top; b++) {
      if(tile & (1u << b)) {
         q.tile_out[n++] = (uint8_t)b;
      } else if(b < bits) {
         q.rest_out[q.nrest] = (uint8_t)b;
         q.rest_src[q.nrest++] = src[b];
      }
   }
   n = 0;
   for(int sb = 0; sb < top; sb++) {
      const int b = out_of[sb];
      if(!(tile & (1u << b))) continue;
      q.load_src[n] = (uint8_t)sb;
      q.load_tile[n++] = (uint8_t)__builtin_popcount(tile & ((1u << b) - 1u));
   }
   const uint64_t blocks = (p.total + kTile - 1) / kTile;
   if(blocks > 0x7fffffffull) return hipErrorInvalidValue;
   void* argv[] = { &q };
   return hipLaunchKernel(reinterpret_cast<const void*>(&plan_tile_kernel), dim3((unsigned)blocks), dim3(256), argv, 0, s);
}

}  // namespace fufft
