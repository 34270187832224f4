// GEMMs whose 256 x 256 tiles would leave most compute units idle (text rows, text encoders,
// short prompts, narrow outputs): the same C = epilogue(A W^T + bias) and element types as
// gemm.hip, in smaller tiles and, where those still leave units idle, with K cut into pieces.
//
// What bounds them: the bytes each compute unit pulls from L2 into its LDS (about 57 B/ns with
// every unit pulling), since a tile reads (BM + BN) K elements for BM BN K products. A launch of
// 24 tiles of 256 x 256 (512 x 3072 x 4096) runs 24 such streams; 96 tiles of 128 x 128 cut in
// two pieces run 192, for twice the bytes in all. The planner at the end of this file weighs the
// two.
//
// A workgroup is 8 wavefronts over a BM x BN tile, in a 2 x 4 grid (4 x 2 for 256 rows: 64 x 64
// each, the fewest LDS bytes per product) of MFMA tiles of 32 x 32 (operand roles and LDS swizzle
// as in gemm.hip: W first, A second, a 128-byte K stage per row, chunk c of row r at c ^ swz8(r)).
// Stages go through a ring of NSLOT
// slots filled by direct-to-LDS loads, NSLOT - 1 of them in flight: these launches have one
// workgroup per compute unit, so the ring alone has to cover the latency of cold weights.
// One barrier per stage, before its last K step, whose fragments are in registers by then: each
// wave has waited for its own loads of the next stage (the younger ones stay in flight), so the
// barrier publishes that stage and frees this one's slot for the loads of stage kt + NSLOT.
//
// fp32 operands run here at every size (v_mfma_f32_32x32x2_f32, a stage of 32 floats per row,
// lane half h of a fragment taking floats 16 h .. 16 h + 15 in turn), bound by the matrix cores:
// 128 x 128 takes 4096 cycles of MFMA per SIMD and stage for 32 KB. What keeps them fed is other
// workgroups on the unit while one is at its barrier, so these tiles take two slots of a ring
// each (two workgroups per unit at 128 x 128, five at 64 x 64): four linears of 452 rows (4096 x
// 12288, 4096 x 4096, 4096 x 20480, 10240 x 4096) 1867 us in the register-staged kernel
// (gemm_f32.hip, which the convolutions still use, with the same K order and so the same bits),
// 1667 with rings of 4 and 5 slots, 1510 now; 1024 rows of 4096 x 12288 897 -> 749 us (138 TFLOP/s).
//
// K pieces: piece c of a tile writes its fp32 sums to part[c][m][n]; gemm_small_reduce adds the
// pieces in order and runs the epilogue. Nothing is kept between launches and nobody waits, so
// any scratch buffer serves, on any stream and under graph capture.
#include <algorithm>

#include "common.hpp"
#include "gemm_small.hpp"

namespace dlt {

struct SmallArgs {
  const uint8_t* a;
  const uint8_t* w;
  uint8_t* c;
  const void* bias;  // bf16 (F32: fp32), as gate, res and C
  const void* gate;
  const void* res;
  const uint8_t* a_scale;
  const uint8_t* w_scale;
  int64_t lda, ldw, ldc, ldr, gate_stride, rows_per_batch;  // element strides
  int m, n, k;
  int tiles_m, tiles_n;
  int pieces, piece_stages;  // K pieces per tile, stages per piece (the last may be shorter)
  float* part;               // fp32 sums [pieces][m][n] (pieces > 1)
};

// direct-to-LDS load of 16 bytes per lane (as attention.hip's dma16, with a scalar offset):
// untracked by the compiler, waited for by the K loop's own vmcnt
typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void dma16s(i32x4 r, const uint8_t* lds_ptr, uint32_t voff,
                                       uint32_t soff) {
  const uint32_t la = (uint32_t)reinterpret_cast<uintptr_t>((lds_void_t*)lds_ptr);
  asm volatile("s_nop 4\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(la), "v"(voff), "s"(r), "s"(soff)
               : "memory", "m0");
}
__device__ __forceinline__ i32x4 rsrc_of(const void* base, int64_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint32_t n = bytes > 0xffffffffLL ? 0xffffffffu : (uint32_t)bytes;
  return i32x4{(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffffu), (int)n, 0x00020000};
}
template <int VM>
__device__ __forceinline__ void wait_vm() {
  static_assert(VM >= 0 && VM < 64, "vmcnt field");
  __builtin_amdgcn_s_waitcnt(0x0070 | (VM & 15) | ((VM >> 4) << 14));  // and lgkmcnt(0)
}
__device__ __forceinline__ int swz8s(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// v (8 columns from n on of row m, fp32 sums) through the epilogue into C: the math of gemm.hip.
template <SmallElem E, bool GATE>
__device__ __forceinline__ void small_store8(const SmallArgs& a, int64_t m, int64_t n, float* v) {
  if (n >= a.n) return;
  const bool full = n + 8 <= a.n;  // n % 4 == 0: a chunk is full or half full
  if constexpr (E == SmallElem::F32) {
    const float* bias = reinterpret_cast<const float*>(a.bias);
    const float* res = reinterpret_cast<const float*>(a.res);
    float* dst = reinterpret_cast<float*>(a.c) + m * a.ldc + n;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h == 1 && !full) break;
      f32x4 x = {v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
      if (bias) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(bias + n + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += b[e];
      }
      if (res) {
        const f32x4 r = *reinterpret_cast<const f32x4*>(res + m * a.ldr + n + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = r[e] + x[e];
      }
      *reinterpret_cast<f32x4*>(dst + 4 * h) = x;
    }
    return;
  }
  auto load8 = [&](const bf16* p, float* o) {
    const u32x2 lo = *reinterpret_cast<const u32x2*>(p);
    const u32x2 hi = full ? *reinterpret_cast<const u32x2*>(p + 4) : u32x2{0u, 0u};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = bf16bits_to_f32(e & 1 ? lo[e >> 1] >> 16 : lo[e >> 1] & 0xffffu);
      o[4 + e] = bf16bits_to_f32(e & 1 ? hi[e >> 1] >> 16 : hi[e >> 1] & 0xffffu);
    }
  };
  if constexpr (E == SmallElem::FP8) {
    const float* ws = reinterpret_cast<const float*>(a.w_scale) + n;
    const float sa = reinterpret_cast<const float*>(a.a_scale)[m];
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(ws);
    const f32x4 w1 = full ? *reinterpret_cast<const f32x4*>(ws + 4) : f32x4{};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * (sa * (e < 4 ? w0[e] : w1[e - 4]));
  }
  if (a.bias) {
    float b[8];
    load8(reinterpret_cast<const bf16*>(a.bias) + n, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += b[e];
  }
  if constexpr (GATE) {
    float g[8], r[8];
    load8(reinterpret_cast<const bf16*>(a.gate) + m / a.rows_per_batch * a.gate_stride + n, g);
    load8(reinterpret_cast<const bf16*>(a.res) + m * a.ldr + n, r);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = r[e] + g[e] * v[e];
  }
  bf16* dst = reinterpret_cast<bf16*>(a.c) + m * a.ldc + n;
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
  if (full && ((uintptr_t)dst & 15) == 0) {
    *reinterpret_cast<u32x4*>(dst) = o;
  } else {
    *reinterpret_cast<u32x2*>(dst) = u32x2{o[0], o[1]};
    if (full) *reinterpret_cast<u32x2*>(dst + 4) = u32x2{o[2], o[3]};
  }
}

template <SmallElem E, int BM, int BN, int NSLOT, bool GATE>
__global__ __launch_bounds__(BN == 64 ? 256 : 512, 1) void gemm_small_kernel(
    const SmallArgs args) {
  constexpr bool F32 = E == SmallElem::F32;
  constexpr int EB = F32 ? 4 : E == SmallElem::BF16 ? 2 : 1;
  constexpr int NW = BN == 64 ? 4 : 8, NT = NW * 64;  // wavefronts, threads
  constexpr int WAVES_M = BM == 256 ? 4 : 2, WAVES_N = NW / WAVES_M;
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  constexpr int TI = WTM / 32, TJ = WTN / 32;     // MFMA tiles per wave
  constexpr int NKS = EB > 1 ? 4 : 2;  // K steps per stage (F32: of 4 MFMAs each)
  constexpr int NA = EB > 1 ? 1 : 2;   // 16-byte LDS reads per fragment
  constexpr int SA = BM / 8 / NW, SW = BN / 8 / NW, LPS = SA + SW;  // 1 KB loads per wave and stage
  constexpr int SLOT = (BM + BN) * 128;
  // MX: E8M0 scales of 4 stages (16 bytes) per row, a ring of two such blocks
  constexpr int SC = E == SmallElem::MX ? (BM + BN) * 16 : 0;
  static_assert(NSLOT * SLOT >= BM * BN * 4, "the epilogue stages the fp32 tile in the ring");
  static_assert(E != SmallElem::MX || NSLOT <= 5, "scale blocks land within 4 stages");
  __shared__ __attribute__((aligned(16))) uint8_t lds[NSLOT * SLOT + 2 * SC];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int frow = lane & 31, fhalf = lane >> 5;

  // work item (piece, column tile, row tile), rows fastest: ids are dealt round-robin over the
  // 8 XCDs, and each XCD takes a contiguous run, so the row tiles that share a slice of W and
  // the columns that share a slice of A meet in one L2
  int item;
  {
    const int total = gridDim.x, x = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int per = total >> 3, rem = total & 7;
    item = x * per + min(x, rem) + j;
  }
  const int tm = item % args.tiles_m, rest = item / args.tiles_m;
  const int tn = rest % args.tiles_n, piece = rest / args.tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = args.m, N = args.n;
  const int nk = (args.k + 128 / EB - 1) / (128 / EB);  // F32: the last stage may be partial
  const int kbeg = piece * args.piece_stages;
  const int nkt = min(args.piece_stages, nk - kbeg);

  const int64_t arow = args.lda * EB, wrow = args.ldw * EB;
  // the buffers end with the tile's last row, not a row stride after it (rows may be a column
  // range of wider ones), and never reach kOut: gemm.hip admits operands of up to 2^32 - 16 bytes,
  // fp32 rows are below 2^24
  constexpr uint32_t kOut = 0xfffffff0u;
  const int arows = min(M - m0, BM), wrows = min(N - n0, BN);
  const i32x4 ra = rsrc_of(args.a + m0 * arow, (arows - 1) * arow + (int64_t)args.k * EB);
  const i32x4 rw = rsrc_of(args.w + n0 * wrow, (wrows - 1) * wrow + (int64_t)args.k * EB);
  // lane l of a 1 KB load fills slab row l / 8, chunk l % 8; rows past M or N read zero, at kOut:
  // where rows are 16 MB and more apart (one token of each batch element) their own offsets would
  // wrap to ones that another row covers
  uint32_t aoff[4], woff[4];
  auto row_off = [&](int r, int rows, int64_t row) {
    const uint32_t o = (uint32_t)r * (uint32_t)row + (uint32_t)(((lane & 7) ^ swz8s(r)) << 4);
    return r < rows ? o : kOut;
  };
#pragma unroll
  for (int i = 0; i < SA; ++i) aoff[i] = row_off((wave * SA + i) * 8 + (lane >> 3), arows, arow);
#pragma unroll
  for (int i = 0; i < SW; ++i) woff[i] = row_off((wave * SW + i) * 8 + (lane >> 3), wrows, wrow);
  const int ksb = args.k / 32;  // MX: scale bytes per row
  i32x4 rsa = ra, rsw = rw;
  if constexpr (E == SmallElem::MX) {
    rsa = rsrc_of(args.a_scale + (int64_t)m0 * ksb, (int64_t)(M - m0) * ksb);
    rsw = rsrc_of(args.w_scale + (int64_t)n0 * ksb, (int64_t)(N - n0) * ksb);
  }
  // MX scale block q (stages 4 q .. 4 q + 3 of the piece) into ring slot q % 2; waves below
  // (BM + BN) / 64 load 64 rows each. The whole offset is per lane, so the range check covers
  // it (bytes past the array read zero).
  auto issue_scales = [&](int q) {
    if constexpr (E == SmallElem::MX) {
      uint8_t* dst = lds + NSLOT * SLOT + (q & 1) * SC + wave * 1024;
      const uint32_t kofs = (uint32_t)((kbeg >> 2) + q) * 16;
      if (wave < BM / 64)
        dma16s(rsa, dst, (uint32_t)(wave * 64 + lane) * ksb + kofs, 0);
      else if (wave < (BM + BN) / 64)
        dma16s(rsw, dst, (uint32_t)((wave - BM / 64) * 64 + lane) * ksb + kofs, 0);
    }
  };
  // stage kt's loads into slot st; past the piece's last stage they are issued with an offset
  // beyond all but the largest buffers (zeros, no memory traffic), so every barrier waits with one
  // vmcnt; what a larger one returns there is not used
  auto issue = [&](int kt, int st) {
    const uint32_t kb = kt < nkt ? (uint32_t)(kbeg + kt) * 128u : 0u;
    const uint32_t off = kt < nkt ? 0u : 0x80000000u;
    uint8_t* d = lds + st * SLOT;
    // F32: K is a multiple of 4, so a lane's 16 bytes are all inside K or all past it
    auto at = [&](uint32_t o, int slab) {
      if constexpr (F32) {
        const int r = slab * 8 + (lane >> 3);
        const int kk = (kbeg + kt) * 32 + ((lane & 7) ^ swz8s(r)) * 4;
        return kt < nkt && kk < args.k ? o : kOut;
      }
      return o | off;
    };
#pragma unroll
    for (int i = 0; i < SA; ++i)
      dma16s(ra, d + (wave * SA + i) * 1024, at(aoff[i], wave * SA + i), kb);
#pragma unroll
    for (int i = 0; i < SW; ++i)
      dma16s(rw, d + BM * 128 + (wave * SW + i) * 1024, at(woff[i], wave * SW + i), kb);
  };

  f32x16 acc[4][4];  // [i < TI][j < TJ]
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16{};

  // fragments of one K step, two sets: the next step's are read while this one's MFMAs run
  i32x4 fa[2][4][2], fw[2][4][2];  // [set][tile][16-byte half]
  auto read_frags = [&](const uint8_t* stage, int ks, int set) {
#pragma unroll
    for (int h = 0; h < NA; ++h) {
      const int ch = F32 ? 4 * fhalf + ks : 2 * NA * ks + 2 * h + fhalf;
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int r = wn * WTN + j * 32 + frow;
        fw[set][j][h] = *reinterpret_cast<const i32x4*>(stage + BM * 128 + r * 128 +
                                                        ((ch ^ swz8s(r)) << 4));
      }
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int r = wm * WTM + i * 32 + frow;
        fa[set][i][h] =
            *reinterpret_cast<const i32x4*>(stage + r * 128 + ((ch ^ swz8s(r)) << 4));
      }
    }
  };
  // MX: the stage's scale word per row, shifted so that bytes 0 and 2 are this lane group's
  // K-blocks of K steps 0 and 1
  uint32_t sca[2][4], scw[2][4];  // [stage parity]
  auto read_scales = [&](int kt, int par) {
    if constexpr (E == SmallElem::MX) {
      const uint8_t* sc = lds + NSLOT * SLOT + ((kt >> 2) & 1) * SC + (kt & 3) * 4;
#pragma unroll
      for (int i = 0; i < TI; ++i)
        sca[par][i] = *reinterpret_cast<const uint32_t*>(sc + (wm * WTM + i * 32 + frow) * 16) >>
                      (8 * fhalf);
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        scw[par][j] =
            *reinterpret_cast<const uint32_t*>(sc + (BM + wn * WTN + j * 32 + frow) * 16) >>
            (8 * fhalf);
    }
  };
  auto mma = [&](int ks, int set) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const i32x4* w = fw[set][j];
        const i32x4* x = fa[set][i];
        if constexpr (F32) {
          const f32x4 wv = __builtin_bit_cast(f32x4, w[0]), xv = __builtin_bit_cast(f32x4, x[0]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[e], xv[e], acc[i][j], 0, 0, 0);
        } else if constexpr (E == SmallElem::BF16) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[0]),
                                                              __builtin_bit_cast(bf16x8, x[0]),
                                                              acc[i][j], 0, 0, 0);
        } else {
          const i32x8 w8 = {w[0][0], w[0][1], w[0][2], w[0][3], w[1][0], w[1][1], w[1][2], w[1][3]};
          const i32x8 a8 = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
          if constexpr (E == SmallElem::FP8)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8, a8, acc[i][j], 0, 0, 0,
                                                                        0, 0, 0);
          else if (ks == 0)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                w8, a8, acc[i][j], 0, 0, 0, (int)scw[0][j], 0, (int)sca[0][i]);
          else
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                w8, a8, acc[i][j], 0, 0, 2, (int)scw[0][j], 2, (int)sca[0][i]);
        }
      }
  };

  issue_scales(0);
  issue_scales(1);
#pragma unroll
  for (int s = 0; s < NSLOT; ++s) issue(s, s);
  wait_vm<(NSLOT - 1) * LPS>();  // stage 0 (and the scale blocks, issued before it)
  asm volatile("s_barrier" ::: "memory");
  read_frags(lds, 0, 0);
  read_scales(0, 0);
  int st = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    const int nst = st == NSLOT - 1 ? 0 : st + 1;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int set = ks & 1;
      if (ks == NKS - 1) {
        // stage kt + 1 has landed (the NSLOT - 2 younger ones may be in flight; a scale load
        // among them only makes the wait stricter) and this wave's reads of stage kt are done
        wait_vm<(NSLOT - 2) * LPS>();
        asm volatile("s_barrier" ::: "memory");
        // block q = (kt + 1) / 4 starts with the next stage; block q - 1, whose slot block q + 1
        // takes, was last read for this stage, before the barrier. q + 1 is first read behind
        // the barrier of four stages on, with at most NSLOT - 2 younger stages in flight.
        if (E == SmallElem::MX && (kt & 3) == 3) issue_scales(((kt + 1) >> 2) + 1);
        issue(kt + NSLOT, st);
        read_frags(lds + nst * SLOT, 0, set ^ 1);  // past the last stage: zeros nobody uses
        read_scales(kt + 1, 1);
      } else {
        read_frags(lds + st * SLOT, ks + 1, set ^ 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(ks, set);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (E == SmallElem::MX) {
#pragma unroll
      for (int i = 0; i < TI; ++i) sca[0][i] = sca[1][i];
#pragma unroll
      for (int j = 0; j < TJ; ++j) scw[0][j] = scw[1][j];
    }
    st = nst;
  }

  // ---- the fp32 tile through the idle ring: 16-byte chunk c of row r at c ^ (r & CM), then
  // BN / 8 lanes per row take 8 columns each (whole lines per store)
  wait_vm<0>();
  __syncthreads();
  float* tile = reinterpret_cast<float*>(lds);
  constexpr int CM = BN / 4 < 32 ? BN / 4 - 1 : 31;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const int r = wm * WTM + i * 32 + frow;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c4 = (wn * WTN + j * 32 + q * 8 + fhalf * 4) >> 2;
        const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                         acc[i][j][4 * q + 3]};
        *reinterpret_cast<f32x4*>(tile + r * BN + ((c4 ^ (r & CM)) << 2)) = v;
      }
    }
  __syncthreads();
  constexpr int LPR = BN / 8, RPP = NT / LPR;  // lanes per row, rows per pass
  const int ch = tid % LPR, rsub = tid / LPR;
  const int64_t n = n0 + ch * 8;
#pragma unroll 4
  for (int r = rsub; r < BM; r += RPP) {
    const int64_t m = m0 + r;
    if (m >= M) break;
    const f32x4 y0 = *reinterpret_cast<const f32x4*>(tile + r * BN + (((2 * ch) ^ (r & CM)) << 2));
    const f32x4 y1 =
        *reinterpret_cast<const f32x4*>(tile + r * BN + (((2 * ch + 1) ^ (r & CM)) << 2));
    if (args.pieces > 1) {
      float* p = args.part + ((int64_t)piece * M + m) * N + n;
      if (n < N) *reinterpret_cast<f32x4*>(p) = y0;
      if (n + 4 < N) *reinterpret_cast<f32x4*>(p + 4) = y1;
    } else {
      float v[8] = {y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
      small_store8<E, GATE>(args, m, n, v);
    }
  }
}

// C = epilogue(sum of the K pieces in order), 8 columns per thread.
template <SmallElem E, bool GATE>
__global__ __launch_bounds__(256) void gemm_small_reduce(const SmallArgs args) {
  const int chunks = (args.n + 7) >> 3;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)args.m * chunks) return;
  const int64_t m = i / chunks, n = (i % chunks) * 8;
  const bool full = n + 8 <= args.n;
  const float* p = args.part + m * args.n + n;
  const int64_t step = (int64_t)args.m * args.n;
  float v[8] = {};
#pragma unroll 4
  for (int c = 0; c < args.pieces; ++c, p += step) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(p);
    const f32x4 y = full ? *reinterpret_cast<const f32x4*>(p + 4) : f32x4{};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] += x[e];
      v[4 + e] += y[e];
    }
  }
  small_store8<E, GATE>(args, m, n, v);
}

// Estimated times on MI355X, in us, from sweeps over 16 to 3000 rows of the layers' widths:
//  - a workgroup takes kStage per K stage (bf16, fp8, MXFP8; 64-, 128- and 256-row tiles; the MX
//    scales cost the small tiles LDS reads) plus 5 for its first loads and its output; a launch runs
//    ceil(workgroups / units) rounds of that, but no faster than its weights come from HBM;
//  - fp32 (64 x 64 and 128 x 128 tiles): a compute unit works through its workgroups' stages two
//    or more workgroups at a time, kStageF32 each with one, two or more of them on the unit
//    (matrix-core time 0.43 and 1.74 at 2.35 GHz);
//  - cutting K adds the reduce launch and the sums' trip out and back at about 5 TB/s.
// What the choices measured (bf16, 3072 x 3072 / 12288 x 3072 /
// 5120 x 5120, 256 x 256 tiles -> the plan's): 64 rows 57 -> 16, 65 -> 23, 50 -> 18; 512 rows
// 62 -> 19, 77 -> 55, 74 -> 44; 1024 rows 66 -> 27, 114 -> 97, 94 -> 75; fp8 12288 x 3072 at 16,
// 512 and 1024 rows 51 -> 18, 60 -> 32, 78 -> 46. Past 4096 rows the 256 x 256 tiles fill the
// chip.
SmallPlan small_plan(SmallElem e, int64_t m, int64_t n, int64_t k, int cus, int64_t scratch,
                     double big_us) {
  SmallPlan best = {0, 0, 0, 0};
  const bool f32 = e == SmallElem::F32;
  if (cus <= 0 || m <= 0 || (m > 4096 && !f32)) return best;
  const int eb = f32 ? 4 : e == SmallElem::BF16 ? 2 : 1;
  const int nk = (int)((k * eb + 127) / 128), gran = e == SmallElem::MX ? 4 : 1;
  static const int kRows[3] = {64, 128, 256};
  static const double kStage[3][3] = {{0.36, 0.52, 0.90}, {0.30, 0.43, 0.88}, {0.38, 0.60, 0.90}};
  static const double kStageF32[2][3] = {{0.62, 0.53, 0.505}, {2.05, 1.95, 1.93}};
  const double hbm_us = (double)n * k * eb / 4.5e6;
  double best_us = 0.95 * big_us;  // within the estimates' error of each other: leave it
  for (int i = 0; i < (f32 ? 2 : 3); ++i) {
    const int bn = f32 && i == 0 ? 64 : 128;
    const int64_t tiles = ((m + kRows[i] - 1) / kRows[i]) * ((n + bn - 1) / bn);
    if (tiles > 4 * cus && !f32) continue;
    for (int pieces = 1; pieces <= 16; ++pieces) {
      const int ps = ((nk + pieces - 1) / pieces + gran - 1) / gran * gran;
      if ((nk + ps - 1) / ps != pieces) continue;  // rounding left a piece without stages
      if (pieces > 1 && (ps < 4 || pieces * m * n * 4 > scratch)) continue;
      if (pieces > 1 && tiles * pieces > 4 * cus) break;
      const int64_t rounds = (tiles * pieces + cus - 1) / cus;
      double us = f32 ? rounds * ps * kStageF32[i][std::min<int64_t>(rounds, 3) - 1] + 5.0
                      : rounds * (ps * kStage[(int)e][i] + 5.0);
      us = std::max(us, hbm_us);
      if (pieces > 1) us += 3.0 + (double)pieces * m * n * 8 / 5e6;
      if (us < best_us) {
        best_us = us;
        best = {kRows[i], bn, pieces, ps};
      }
    }
  }
  return best;
}

template <SmallElem E, bool GATE>
static void launch_small(const SmallArgs& a, const SmallPlan& p, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n * a.pieces)), block(512);
  if constexpr (E == SmallElem::F32) {
    if (p.bm == 64)
      hipLaunchKernelGGL((gemm_small_kernel<E, 64, 64, 2, GATE>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((gemm_small_kernel<E, 128, 128, 2, GATE>), grid, block, 0, s, a);
  } else {
    if (p.bm == 64)
      hipLaunchKernelGGL((gemm_small_kernel<E, 64, 128, 5, GATE>), grid, block, 0, s, a);
    else if (p.bm == 128)
      hipLaunchKernelGGL((gemm_small_kernel<E, 128, 128, 4, GATE>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((gemm_small_kernel<E, 256, 128, 3, GATE>), grid, block, 0, s, a);
  }
  if (p.pieces > 1) {
    const int64_t chunks = (int64_t)a.m * ((a.n + 7) / 8);
    hipLaunchKernelGGL((gemm_small_reduce<E, GATE>), dim3((unsigned)((chunks + 255) / 256)),
                       dim3(256), 0, s, a);
  }
}

void gemm_small(SmallElem e, const SmallPlan& plan, const difflet_gemm_problem& q, int64_t n,
                int64_t k, bool gate, int64_t rows_per_batch, void* scratch, hipStream_t s) {
  SmallArgs a = {};
  a.a = (const uint8_t*)q.a;
  a.w = (const uint8_t*)q.w;
  a.c = (uint8_t*)q.c;
  a.bias = q.bias;
  a.gate = q.gate;
  a.res = q.residual;
  a.a_scale = (const uint8_t*)q.a_scale;
  a.w_scale = (const uint8_t*)q.w_scale;
  a.lda = q.lda;
  a.ldw = q.ldw;
  a.ldc = q.ldc;
  a.ldr = q.ldr;
  a.gate_stride = q.gate_stride;
  a.rows_per_batch = rows_per_batch;
  a.m = (int)q.m;
  a.n = (int)n;
  a.k = (int)k;
  a.tiles_m = (int)((q.m + plan.bm - 1) / plan.bm);
  a.tiles_n = (int)((n + plan.bn - 1) / plan.bn);
  a.pieces = plan.pieces;
  a.piece_stages = plan.piece_stages;
  a.part = (float*)scratch;
  if (e == SmallElem::F32) {
    launch_small<SmallElem::F32, false>(a, plan, s);
    return;
  }
  auto go = [&](auto et) {
    constexpr SmallElem E = decltype(et)::value;
    if (gate) launch_small<E, true>(a, plan, s);
    else launch_small<E, false>(a, plan, s);
  };
  using std::integral_constant;
  if (e == SmallElem::BF16) go(integral_constant<SmallElem, SmallElem::BF16>{});
  else if (e == SmallElem::FP8) go(integral_constant<SmallElem, SmallElem::FP8>{});
  else go(integral_constant<SmallElem, SmallElem::MX>{});
}

}  // namespace dlt
