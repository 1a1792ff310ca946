// rows.hip -- grouped INT4 GEMMs for token groups of few rows and for every
// scale-group size (a multiple of 32 dividing K), any K % 32 == 0 and any
// number of weight rows.
//
// Work decomposition.  One work-group computes 32 expert-sorted rows of one
// expert times 128 weight rows (GATEUP: 64 gate rows and the matching up rows,
// SiLU(gate) * up written to `mid`), its four waves each 32 of the weight rows
// over the whole contraction.
//
// Data movement.  The contraction runs in chunks of 128 k: 32 activation rows x
// 256 B (gathered for GATEUP) and 128 packed weight rows x 64 B are copied
// straight from global memory into LDS, double-buffered, XOR-swizzled in
// 16-byte columns (the operand reads are free of bank conflicts).  32 KiB of
// LDS and at most 128 registers put four work-groups on a CU, so that one's
// copies are in flight while another multiplies.
//
// Bound.  With few rows per expert every weight is used once or twice, and a
// chunk's copies, its dequantisation (14 VALU instructions per 8 weights) and
// its LDS reads cost about the same.  Qwen3 shape at 187 tokens (105 token
// groups), gate/up: 52 us, the matrix pipes busy 15 % of it and 1.15 times the
// weights fetched; when it took 61 us, 39 with only the copies left in and 46 with
// only the arithmetic.  Tiles of 16 or 64 rows, or of 256 weight rows, measured the
// same or slower there (109 - 123 us a layer against 111), and so did weights
// copied two chunks at a time in whole 128-byte lines (113).  Three or four stages
// instead of two, with three or two work-groups per CU: 95 -> 107 / 121 us (group
// 64 at 48 tokens 67 -> 74 / 81): waves per SIMD hide more than copies in flight.
//
// Arithmetic.  Step s of a chunk covers k = 32 s .. 32 s + 31, so every step
// lies inside one scale group: lane (r, q) of the MFMA 16x16x32 operands holds
// k = 32 s + 8 q .. + 7 of row r (16 bytes of activations, one dword of packed
// nibbles), or another 8 k of the same scale group where a group holds several
// steps.  Nibbles become exact 16-bit floats of q - 8 (bf16: of (q - 8) / 16, the
// 16 folded into the scale), a scale group's steps accumulate in fp32 and the
// group's fp16 scale multiplies the sum in fp32.
#include "exq_internal.h"

#include "dev_util.h"

namespace exq {
namespace {

using namespace dev;

constexpr int RTH = 256;            // threads per work-group
constexpr int RKC = 128;            // contraction per chunk
constexpr int MT = 2, NTW = 2;      // 16-row tiles of activations, of weights per wave
constexpr int TN = 64 * NTW;        // weight rows per work-group
static_assert(16 * MT == kTokenGroupRows, "a token group is one tile of rows");

// Swizzles of the staged rows (their low four bits) in 16-byte columns:
// activations 16 columns per row, packed weights 4.  gfx950 serves a
// ds_read_b128 in four cycles of 256 bytes; the lanes served together have
// equal bit 5 and equal parity of bits 2..4, and under these maps they cover
// 16 distinct 16-byte units (activations, column 4 s + q); a ds_read_b32 of
// the weights (column s, dword q) covers 64 distinct banks.
__device__ __forceinline__ int ra_swz(int r) {
  return (r & 3) | ((r >> 1) & 4) | (((r << 1) ^ r) & 8);
}
__device__ __forceinline__ int rb_swz(int r) {
  return ((r >> 3) & 1) | ((((r >> 2) ^ (r >> 3)) & 1) << 1);
}

// 16 bytes per lane from the lane's address into LDS at lds + 16 * lane.
__device__ __forceinline__ void gdma16(const void* p, unsigned char* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_global_load_lds((gptr_t)p, (lptr_t)lds, 16, 0, 0);
#endif
}
// The same through a buffer resource at voff + soff (soff wave-uniform); AUX 2:
// nontemporal.
template <int AUX = 0>
__device__ __forceinline__ void bdma16(__amdgpu_buffer_rsrc_t r, unsigned char* lds, int voff,
                                       int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lptr_t)lds, 16, voff, soff, 0, AUX);
#endif
}

// Buffer resource whose size is a plain 32-bit product (make_rsrc's 64-bit
// clamp is a vector compare, which costs the uniformity of what follows).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc32(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}

// 8 packed nibbles (low nibble = even k) -> 8 exact 16-bit floats in natural k
// order: q - 8 (f16), (q - 8) / 16 (bf16, v_cvt_off_f32_i4).
template <bool BF>
__device__ __forceinline__ uint4 deq_signed(uint32_t p, uint32_t mask, uint32_t magic) {
  uint4 o;
  if constexpr (BF) {
    uint32_t l = p ^ 0x88888888u;  // two's complement nibbles
    uint32_t h = l >> 4;
    asm volatile("" : "+v"(l), "+v"(h));  // byte selects stay inside the conversions
    auto pk = [](uint32_t a, uint32_t b) {
      typedef float f32x2_t __attribute__((ext_vector_type(2)));
      const f32x2_t v = {__builtin_amdgcn_cvt_off_f32_i4((int)a),
                         __builtin_amdgcn_cvt_off_f32_i4((int)b)};
      return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    };
    o.x = pk(l & 0xffu, h & 0xffu);
    o.y = pk((l >> 8) & 0xffu, (h >> 8) & 0xffu);
    o.z = pk((l >> 16) & 0xffu, (h >> 16) & 0xffu);
    o.w = pk(l >> 24, h >> 24);
  } else {
    // 1024 + n in each half (v_perm_b32, v_and_or_b32), minus 1032: exact
    const uint32_t h = p >> 4;
    const f16x2_t off = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    auto pk = [&](uint32_t sel) {
      const uint32_t u = (__builtin_amdgcn_perm(h, p, sel) & mask) | magic;
      return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2_t, u) + off);
    };
    o.x = pk(0x0c040c00u);
    o.y = pk(0x0c050c01u);
    o.z = pk(0x0c060c02u);
    o.w = pk(0x0c070c03u);
  }
  return o;
}

// Unit (token group, weight tile) of work-group bid over n token groups from t0
// (unit_order.h).
__device__ __forceinline__ bool rows_unit(const GemmArgs& a, int t0, int n, int NT, int bid,
                                          TgEntry& te, int& nt, bool* once = nullptr) {
  int tgi;
  if (!rows_unit_of(bid, n, NT, tgi, nt)) return false;
  te = a.tg[t0 + tgi];
  if (once)  // the expert's only group (an expert's groups are neighbours in the list)
    *once = (tgi == 0 || a.tg[t0 + tgi - 1].e != te.e) &&
            (tgi + 1 >= n || a.tg[t0 + tgi + 1].e != te.e);
  return te.cnt > 0;
}

// Steps per scale group known at compile time: 1 (group 32), 2 (64), 4 (128 and
// its multiples: a scale per chunk), with K % 128 == 0; 0: any group size and
// any K % 32 == 0.
template <bool BF, int MODE, int SPG>
__device__ __forceinline__ void rows_body(const GemmArgs& a, int n_tiles,
                                          unsigned char* const (&sA)[2],
                                          unsigned char* const (&sB)[2]) {
  constexpr int HN = TN / 2, HALF = NTW / 2;
  constexpr int QA = MT;        // activation copies per wave and chunk (4 rows each)
  constexpr int QB = NTW;       // weight copies per wave and chunk (16 rows each)
  constexpr float kFold = BF ? 16.f : 1.f;

  TgEntry te;
  int nt;
  // INT4 groups [hdr[1], hdr[0])
  if (!rows_unit(a, a.hdr[1], a.hdr[0] - a.hdr[1], n_tiles, blockIdx.x, te, nt)) return;
  nt = uni_i(nt);
  const int cnt = uni_i(te.cnt), pos0 = uni_i(te.pos0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int K = a.K;
  const int nch = (K + RKC - 1) / RKC;
  const int ngs = K / a.group_size, spg = a.group_size / 32;
  const int n_out = MODE == MODE_GATEUP ? a.inter : a.n_rows;  // output columns
  const int rowbytes = K / 2;

  // The tile's weight rows: GATEUP gate rows c0 .. c0 + HN - 1 and the up rows
  // of the same columns, otherwise rows c0 .. c0 + TN - 1; rows past the end
  // repeat the last one and are not stored.
  const int c0 = nt * (MODE == MODE_GATEUP ? HN : TN);
  const int e = uni_i(te.e);
  const int widx = a.w.index ? uni_i(a.w.index[e]) : e;
  const int64_t row0 = (int64_t)widx * a.n_rows + c0;
  const int left = n_out - c0, full = MODE == MODE_GATEUP ? HN : TN;
  const int have = left < full ? left : full;  // rows of each half / of all
  auto lrow = [&](int rho) {  // row within its half (GATEUP) or tile
    const int l = MODE == MODE_GATEUP && rho >= HN ? rho - HN : rho;
    return l < have ? l : have - 1;
  };
  const int64_t up = MODE == MODE_GATEUP ? (int64_t)a.inter : 0;
  // each wave copies rows of one half: one resource per wave, its base uniform
  const int64_t wbase = row0 + (MODE == MODE_GATEUP && wave >= 2 ? up : 0);
  const __amdgpu_buffer_rsrc_t wr = rsrc32(a.w.i4 + wbase * rowbytes, have * rowbytes);
  const __amdgpu_buffer_rsrc_t sg = rsrc32(a.w.i4_scales + row0 * ngs, have * ngs * 2);
  const __amdgpu_buffer_rsrc_t su = rsrc32(a.w.i4_scales + (row0 + up) * ngs, have * ngs * 2);

  // ---- copies: wave's instruction q fills LDS rows 4j.. (activations, j = wave
  // QA + q, 16 columns each) / 8j.. (weights, j = wave QB + q, 8 columns each)
  const uint16_t* pA[QA];
  int cA[QA];
#pragma unroll
  for (int q = 0; q < QA; ++q) {
    const int m = (wave * QA + q) * 4 + (lane >> 4);
    const int mm = m < cnt ? m : cnt - 1;  // rows past the group repeat its last row
    const int64_t row = MODE == MODE_GATEUP || (MODE == MODE_PLAIN && a.gather)
                            ? a.row_slot[pos0 + mm] / a.slot_div
                            : pos0 + mm;
    cA[q] = ((lane & 15) ^ ra_swz(m & 15)) * 8;  // k of this lane's piece in the chunk
    pA[q] = a.x + row * a.x_stride + cA[q];
  }
  int vB[QB], cB[QB];
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    const int rho = (wave * QB + q) * 16 + (lane >> 2);
    cB[q] = (lane & 3) ^ rb_swz(rho & 15);
    vB[q] = lrow(rho) * rowbytes + cB[q] * 16;
  }
  auto brow = [&](int t) {  // first LDS weight row of this wave's tile t
    if constexpr (MODE == MODE_GATEUP)
      return t < HALF ? wave * HALF * 16 + t * 16 : HN + wave * HALF * 16 + (t - HALF) * 16;
    else
      return wave * NTW * 16 + t * 16;
  };

  auto copy_a = [&](unsigned char* A, int ch) {
    if (ch >= nch) return;
#pragma unroll
    for (int q = 0; q < QA; ++q) {
      // past the row's end (a last chunk shorter than 128 k) the lane reads the
      // chunk's start again: those steps are not multiplied
      const bool in = SPG != 0 || ch * RKC + cA[q] < K;
      gdma16(pA[q] + (int64_t)ch * RKC - (in ? 0 : cA[q]), A + (wave * QA + q) * 1024);
    }
  };
  // (No copy or load here has a scalar offset at or past its resource's end: the
  // range check of the lanes' offsets against size - scalar offset would be
  // against a negative number.)
  auto copy_b = [&](unsigned char* B, int ch) {
    if (ch >= nch) return;
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      // past the row's end in a short last chunk: nothing to fetch
      const int v = SPG != 0 || ch * RKC + cB[q] * 32 < K ? vB[q] : OOB_OFF;
      bdma16(wr, B + (wave * QB + q) * 1024, v, uni_i(ch * (RKC / 2)));
    }
  };

  // ---- scales: 16 consecutive groups of the lane's weight rows at a time, four
  // per lane (kq holds groups 4 kq .. 4 kq + 3 of the window as two dwords); a
  // group's scale is read from the holding lanes with ds_bpermute.  Loading each
  // chunk's scales by itself cost a quarter of the kernel (2-byte loads from 16
  // rows per instruction: Qwen3 gate/up at 187 tokens 59.7 -> 45.6 us without
  // them).
  int vS[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) vS[t] = (lrow(brow(t) + r16) * ngs + kq * 4) * 2;
  uint32_t sc0[NTW], sc1[NTW], sn0[NTW], sn1[NTW];  // this window's and the next one's dwords
  int win = 0;
  auto load_window = [&](uint32_t (&d0)[NTW], uint32_t (&d1)[NTW], int w) {
    // a window past the row's last group (never used) reads window 0 again
    const int off = uni_i(w * 16 < ngs ? w * 32 : 0);
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      const __amdgpu_buffer_rsrc_t sr = MODE == MODE_GATEUP && t >= HALF ? su : sg;
      const uint32_t h0 = __builtin_amdgcn_raw_buffer_load_b16(sr, vS[t], off, 0);
      const uint32_t h1 = __builtin_amdgcn_raw_buffer_load_b16(sr, vS[t] + 2, off, 0);
      const uint32_t h2 = __builtin_amdgcn_raw_buffer_load_b16(sr, vS[t] + 4, off, 0);
      const uint32_t h3 = __builtin_amdgcn_raw_buffer_load_b16(sr, vS[t] + 6, off, 0);
      d0[t] = h0 | (h1 << 16);
      d1[t] = h2 | (h3 << 16);
    }
  };
  // before chunk ch: its steps end at most four groups, so they lie in the
  // window of its first one and the next
  auto advance_window = [&](int ch) {
    const int w = ch * 4 / spg >> 4;
    if (w == win) return;  // wave-uniform
    win = w;
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      sc0[t] = sn0[t];
      sc1[t] = sn1[t];
    }
    load_window(sn0, sn1, w + 1);
  };
  auto scale = [&](int t, int g) {
    const int i = g & 15;
    uint32_t v0 = sc0[t], v1 = sc1[t];
    if (SPG == 0 && (g >> 4) != win) {  // (whole groups per pair never straddle)
      v0 = sn0[t];
      v1 = sn1[t];
    }
    const uint32_t v = i & 2 ? v1 : v0;
    const uint32_t b = (uint32_t)__builtin_amdgcn_ds_bpermute(((i >> 2) * 16 + r16) * 4, (int)v);
    return f16_bits_to_f32((b >> (16 * (i & 1))) & 0xffffu) * kFold;
  };

  const uint32_t dq_mask = __builtin_amdgcn_readfirstlane(0x000F000Fu);
  uint32_t dq_magic = 0x64006400u;
  asm volatile("" : "+v"(dq_magic));

  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t tot[MT][NTW], acc[MT][NTW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NTW; ++t) tot[mt][t] = acc[mt][t] = zero;

  auto flush = [&](int g) {
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      const float sc = scale(t, g);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        tot[mt][t] += sc * acc[mt][t];
        acc[mt][t] = zero;
      }
    }
  };
  // LDS reads of step s: A at column 4 s + kq of row r16 (+ 4 KiB per m-tile), B
  // at column s, dword kq of weight row brow(t) + r16.  Where a scale group holds
  // several steps (group 64, multiples of 128) the order of k inside it is free,
  // and a lane's weights for those steps are one read: k = 64 h + 16 kq + 8 j (step
  // s = 2 h + j, 8 bytes) or k = 32 kq + 8 s (16 bytes), A read at the same k.  These
  // reads are free of bank conflicts under the maps above, but for group 64 outside
  // gate/up: the 8-byte reads of a wave's two neighbouring weight tiles become one
  // instruction there, 22 % of the LDS cycles conflicts.  With the loop as
  // one body per stage (fewer registers): Qwen3 shape at 187 tokens 98.4 -> 95.0 us
  // a layer, Mixtral at 100 tokens 315 -> 308, group 96 at 64 tokens 75 -> 70.5,
  // group 64 the same.
  const int asw = ra_swz(r16), bsw = rb_swz(r16);
  auto chunk = [&](const unsigned char* A, const unsigned char* B, int ch) {
    uint32_t bw[NTW][4];
    if constexpr (SPG == 4) {
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const uint4 v =
            *reinterpret_cast<const uint4*>(B + (brow(t) + r16) * 64 + ((kq ^ bsw) * 16));
        bw[t][0] = v.x, bw[t][1] = v.y, bw[t][2] = v.z, bw[t][3] = v.w;
      }
    } else if constexpr (SPG == 2) {
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint2 v = *reinterpret_cast<const uint2*>(
              B + (brow(t) + r16) * 64 + (((2 * h + (kq >> 1)) ^ bsw) * 16) + (kq & 1) * 8);
          bw[t][2 * h] = v.x, bw[t][2 * h + 1] = v.y;
        }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (SPG == 0 && ch * 4 + s >= K / 32) break;  // wave-uniform: end of the contraction
      uint4 af[MT], bf[NTW];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int col = SPG == 4   ? 4 * kq + s
                        : SPG == 2 ? 8 * (s >> 1) + 2 * kq + (s & 1)
                                   : 4 * s + kq;
        af[mt] = *reinterpret_cast<const uint4*>(A + (mt * 16 + r16) * 256 + ((col ^ asw) * 16));
      }
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        if constexpr (SPG != 4 && SPG != 2)
          bw[t][s] = *reinterpret_cast<const uint32_t*>(B + (brow(t) + r16) * 64 +
                                                        ((s ^ bsw) * 16) + kq * 4);
        bf[t] = deq_signed<BF>(bw[t][s], dq_mask, dq_magic);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < NTW; ++t) acc[mt][t] = dmfma<BF>(af[mt], bf[t], acc[mt][t]);

      if constexpr (SPG == 4) {
        if (s == 3) flush(ch * RKC / a.group_size);
      } else if constexpr (SPG != 0) {
        if ((s + 1) % SPG == 0) flush(ch * (4 / SPG) + s / SPG);
      } else {
        const int st = ch * 4 + s;
        if ((st + 1) % spg == 0) flush(st / spg);
      }
    }
  };

  // Every copy of this wave has landed and its LDS reads are done; behind the
  // barrier every wave's are, and what they read may be overwritten.  (The
  // builtin wait is known to the compiler's own wait insertion, which otherwise
  // waits again at the chunk's first LDS read.)
  auto barrier = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  load_window(sc0, sc1, 0);
  load_window(sn0, sn1, 1);
  copy_a(sA[0], 0);
  copy_b(sB[0], 0);
  for (int ch0 = 0; ch0 < nch; ch0 += 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // the stage is a constant in each copy of the body
      const int ch = ch0 + i;
      if (ch >= nch) break;
      barrier();
      advance_window(ch);
      copy_b(sB[1 - i], ch + 1);
      copy_a(sA[1 - i], ch + 1);
      __builtin_amdgcn_sched_barrier(0);
      chunk(sA[i], sB[i], ch);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy outlives the work-group

  // D layout: lane (r16, kq) holds rows 4 kq + i of each tile, column r16
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + kq * 4 + i;
      if (m >= cnt) continue;
      const int pos = pos0 + m;
      if constexpr (MODE == MODE_GATEUP) {
        uint16_t* mid = reinterpret_cast<uint16_t*>(a.out) + (int64_t)pos * a.out_stride + c0;
#pragma unroll
        for (int t = 0; t < HALF; ++t)
          if (brow(t) + r16 < have)
            mid[brow(t) + r16] =
                (uint16_t)to_act_bits<BF>(silu_f32(tot[mt][t][i]) * tot[mt][t + HALF][i]);
      } else if constexpr (MODE == MODE_PLAIN) {
        uint16_t* c = reinterpret_cast<uint16_t*>(a.out) + (int64_t)pos * a.out_stride + c0;
#pragma unroll
        for (int t = 0; t < NTW; ++t)
          if (brow(t) + r16 < have) c[brow(t) + r16] = (uint16_t)to_act_bits<BF>(tot[mt][t][i]);
      } else {
        float* part =
            reinterpret_cast<float*>(a.out) + (int64_t)a.row_slot[pos] * a.out_stride + c0;
#pragma unroll
        for (int t = 0; t < NTW; ++t)
          if (brow(t) + r16 < have) part[brow(t) + r16] = tot[mt][t][i];
      }
    }
  }
}

template <bool BF, int MODE, int SPG>
__global__ void __launch_bounds__(RTH, 4) rows_kernel(GemmArgs a, int n_tiles) {
  __shared__ __attribute__((aligned(1024))) unsigned char sA0[MT * 4096];
  __shared__ __attribute__((aligned(1024))) unsigned char sA1[MT * 4096];
  __shared__ __attribute__((aligned(1024))) unsigned char sB0[NTW * 4096];
  __shared__ __attribute__((aligned(1024))) unsigned char sB1[NTW * 4096];
  unsigned char* const sA[2] = {sA0, sA1};
  unsigned char* const sB[2] = {sB0, sB1};
  rows_body<BF, MODE, SPG>(a, n_tiles, sA, sB);
}

// Unquantised weights: C = A x W^T with the same 32-row x 128-weight-row
// work-groups, in chunks of 64 k (32 rows x 128 B and 128 rows x 128 B, whole
// cache lines; 40 KiB of LDS for two stages, four work-groups per CU with 64 KiB
// of weights in flight).  Lane (r, q) at k-step s holds k = 32 s + 8 q .. + 7 of
// both operands, both LDS images swizzled by w_swz (free of bank conflicts);
// the fp32 accumulators run over the whole contraction.
//
// Bound: HBM, the weights of the active experts read once.  OLMoE shape (K =
// 2048, 2048 weight rows) at 96 tokens: 115 us on the 128 x 128 tiles (whose
// activation rows are mostly padding there) -> 107 us.  An expert with one token
// group has its weights copied with the nontemporal hint, as only this work-group
// reads them: the layer 196 -> 178 us (Qwen3 shape at 40 tokens 137 -> 126).
// Weights that several groups share stay cached: the hint on them too cost 188 us
// there and 244 -> 258 at 250 tokens.  The INT4 kernel's 64-byte row pieces are
// half lines, and the hint loses the other half: 95 -> 105 us at 187 tokens.
constexpr int WKC = 64;
__device__ __forceinline__ int w_swz(int r) { return (r >> 1) & 7; }

template <bool BF>
__global__ void __launch_bounds__(RTH, 4) rows_bf16_kernel(GemmArgs a, int n_tiles) {
  __shared__ __attribute__((aligned(1024))) unsigned char sA0[MT * 16 * WKC * 2];
  __shared__ __attribute__((aligned(1024))) unsigned char sA1[MT * 16 * WKC * 2];
  __shared__ __attribute__((aligned(1024))) unsigned char sB0[TN * WKC * 2];
  __shared__ __attribute__((aligned(1024))) unsigned char sB1[TN * WKC * 2];
  static_assert(MT == 2, "one activation copy per wave and chunk");
  constexpr int QB = TN / 32;  // weight copies per wave and chunk (8 rows each)
  TgEntry te;
  int nt;
  bool once;
  if (!rows_unit(a, 0, a.hdr[2], n_tiles, blockIdx.x, te, nt, &once)) return;  // BF16 groups
  nt = uni_i(nt);
  const bool nontemporal = uni_i(once ? 1 : 0) != 0;
  const int cnt = uni_i(te.cnt), pos0 = uni_i(te.pos0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int K = a.K, nch = K / WKC;  // an even number of chunks: K % 128 == 0
  const int c0 = nt * TN;
  const int left = a.n_rows - c0;
  const int have = left < TN ? left : TN;
  const int e = uni_i(te.e);
  const int64_t row0 = (int64_t)(a.w.index ? uni_i(a.w.index[e]) : e) * a.n_rows + c0;
  const __amdgpu_buffer_rsrc_t wr = rsrc32(a.w.bf16 + row0 * K, have * K * 2);

  // copies: 8 rows x 8 columns of 16 bytes per instruction
  const int m = wave * 8 + (lane >> 3);
  const int mm = m < cnt ? m : cnt - 1;  // rows past the group repeat its last row
  const int64_t xrow = a.gather ? a.row_slot[pos0 + mm] / a.slot_div : pos0 + mm;
  const uint16_t* pA = a.x + xrow * a.x_stride + ((lane & 7) ^ w_swz(m & 15)) * 8;
  int vB[QB];
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    const int rho = (wave * QB + q) * 8 + (lane >> 3);
    const int l = rho < have ? rho : have - 1;  // rows past the end repeat the last one
    vB[q] = l * K * 2 + ((lane & 7) ^ w_swz(rho & 15)) * 16;
  }
  auto copy = [&](unsigned char* A, unsigned char* B, int ch) {
    if (ch >= nch) return;
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      if (nontemporal)
        bdma16<2>(wr, B + (wave * QB + q) * 1024, vB[q], uni_i(ch * WKC * 2));
      else
        bdma16(wr, B + (wave * QB + q) * 1024, vB[q], uni_i(ch * WKC * 2));
    }
    gdma16(pA + (int64_t)ch * WKC, A + wave * 1024);
  };
  f32x4_t acc[MT][NTW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NTW; ++t) acc[mt][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int swz = w_swz(r16);
  auto chunk = [&](const unsigned char* A, const unsigned char* B) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint4 af[MT], bf[NTW];
      const int col = ((4 * s + kq) ^ swz) * 16;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        af[mt] = *reinterpret_cast<const uint4*>(A + (mt * 16 + r16) * 128 + col);
#pragma unroll
      for (int t = 0; t < NTW; ++t)
        bf[t] = *reinterpret_cast<const uint4*>(B + ((wave * NTW + t) * 16 + r16) * 128 + col);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NTW; ++t) acc[mt][t] = dmfma<BF>(af[mt], bf[t], acc[mt][t]);
    }
  };
  auto barrier = [&]() {  // as in rows_body
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  copy(sA0, sB0, 0);
  for (int ch = 0; ch < nch; ch += 2) {
    barrier();
    copy(sA1, sB1, ch + 1);
    __builtin_amdgcn_sched_barrier(0);
    chunk(sA0, sB0);
    barrier();
    copy(sA0, sB0, ch + 2);
    __builtin_amdgcn_sched_barrier(0);
    chunk(sA1, sB1);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int mr = mt * 16 + kq * 4 + i;
      if (mr >= cnt) continue;
      uint16_t* c = reinterpret_cast<uint16_t*>(a.out) + (int64_t)(pos0 + mr) * a.out_stride + c0;
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const int col = (wave * NTW + t) * 16 + r16;
        if (col < have) c[col] = (uint16_t)to_act_bits<BF>(acc[mt][t][i]);
      }
    }
  }
}

template <int MODE, int SPG>
int launch_spg(bool bf, const GemmArgs& a, int64_t grid, int n_tiles, hipStream_t s) {
  const dim3 g((unsigned)grid), b(RTH);
  if (bf)
    hipLaunchKernelGGL((rows_kernel<true, MODE, SPG>), g, b, 0, s, a, n_tiles);
  else
    hipLaunchKernelGGL((rows_kernel<false, MODE, SPG>), g, b, 0, s, a, n_tiles);
  return check_launch("rows_kernel");
}

template <int MODE>
int launch_mode(bool bf, const GemmArgs& a, int64_t tg_cap, hipStream_t s) {
  const int n_tiles = (int)(MODE == MODE_GATEUP ? cdiv(a.inter, TN / 2) : cdiv(a.n_rows, TN));
  const int64_t grid = 8 * cdiv(tg_cap, 8) * n_tiles;
  if (grid <= 0) return EXQ_SUCCESS;
  if (grid > INT32_MAX) return set_error(EXQ_ERROR_UNSUPPORTED, "rows_gemm: problem too large");
  const bool whole = a.K % RKC == 0;
  if (whole && a.group_size % 128 == 0) return launch_spg<MODE, 4>(bf, a, grid, n_tiles, s);
  if (whole && a.group_size == 64) return launch_spg<MODE, 2>(bf, a, grid, n_tiles, s);
  if (whole && a.group_size == 32) return launch_spg<MODE, 1>(bf, a, grid, n_tiles, s);
  return launch_spg<MODE, 0>(bf, a, grid, n_tiles, s);
}

}  // namespace

bool general_shape(int64_t K, int64_t group_size) {
  return K >= 32 && K % 32 == 0 && group_size >= 32 && group_size % 32 == 0 &&
         K % group_size == 0;
}

int launch_rows_gemm(int mode, bool bf, const GemmArgs& a, int64_t tg_cap, hipStream_t s) {
  if (a.K > (1 << 24))  // 32-bit offsets inside a tile's weight rows
    return set_error(EXQ_ERROR_UNSUPPORTED, "rows_gemm: contraction of %d too long", a.K);
  if (mode == MODE_GATEUP) return launch_mode<MODE_GATEUP>(bf, a, tg_cap, s);
  if (mode == MODE_DOWN) return launch_mode<MODE_DOWN>(bf, a, tg_cap, s);
  return launch_mode<MODE_PLAIN>(bf, a, tg_cap, s);
}

int launch_rows_gemm_bf16(bool bf, const GemmArgs& a, int64_t tg_cap, hipStream_t s) {
  if (a.K > (1 << 22))  // 32-bit offsets inside a tile's weight rows
    return set_error(EXQ_ERROR_UNSUPPORTED, "rows_gemm: contraction of %d too long", a.K);
  const int n_tiles = (int)cdiv(a.n_rows, TN);
  const int64_t grid = 8 * cdiv(tg_cap, 8) * n_tiles;
  if (grid <= 0) return EXQ_SUCCESS;
  if (grid > INT32_MAX) return set_error(EXQ_ERROR_UNSUPPORTED, "rows_gemm: problem too large");
  const dim3 g((unsigned)grid), b(RTH);
  if (bf)
    hipLaunchKernelGGL(rows_bf16_kernel<true>, g, b, 0, s, a, n_tiles);
  else
    hipLaunchKernelGGL(rows_bf16_kernel<false>, g, b, 0, s, a, n_tiles);
  return check_launch("rows_bf16_kernel");
}

}  // namespace exq
