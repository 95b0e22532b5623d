// LDS tile helpers shared by the flash-attention kernels (flash_attn.hip: head size 128, flash_attn_d256.hip: 256).
// Tiles use 256-byte rows (128 bf16) with the 16-byte-chunk XOR swizzle
//   off(row, ch) = 256*row + 16*(ch ^ (((row&3)<<2) | ((row>>2)&3)))
// which is conflict-free for both ds_read_b128 row reads and transposed reads.
#pragma once
#include "common.hpp"

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

DEVINL f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// (exponentials go through fast_exp2 of common.hpp: v_exp_f32 directly; exp2f() expands to a denormal-safe
// sequence (scale, v_exp, ldexp, compare) that the compiler then guards with per-element branches)
DEVINL int swz_off(int row, int ch) {  // byte offset of 16-byte chunk `ch` of `row`
  return 256 * row + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3)));
}
// Transposed read of a 4-row x 16-col block: every lane supplies the address of
// (row0 + q, col0 + 4p) with its group-lane index 4q+p and receives column `i` of the four
// rows. `base` is the LDS tile, rows are 256 bytes, col0 must be a multiple of 16.
DEVINL bf16x4 tr_read(const char* tile, int row0, int col0, int gl) {
  const int q = gl >> 2, p = gl & 3;
  const int ch = (col0 >> 3) + (p >> 1);
  const char* a = tile + swz_off(row0 + q, ch) + 8 * (p & 1);
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(a));
}
// The same read split in two: the address (loop-invariant when a tile is restaged in place) and the load.
DEVINL const char* tr_addr(const char* tile, int row0, int col0, int gl) {
  const int q = gl >> 2, p = gl & 3;
  const int ch = (col0 >> 3) + (p >> 1);
  return tile + swz_off(row0 + q, ch) + 8 * (p & 1);
}
DEVINL bf16x4 tr_load(const char* a) { return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(a)); }
DEVINL bf16x8 cat4(bf16x4 a, bf16x4 b) {
  bf16x8 r;
  r[0] = a[0]; r[1] = a[1]; r[2] = a[2]; r[3] = a[3];
  r[4] = b[0]; r[5] = b[1]; r[6] = b[2]; r[7] = b[3];
  return r;
}
DEVINL bf16x8 lds_row_read(const char* tile, int row, int ch) {
  return *reinterpret_cast<const bf16x8*>(tile + swz_off(row, ch));
}
DEVINL void lds_row_write(char* tile, int row, int ch, bf16x8 v) {
  *reinterpret_cast<bf16x8*>(tile + swz_off(row, ch)) = v;
}

// ---- gradients of rows that belong to no sequence: zero. A backward's first kernel visits every (token t, head h), `at`: the
// 8 values of a head that this lane is responsible for.
struct FlashGrads {
  bf16_t *dq, *dk, *dv;
  int64_t dq_stride, dk_stride, dv_stride, total_q, total_k;
  const int *cu_q, *cu_k;
  int nbatch, Hkv;
};
DEVINL void flash_zero_uncovered(const FlashGrads& g, int64_t t, int h, int D, int at) {
  const bf16x8 zero = {};
  const size_t col = (size_t)h * D + at;
  if (t < g.total_q && (t < g.cu_q[0] || t >= g.cu_q[g.nbatch])) st8(g.dq + t * g.dq_stride + col, zero);
  if (h < g.Hkv && t < g.total_k && (t < g.cu_k[0] || t >= g.cu_k[g.nbatch])) {
    st8(g.dk + t * g.dk_stride + col, zero);
    st8(g.dv + t * g.dv_stride + col, zero);
  }
}

// ---- staging of 64-row tiles by LDS-DMA. One wave instruction (16 bytes a lane) fills four consecutive 256-byte rows of a
// tile linearly; the swizzle sits on the source address: lane -> row (lane >> 4) of the four, physical chunk lane & 15.
typedef __attribute__((address_space(3))) void* dma_lptr_t;
// In assembly, because behind the builtin the compiler cannot tell the reads of one buffer from the pending writes of the other and
// puts a wait for all of them in front of the first read: the tile after this one was waited for before this one was computed.
// Nothing comes back into registers; what waits is `dma_arrive`, in front of every read of a tile. With `dma_pin` and the row
// statistics of a slice chosen behind its arrival, us, forward / backward, 12 query heads on 2: 25 sequences of up to 1133 tokens 154 -> 143 /
// 580 -> 514, one of 24576 1842 -> 1784 / 6307 -> 5853; 16 heads, 8 of 2048 206 -> 177 / 671 -> 604; short ones level.
// The destination goes through m0, which the compiler does not let assembly clobber: it is put back, and a load of the compiler's own
// that takes it right behind finds it settled. Once for all pieces of a tile, 1 KiB apart: once for each took 0.5 to 1 % of a pass.
#define DMA_FIRST "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %2"
#define DMA_NEXT(off) "\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 " off ", %2"
#define DMA_LAST "\n\ts_mov_b32 m0, %0\n\ts_nop 0"
DEVINL void dma16(const char* base, const unsigned (&off)[4], const void* lds) {
  const unsigned at = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(dma_lptr_t)lds);
  unsigned m0;
  asm volatile(DMA_FIRST DMA_NEXT("%4") DMA_NEXT("%5") DMA_NEXT("%6") DMA_LAST
               : "=&s"(m0) : "s"(at), "s"(base), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]) : "memory", "scc");
}
DEVINL void dma16(const char* base, const unsigned (&off)[2], const void* lds) {
  const unsigned at = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(dma_lptr_t)lds);
  unsigned m0;
  asm volatile(DMA_FIRST DMA_NEXT("%4") DMA_LAST : "=&s"(m0) : "s"(at), "s"(base), "v"(off[0]), "v"(off[1]) : "memory", "scc");
}
#undef DMA_FIRST
#undef DMA_NEXT
#undef DMA_LAST
// Registers that were loaded ahead of a loop of tiles are waited for here, once, not at their first use in every round of it
template <int N>
DEVINL void dma_pin(bf16x8 (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}
// Rows 16 w + 4 i + (lane >> 4), i = 0..3, of a tile of 64 rows go through wave w of four. `off`: this lane's byte offsets of
// the four pieces for rows `stride` elements apart.
constexpr int64_t FLASH_MAX_STRIDE = 1 << 24;  // elements: the byte offsets of 64 rows fit 32 bits
DEVINL void dma_offsets(unsigned (&off)[4], int wave, int lane, int64_t stride) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * wave + 4 * i + (lane >> 4), chunk = (lane & 15) ^ (((lane >> 4) << 2) | i);
    off[i] = (unsigned)(row * stride + chunk * 8) * 2;
  }
}
// base: row 0 of the tile (uniform); rows from `rows` on repeat row rows - 1. The base is kept in scalar registers (the
// compiler would otherwise carry one 64-bit pointer a piece and lane through the loop).
DEVINL void dma_tile(const bf16_t* base, const unsigned (&off)[4], int64_t stride, int rows, char* tile, int wave, int lane) {
  char* dst = tile + wave * 4096;
  const char* b = reinterpret_cast<const char*>(base);
  asm volatile("" : "+s"(b));
  if (rows >= 64) {
    dma16(b, off, dst);
  } else {
    unsigned last[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * wave + 4 * i + (lane >> 4), over = row < rows ? 0 : row - (rows - 1);
      // (same chunk order as row `row` would have: the swizzle belongs to the place in the tile)
      last[i] = off[i] - (unsigned)(over * stride) * 2;
    }
    dma16(b, last, dst);
  }
}
// every DMA of this wave has landed; then all waves have said so (and have finished reading the other buffer)
DEVINL void dma_arrive() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 32-row tiles, two pieces of each wave of four: rows 8 w + 4 i + (lane >> 4), i = 0, 1
DEVINL void dma_offsets32(unsigned (&off)[2], int wave, int lane, int64_t stride) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * wave + 4 * i + (lane >> 4), chunk = (lane & 15) ^ (((lane >> 4) << 2) | ((2 * wave + i) & 3));
    off[i] = (unsigned)(row * stride + chunk * 8) * 2;
  }
}
DEVINL void dma_tile32(const bf16_t* base, const unsigned (&off)[2], int64_t stride, int rows, char* tile, int wave, int lane) {
  char* dst = tile + wave * 2048;
  const char* b = reinterpret_cast<const char*>(base);
  asm volatile("" : "+s"(b));
  if (rows >= 32) {
    dma16(b, off, dst);
  } else {
    unsigned last[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 8 * wave + 4 * i + (lane >> 4), over = row < rows ? 0 : row - (rows - 1);
      last[i] = off[i] - (unsigned)(over * stride) * 2;
    }
    dma16(b, last, dst);
  }
}

// Byte offsets inside a tile of this lane's fragment reads. row(s): row r = lane & 31 of a 32-row block, chunk 2 s + hf (add
// 8192 per block); tr0(db), tr1(db): rows 4 hf + .. (second: + 8), 16-column block 2 db + (grp & 1), transposed (add 4096 per
// 16 rows). The chunk's bits of s and db do not meet the swizzle's carry: one register each and an exclusive or.
struct FragOffsets {
  int r0, t0, t1;
  DEVINL FragOffsets(int lane) {
    const int hf = lane >> 5, gl = lane & 15, grp = lane >> 4, ch = 2 * (grp & 1) + ((gl & 3) >> 1);
    r0 = swz_off(lane & 31, hf);
    t0 = swz_off(4 * hf + (gl >> 2), ch) + 8 * (gl & 1);
    t1 = swz_off(8 + 4 * hf + (gl >> 2), ch) + 8 * (gl & 1);
  }
  DEVINL int row(int s) const { return r0 ^ (s << 5); }
  DEVINL int tr0(int db) const { return t0 ^ (db << 6); }
  DEVINL int tr1(int db) const { return t1 ^ (db << 6); }
};
