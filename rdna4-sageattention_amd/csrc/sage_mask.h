// Attention masks (bool, or additive bf16 / fp16): the device work that turns a torch mask into the tables the
// attention kernel's mask variant reads (MaskTabs in sage_host.h).  It runs as extra workgroups of sage_forward's
// two quantization launches (no launch of its own): the bits, classes and bias values in the first, the
// per-workgroup tile ranges in the second, which stream order places after the first.
#pragma once

#include "sage_common.h"
#include "sage_host.h"

namespace sage {

// Everything the two kinds of mask workgroups need.  prep_blocks / range_blocks = 0: no mask work (the dense call).
struct MaskPrep {
  const void* mask;         // element (b, h, row, key) at mask + b*msb + h*msh + row*msq + key (element strides)
  int mdt;                  // SAGE_DTYPE_BOOL (nonzero byte = attend) or SAGE_DTYPE_BF16 / SAGE_DTYPE_F16 (additive)
  int64_t msb, msh, msq;
  int mh, mq, mg, nt, nrb;  // table extents (sage_mask.hip: mask_shape)
  int Sq, Skv, causal;
  int a4;                   // bool rows aligned to a run of 4 keys (4 bytes): one load per run
  uint32_t* bits;
  uint16_t* bias;           // 16-bit masks: the 64 values of every row's partial last tile (-inf past kv_len)
  int* cls;
  int2* range;
  int nrange;               // mb * mh * nrb
  int prep_blocks, range_blocks;
};

typedef unsigned short v2us __attribute__((ext_vector_type(2)));

// 1 in each 16-bit half of x that is not 0
__device__ __forceinline__ uint32_t nonzero_halves(uint32_t x) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(v2us, x), v2us{1, 1}));
}

// The visibility word of the lane's 32 keys of a bool mask (bit order below); keys past `lim` are not visible.
__device__ __forceinline__ uint32_t mask_bool_word(const MaskPrep& p, const uint8_t* row, int k0, int lim) {
  uint32_t b4[8], w = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int kj = k0 + 8 * j;
    if (p.a4 && kj + 3 < p.Skv) {
      b4[j] = *reinterpret_cast<const uint32_t*>(row + kj);
    } else {
      b4[j] = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (kj + i < p.Skv) b4[j] |= (uint32_t)row[kj + i] << (8 * i);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool vis = ((b4[j] >> (8 * i)) & 0xFFu) != 0 && k0 + 8 * j + i <= lim;
      w |= (uint32_t)vis << (4 * j + i);
    }
  return w;
}

// One wave per (mask batch-head, 32-row group, tile); a block is 4 waves on 4 consecutive tiles.  Lane (row r =
// lane % 32 of the group, half hf = lane / 32) writes the visibility word of its 32 keys: bits 4 j + i for key
// 64 t + 8 j + 4 hf + i.  Bool masks: the lane reads those keys (8 runs of 4); a key is visible when its byte is
// nonzero.  16-bit (additive) masks: the two lanes of a row read alternate 16-byte chunks (8 keys each) and exchange
// the half-words the other one needs; a key is visible when its value is not -inf; the values a lane reads are also
// "zero" (every one +-0) or "general" (some value neither 0 nor -inf).  Keys past kv_len and, causal, past the
// bottom-right diagonal are -inf.  Wave ballots give the class: 0 no row sees a key, 1 every key of every row visible
// with a zero bias, 2 visibility only (bool masks, or 16-bit values all 0 / -inf), 3 a general bias.  The attention
// reads the values of class-3 tiles from the mask itself; only those of a partial last tile are copied here, padded
// with -inf, so that it never reads past a row's end.  Rows past q_len (and, for a mask without rows, every row but 0)
// count as neither seeing nor missing a key.  block < mb * mh * mg * ceil(nt / 4).
//
// A 16-bit mask is read once here (HBM bound) and once by the attention.
__device__ __forceinline__ void mask_prep_block(const MaskPrep& p, int block) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 31, hf = lane >> 5;
  const int ntb = (p.nt + 3) >> 2;
  const int t = (block % ntb) * 4 + wave;
  const int rest = block / ntb;
  const int g = rest % p.mg;
  const int mbh = rest / p.mg;
  if (t >= p.nt) return;  // the whole wave
  const int mbi = mbh / p.mh, mhi = mbh % p.mh;
  const int q = g * 32 + r;  // table row (mq == 1: row 0 only)
  const bool real = p.mq == 1 ? r == 0 : q < p.Sq;
  uint32_t w = 0;
  bool zero = true, general = false;
  v4i c[4] = {};  // 16-bit masks: the lane's chunks, keys [64 t + 16 i + 8 hf, + 8)
  const bool part = (t + 1) * 64 > p.Skv;
  if (real) {
    const int lim = p.causal ? min(p.Skv - 1, q + (p.Skv - p.Sq)) : p.Skv - 1;  // last key the row may see
    const int64_t rowoff = mbi * p.msb + mhi * p.msh + (int64_t)q * p.msq;
    if (p.mdt == SAGE_DTYPE_BOOL) {
      w = mask_bool_word(p, static_cast<const uint8_t*>(p.mask) + rowoff, t * 64 + 4 * hf, lim);
    } else {
      const uint32_t ninf = p.mdt == SAGE_DTYPE_BF16 ? 0xFF80u : 0xFC00u;
      const uint16_t* row = static_cast<const uint16_t*>(p.mask) + rowoff + t * 64 + 8 * hf;
      const int left = lim - t * 64 - 8 * hf;  // the lane's key 16 i + e is visible when 16 i + e <= left
      if (!part) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = load16_2aligned(row + 16 * i);
      } else {
        const int in_row = p.Skv - 1 - t * 64 - 8 * hf;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t e[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) e[u] = 16 * i + u <= in_row ? (uint32_t)row[16 * i + u] : ninf;
#pragma unroll
          for (int d = 0; d < 4; ++d) c[i][d] = (int)(e[2 * d] | (e[2 * d + 1] << 16));
        }
      }
      if (p.causal && t * 64 + 63 > g * 32 + (p.Skv - p.Sq)) {  // wave-uniform: the tile crosses some row's diagonal
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            uint32_t x = (uint32_t)c[i][d];
            if (16 * i + 2 * d > left) x = (x & 0xFFFF0000u) | ninf;
            if (16 * i + 2 * d + 1 > left) x = (x & 0xFFFFu) | (ninf << 16);
            c[i][d] = (int)x;
          }
        }
      }
      uint32_t anynz = 0, gen = 0, lo = 0, hi = 0;  // lo / hi: visibility of the chunks' first / last 4 keys
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t nz = nonzero_halves((uint32_t)c[i][d] & 0x7FFF7FFFu);
          const uint32_t vis = nonzero_halves((uint32_t)c[i][d] ^ (ninf * 0x10001u));
          anynz |= nz;
          gen |= nz & vis;
          const uint32_t two = (vis | (vis >> 15)) & 3u;
          if (d < 2)
            lo |= two << (8 * i + 2 * d);
          else
            hi |= two << (8 * i + 2 * (d - 2));
        }
      }
      zero = anynz == 0;
      general = gen != 0;
      // lane hf holds the chunks j = 2 i + hf (bits 4 j): its own half of them is the word's, the other half goes to
      // the row's other lane
      const auto x = __builtin_amdgcn_permlane32_swap(lo << (4 * hf), hi << (4 * hf), false, false);
      w = x[0] | x[1];
    }
    p.bits[((int64_t)mbh * p.mq + q) * p.nt * 2 + t * 2 + hf] = w;
  }
  const uint64_t any = __ballot(real && w != 0);
  const uint64_t all = __ballot(!real || (w == 0xFFFFFFFFu && zero));
  const uint64_t gen = __ballot(real && general);
  const int cls = any == 0 ? 0 : gen != 0 ? 3 : all == ~0ull ? 1 : 2;
  if (cls == 3 && part && real) {  // wave-uniform class
    uint16_t* dst = p.bias + ((int64_t)mbh * p.mq + q) * 64 + 8 * hf;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<v4i*>(dst + 16 * i) = c[i];
  }
  if (lane == 0) p.cls[((int64_t)mbh * p.mg + g) * p.nt + t] = cls;
}

// One wave per (mask batch-head, 128-row block): the first and one past the last tile whose class is not 0 in any of
// the block's four 32-row groups (groups past the last one repeat it), (nt, 0) when there is none.  Lanes scan the
// 4 x nt classes with all their loads in flight, then a wave reduction.  block < ceil(nrange / 4).
__device__ __forceinline__ void mask_range_block(const MaskPrep& p, int block) {
  const int wid = block * 4 + (int)(threadIdx.x >> 6);
  if (wid >= p.nrange) return;  // the whole wave
  const int lane = threadIdx.x & 63;
  const int mbh = wid / p.nrb, rb = wid % p.nrb;
  int lo = p.nt, hi = -1;
  for (int i = lane; i < 4 * p.nt; i += 64) {
    const int g = min(rb * 4 + i / p.nt, p.mg - 1), t = i % p.nt;
    if (p.cls[((int64_t)mbh * p.mg + g) * p.nt + t] != 0) {
      lo = min(lo, t);
      hi = max(hi, t);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  if (lane == 0) p.range[wid] = make_int2(lo, hi + 1);
}

}  // namespace sage
