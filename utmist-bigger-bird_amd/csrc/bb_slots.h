// Key slots of the decode kernels: 8 lanes per cached row, 8 rows per wave; reductions on VALU lane moves.
#pragma once
#include "bb_common.h"

namespace bb {
namespace {

// fp32 c + a.x b.x + a.y b.y over packed 16-bit pairs (one v_dot2c_f32_{bf16,f16}).
template <bool F16>
BB_DEV float dot2(uint32_t a, uint32_t b, float c) {
  typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2_t;
  if constexpr (F16)
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, a), __builtin_bit_cast(f16x2_t, b), c, false);
  else return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}

// The decode kernels read each cached row with the 8 lanes of a key slot. Lane `sub` holds the 16-byte pieces
// sub, sub + 8, ... of the row (element offset piece_off(sub, e0)), so that each load instruction of the slot covers
// whole 128-byte spans of the row: the rows are read once per step, with non-temporal loads (global_load ... nt),
// which stream at about 7.1 TB/s where plain loads reach 6.2-6.3 (16-byte reads over 4 GiB, measured) but which
// fetch whole lines for every instruction, so a lane layout that left half-lines per instruction read them twice.
constexpr int kSlotLanes = 8;
BB_DEV int piece_off(int sub, int e0) { return 8 * (sub + kSlotLanes * e0); }
// Sum over the kSlotLanes = 8 lanes of a key slot (lane bits 0..2), the same value in every lane of the slot, on DPP
// lane moves inside the VALU: quad_perm [1, 0, 3, 2], quad_perm [2, 3, 0, 1], then row_half_mirror (lane i of an
// 8-lane half row reads lane 7 - i, which lies in the other quad and holds that quad's sum). The additions pair the
// same values as a butterfly over lane xor 1, 2, 4, and each lane adds the pair in either order, so every lane holds
// the same bits. (__shfl_xor goes through the LDS crossbar, ds_bpermute, with a wait per round.)
template <int CTRL>
BB_DEV float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
BB_DEV float slot_sum8(float v) {
  static_assert(kSlotLanes == 8, "the DPP pattern reduces 8-lane slots");
  v += dpp_mov<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_mov<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_mov<0x141>(v);  // row_half_mirror
  return v;
}
BB_DEV u32x4_t ld16_nt(const void* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p)); }

// Sum and maximum over the 8 key slots of a wave (lane bits 3..5), the same bits in every lane: row_ror 8, then the
// permlane16 and permlane32 swaps, all inside the VALU (a __shfl_xor is an LDS crossbar round trip per value).
BB_DEV float slots_sum(float v) {
  v += dpp_mov<0x128>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_sum(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}
BB_DEV float slots_max(float v) {
  v = fmaxf(v, dpp_mov<0x128>(v));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_max(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
}
}  // namespace
}  // namespace bb
