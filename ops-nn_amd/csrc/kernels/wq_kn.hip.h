// Dequantisation of weights in [K, N] storage: an 8 x 8 block (8 rows of k, 8 neighbouring columns) of one lane, dequantised along
// the columns -- that is how the codes and the scales lie -- and delivered per column as 8 consecutive k.
#pragma once
#include "wqmm_common.hip.h"

namespace opsnn {

// q[i]: the codes of row i (int4: one dword, low nibble first; int8: two dwords); sc, of: the 8 columns' scales and offsets in
// x's type, two per dword; o[column][pair of k].  The arithmetic and its two roundings are those of dequant8 in
// wqmm_stream.hip.h; the 8 x 8 transposition is one byte permute per pair of weights (bf16: the packing conversion itself).
template <int XDT, int WBITS, bool HAS_OFF>
__device__ __forceinline__ void dequant_8x8(const uint32_t (&q)[8][WBITS / 4], const uint32_t (&scw)[4], const uint32_t (&ofw)[4], uint32_t (&o)[8][4])
{
    constexpr int DW = WBITS / 4;
    if constexpr (XDT == DT_F16) {
        // per row of k: four pairs of columns -- int4: (0,4) (1,5) (2,6) (3,7), the order of the nibble splice; int8: (0,1) ...
        h2 sc[4], of[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            uint32_t s = scw[t], f = ofw[t];
            if constexpr (WBITS == 4) {   // halves t and t + 4
                const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
                s = __builtin_amdgcn_perm(scw[2 + t / 2], scw[t / 2], sel);
                f = __builtin_amdgcn_perm(ofw[2 + t / 2], ofw[t / 2], sel);
            }
            sc[t] = __builtin_bit_cast(h2, s);
            of[t] = __builtin_bit_cast(h2, f);
        }
        const h2 c1032 = {(_Float16)-1032.0f, (_Float16)-1032.0f}, c72 = {(_Float16)-72.0f, (_Float16)-72.0f}, r16 = {(_Float16)0.0625f, (_Float16)0.0625f};
        const h2 c1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            uint32_t row[2][4];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                h2 t[4];
                if constexpr (WBITS == 4) {
                    const uint32_t u = q[i + r][0], u8 = u >> 8;
                    t[0] = __builtin_bit_cast(h2, (u & 0x000F000Fu) ^ 0x64086408u) + c1032;
                    t[1] = __builtin_elementwise_fma(__builtin_bit_cast(h2, (u & 0x00F000F0u) ^ 0x64806480u), r16, c72);
                    t[2] = __builtin_bit_cast(h2, (u8 & 0x000F000Fu) ^ 0x64086408u) + c1032;
                    t[3] = __builtin_elementwise_fma(__builtin_bit_cast(h2, (u8 & 0x00F000F0u) ^ 0x64806480u), r16, c72);
                } else {
                    const uint32_t qa = q[i + r][0] ^ 0x80808080u, qb = q[i + r][DW - 1] ^ 0x80808080u, magic = 0x64646464u;
                    t[0] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(magic, qa, 0x04010400u)) + c1152;
                    t[1] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(magic, qa, 0x04030402u)) + c1152;
                    t[2] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(magic, qb, 0x04010400u)) + c1152;
                    t[3] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(magic, qb, 0x04030402u)) + c1152;
                }
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    if constexpr (HAS_OFF) t[c] = t[c] + of[c];
                    row[r][c] = u32(t[c] * sc[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int a = WBITS == 4 ? c : 2 * c, b = WBITS == 4 ? c + 4 : 2 * c + 1;
                o[a][i / 2] = __builtin_amdgcn_perm(row[1][c], row[0][c], 0x05040100u);
                o[b][i / 2] = __builtin_amdgcn_perm(row[1][c], row[0][c], 0x07060302u);
            }
        }
    } else {
        // (4 bits: signed bytes of 16 times the weight, as in dequant8)
        uint32_t even[8], odd[8];
#pragma unroll
        for (int i = 0; i < 8; i++) { odd[i] = q[i][0] & 0xf0f0f0f0u; even[i] = (q[i][0] << 4) & 0xf0f0f0f0u; }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float sc1 = u2f((j & 1) ? scw[j / 2] & 0xffff0000u : scw[j / 2] << 16), scf = WBITS == 4 && !HAS_OFF ? 0.0625f * sc1 : sc1, off = u2f((j & 1) ? ofw[j / 2] & 0xffff0000u : ofw[j / 2] << 16);
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                float w[2];
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    if constexpr (WBITS == 4) w[r] = (float)((int)((j & 1 ? odd : even)[i + r] << (24 - 8 * (j >> 1))) >> 24);
                    else w[r] = (float)((int)(q[i + r][j / 4 * (DW - 1)] << (24 - 8 * (j & 3))) >> 24);
                }
                if constexpr (HAS_OFF) {
                    const float one = WBITS == 4 ? 0.0625f : 1.0f;
                    const uint32_t pk = pack2_bf16((v2f){__builtin_fmaf(w[0], one, off), __builtin_fmaf(w[1], one, off)});
                    w[0] = u2f(pk << 16);
                    w[1] = u2f(pk & 0xffff0000u);
                }
                o[j][i / 2] = pack2_bf16((v2f){w[0] * scf, w[1] * scf});
            }
        }
    }
}

}  // namespace opsnn
