// Rotation of K head rows whose 16-byte units do not map onto the lanes of a
// wavefront: rows of any 16-byte multiple (heads of 80, 96 or 192 values, 576
// wide latent rows) and rotary halves that end inside a unit (20 of 80 values).
//
// A workgroup takes up to kRowUnits units of whole rows, loads them in memory
// order, keeps a copy in LDS and reads a unit's partners, half a rotary width
// away in the same row, from that copy. So the accesses to memory are those
// of a plain copy whatever the row width; reading both halves of a pair by one
// lane instead splits every row into two streams of half a row.
#pragma once

#include <hip/hip_runtime.h>

#include "elem.h"

namespace daric {

constexpr int kRowThreads = 256;
constexpr int kRowUnroll = 4;
constexpr int kRowUnits = kRowThreads * kRowUnroll;   // 16 KiB
constexpr int kRowMaxHalf = 256;                      // rotary_dim / 2 limit of the LDS cos/sin table

// ALIGNED: the pairs' members (NeoX: the rotary half; GPT-J: the rotary dims)
// are whole units. Otherwise a unit may hold values of both halves, or values
// past the rotary dims, which keep their bits.
template <int KIND, bool NEOX, bool ALIGNED>
struct RowRotation {
    using E = Elem<KIND>;
    static constexpr int VE = E::VE;
    static constexpr int EPW = E::EPW;
    static constexpr int ES = KIND == kE4M3 ? 1 : 2;

    // (cos, sin) of every pair. ALIGNED tables are transposed so that lanes of
    // consecutive units read consecutive entries: NeoX float4 j (pairs 2j and
    // 2j + 1 of a unit) of unit k at j * units + k, GPT-J pair j of unit k at
    // j * units + k.
    static __device__ __forceinline__ void fill(float4* table, int half, float delta,
                                                const float* __restrict__ inv_freq) {
        float* t = reinterpret_cast<float*>(table);
        for (int i = threadIdx.x; i < half; i += kRowThreads) {
            float sn, c;
            sincosf(delta * inv_freq[i], &sn, &c);
            int at = 2 * i;
            if (ALIGNED && NEOX) {
                const int f = i >> 1;
                at = 4 * ((f % (VE / 2)) * (half / VE) + f / (VE / 2)) + 2 * (i & 1);
            } else if (ALIGNED) {
                at = 2 * ((i % (VE / 2)) * (half / (VE / 2)) + i / (VE / 2));
            }
            t[at] = c;
            t[at + 1] = sn;
        }
    }

    // Units of a row that hold rotated values.
    static __host__ __device__ __forceinline__ int rotated_units(int R) { return (R + VE - 1) / VE; }

    // Unit k of a row after the rotation; v: its bits; row: the LDS copy of the
    // row's first unit (NeoX).
    static __device__ __forceinline__ u32x4 turn(const u32x4& v, const u32x4* row, int k, const float4* table, int half) {
        u32x4 out;
        if constexpr (ALIGNED && NEOX) {
            const int nr = half / VE;
            const bool first = k < nr;
            const int kk = first ? k : k - nr;
            const u32x4 pv = row[first ? k + nr : kk];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float x[EPW], y[EPW];
                E::unpack_word(v[w], x);
                E::unpack_word(pv[w], y);
#pragma unroll
                for (int h = 0; h < EPW / 2; ++h) {
                    const float4 t = table[(w * (EPW / 2) + h) * nr + kk];
                    const float s0 = first ? -t.y : t.y, s1 = first ? -t.w : t.w;
                    x[2 * h] = x[2 * h] * t.x + y[2 * h] * s0;
                    x[2 * h + 1] = x[2 * h + 1] * t.z + y[2 * h + 1] * s1;
                }
                out[w] = E::pack_word(x);
            }
        } else if constexpr (NEOX) {
            const uint8_t* bytes = reinterpret_cast<const uint8_t*>(row);
            const float2* cs = reinterpret_cast<const float2*>(table);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int e0 = k * VE + w * EPW;
                uint32_t pw = 0, keep = 0;
#pragma unroll
                for (int e = 0; e < EPW; ++e) {
                    const int at = e0 + e;
                    if (at >= 2 * half) {
                        keep |= (ES == 2 ? 0xffffu : 0xffu) << (8 * ES * e);
                        continue;
                    }
                    const int pe = at < half ? at + half : at - half;
                    const uint32_t b = ES == 2 ? reinterpret_cast<const uint16_t*>(bytes)[pe] : bytes[pe];
                    pw |= b << (8 * ES * e);
                }
                float x[EPW], y[EPW];
                E::unpack_word(v[w], x);
                E::unpack_word(pw, y);
#pragma unroll
                for (int e = 0; e < EPW; ++e) {
                    const int at = e0 + e;
                    const bool first = at < half;
                    const float2 t = cs[min(first ? at : at - half, half - 1)];
                    x[e] = x[e] * t.x + y[e] * (first ? -t.y : t.y);
                }
                out[w] = (E::pack_word(x) & ~keep) | (v[w] & keep);
            }
        } else {
            const float2* cs = reinterpret_cast<const float2*>(table);
            const int units = half / (VE / 2);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float x[EPW];
                E::unpack_word(v[w], x);
                uint32_t keep = 0;
#pragma unroll
                for (int m = 0; m < EPW / 2; ++m) {
                    const int j = w * (EPW / 2) + m;       // the unit's pair
                    const int pair = k * (VE / 2) + j;
                    if (!ALIGNED && pair >= half) {
                        keep |= (ES == 2 ? 0xffffffffu : 0xffffu) << (16 * m);
                        continue;
                    }
                    const float2 t = cs[ALIGNED ? j * units + k : pair];
                    const float x1 = x[2 * m], x2 = x[2 * m + 1];
                    x[2 * m] = x1 * t.x - x2 * t.y;
                    x[2 * m + 1] = x2 * t.x + x1 * t.y;
                }
                out[w] = ALIGNED ? E::pack_word(x) : (E::pack_word(x) & ~keep) | (v[w] & keep);
            }
        }
        return out;
    }
};

}  // namespace daric
