// What a step does for one token in front of the attention over latents (attn_latent.hip), by one workgroup: the cache row and
// the rotated parts of its queries.  Used by a launch of its own and by the decode launch that also expands the queries.
#pragma once

#include "common.h"
#include "pta_kernels.h"

struct LatentToken {
    const void* down_rows;  // [M, R + dr], rows ld apart
    long ld;
    const float* w_norm;
    float eps;
    const float* inv_freq;
    int inv_freq_ld;
    float cs_scale;
    int rot_n, pairing;
    const int* token_pos;
    const int* token_seq;
    const int* block_table;
    int bt_stride, H, dn, dr, R, write_cache;
};

// element i of a rotated part v, rotated by the position (freq null: as it is)
template <typename T>
__device__ __forceinline__ float latent_rotated(const LatentToken& a, const float* freq, int pos, const T* v, int i) {
    const float x = Io<T>::ld(v + i);
    if (!freq || i >= a.rot_n) return x;
    int pair, fi;  // the element that it is paired with; the sign of the sine term
    float sign;
    if (a.pairing == PTA_PAIR_INTERLEAVED) { pair = i ^ 1; fi = i >> 1; sign = (i & 1) ? 1.f : -1.f; }
    else { const int half = a.rot_n >> 1; pair = i < half ? i + half : i - half; fi = i < half ? i : i - half; sign = i < half ? -1.f : 1.f; }
    float sn, c;
    sincosf((float)pos * freq[fi], &sn, &c);
    return x * (c * a.cs_scale) + sign * Io<T>::ld(v + pair) * (sn * a.cs_scale);
}

__device__ __forceinline__ const float* latent_freq(const LatentToken& a, int m) {
    return a.inv_freq ? a.inv_freq + (a.inv_freq_ld ? (long)a.token_seq[m] * a.inv_freq_ld : 0) : nullptr;
}

// Token m's cache row from down_rows[m] = R + dr elements:
//  - latent c = down[:R] / sqrt(mean(down[:R]^2) + eps) * w_norm -> [0, R)
//  - shared key part down[R:], its first rot_n elements rotated by the token's position -> [R, R + dr)
// red: 16 floats of LDS.
template <typename T>
__device__ __forceinline__ void latent_row(const LatentToken& a, int m, T* __restrict__ k_pool, float* red) {
    const int pos = a.token_pos[m];
    const T* down = (const T*)a.down_rows + (long)m * a.ld;
    const float* freq = latent_freq(a, m);
    const long page = a.block_table[(long)a.token_seq[m] * a.bt_stride + pos / PTA_PAGE];
    float ss = 0.f;
    for (int i = threadIdx.x; i < a.R; i += blockDim.x) { const float v = Io<T>::ld(down + i); ss += v * v; }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)a.R + a.eps);
    T* dst = k_pool + (page * PTA_PAGE + pos % PTA_PAGE) * (long)(a.R + a.dr);
    for (int i = threadIdx.x; i < a.R; i += blockDim.x) Io<T>::st(dst + i, Io<T>::ld(down + i) * inv * a.w_norm[i]);
    for (int i = threadIdx.x; i < a.dr; i += blockDim.x) Io<T>::st(dst + a.R + i, latent_rotated(a, freq, pos, down + a.R, i));
}

// each head's rotated query part (q_rows[m] = H * (dn + dr) elements, rows q_ld apart), rotated likewise -> q_full[m, h, R:] (32-bit)
template <typename T>
__device__ __forceinline__ void latent_rotations(const LatentToken& a, int m, float* __restrict__ q_full, const T* __restrict__ q_rows, long q_ld) {
    const int pos = a.token_pos[m], D = a.R + a.dr;
    const T* row = q_rows + (long)m * q_ld;
    const float* freq = latent_freq(a, m);
    for (int i = threadIdx.x; i < a.H * a.dr; i += blockDim.x) {
        const int h = i / a.dr, e = i - h * a.dr;
        q_full[((long)m * a.H + h) * D + a.R + e] = latent_rotated(a, freq, pos, row + (long)h * (a.dn + a.dr) + a.dn, e);
    }
}

// the entry points' arguments checked and put together; nonzero with the reason in pta_last_error
static inline int latent_token_args(const char* what, LatentToken& t, const float* q_full, const void* k_pool, const void* q_rows,
                                    long q_ld, const void* down, long ld, const float* w_norm, float eps, const PtaRotation* rot,
                                    const int* token_pos, const int* token_seq, const int* block_table, int bt_stride, int M, int H,
                                    int dn, int dr, int R, int write_cache) {
    PTA_REQUIRE(M > 0 && H > 0 && dn > 0 && dr >= 0 && R > 0, "%s: sizes must be positive", what);
    PTA_REQUIRE(q_full && q_rows && token_pos && token_seq && (!write_cache || (k_pool && down && w_norm && block_table)), "%s: null pointer", what);
    PTA_REQUIRE(q_ld >= (long)H * (dn + dr) && (!write_cache || ld >= (long)R + dr), "%s: rows lie closer together than they are long", what);
    const float* inv_freq = rot ? rot->inv_freq : nullptr;
    int rot_n = 0, pairing = PTA_PAIR_HALF, freq_ld = 0;
    float cs = 1.f;
    if (inv_freq) {
        rot_n = rot->rotary_dim, pairing = rot->pairing, freq_ld = rot->inv_freq_ld, cs = rot->cs_scale;
        PTA_REQUIRE(rot_n >= 2 && rot_n % 2 == 0 && rot_n <= dr,
                    "%s: %d rotated elements must be even and at most the rotated part's %d", what, rot_n, dr);
        PTA_REQUIRE(pairing == PTA_PAIR_HALF || pairing == PTA_PAIR_INTERLEAVED, "%s: unknown pairing %d", what, pairing);
    }
    t = LatentToken{down, ld, w_norm, eps, inv_freq, freq_ld, cs, rot_n, pairing, token_pos, token_seq, block_table, bt_stride, H, dn, dr, R, write_cache};
    return 0;
}
