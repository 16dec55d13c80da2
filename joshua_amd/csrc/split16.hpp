// Attention of many tokens on the f16 matrix cores at f32 precision (kernels in kernels_split16.hpp): the decoder's over an
// f32 cache of keys and values, and latent attention with the cached latents expanded to keys and values per head.
#pragma once
#include "core.hpp"

namespace jqh {

// What one latent attention object keeps: its up-projection as matrix-core operands, and the buffers of a call.
struct Split16Latent;
bool split16_latent_fits(size_t nope, size_t rope, size_t vh, size_t lkv);
// wkv: [n_head * 256][512] f32 on the device; kv_norm: the latent's norm weights on the host.  Where there is no memory for
// the operands (half a megabyte a head) *out is null, and the object's calls are absorbed ones.
int split16_latent_create(size_t n_head, size_t n_ctx, const float *wkv, const float *kv_norm, Split16Latent **out);
void split16_latent_free(Split16Latent *s);
// The cached tokens from `pos` on are about to be written by work on that stream: their keys and values, if they were
// expanded, are not those of the cache any more.
void split16_latent_overwrites(Split16Latent *s, size_t pos, hipStream_t stream);
// Whether a call of S tokens behind `pos` is cheaper with expanded keys and values than absorbed; `fresh`: where none of those
// in front are expanded already.
bool split16_latent_pays(const Split16Latent *s, size_t S, size_t pos, bool fresh);
// out[t][n_head * 128] for S tokens at positions pos .. over the cached latents and rotated rope keys of pos + S tokens;
// q [t][n_head * 192] rotated.  0: done, 1: failed, -1: no memory for the expanded keys and values (then not asked for again).
int split16_latent_attention(Split16Latent *s, const float *q, size_t S, size_t pos, const float *lat, const float *kpe, float scale,
                             float *out, hipStream_t stream);

// The decoder's: a copy of one layer's cache as operands, made anew by each call.
struct Split16Cache {
    uint8_t *ws = nullptr;
    void *info = nullptr;  // [kv head][tile]: scales
    bool refused = false;  // there was no memory for them
};
void split16_cache_free(Split16Cache *c);
bool split16_attention_fits(int d, int heads, int kv_heads);
// out[t][heads * 128] for T tokens at positions pos .. over kc, vc [kv_heads][n_ctx][128]; a token's heads start q_stride
// floats apart.  0: done, 1: failed, -1: no memory for the copy (then not asked for again).
int split16_attention(Split16Cache *c, const float *q, int q_stride, int T, int pos, const float *kc, const float *vc, int heads, int kv_heads,
                      int n_ctx, float *out, hipStream_t stream);

}  // namespace jqh
