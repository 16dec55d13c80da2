// Host side of the attention kernels on split f16 operands.
#include "split16.hpp"

#include "kernels_split16.hpp"

namespace jqh {

namespace {

size_t tiles_of(size_t tokens) { return (tokens + jq::S16_TILE - 1) / jq::S16_TILE; }

// hipMalloc that leaves no error behind; `refused` is set where there is no memory.
bool have(void **p, size_t bytes, bool *refused) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return true;
    *p = nullptr;
    *refused |= e == hipErrorOutOfMemory;
    (void)hipGetLastError();
    return false;
}

// Whether the stream is being captured; also where it does not say (the null stream beside another's capture).
bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) == hipSuccess) return capture != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

}  // namespace

struct Split16Latent {
    size_t n_head, n_ctx, ws_bytes = 0;  // (0: not asked for yet)
    bool refused = false;                // there was no memory for the buffers below
    int ec;                              // exponent of the latents' scale
    uint8_t *wfrags = nullptr;
    float2 *fac = nullptr;
    uint8_t *cf = nullptr, *rf = nullptr, *ws = nullptr;  // latents, rope keys, a group of heads' keys and values
    jq::S16Tile *info = nullptr;
    // Tokens whose keys and values lie in ws, where it holds all heads over the whole context: a part of the cache like the latents
    // they are made of, which a call adds its own tokens to.  4096 tokens in chunks of 512: 7.0 ms with every chunk expanding all in
    // front of it again, 5.3 without.
    size_t ready = 0;
    // A call of this object was captured: its replays write tokens without this knowing, and each has to leave the keys and values
    // of all tokens in front of it, so that from then on every call expands them all.
    bool captured = false;
};

bool split16_latent_fits(size_t nope, size_t rope, size_t vh, size_t lkv) {
    return nope == jq::S16_HEAD && vh == jq::S16_HEAD && rope == jq::S16_ROPE && lkv == jq::S16_LKV;
}

// Bytes of an object's keys and values: those of all heads over the whole context, so that no later call allocates, up to
// 512 MiB (what the absorbed form's scratch takes for 1000 tokens of 128 heads); longer contexts take the heads in groups.
// 512 tokens of DeepSeek-V3's size behind 8000, 512 MiB against 256: 2.5 and 3.9 ms.
static size_t latent_ws_bytes(const Split16Latent *s) {
    return s->ws_bytes ? s->ws_bytes : std::min(s->n_head * tiles_of(s->n_ctx) * jq::S16_KV_TILE, (size_t)512 << 20);
}

// Heads of a group of a call over nt tiles: as even as fits, by eights where they fit (a head then keeps to one XCD); 0 where
// not one fits.
static size_t latent_group(const Split16Latent *s, size_t nt) {
    const size_t fit = std::min(s->n_head, latent_ws_bytes(s) / (nt * jq::S16_KV_TILE));
    if (fit == 0) return 0;
    const size_t groups = (s->n_head + fit - 1) / fit, even = (s->n_head + groups - 1) / groups, eights = (even + 7) / 8 * 8;
    return eights <= fit ? eights : even;
}

static bool latent_keeps(const Split16Latent *s) { return !s->captured && latent_ws_bytes(s) >= s->n_head * tiles_of(s->n_ctx) * jq::S16_KV_TILE; }
// The first tile that a call has to expand.
static size_t latent_first_tile(const Split16Latent *s) { return latent_keeps(s) ? s->ready / jq::S16_TILE : 0; }

void split16_latent_overwrites(Split16Latent *s, size_t pos, hipStream_t stream) {
    s->ready = std::min(s->ready, pos);
    if (s->captured) return;
    s->captured = capturing(stream);
}

// Both sides in us, fitted to calls of 48 to 1024 tokens behind 0 to 32000 with 128 and 32 heads (within 10 %, the absorbed
// form's vector kernel, for head counts that are no multiple of 32, within 25 %).  Expanded, a group of g heads: 0.0266 a tile and
// head to expand and, a workgroup walking all tiles, 1.76 a tile while there is one to a compute unit.  128 heads, absorbed /
// expanded in groups as here: 48 tokens behind 0, 4000, 8000, 16000: 139 / 32, 829 / 671, 1527 / 1690, 2924 / 5045; 128 tokens behind
// 4000, 8000, 16000: 1707 / 718, 3105 / 1735, 5881 / 5112; 512 tokens behind 4000, 16000: 7016 / 1037, 23784 / 5423.
bool split16_latent_pays(const Split16Latent *s, size_t S, size_t pos, bool fresh) {
    const size_t nt = tiles_of(pos + S), made = fresh ? 0 : latent_first_tile(s), g = latent_group(s, nt), nh = s->n_head;
    if (g == 0 || s->refused) return false;
    const double wgs = (double)(g * ((S + 127) / 128)), keys = (double)pos + (double)S / 2;
    const double expanded = (double)((nh + g - 1) / g) * (20.0 + (double)nt * 1.76 * std::max(1.0, wgs / 233.0) + (double)(nt - made) * 0.0266 * (double)g);
    const double walk = nh % 32 == 0 ? 0.174 * std::ceil((double)(S * nh) / (32 * 256)) : 0.27 * std::max(1.0, 0.75 * (double)(S * ((nh + 7) / 8)) / 256);
    return expanded < 0.92 * (35.0 + 0.017 * (double)(S * nh) + walk * keys);  // (level with it: the form that needs no buffer)
}

int split16_latent_create(size_t n_head, size_t n_ctx, const float *wkv, const float *kv_norm, Split16Latent **out) {
    std::unique_ptr<Split16Latent, void (*)(Split16Latent *)> s(new Split16Latent{n_head, n_ctx}, split16_latent_free);
    float wmax = 0.0f;
    for (int i = 0; i < jq::S16_LKV; i++) wmax = std::max(wmax, fabsf(kv_norm[i]));
    // a normed latent's 2-norm is at most sqrt(512) times the largest norm weight
    const float cmax = std::min(std::max(sqrtf((float)jq::S16_LKV) * wmax, 1e-20f), 1e20f);
    int e;
    (void)frexpf(cmax, &e);  // cmax < 2^e
    s->ec = 14 - e;
    *out = nullptr;
    if (!have((void **)&s->wfrags, n_head * 2 * (jq::S16_LKV / 16) * 8 * jq::S16_FRAG, &s->refused) ||
        !have((void **)&s->fac, n_head * 2 * sizeof(float2), &s->refused))
        return 0;
    hipLaunchKernelGGL(jq::s16_up_projection, dim3(2, (unsigned)n_head), dim3(256), 0, nullptr, wkv, s->wfrags, s->fac, cmax, s->ec);
    HIP_TRY(hipGetLastError());
    *out = s.release();
    return 0;
}

void split16_latent_free(Split16Latent *s) {
    if (!s) return;
    for (void *p : {(void *)s->wfrags, (void *)s->fac, (void *)s->cf, (void *)s->rf, (void *)s->ws, (void *)s->info})
        if (p) (void)hipFree(p);
    delete s;
}

int split16_latent_attention(Split16Latent *s, const float *q, size_t S, size_t pos, const float *lat, const float *kpe, float scale,
                             float *out, hipStream_t stream) {
    const size_t all = tiles_of(s->n_ctx), nt = tiles_of(pos + S);
    if (s->refused) return -1;
    if (!s->ws) {
        // nothing can be allocated while the stream is captured: this call is absorbed, and a later one asks
        if (capturing(stream)) return -1;
        size_t want = latent_ws_bytes(s);
        bool none = false;
        const bool rest = (s->cf || have((void **)&s->cf, all * (jq::S16_LKV / 16) * 2 * jq::S16_FRAG, &s->refused)) &&
                          (s->rf || have((void **)&s->rf, all * jq::S16_ROPE_TILE, &s->refused)) &&
                          (s->info || have((void **)&s->info, all * sizeof(jq::S16Tile), &s->refused));
        while (rest && !have((void **)&s->ws, want, &none)) {  // half as much, down to one head
            if (!none || want / 2 < all * jq::S16_KV_TILE) break;
            want /= 2;
        }
        s->refused |= none && !s->ws;
        if (!s->ws) return -1;
        s->ws_bytes = want;
    }
    const size_t group = latent_group(s, nt);
    if (group == 0) return -1;
    // tiles from t0 on are to be made, the heads' tiles lie `stride` apart
    const bool keeps = latent_keeps(s);
    const size_t t0 = latent_first_tile(s), stride = keeps ? all : nt, made = nt - t0;
    hipLaunchKernelGGL(jq::s16_latent_tiles, dim3((unsigned)made), dim3(256), 0, stream, lat, kpe, (int)t0, (int)(pos + S), ldexpf(1.0f, s->ec),
                       s->cf, s->rf, s->info);
    HIP_TRY(hipGetLastError());
    for (size_t h0 = 0; h0 < s->n_head; h0 += group) {
        const size_t hg = std::min(group, s->n_head - h0);
        hipLaunchKernelGGL(jq::s16_expand, dim3((unsigned)(2 * hg * ((made + 3) / 4))), dim3(256), 0, stream, (const uint8_t *)s->wfrags,
                           (const float2 *)s->fac, (const uint8_t *)s->cf, (int)h0, (int)hg, (int)t0, (int)made, (int)stride, s->ws);
        HIP_TRY(hipGetLastError());
        jq::S16Attention a{};
        a.q = q + h0 * (jq::S16_HEAD + jq::S16_ROPE), a.q_stride = (int)(s->n_head * (jq::S16_HEAD + jq::S16_ROPE)), a.q_head = jq::S16_HEAD + jq::S16_ROPE;
        a.kv = s->ws, a.info = s->info, a.fac = s->fac + 2 * h0, a.rope = s->rf;
        a.out = out + h0 * jq::S16_HEAD, a.out_stride = (int)(s->n_head * jq::S16_HEAD);
        a.T = (int)S, a.pos0 = (int)pos, a.n_tiles = (int)stride, a.heads = (int)hg, a.group = 1, a.blocks = (int)((S + 127) / 128);
        a.scale_log2e = scale * 1.44269504088896340736f;
        hipLaunchKernelGGL((jq::s16_attention<true, 1>), dim3((unsigned)(hg * a.blocks)), dim3(256), 0, stream, a);
        HIP_TRY(hipGetLastError());
    }
    if (keeps) s->ready = pos + S;
    return 0;
}

void split16_cache_free(Split16Cache *c) {
    if (c->ws) (void)hipFree(c->ws);
    if (c->info) (void)hipFree(c->info);
    *c = {};
}

bool split16_attention_fits(int d, int heads, int kv_heads) {
    const int g = heads / kv_heads;
    return d == 128 && heads % kv_heads == 0 && (g == 1 || g == 2 || g % 4 == 0);
}

int split16_attention(Split16Cache *c, const float *q, int q_stride, int T, int pos, const float *kc, const float *vc, int heads, int kv_heads,
                      int n_ctx, float *out, hipStream_t stream) {
    const size_t all = tiles_of((size_t)n_ctx);
    if (c->refused) return -1;
    if (!c->ws && !have((void **)&c->ws, (size_t)kv_heads * all * jq::S16_KV_TILE, &c->refused)) return -1;
    if (!c->info && !have((void **)&c->info, (size_t)kv_heads * all * sizeof(jq::S16Tile), &c->refused)) return -1;
    const int nt = (int)tiles_of((size_t)pos + T), g = heads / kv_heads, wh = std::min(g, 4);
    hipLaunchKernelGGL(jq::s16_kv_tiles, dim3((unsigned)nt, (unsigned)kv_heads), dim3(256), 0, stream, kc, vc, n_ctx, pos + T, c->ws, (jq::S16Tile *)c->info);
    HIP_TRY(hipGetLastError());
    jq::S16Attention a{};
    a.q = q, a.q_stride = q_stride, a.q_head = 128;
    a.kv = c->ws, a.info = (const jq::S16Tile *)c->info;
    a.out = out, a.out_stride = heads * 128;
    a.T = T, a.pos0 = pos, a.n_tiles = nt, a.heads = heads, a.group = g;
    const int tb = 32 * (4 / wh);
    a.blocks = (T + tb - 1) / tb;
    a.scale_log2e = (float)(1.4426950408889634 / sqrt(128.0));
    const dim3 grid((unsigned)(heads / wh * a.blocks));
    if (wh == 4) hipLaunchKernelGGL((jq::s16_attention<false, 4>), grid, dim3(256), 0, stream, a);
    else if (wh == 2) hipLaunchKernelGGL((jq::s16_attention<false, 2>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((jq::s16_attention<false, 1>), grid, dim3(256), 0, stream, a);
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace jqh
