// gmoe_attn.hip — grouped-query decode attention over a paged KV cache.
//
// Reference: LlamaBackend::attend_one (garuda/src/llama/mod.rs:766-821) and
// KVCacheState (cache/mod.rs:143-600). Per token: rotate q (every query head) and k
// (every kv head) by the token's position (simd::rope, simd/mod.rs:196-206), append k
// and v to the sequence's cache, and for each query head h attend over positions
// [start, pos] of kv head h / group: scores = q·k * (1/sqrt(hd)), softmax (simd.rs
// :132-158), context = sum of p_j * v_j. f32 throughout; the reductions run in
// parallel, so results match the reference within the layer tolerance.
//
// Device layout. Pages of `bs` positions: keys [n_kv][bs][hd] then values in the same
// layout, f32, so one kv head's rows of a page are contiguous. Each (sequence, layer) has
// a page table of `ppseq` page ids. A call's entries
// are tokens, each with its sequence's page table, its position and the position
// attention starts at; entries of one sequence come in position order, and where a call has
// several of one sequence the append kernel writes every entry's k and v before any attends
// (causal within the call).
// Calls of several tokens of a sequence (prompts) run tiles of rows on MFMA (k_attn_tile).
#include "gmoe_device.h"

namespace gmoe {

// simd::rope for pair i of a head at position pos: the frequency theta^(-2i/hd) and
// the angle in f32 as the reference forms them.
__device__ __forceinline__ void rope_pair(float& a, float& b, uint32_t i, uint32_t hd, uint32_t pos, float theta) {
  const float freq = 1.0f / powf(theta, (2.0f * (float)i) / (float)hd);
  const float ang = (float)pos * freq;
  float s, c;
  sincosf(ang, &s, &c);
  const float x = a, y = b;
  a = x * c - y * s;
  b = x * s + y * c;
}

__device__ __forceinline__ AttnEntry entry(const AttnArgs& a, uint32_t i) { return a.ent ? a.ent[i] : a.inl[i]; }

// Key row of position p, kv head h (the value row is bs * kv_dim floats further on).
__device__ __forceinline__ const float* key_row(const AttnArgs& a, const AttnEntry& e, uint32_t p, uint32_t h) {
  return a.pool + (size_t)e.pages[p / a.bs] * a.page_floats + ((size_t)h * a.bs + p % a.bs) * a.hd;
}

// grid (n, ceil(pairs / 256)), pairs = (n_heads + n_kv) * hd / 2
// (x, y) = elements 2j, 2j+1 from p, each the sum of nsl K slices `stride` floats apart in
// slice order when nsl > 1 (k_reduce_parts's sum); the slice loads are issued together
// (indices clamped, the surplus ones not added)
__device__ __forceinline__ void ld_pair(const float* p, uint32_t j, uint32_t nsl, uint64_t stride, float& x, float& y) {
  if (nsl <= 1) {
    x = p[2 * j];
    y = p[2 * j + 1];
    return;
  }
  float vx[kMaxKsg], vy[kMaxKsg];
#pragma unroll
  for (uint32_t g = 0; g < kMaxKsg; g++) {
    const float* s = p + min(g, nsl - 1) * stride;
    vx[g] = s[2 * j];
    vy[g] = s[2 * j + 1];
  }
  x = vx[0];
  y = vy[0];
#pragma unroll
  for (uint32_t g = 1; g < kMaxKsg; g++)
    if (g < nsl) {
      x += vx[g];
      y += vy[g];
    }
}

__global__ void __launch_bounds__(256) k_rope_append(AttnArgs a) {
  const uint32_t i = blockIdx.x, half = a.hd / 2, kvd = a.n_kv * a.hd;
  const uint32_t pr = blockIdx.y * 256 + threadIdx.x, qpairs = a.n_heads * half;
  const AttnEntry e = entry(a, i);
  const uint32_t page = e.page, slot = e.pos % a.bs;
  if (e.fresh && pr == 0) e.pages[e.pos / a.bs] = page;  // read by the attention kernel after this one
  float* kp = a.pool + (size_t)page * a.page_floats + (size_t)slot * a.hd;  // head h at + h * bs * hd
  float* vp = kp + (size_t)a.bs * kvd;
  if (pr < qpairs) {
    const uint32_t h = pr / half, j = pr % half;
    const float* src = a.q + (size_t)i * a.q_stride + h * a.hd;
    float x, y;
    ld_pair(src, j, a.nsl, a.sl_stride, x, y);
    rope_pair(x, y, j, a.hd, e.pos, a.theta);
    float* dst = a.qr + (size_t)i * a.n_heads * a.hd + h * a.hd;
    dst[2 * j] = x;
    dst[2 * j + 1] = y;
  } else if (pr < qpairs + a.n_kv * half) {
    const uint32_t p2 = pr - qpairs, h = p2 / half, j = p2 % half;
    const float* src = a.k + (size_t)i * a.kv_stride + h * a.hd;
    float x, y;
    ld_pair(src, j, a.nsl, a.sl_stride, x, y);
    rope_pair(x, y, j, a.hd, e.pos, a.theta);
    const size_t hoff = (size_t)h * a.bs * a.hd;
    kp[hoff + 2 * j] = x;
    kp[hoff + 2 * j + 1] = y;
    const float* vs = a.v + (size_t)i * a.kv_stride + h * a.hd;
    float vx, vy;
    ld_pair(vs, j, a.nsl, a.sl_stride, vx, vy);
    vp[hoff + 2 * j] = vx;
    vp[hoff + 2 * j + 1] = vy;
  }
}

// k_rope_append for calls of many tokens, gridDim.y workgroups a token: a thread makes its
// pair's angle once for every head it rotates (the powf and sincosf were most of the
// launch), with up to kRopeHeads heads' loads issued before it. Copies the call's entries
// and tiles to the device for the launches after it.
constexpr uint32_t kRopeHeads = 8;
__global__ void __launch_bounds__(256) k_rope_rows(AttnArgs a) {
  const uint32_t i = blockIdx.x, t = threadIdx.x, half = a.hd / 2, ng = 256 / half, j = t % half, g = t / half;
  const AttnEntry e = a.hent[i];
  if (t == 0 && blockIdx.y == 0) {
    const_cast<AttnEntry*>(a.ent)[i] = e;
    if (i < a.ntile) const_cast<AttnTile*>(a.tiles)[i] = a.htile[i];
    if (i < a.npick) const_cast<uint32_t*>(a.pick)[i] = a.hpick[i];
  }
  const uint32_t slot = e.pos % a.bs, kvd = a.n_kv * a.hd, nh = a.n_heads + a.n_kv, step = ng * gridDim.y;
  if ((e.fresh & 1) && t == 0 && blockIdx.y == 0) e.pages[e.pos / a.bs] = e.page;  // read by the attention kernel after this one
  float* kp = a.pool + (size_t)e.page * a.page_floats + (size_t)slot * a.hd;  // head h at + h * bs * hd
  float* vp = kp + (size_t)a.bs * kvd;
  const float* vs = a.v + (size_t)i * a.kv_stride;
  float x[kRopeHeads], y[kRopeHeads], cs = 0.0f, sn = 0.0f;
  for (uint32_t h0 = g + ng * blockIdx.y; g < ng && h0 < nh; h0 += kRopeHeads * step) {
#pragma unroll
    for (uint32_t b = 0; b < kRopeHeads; b++) {
      const uint32_t h = min(h0 + b * step, nh - 1);
      const float* src = h < a.n_heads ? a.q + (size_t)i * a.q_stride + h * a.hd
                                       : a.k + (size_t)i * a.kv_stride + (h - a.n_heads) * a.hd;
      x[b] = src[2 * j];
      y[b] = src[2 * j + 1];
    }
    if (h0 < step) {
      const float freq = 1.0f / powf(a.theta, (2.0f * (float)j) / (float)a.hd);
      sincosf((float)e.pos * freq, &sn, &cs);
    }
#pragma unroll
    for (uint32_t b = 0; b < kRopeHeads; b++) {
      const uint32_t h = h0 + b * step;
      if (h < nh) {
        float* dst = h < a.n_heads ? a.qr + ((size_t)i * a.n_heads + h) * a.hd : kp + (size_t)(h - a.n_heads) * a.bs * a.hd;
        dst[2 * j] = x[b] * cs - y[b] * sn;
        dst[2 * j + 1] = x[b] * sn + y[b] * cs;
      }
    }
  }
  for (uint32_t z = t + 256 * blockIdx.y; z < kvd; z += 256 * gridDim.y)
    vp[(size_t)(z / a.hd) * a.bs * a.hd + z % a.hd] = vs[z];
}

__device__ __forceinline__ float wave_max(float v) { return wave64_max(v); }
__device__ __forceinline__ float wave_sum(float v) { return wave64_sum(v); }

// grid (n, n_kv, nchunk), 256 threads: one chunk of kAttnChunk positions for the
// `group` query heads of one kv head. Thread t takes position j = t / 4 of the chunk and
// every fourth float4 column of its key and value rows from column t % 4 on, loaded from
// the page at once (the value loads' latency hides behind the scores). Scores: the
// thread's columns dotted with each head's q (in LDS), the four partial dots added by
// lane shuffles. The values go to an LDS tile [kAttnChunk][hd]; per head the chunk's max
// m, the sum l of exp(s - m) and o = sum of exp(s - m) * v go to part, o by float4
// columns with the positions split over the spare threads (parts added in order).
// Dynamic LDS: tile, q [G][hd], p [G][kAttnChunk], (m, l) [kAttnMaxGroup][2], o parts [256] float4.
//
// ROPE (calls whose entries are all of different sequences: decode steps): no
// k_rope_append before it. While the chunk's rows are on their way, hd / 2 threads make the
// position's angles (powf and sincosf, once a pair for every head) and the workgroup
// rotates its q heads into LDS; the chunk that holds the new position also rotates and
// stores that key and its value, and scores them from LDS. No other workgroup reads that
// row, nor the page table's entry of a fresh page, which only it uses: positions before a
// fresh page's first sit on other pages. The same operations as k_rope_append's, so the
// same bits. A call of one chunk (ONE) writes the context itself, as k_attn_combine would.
// Eight sequences over a window of 2048, four layers: 181.1 -> 170.8 us (the launch saved
// and its gap, 35 us a layer here being the pages' 134 MB at 3.8 TB/s). The synthetic
// engine's steps (one sequence, spans below 64: three launches a layer become one): 24
// steps after a prompt of 16 in 8856 -> 8100 us.
inline uint32_t attn_lds_bytes(uint32_t G, uint32_t hd) {
  return (kAttnChunk * hd + G * hd + G * kAttnChunk + 2 * kAttnMaxGroup) * 4 + 256 * 16;
}

static_assert(kAttnChunk * 4 == 256, "four threads per position of a chunk");

template <int MAXHD, bool ROPE, bool ONE>
__global__ void __launch_bounds__(256) k_attn_partial(AttnArgs a) {
  constexpr int NR = MAXHD / 16;  // float4 columns of a row per thread
  extern __shared__ float4 lds_v4[];
  float* lds_f = reinterpret_cast<float*>(lds_v4);
  const uint32_t i = !ROPE && a.pick ? a.pick[blockIdx.x] : blockIdx.x, h = blockIdx.y, c = blockIdx.z, t = threadIdx.x;
  const uint32_t G = a.n_heads / a.n_kv, hd = a.hd, kvd = a.n_kv * hd, q4 = hd / 4;
  float* tile = lds_f;                  // [kAttnChunk][hd] values
  float* qs = tile + kAttnChunk * hd;   // [G][hd]
  float* psb = qs + G * hd;             // [G][kAttnChunk]
  float* mlb = psb + G * kAttnChunk;    // [kAttnMaxGroup][2]
  float4* og = reinterpret_cast<float4*>(mlb + 2 * kAttnMaxGroup);  // [256]
  auto ps = [&](uint32_t g, uint32_t j) -> float& { return psb[g * kAttnChunk + j]; };
  auto ml = [&](uint32_t g, uint32_t k) -> float& { return mlb[2 * g + k]; };
  const AttnEntry e = entry(a, i);
  const uint32_t end = e.pos + 1, p0 = e.start + c * kAttnChunk;
  float* out = a.part + (((size_t)blockIdx.x * a.n_heads + h * G) * a.nchunk + c) * (hd + 2);
  const size_t gstride = (size_t)a.nchunk * (hd + 2);
  if (p0 >= end) {  // past the entry's span: an empty chunk
    if (t < G) {
      out[t * gstride + hd] = -INFINITY;
      out[t * gstride + hd + 1] = 0.0f;
    }
    return;
  }
  const uint32_t cnt = min(kAttnChunk, end - p0);
  const uint32_t j = t >> 2, qq = t & 3;
  const bool rowok = j < cnt;
  const bool last = ROPE && p0 + cnt == end, rownew = last && j == cnt - 1;  // the new position's chunk and row
  const bool rowold = rowok && !rownew;
  float4 kreg[NR], vreg[NR];
  {
    const float* kr = rowold ? key_row(a, e, p0 + j, h) : a.pool;
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const uint32_t col = qq + 4 * r;
      kreg[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      vreg[r] = kreg[r];
      if (rowold && col < q4) {
        kreg[r] = *reinterpret_cast<const float4*>(kr + 4 * col);
        vreg[r] = *reinterpret_cast<const float4*>(kr + (size_t)a.bs * kvd + 4 * col);
      }
    }
  }
  if constexpr (ROPE) {
    const uint32_t half = hd / 2, npair = G * half;
    float2* ang = reinterpret_cast<float2*>(og);  // [half] (cos, sin), then the new key and value: 3 hd floats of og
    float2 *kn = ang + half, *vn = kn + half;
    const float* qsrc = a.q + (size_t)i * a.q_stride + (size_t)h * G * hd;
    float x = 0.0f, y = 0.0f, nx = 0.0f, ny = 0.0f;
    if (t < npair) ld_pair(qsrc + (t / half) * hd, t % half, a.nsl, a.sl_stride, x, y);
    if (last && t < hd) {
      const float* src = (t < half ? a.k : a.v) + (size_t)i * a.kv_stride + h * hd;
      ld_pair(src, t % half, a.nsl, a.sl_stride, nx, ny);
    }
    if (t < half) {
      const float freq = 1.0f / powf(a.theta, (2.0f * (float)t) / (float)hd);
      float sn, cs;
      sincosf((float)e.pos * freq, &sn, &cs);
      ang[t] = make_float2(cs, sn);
    }
    __syncthreads();
    for (uint32_t pr = t; pr < npair; pr += 256) {
      if (pr != t) ld_pair(qsrc + (pr / half) * hd, pr % half, a.nsl, a.sl_stride, x, y);
      const float2 cs = ang[pr % half];
      reinterpret_cast<float2*>(qs)[pr] = make_float2(x * cs.x - y * cs.y, x * cs.y + y * cs.x);
    }
    if (last && t < hd) {
      float* kp = a.pool + (size_t)e.page * a.page_floats + ((size_t)h * a.bs + e.pos % a.bs) * hd;
      if (e.fresh && h == 0 && t == 0) e.pages[e.pos / a.bs] = e.page;  // for the calls after this one
      float2 w = make_float2(nx, ny);
      if (t < half) {
        const float2 cs = ang[t];
        w = make_float2(nx * cs.x - ny * cs.y, nx * cs.y + ny * cs.x);
        kn[t] = w;
      } else {
        vn[t - half] = w;
        kp += (size_t)a.bs * kvd;
      }
      kp[2 * (t % half)] = w.x;
      kp[2 * (t % half) + 1] = w.y;
    }
    __syncthreads();
    if (rownew) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const uint32_t col = qq + 4 * r;
        if (col < q4) {
          const float2 k0 = kn[2 * col], k1 = kn[2 * col + 1], v0 = vn[2 * col], v1 = vn[2 * col + 1];
          kreg[r] = make_float4(k0.x, k0.y, k1.x, k1.y);
          vreg[r] = make_float4(v0.x, v0.y, v1.x, v1.y);
        }
      }
    }
  } else {
    const float4* qsrc = reinterpret_cast<const float4*>(a.qr + (size_t)i * a.n_heads * hd + (size_t)h * G * hd);
    for (uint32_t x = t; x < G * q4; x += 256) reinterpret_cast<float4*>(qs)[x] = qsrc[x];
    __syncthreads();
  }
  // scores of position j, every head of the group
  float acc[kAttnMaxGroup];
#pragma unroll
  for (int g = 0; g < kAttnMaxGroup; g++) acc[g] = 0.0f;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const uint32_t col = qq + 4 * r;
    if (col < q4) {
      const float4 kv = kreg[r];
#pragma unroll
      for (int g = 0; g < kAttnMaxGroup; g++) {
        if ((uint32_t)g < G) {
          const float4 qv = reinterpret_cast<const float4*>(qs + g * hd)[col];
          float v = acc[g];
          v = fmaf(qv.x, kv.x, v);
          v = fmaf(qv.y, kv.y, v);
          v = fmaf(qv.z, kv.z, v);
          v = fmaf(qv.w, kv.w, v);
          acc[g] = v;
        }
      }
    }
  }
#pragma unroll
  for (int g = 0; g < kAttnMaxGroup; g++) {
    if ((uint32_t)g < G) {
      float v = acc[g];
      v += dpp_f<kDppXor1>(v);
      v += dpp_f<kDppXor2>(v);
      if (qq == 0) ps(g, j) = rowok ? v * a.scale : -INFINITY;
    }
  }
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const uint32_t col = qq + 4 * r;
    if (rowok && col < q4) reinterpret_cast<float4*>(tile + j * hd)[col] = vreg[r];
  }
  __syncthreads();
  // per head: max and sum over the chunk, one wave per head in turn. A NaN or +inf score
  // makes the reference's softmax uniform over the whole span (simd/mod.rs:132-158): the
  // chunk's max is then NaN, which the combine reads as that mark.
  const uint32_t lane = t & 63, w = t >> 6;
  for (uint32_t g = w; g < G; g += 4) {
    const float sc = ps(g, lane);  // kAttnChunk == 64: one position a lane
    const bool bad = __ballot(lane < cnt && (sc != sc || sc == INFINITY)) != 0ull;
    const float m = wave_max(sc);
    const float pv = lane < cnt && !bad ? gm_expf(sc - m) : 0.0f;
    ps(g, lane) = pv;
    const float l = wave_sum(pv);
    if (lane == 0) {
      ml(g, 0) = bad ? __int_as_float(0x7fc00000) : m;
      ml(g, 1) = l;
    }
  }
  __syncthreads();
  // o: item = (head, float4 column); with few items the positions split into parts
  const uint32_t items = G * q4;
  const float4* tile4 = reinterpret_cast<const float4*>(tile);
  auto pv_sum = [&](uint32_t item, uint32_t j0, uint32_t j1) {
    const uint32_t g = item / q4, d4 = item % q4;
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t jj = j0; jj < j1; jj++) {
      const float p = ps(g, jj);
      const float4 v = tile4[jj * q4 + d4];
      o.x = fmaf(p, v.x, o.x);
      o.y = fmaf(p, v.y, o.y);
      o.z = fmaf(p, v.z, o.z);
      o.w = fmaf(p, v.w, o.w);
    }
    return o;
  };
  auto put = [&](uint32_t item, float4 o) {
    if constexpr (ONE) {
      const uint32_t g = item / q4, col = 4 * (item % q4);
      const float m = ml(g, 0), l = ml(g, 1);
      if (m != m || m == -INFINITY) {  // attn_uniform's plain mean, from the tile
        const float u = fdiv(1.0f, (float)cnt);
        o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (uint32_t jj = 0; jj < cnt; jj++) {
          const float4 v = tile4[jj * q4 + item % q4];
          o = make_float4(o.x + v.x * u, o.y + v.y * u, o.z + v.z * u, o.w + v.w * u);
        }
      } else {  // 0 + o, as the combine's first chunk gives (a -0 sum becomes +0)
        o = make_float4((0.0f + o.x) / l, (0.0f + o.y) / l, (0.0f + o.z) / l, (0.0f + o.w) / l);
      }
      float* dst = a.ctx + ((size_t)i * a.n_heads + h * G + g) * hd + col;
      dst[0] = o.x; dst[1] = o.y; dst[2] = o.z; dst[3] = o.w;
      return;
    }
    float* dst = out + (item / q4) * gstride + 4 * (item % q4);
    dst[0] = o.x; dst[1] = o.y; dst[2] = o.z; dst[3] = o.w;
  };
  if (items <= 128) {
    const uint32_t parts = items <= 64 ? 4u : 2u, span = kAttnChunk / parts;
    if (t < items * parts) {
      const uint32_t part = t / items, j0 = part * span;
      og[t] = pv_sum(t % items, min(j0, cnt), min(j0 + span, cnt));
    }
    __syncthreads();
    if (t < items) {
      float4 o = og[t];
      for (uint32_t part = 1; part < parts; part++) {
        const float4 v = og[part * items + t];
        o.x += v.x; o.y += v.y; o.z += v.z; o.w += v.w;
      }
      put(t, o);
    }
  } else {
    for (uint32_t x = t; x < items; x += 256) put(x, pv_sum(x, 0, cnt));
  }
  if (!ONE && t < G) {
    out[t * gstride + hd] = ml(t, 0);
    out[t * gstride + hd + 1] = ml(t, 1);
  }
}

// The reference's softmax falls back to uniform weights when a score is NaN or +inf, or
// every score is -inf (simd/mod.rs:132-158); the context is then the values' plain mean,
// summed as add_scaled does (out += v * (1 / len), positions in order). Column d of
// query head hh; runs only on that rare input.
__device__ float attn_uniform(const AttnArgs& a, uint32_t i, uint32_t hh, uint32_t d) {
  const AttnEntry e = entry(a, i);
  const uint32_t kh = hh / (a.n_heads / a.n_kv), len = e.pos + 1 - e.start;
  const float u = fdiv(1.0f, (float)len);
  const size_t voff = (size_t)a.bs * a.n_kv * a.hd;
  float acc = 0.0f;
  for (uint32_t p = e.start; p <= e.pos; p++) acc = acc + key_row(a, e, p, kh)[voff + d] * u;
  return acc;
}

// grid (n, n_heads), 256 threads: the chunks merged, context = o / l, in one pass.
// Thread (g, d) with g < 256 / hd runs over the chunks c = g, g + 256 / hd, ... of column
// d (16 chunks in flight) with a running max: (M, L, O) is rescaled when a chunk's max
// exceeds M. The groups are then merged in group order. A chunk marked NaN (a NaN or
// +inf score), or no finite score at all, gives the uniform weights of attn_uniform.
// PICK: the entries of a.pick.
template <bool PICK>
__global__ void __launch_bounds__(256) k_attn_combine(AttnArgs a) {
  __shared__ float gm[256], gl[256], go[256];
  const uint32_t i = PICK ? a.pick[blockIdx.x] : blockIdx.x, hh = blockIdx.y, t = threadIdx.x, hd = a.hd, row = hd + 2, nc = a.nchunk;
  const float* base = a.part + ((size_t)blockIdx.x * a.n_heads + hh) * nc * row;
  const uint32_t ng = 256 / hd, g = t / hd, d = t % hd;
  float M = -INFINITY, L = 0.0f, O = 0.0f;
  bool bad = false;
  if (g < ng) {
    constexpr int kIn = 16;
    for (uint32_t c0 = g; c0 < nc; c0 += kIn * ng) {
      float mv[kIn], lv[kIn], pv[kIn];
#pragma unroll
      for (int r = 0; r < kIn; r++) {
        const uint32_t c = c0 + r * ng;
        mv[r] = -INFINITY;
        if (c < nc) {
          const float* rc = base + (size_t)c * row;
          mv[r] = rc[hd];
          lv[r] = rc[hd + 1];
          pv[r] = rc[d];
        }
      }
#pragma unroll
      for (int r = 0; r < kIn; r++) {
        if (mv[r] != mv[r]) {  // a NaN or +inf score in that chunk
          bad = true;
          continue;
        }
        if (mv[r] == -INFINITY) continue;  // an empty chunk
        if (mv[r] > M) {
          const float f = gm_expf(M - mv[r]);  // 0 while M is -inf
          L = fmaf(L, f, lv[r]);
          O = fmaf(O, f, pv[r]);
          M = mv[r];
        } else {
          const float f = gm_expf(mv[r] - M);
          L = fmaf(lv[r], f, L);
          O = fmaf(pv[r], f, O);
        }
      }
    }
  }
  gm[t] = bad ? __int_as_float(0x7fc00000) : M;
  gl[t] = L;
  go[t] = O;
  __syncthreads();
  if (t < hd) {
    float Mt = gm[t], Lt = gl[t], Ot = go[t];
    bool bad_t = Mt != Mt;
    if (bad_t) Mt = -INFINITY;
    for (uint32_t k = 1; k < ng; k++) {
      const float m2 = gm[k * hd + t];
      if (m2 != m2) {
        bad_t = true;
        continue;
      }
      if (m2 == -INFINITY) continue;
      if (m2 > Mt) {
        const float f = gm_expf(Mt - m2);
        Lt = fmaf(Lt, f, gl[k * hd + t]);
        Ot = fmaf(Ot, f, go[k * hd + t]);
        Mt = m2;
      } else {
        const float f = gm_expf(m2 - Mt);
        Lt = fmaf(gl[k * hd + t], f, Lt);
        Ot = fmaf(go[k * hd + t], f, Ot);
      }
    }
    a.ctx[(size_t)i * a.n_heads * hd + hh * hd + t] =
        bad_t || Mt == -INFINITY ? attn_uniform(a, i, hh, t) : Ot / Lt;
  }
}

// ---------------------------------------------------------------------------------
// Tiled attention: runs of tokens of one sequence (a prompt's positions).
//
// One workgroup per (kv head, tile of 256 (token, query head) rows, split of the keys), 8
// waves of 32 rows. The single-token kernels read a kv head's keys and values once for
// every token; here a 32-key tile in LDS serves 256 rows. The products run on bf16 MFMA at
// f32 precision: an f32 is the sum of three bf16 of 8 bits each (split_planes, exact), and of
// the nine products of two such sums the six down to 2^-16 of the first are taken. Each plane
// is rounded to nearest, so the second is at most 2^-8 of the value and the third 2^-16, of
// either sign: the three products left out are at most 2^-23 of the first (typically a
// tenth of that) and cancel over a sum. (Truncated planes left up to 2^-21 out, always of
// the product's sign.) Six passes of v_mfma_f32_32x32x16_bf16 take 3/8 of the cycles of
// v_mfma_f32_32x32x2_f32.
//   S^T = K Q^T: A = the keys (row l % 32), B = the wave's queries, so lane l holds the
//     scores of query l % 32 for keys 8 (r / 4) + 4 (l / 32) + r % 4, r = 0..15;
//   O^T = V^T P^T: with those keys taken in that order, lane l's own 16 probabilities are
//     the B operand as they stand; A is V^T (row d = l % 32), transposed while staged.
// So a row's softmax state sits in two lanes (l, l ^ 32), and no probability moves.
// Grid x is the kv head: workgroups go round-robin over the 8 XCDs, so with 8 kv heads a
// head's keys and values are read into one XCD's L2.
//
// Measured (a 1500-token prompt in 256-token calls, 32 heads on 8 of 128): 35 us a call on
// average, against 198 us of k_attn_partial; its products are 5.9 GFLOP at 1400 keys, 35
// GFLOP in six passes. A 32-key tile takes 3.9 us where its MFMAs take 2.6 (8 waves); 6 us
// of a call are its start (tile, pages, first keys, queries) and its partial rows. With f32
// MFMA instead the same call took 54 us. Row sums: the tile's products are summed by
// themselves, smallest planes first, then added to the row's in one rounding (with one long
// chain the error against 64 bits was 1.8 times as large).
//
// Non-finite input: 0 * inf and inf - inf make NaNs of what f32 products would leave alone
// (keys beside a row's span, -inf scores), so a row that meets a non-finite score or ends
// with a non-finite sum is marked and summed by itself (attn_row).
//
// The softmax runs in base 2 (v_exp_f32 on scores scaled by log2 e). Against 64 bits, relative
// (2-norm), single-token kernels and this one: 32 heads on 8 of 128, 17 tokens 1.05e-7 and 0.82e-7,
// 256 tokens 1.62e-7 and 1.30e-7, 1500 tokens 1.85e-7 and 1.57e-7; 8 heads on 2 of 32 1.55e-7 and 1.38e-7
// at 1500; queries 16 times as large (scores to about 100) 6.7e-7 and 5.9e-7.
// ---------------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Two f32 rounded to a pair of bf16, and back.
__device__ __forceinline__ uint32_t bf_pair(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
// N values (even) as three planes of bf16 pairs: each plane what is left of the value after
// the ones before it (exact: 24 bits in three signed 8-bit parts), rounded to nearest.
template <int N>
__device__ __forceinline__ void split_planes(const float* x, uint32_t (*w)[N / 2]) {
#pragma unroll
  for (int i = 0; i < N / 2; i++) {
    float lo = x[2 * i], hi = x[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; p++) {
      w[p][i] = bf_pair(lo, hi);
      lo -= __uint_as_float(w[p][i] << 16);
      hi -= __uint_as_float(w[p][i] & 0xffff0000u);
    }
  }
}
__device__ __forceinline__ bf16x8 frag4(const uint32_t* w) {
  return __builtin_bit_cast(bf16x8, u32x4{w[0], w[1], w[2], w[3]});
}
__device__ __forceinline__ f32x16 mfma_bf(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// c += the five smaller products of a * b, two values split in three planes.
__device__ __forceinline__ f32x16 mfma_rest(const bf16x8* a, const bf16x8* b, f32x16 c) {
  c = mfma_bf(a[2], b[0], c);
  c = mfma_bf(a[0], b[2], c);
  c = mfma_bf(a[1], b[1], c);
  c = mfma_bf(a[1], b[0], c);
  return mfma_bf(a[0], b[1], c);
}

// A split's max may be a mark: a row for attn_row (a NaN pattern no max can be).
constexpr uint32_t kMarkSerial = 0x7fc00001u;

__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }

template <int NT>  // head_dim = 32 NT
__global__ void __launch_bounds__(512, 2) k_attn_tile(AttnArgs a) {
  constexpr uint32_t HD = 32 * NT, KT = kAttnTileKeys, KS = HD / 16;
  // a buffer: keys [plane][key][HD], 16-byte column x at x ^ (key % KX); values transposed
  // [plane][d][KT] in rows of 80 bytes (which spread a column's 16-byte reads over all
  // banks). Two buffers: the next tile is loaded while this one's products run (to LDS, a
  // thread's own 16 bytes at a time: the registers are full), then split and written, with
  // one barrier a tile.
  constexpr uint32_t KX = NT == 4 ? 16 : NT == 2 ? 8 : 4, KPL = KT * HD * 2, VP = 2 * KT + 16, VPL = HD * VP;
  constexpr uint32_t BUF = 3 * (KPL + VPL);
  constexpr int NK = (NT + 1) / 2;  // key float4 a thread
  static_assert(KT == 32 && kAttnTileRows == 256, "one MFMA row tile of keys, eight of rows");
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * BUF];
  __shared__ float4 raw[NK + 2 < 4 ? 2048 : (NK + 2) * 512];  // at least 4 KB a wave for the output
  __shared__ uint32_t tab[2][KT];  // pool rows (of HD floats) of a tile's keys
  const uint32_t h = blockIdx.x, c = blockIdx.z, tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hf = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t G = a.n_heads / a.n_kv;
  const AttnTile* T = a.tiles + blockIdx.y;
  auto uni = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane(v); };
  const uint32_t i0 = uni(T->i0), r0 = uni(T->r0), nr = uni(T->nr);
  const uint32_t pos0 = uni(T->pos0), start1 = uni(T->start1);
  const uint32_t k0 = uni(T->start0) + c * a.skeys, k1 = min(uni(T->pos1) + 1, k0 + a.skeys);
  const uint32_t row = 32 * wave + l32, rr = r0 + min(row, nr - 1), i = i0 + rr / G;
  const uint32_t head = h * G + rr % G, rows = a.n * a.n_heads;
  const uint32_t prow = c * rows + i * a.n_heads + head;  // the row's partial
  float* pml = a.part + (size_t)a.nchunk * rows * HD;
  const bool mine = row < nr;
  if (k0 >= k1) {  // past the tile's span: an empty split
    if (mine && hf == 0) {
      pml[2 * (size_t)prow] = -INFINITY;
      pml[2 * (size_t)prow + 1] = 0.0f;
    }
    return;
  }
  const uint32_t pos = a.ent[i].pos, start = a.ent[i].start;
  const uint32_t* pages = T->pages;
  const uint32_t prows = 2 * a.bs * a.n_kv;  // pool rows of a page
  // page and row in it of a key position (the product waits for the page's load)
  auto look = [&](uint32_t p, uint32_t& page, uint32_t& off) {
    const uint32_t q = min(p, k1 - 1), pg = q / a.bs;
    page = pages[pg];
    off = h * a.bs + (q - pg * a.bs);
  };
  if (tid < 2 * KT) {
    uint32_t page, off;
    look(k0 + tid, page, off);
    tab[tid / KT][tid % KT] = page * prows + off;
  }
  f32x16 o[NT], zero;
#pragma unroll
  for (int r = 0; r < 16; r++) zero[r] = 0.0f;
#pragma unroll
  for (int t = 0; t < NT; t++) o[t] = zero;
  float M = -INFINITY, L = 0.0f;  // M in units of log2, as the scores below
  bool odd = false;               // a non-finite score was seen
  const float sc2 = a.scale * 0x1.715476p+0f;  // log2 e
  // staging: the thread's keys (float4 kx of keys it / (8 NT)), and of the values a pair of
  // keys kp and four columns dq
  const uint32_t kp = lane % 16, dq = 4 * wave + lane / 16;
  const uint32_t vwo = 3 * KPL + 4 * dq * VP + 16 * (2 * (kp / 8) + (kp / 2) % 2) + 8 * ((kp / 4) % 2) + 4 * (kp % 2);
  const bool vmine = wave < 2 * NT;
  const float4* vpool = reinterpret_cast<const float4*>(a.pool + (size_t)a.bs * a.n_kv * HD);
  auto load = [&](uint32_t b) {
    auto lds16 = [&](const float4* src, uint32_t j) {
      __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)(raw + 512 * j + 64 * wave), 16, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < NK; j++) {
      const uint32_t it = j * 512 + tid, key = it / (8 * NT), x = it % (8 * NT);
      if ((j + 1) * 512 <= 256 * NT || 64 * wave < 256 * NT - j * 512)
        lds16(reinterpret_cast<const float4*>(a.pool + (size_t)tab[b][key] * HD) + x, j);
    }
    if (vmine)
#pragma unroll
      for (uint32_t j = 0; j < 2; j++) lds16(vpool + (size_t)tab[b][2 * kp + j] * (HD / 4) + dq, NK + j);
  };
  auto store = [&](uint8_t* buf) {
#pragma unroll
    for (int j = 0; j < NK; j++) {
      const uint32_t it = j * 512 + tid, key = it / (8 * NT), x = it % (8 * NT);
      if ((j + 1) * 512 <= 256 * NT || 64 * wave < 256 * NT - j * 512) {
        const float4 kv = raw[512 * j + tid];
        const float v[4] = {kv.x, kv.y, kv.z, kv.w};
        uint32_t w[3][2];
        split_planes<4>(v, w);
        uint8_t* dst = buf + key * HD * 2 + (((x / 2) ^ (key % KX)) * 16 + 8 * (x % 2));
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<u32x2*>(dst + p * KPL) = u32x2{w[p][0], w[p][1]};
      }
    }
    if (vmine) {
      const float4 v0 = raw[512 * NK + tid], v1 = raw[512 * (NK + 1) + tid];
      const float v[4][2] = {{v0.x, v1.x}, {v0.y, v1.y}, {v0.z, v1.z}, {v0.w, v1.w}};
#pragma unroll
      for (int d = 0; d < 4; d++) {
        uint32_t w[3][1];
        split_planes<2>(v[d], w);
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<uint32_t*>(buf + vwo + d * VP + p * VPL) = w[p][0];
      }
    }
  };
  float4 qx[2 * KS];
  {
    const float4* qs = reinterpret_cast<const float4*>(a.qr + ((size_t)i * a.n_heads + head) * HD);
#pragma unroll
    for (uint32_t s = 0; s < KS; s++) {
      qx[2 * s] = qs[4 * s + 2 * hf];
      qx[2 * s + 1] = qs[4 * s + 2 * hf + 1];
    }
  }
  __syncthreads();
  load(0);
  bf16x8 q[KS][3];
#pragma unroll
  for (uint32_t s = 0; s < KS; s++) {
    const float4 x = qx[2 * s], y = qx[2 * s + 1];
    const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
    uint32_t w[3][4];
    split_planes<8>(v, w);
#pragma unroll
    for (int p = 0; p < 3; p++) q[s][p] = frag4(w[p]);
  }
  __builtin_amdgcn_s_waitcnt(0);
  store(lds);
  __syncthreads();

  uint32_t tb = 0;
  for (uint32_t kb = k0; kb < k1; kb += KT, tb ^= 1) {
    const bool more = kb + KT < k1;
    uint32_t page = 0, off = 0;
    if (more) {
      if (tid < KT) look(kb + 2 * KT + tid, page, off);
      load(tb ^ 1);
    }
    const uint8_t* buf = lds + tb * BUF;
    if (32 * wave < nr) {
      f32x16 s = zero, sr = zero;  // the products of the first planes, and of the others
#pragma unroll
      for (uint32_t st = 0; st < KS; st++) {
        bf16x8 kf[3];
#pragma unroll
        for (int p = 0; p < 3; p++)
          kf[p] = *reinterpret_cast<const bf16x8*>(buf + l32 * HD * 2 + p * KPL + ((2 * st + hf) ^ (l32 % KX)) * 16);
        sr = mfma_rest(kf, q[st], sr);
        s = mfma_bf(kf[0], q[st][0], s);
      }
      float mt = -INFINITY;
#pragma unroll
      for (uint32_t r = 0; r < 16; r++) {
        s[r] = (s[r] + sr[r]) * sc2;
        odd |= __builtin_amdgcn_classf(s[r], 0x207);  // NaN or infinite
      }
      if (kb + KT > min(pos0 + 1, k1) || kb < start1) {  // keys that some row does not attend to
        const uint32_t p0 = kb + 4 * hf, hi = min(pos + 1, k1);
#pragma unroll
        for (uint32_t r = 0; r < 16; r++) {
          const uint32_t p = p0 + 8 * (r / 4) + r % 4;
          s[r] = p >= hi || p < start ? -INFINITY : s[r];
        }
      }
#pragma unroll
      for (uint32_t r = 0; r < 16; r++) mt = fmaxf(mt, s[r]);
      mt = fmaxf(M, fmaxf(mt, other_half(mt)));
      const float mu = mt == -INFINITY ? 0.0f : mt;
      const float f = __builtin_amdgcn_exp2f(M - mu);
      M = mt;
      float pv[16], ps = 0.0f;
#pragma unroll
      for (uint32_t r = 0; r < 16; r++) {
        pv[r] = __builtin_amdgcn_exp2f(s[r] - mu);
        ps += pv[r];
      }
      L = fmaf(L, f, ps);
      uint32_t w[2][3][4];
      bf16x8 pf[2][3];
#pragma unroll
      for (int st = 0; st < 2; st++) {
        split_planes<8>(pv + 8 * st, w[st]);
#pragma unroll
        for (int p = 0; p < 3; p++) pf[st][p] = frag4(w[st][p]);
      }
      // the tile's sum by itself, then one rounding into the row's: a long chain of them
      // cost more than the products' own
#pragma unroll
      for (int t = 0; t < NT; t++) {
        f32x16 d = zero;
        bf16x8 vf[2][3];
#pragma unroll
        for (int st = 0; st < 2; st++) {
#pragma unroll
          for (int p = 0; p < 3; p++)
            vf[st][p] = *reinterpret_cast<const bf16x8*>(buf + 3 * KPL + (l32 + 32 * t) * VP + p * VPL + 16 * hf + 32 * st);
          d = mfma_rest(vf[st], pf[st], d);
        }
        d = mfma_bf(vf[0][0], pf[0][0], d);
        d = mfma_bf(vf[1][0], pf[1][0], d);
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = fmaf(o[t][r], f, d[r]);
      }
    }
    if (more) {
      __builtin_amdgcn_s_waitcnt(0);  // the wave's own loads, in LDS
      if (tid < KT) tab[tb][tid] = page * prows + off;
      store(lds + (tb ^ 1) * BUF);
    }
    __syncthreads();
  }
  L += other_half(L);
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) odd |= __builtin_amdgcn_classf(o[t][r], 0x207);
  odd |= other_half(odd ? 1.0f : 0.0f) != 0.0f;
  if (mine && hf == 0) {
    pml[2 * (size_t)prow] = odd ? __uint_as_float(kMarkSerial) : M;
    pml[2 * (size_t)prow + 1] = L;
  }
  // through LDS, 32 columns at a time, so that a row's 128 bytes go out together (lane l
  // holds 16-byte pieces of row l % 32); the wave's own 4 KB of raw, 16-byte column x of
  // row j at x ^ (j % 8)
  float4* w4 = raw + 256 * wave;
  const uint32_t orow = lane / 8, ox = lane % 8;
#pragma unroll
  for (uint32_t t = 0; t < NT; t++) {
#pragma unroll
    for (uint32_t j = 0; j < 4; j++)
      w4[8 * l32 + ((2 * j + hf) ^ (l32 % 8))] = make_float4(o[t][4 * j], o[t][4 * j + 1], o[t][4 * j + 2], o[t][4 * j + 3]);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t x = 8 * j + orow;
      const uint32_t to = __shfl(prow, x, 64);
      if (32 * wave + x < nr) reinterpret_cast<float4*>(a.part + (size_t)to * HD)[8 * t + ox] = w4[8 * x + (ox ^ (x % 8))];
    }
  }
}

// attn_uniform's four columns from d on.
__device__ float4 attn_uniform4(const AttnArgs& a, uint32_t i, uint32_t hh, uint32_t d) {
  const AttnEntry e = entry(a, i);
  const uint32_t kh = hh / (a.n_heads / a.n_kv);
  const float u = fdiv(1.0f, (float)(e.pos + 1 - e.start));
  const size_t voff = (size_t)a.bs * a.n_kv * a.hd + d;
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (uint32_t p = e.start; p <= e.pos; p++) {
    const float4 v = *reinterpret_cast<const float4*>(key_row(a, e, p, kh) + voff);
    o = make_float4(o.x + v.x * u, o.y + v.y * u, o.z + v.z * u, o.w + v.w * u);
  }
  return o;
}

// Row hh of token i by the whole workgroup, for the rows that k_attn_tile marks (non-finite
// input): chunks of kAttnChunk positions as the single-token kernels cut them, scores four
// threads a position, values a thread per (every q4-th position, float4 column x = t % q4),
// in f32. sc [kAttnChunk], po [256] in LDS. Returns false where the softmax falls back to
// uniform weights (a NaN or +inf score, or none above -inf), as soon as that is known;
// otherwise threads x < q4 have the row's columns 4 x .. 4 x + 3 in w.
__device__ bool attn_row(const AttnArgs& a, uint32_t i, uint32_t hh, float* sc, float4* po, float4& w) {
  const AttnEntry e = entry(a, i);
  const uint32_t t = threadIdx.x, lane = t & 63, hd = a.hd, q4 = hd / 4, ng = 256 / q4, g = t / q4, x = t % q4;
  const uint32_t kh = hh / (a.n_heads / a.n_kv);
  const size_t voff = (size_t)a.bs * a.n_kv * hd;
  const float4* q = reinterpret_cast<const float4*>(a.qr + ((size_t)i * a.n_heads + hh) * hd);
  float M = -INFINITY, L = 0.0f;
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (uint32_t p0 = e.start; p0 <= e.pos; p0 += kAttnChunk) {
    const uint32_t cnt = min(kAttnChunk, e.pos + 1 - p0), j = t >> 2;
    float s = 0.0f;
    if (j < cnt) {
      const float4* kr = reinterpret_cast<const float4*>(key_row(a, e, p0 + j, kh));
      for (uint32_t c = t & 3; c < q4; c += 4) {
        const float4 kv = kr[c], qv = q[c];
        s = fmaf(kv.x, qv.x, s);
        s = fmaf(kv.y, qv.y, s);
        s = fmaf(kv.z, qv.z, s);
        s = fmaf(kv.w, qv.w, s);
      }
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if ((t & 3) == 0) sc[j] = j < cnt ? s * a.scale : -INFINITY;
    __syncthreads();
    const float v = sc[lane];
    if (__ballot(v != v || v == INFINITY)) return false;  // every wave sees the same scores
    const float mc = wave_max(v);
    if (mc > -INFINITY) {  // a chunk without a score above -inf adds nothing
      const float mn = fmaxf(M, mc), f = gm_expf(M - mn), pv = lane < cnt ? gm_expf(v - mn) : 0.0f;
      M = mn;
      L = fmaf(L, f, wave_sum(pv));
      __syncthreads();
      if (t < kAttnChunk) sc[t] = pv;
      __syncthreads();
      o = make_float4(o.x * f, o.y * f, o.z * f, o.w * f);
      if (g < ng)
        for (uint32_t jj = g; jj < cnt; jj += ng) {
          const float4 vv = *reinterpret_cast<const float4*>(key_row(a, e, p0 + jj, kh) + voff + 4 * x);
          const float pj = sc[jj];
          o = make_float4(fmaf(pj, vv.x, o.x), fmaf(pj, vv.y, o.y), fmaf(pj, vv.z, o.z), fmaf(pj, vv.w, o.w));
        }
    }
    __syncthreads();
  }
  if (M == -INFINITY) return false;
  po[t] = o;
  __syncthreads();
  if (t < q4) {
    for (uint32_t k = 1; k < ng; k++) {
      const float4 b = po[k * q4 + t];
      o = make_float4(o.x + b.x, o.y + b.y, o.z + b.z, o.w + b.w);
    }
    w = make_float4(o.x / L, o.y / L, o.z / L, o.w / L);
  }
  return true;
}

// The splits of a tiled call merged: a thread per four columns of a (token, head) row, the
// splits kIn at a time with a running max. Marked rows, and those without any score above
// -inf, are then summed by the workgroup one after another (attn_row), the uniform ones of
// them by their own threads: 256 tokens over a NaN key 128 tokens in 547 us, in the
// single-token kernels 860 to 1100 (each thread summing its columns' row took 7.2 ms). With
// many splits (40 tokens at 4000, 8 heads on 2 of 32: 63) a batch's loads are in flight
// together: the call 54.5 -> 26 us.
__global__ void __launch_bounds__(256) k_attn_merge(AttnArgs a) {
  __shared__ float4 po[256];
  __shared__ float sc[kAttnChunk];
  __shared__ uint32_t marks;
  const uint32_t rows = a.n * a.n_heads, q4 = a.hd / 4, rpb = 256 / q4, r = threadIdx.x / q4, x = threadIdx.x % q4;
  const uint32_t row = blockIdx.x * rpb + r;
  const bool mine = r < rpb && row < rows && !(a.npick && (a.ent[row / a.n_heads].fresh & kAttnSingle));
  float4 w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  bool serial = false;
  if (threadIdx.x == 0) marks = 0;
  __syncthreads();
  if (mine) {
    constexpr uint32_t kIn = 8;
    const float2* ml = reinterpret_cast<const float2*>(a.part + (size_t)a.nchunk * rows * a.hd) + row;
    const float4* po4 = reinterpret_cast<const float4*>(a.part) + (size_t)row * q4 + x;
    float M = -INFINITY, L = 0.0f;  // M in units of log2
    float4 o = w;
    for (uint32_t c0 = 0; c0 < a.nchunk; c0 += kIn) {
      float2 v[kIn];
      float4 p[kIn];
      float mb = M;
#pragma unroll
      for (uint32_t k = 0; k < kIn; k++) {
        const uint32_t c = min(c0 + k, a.nchunk - 1);
        v[k] = ml[(size_t)c * rows];
        p[k] = po4[(size_t)c * rows * q4];
        if (c0 + k >= a.nchunk) v[k].x = -INFINITY;
        serial |= v[k].x != v[k].x;
        mb = fmaxf(mb, v[k].x);
      }
      if (mb > M) {
        const float f = __builtin_amdgcn_exp2f(M - mb);
        L *= f;
        o = make_float4(o.x * f, o.y * f, o.z * f, o.w * f);
        M = mb;
      }
#pragma unroll
      for (uint32_t k = 0; k < kIn; k++) {
        if (!(v[k].x > -INFINITY)) continue;  // nothing was written for an empty split
        const float f = __builtin_amdgcn_exp2f(v[k].x - M);
        L = fmaf(v[k].y, f, L);
        o = make_float4(fmaf(p[k].x, f, o.x), fmaf(p[k].y, f, o.y), fmaf(p[k].z, f, o.z), fmaf(p[k].w, f, o.w));
      }
    }
    w = make_float4(o.x / L, o.y / L, o.z / L, o.w / L);
    serial |= M == -INFINITY;
    if (serial && x == 0) atomicOr(&marks, 1u << r);
  }
  __syncthreads();
  for (uint32_t left = marks; left; left &= left - 1) {
    const uint32_t r1 = __builtin_ctz(left), row1 = blockIdx.x * rpb + r1;
    float4 w1;
    const bool ok = attn_row(a, row1 / a.n_heads, row1 % a.n_heads, sc, po, w1);
    __syncthreads();
    if (ok) {
      if (threadIdx.x < q4) po[threadIdx.x] = w1;
      __syncthreads();
      if (r == r1) {
        w = po[x];
        serial = false;
      }
      __syncthreads();
    }
  }
  if (!mine) return;
  if (serial) w = attn_uniform4(a, row / a.n_heads, row % a.n_heads, 4 * x);
  reinterpret_cast<float4*>(a.ctx)[(size_t)row * q4 + x] = w;
}

template <bool ROPE, bool ONE>
static void launch_partial(const AttnArgs& a, hipStream_t st) {
  static const bool once =
      hipFuncSetAttribute((const void*)k_attn_partial<128, ROPE, ONE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)attn_lds_bytes(kAttnMaxGroup, 128)) == hipSuccess &&
      hipFuncSetAttribute((const void*)k_attn_partial<kAttnMaxHd, ROPE, ONE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)attn_lds_bytes(kAttnMaxGroup, kAttnMaxHd)) == hipSuccess;
  (void)once;
  const dim3 grid(a.pick ? a.npick : a.n, a.n_kv, a.nchunk);
  const uint32_t lds = attn_lds_bytes(a.n_heads / a.n_kv, a.hd);
  if (a.hd <= 128) hipLaunchKernelGGL((k_attn_partial<128, ROPE, ONE>), grid, dim3(256), lds, st, a);
  else hipLaunchKernelGGL((k_attn_partial<kAttnMaxHd, ROPE, ONE>), grid, dim3(256), lds, st, a);
}

// Whether the context's floats overlap those of `rows` rows of q, k or v (all their slices).
static bool ctx_overlaps(const AttnArgs& a, const float* p, uint32_t width, uint32_t stride) {
  const uintptr_t c0 = (uintptr_t)a.ctx, c1 = c0 + (size_t)a.n * a.n_heads * a.hd * 4, p0 = (uintptr_t)p;
  const uintptr_t p1 = p0 + (((size_t)a.n - 1) * stride + width + (a.nsl > 1 ? (a.nsl - 1) * a.sl_stride : 0)) * 4;
  return c0 < p1 && p0 < c1;
}

hipError_t launch_attention(const AttnArgs& a, hipStream_t st) {
  // The fused first launch needs every key but an entry's own in the pages already: entries
  // of different sequences. One chunk then needs no other launch, unless the context lies
  // over an input that a workgroup of another head or token has yet to read.
  const uint32_t qd = a.n_heads * a.hd, kvd = a.n_kv * a.hd;
  const bool one = a.nchunk == 1 && !ctx_overlaps(a, a.q, qd, a.q_stride) && !ctx_overlaps(a, a.k, kvd, a.kv_stride) &&
                   !ctx_overlaps(a, a.v, kvd, a.kv_stride);
  if (a.distinct && one) {
    launch_partial<true, true>(a, st);
    return hipGetLastError();
  }
  if (a.distinct) {
    launch_partial<true, false>(a, st);
  } else {
    const uint32_t pairs = (a.n_heads + a.n_kv) * a.hd / 2;
    hipLaunchKernelGGL(k_rope_append, dim3(a.n, (pairs + 255) / 256), dim3(256), 0, st, a);
    launch_partial<false, false>(a, st);
  }
  hipLaunchKernelGGL(k_attn_combine<false>, dim3(a.n, a.n_heads), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_attention_tiled(const AttnArgs& a, const AttnArgs& rest, hipStream_t st) {
  hipLaunchKernelGGL(k_rope_rows, dim3(a.n, 2), dim3(256), 0, st, a);  // every entry's k and v before any attends
  const dim3 grid(a.n_kv, a.ntile, a.nchunk);
  switch (a.hd / 32) {
    case 1: hipLaunchKernelGGL(k_attn_tile<1>, grid, dim3(512), 0, st, a); break;
    case 2: hipLaunchKernelGGL(k_attn_tile<2>, grid, dim3(512), 0, st, a); break;
    case 3: hipLaunchKernelGGL(k_attn_tile<3>, grid, dim3(512), 0, st, a); break;
    default: hipLaunchKernelGGL(k_attn_tile<4>, grid, dim3(512), 0, st, a); break;
  }
  const uint32_t rpb = 256 / (a.hd / 4);
  hipLaunchKernelGGL(k_attn_merge, dim3((a.n * a.n_heads + rpb - 1) / rpb), dim3(256), 0, st, a);
  if (a.npick) {
    launch_partial<false, false>(rest, st);
    hipLaunchKernelGGL(k_attn_combine<true>, dim3(a.npick, a.n_heads), dim3(256), 0, st, rest);
  }
  return hipGetLastError();
}

}  // namespace gmoe
