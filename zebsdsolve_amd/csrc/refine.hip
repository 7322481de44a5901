// Orientation refinement on the detector, fused: one block of 1 to 16 waves (64 lanes each) per
// item runs the seed, every Gauss-Newton iteration, the normalized mutual information and the
// record, in one launch (the reference's detector.wgsl seed, refine_init, sums_rot +
// refine_rot_step per iteration, nmi and collect; src/detector.zig:178-212).
//
// Per iteration each lane adds up its pixels' share of the 19 sums the step needs (1, M, M^2,
// M e, d, M d, e d and the upper triangle of d d', with d = c x grad M(c) for c = q . ray); the
// wave that adds the last pixels sums over the lanes and takes the step for the block. The
// master's gradient field holds (grad M, M) per texel: one bilinear lookup reads both.
// What bounds it: the gathers' cache lines (a step of 64 pixels touches 70 to 100 lines of 128
// bytes, at 64 bytes a clock into the CU's cache) beside 110 vector instructions a step. One wave an
// item, its list and pattern read again in each pass, left most of the chip idle for few or large
// items: 8 items of 120 x 120 took 723 us and take 235, 40 of 240 x 240 3 673 and 569, 4 500 of
// 60 x 60 634 and 513, 16 000 1 944 and 1 716 (5 iterations at 60 x 60, 8 else).
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

#include "common.h"

namespace zb {

struct RefArg {
    float c0[3], c1[3], c2[3];
    float mask[3];
    int h, w, side;
    int iters, nmi_bins, polls, out0;
    float max_step, scale0, scale_min, scale_max;
    float stamp;
    int tiles;  // 8 x 8 tiles of the frame the tile walk lists (0: every tile is walked)
};

// A value every lane holds alike, read from the first lane into a scalar register.
__device__ __forceinline__ float ufloat(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
__device__ __forceinline__ float4 uniform4(float4 v) { return make_float4(ufloat(v.x), ufloat(v.y), ufloat(v.z), ufloat(v.w)); }
// (a number known to the compiler, as an argument)
template <int N>
struct Const {
    static constexpr int value = N;
};
__device__ __forceinline__ float lane_of(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ __forceinline__ float3 f3s(float3 a, float s) { return make_float3(a.x * s, a.y * s, a.z * s); }

__device__ __forceinline__ bool under_mask(const RefArg& a, int r, int c) {
    const float dr = (float)r - a.mask[0], dc = (float)c - a.mask[1];
    return r < a.h && c < a.w && (a.mask[2] <= 0.f || dr * dr + dc * dc <= a.mask[2]);
}

// The masked pixels of the frame as pixel indices, built by each block into LDS (the same list
// for every item): the passes then walk only the pixels under the mask, 64 at a time, instead of
// the whole frame with a quarter of the lanes idle. The order is by 8 x 8 tiles of the frame (in
// row-major tile order, each tile's pixels row-major), so that the 64 lanes of a pass look up a
// compact patch of the detector, whose rays land on nearby texels of the master, rather than a
// row segment, whose rays trace a long curve across it: fewer cache lines per gather (the
// refinement 6.8 % faster than with row-major order). One lane a pixel of the tile, the place in
// the list from the tile's ballot; with several waves each takes a run of the tiles, counted
// first (cnt: an int a wave). TILES: the tiles that hold a masked pixel instead, as tile numbers.
template <int W, bool TILES>
__device__ int build_list(const RefArg& a, unsigned short* list, int* cnt, int wave, int lane) {
    const int tw = (a.w + 7) >> 3, nt = tw * ((a.h + 7) >> 3);
    const int per = (nt + W - 1) / W;
    const int t_lo = min(wave * per, nt), t_hi = min(t_lo + per, nt);
    const int y = lane >> 3, x = lane & 7;
    int at = 0, total = 0;
    auto walk = [&](auto put) {
        int tr = t_lo / tw, tc = t_lo - (t_lo / tw) * tw;
        for (int t = t_lo; t < t_hi; ++t) {
            const int r = tr * 8 + y, c = tc * 8 + x;
            const bool in = under_mask(a, r, c);
            const unsigned long long m = __ballot(in);
            put(t, r, c, in, m);
            at += TILES ? (m ? 1 : 0) : __popcll(m);
            if (++tc == tw) tc = 0, ++tr;
        }
    };
    if constexpr (W > 1) {
        // (counted)
        walk([](int, int, int, bool, unsigned long long) {});
        if (lane == 0) cnt[wave] = at;
        __syncthreads();
        at = 0;
        for (int v = 0; v < W; ++v) {
            const int k = cnt[v];
            if (v < wave) at += k;
            total += k;
        }
    }
    walk([&](int t, int r, int c, bool in, unsigned long long m) {
        if constexpr (TILES) {
            if (m && lane == 0) list[at] = (unsigned short)t;
        } else {
            if (in) list[at + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = (unsigned short)(r * a.w + c);
        }
    });
    if constexpr (W == 1) total = at;
    __syncthreads();
    return total;
}

// An item's masked pixels are taken 64 a step, one a lane. A list form's steps are the list's
// entries in order, cut into chunks of consecutive steps dealt to the block's W waves in turn.
// Each wave looks its chunk's pixels up by itself and keeps what the sums need in registers; the
// sums then run through the chunks in order, handed from wave to wave through LDS, so that each
// lane adds its pixels up in the list's order whatever W is: a record's bits depend neither on the
// launch nor on the batch. (With partial sums a wave the last steps' acceptance, decided in the
// sums' last bits, came out otherwise for some items.) The look-ups are eight parts in nine of a
// pass's instructions and run side by side; the chain of additions is the rest.
//  REF_HELD: at most kHeld steps a wave: each lane holds its pixels' rays and pattern values in
//            registers over all passes;
//  REF_LIST: any number, the list and the pattern read again in each pass;
//  REF_TILES: frames whose pixels pass 16-bit indices or whose list passes LDS: a step is one
//            8 x 8 tile of the frame with the mask tested a pixel, from the list of tiles that hold
//            a masked pixel (every tile where that list passes LDS: tiles = 0), step s to wave s
//            mod W, and each wave's sums are added up on their own.
enum { REF_HELD, REF_LIST, REF_TILES };
constexpr int kHeld = 12;   // steps a lane holds (REF_HELD)
constexpr int kChunk = 6;   // steps of a chunk
// Pixels per lane whose gathers are in flight together: a lane issues the loads of kBatch pixels
// (2 each) before it blends any.
constexpr int kBatch = 3;
constexpr int kPart = 20;  // floats handed over: the 19 sums of a pass and a pad

// The refinement's state (detector.wgsl refine_init), kept in LDS between the passes (its
// registers would be every wave's).
struct Gn {
    float4 cur, qbest;
    float best, mu;
    float3 gbest;
    float hbest[6];
    float last_step, promised, step_size, accepted;
};

template <int W>
struct alignas(16) Shared {
    float4 acc[kPart / 4][64];  // the chain's sums, a lane's own (list forms)
    float part[W][kPart];       // each wave's sums (REF_TILES); each wave's extremes
    Gn gn;
    int cnt[W];
    int turn;  // the chunk whose sums are to be added next, counted over the item's passes
};

struct Held {
    float3 u[kHeld];
    float e[kHeld];
};

// The chunks of n_steps for W waves: as even as whole steps allow, at most kChunk steps each.
struct Chunks {
    int steps, size, count, rounds;
};
template <int W>
__device__ __forceinline__ Chunks chunks_of(int n_px) {
    Chunks c;
    c.steps = (n_px + 63) >> 6;
    c.rounds = max((c.steps + W * kChunk - 1) / (W * kChunk), 1);
    c.size = max((c.steps + W * c.rounds - 1) / (W * c.rounds), 1);
    c.count = max((c.steps + c.size - 1) / c.size, 1);
    return c;
}

// Waits until the chain reaches chunk `id` (its turn comes after finitely many chunks of other
// waves of the block, all resident; the bound only keeps a wave from waiting for ever: one that
// gives up takes the record's stamp away).
// The loop is written out so that a turn that has come leaves it by one branch: the hand-overs are a
// chain, some 300 for an item of 120 x 120, and the compiler's loop with a bound that is an argument and
// a store behind it cost 40 to 60 ns each (one item, 8 iterations: 231 us, with the compiler's 240 to 268).
template <int W>
__device__ __forceinline__ void wait_turn(Shared<W>& sh, int id, int polls, float* stamp) {
    int left = __builtin_amdgcn_readfirstlane(polls), seen, turn;
    const unsigned at = (unsigned)(size_t)(__attribute__((address_space(3))) int*)&sh.turn;
    asm volatile(
        "1:\n"
        "ds_read_b32 %0, %3\n"
        "s_waitcnt lgkmcnt(0)\n"
        "v_readfirstlane_b32 %1, %0\n"
        "s_cmp_eq_u32 %1, %4\n"
        "s_cbranch_scc1 2f\n"
        "s_sleep 1\n"
        "s_sub_u32 %2, %2, 1\n"
        "s_cmp_lg_u32 %2, 0\n"
        "s_cbranch_scc1 1b\n"
        "2:\n"
        : "=&v"(seen), "=&s"(turn), "+s"(left)
        : "v"(at), "s"(id)
        : "memory", "scc");
    if (__builtin_expect(left == 0, 0)) *stamp = __int_as_float(0x7fc00000);  // (no stamp equals a NaN)
}
__device__ __forceinline__ void pass_turn(int* turn, int id, int lane) {
    if (lane == 0) __hip_atomic_store(turn, id + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Steps wave `wave` takes of n_steps dealt one by one.
template <int W>
__device__ __forceinline__ int own_steps(int n_steps, int wave) {
    return (n_steps - wave + W - 1) / W;
}

// The ray of pixel (row, col) from the item's origin t, in the sample frame, of unit length.
__device__ __forceinline__ float3 pixel_ray(const RefArg& a, int row, int col, float3 t) {
    const float fr = (float)row, fc = (float)col;
    return normalize3(make_float3(a.c0[0] * fr + a.c1[0] * fc + t.x, a.c0[1] * fr + a.c1[1] * fc + t.y, a.c0[2] * fr + a.c1[2] * fc + t.z));
}

// A list form's pixel k: its ray and pattern value. The row by a float product (exact below
// 65 536 pixels).
__device__ __forceinline__ float3 list_pixel(const RefArg& a, const unsigned short* list, int k, int n_px, float inv_w, float3 t,
                                             const float* __restrict__ pat, float& e) {
    const int pix = list[min(k, n_px - 1)];
    const int row = (int)(((float)pix + 0.5f) * inv_w);
    e = pat[pix];
    return pixel_ray(a, row, pix - __mul24(row, a.w), t);
}

// The look-ups of one chunk of a list form, kBatch steps in flight: tap(p, ray) issues the loads
// of step p of the batch, keep(i, p, ray, pattern value) takes step i's in.
template <int MODE, int ROUND, typename Tap, typename Keep>
__device__ __forceinline__ void look_up(const RefArg& a, const unsigned short* list, int n_px, float inv_w, float3 t, const float* __restrict__ pat,
                                        const Held& held, int step0, int cnt, int lane, Tap tap, Keep keep) {
#pragma unroll
    for (int i0 = 0; i0 < kChunk; i0 += kBatch) {
        if (i0 < cnt) {
            float3 u[kBatch];
            float e[kBatch];
#pragma unroll
            for (int p = 0; p < kBatch; ++p) {
                if constexpr (MODE == REF_HELD) {
                    u[p] = held.u[ROUND * kChunk + i0 + p];
                    e[p] = held.e[ROUND * kChunk + i0 + p];
                } else {
                    u[p] = list_pixel(a, list, 64 * (step0 + i0 + p) + lane, n_px, inv_w, t, pat, e[p]);
                }
                u[p] = tap(p, u[p]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < kBatch; ++p) keep(i0 + p, p, u[p], e[p]);
        }
    }
}

// One wave's tiles, kBatch in flight: tap(p, ray, pixel) issues the loads of step p of the batch,
// keep(p) takes them in on the lanes whose pixel counts.
template <int W, typename Tap, typename Keep>
__device__ __forceinline__ void walk_tiles(const RefArg& a, const unsigned short* list, int n_tiles, float3 t, int wave, int lane, Tap tap, Keep keep) {
    const int tw = (a.w + 7) >> 3;
    const int own = own_steps<W>(n_tiles, wave);
    for (int i0 = 0; i0 < own; i0 += kBatch) {
        bool ok[kBatch];
#pragma unroll
        for (int p = 0; p < kBatch; ++p) {
            // steps past the end look up the wave's last tile again and add nothing
            const int k = wave + W * min(i0 + p, own - 1);
            const int tile = __builtin_amdgcn_readfirstlane(a.tiles ? (int)list[k] : k);
            const int tr = tile / tw;
            const int r = tr * 8 + (lane >> 3), c = (tile - tr * tw) * 8 + (lane & 7);
            ok[p] = i0 + p < own && under_mask(a, r, c);
            const int rr = min(r, a.h - 1), cc = min(c, a.w - 1);
            tap(p, pixel_ray(a, rr, cc, t), rr * a.w + cc);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < kBatch; ++p)
            if (ok[p]) keep(p);
    }
}

// 20 values summed over the wave's lanes: lane 16 r ends with the sums of v[4 j + {0, 2, 1, 3}[r]],
// j < 5. Two values share a register after each of the first two exchanges (halves, then rows of
// 16), so that the sums take 50 instructions, not the 120 of a butterfly for each.
__device__ __forceinline__ void wave_sums20(const float* v, float* out) {
    float x[10];
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * i]), __float_as_uint(v[2 * i + 1]), false, false);
        x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[2 * j]), __float_as_uint(x[2 * j + 1]), false, false);
        float s = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        s = dpp_add<0x128>(s);  // row_ror:8, 4, 2, 1
        s = dpp_add<0x124>(s);
        s = dpp_add<0x122>(s);
        out[j] = dpp_add<0x121>(s);
    }
}

__device__ __forceinline__ float det3(float3 c0, float3 c1, float3 c2) {
    return c0.x * (c1.y * c2.z - c2.y * c1.z) - c1.x * (c0.y * c2.z - c2.y * c0.z) + c2.x * (c0.y * c1.z - c1.y * c0.z);
}

// The symmetric 3 x 3 system (h: xx, xy, xz, yy, yz, zz) by Cramer's rule (detector.wgsl:519-527).
__device__ __forceinline__ float3 solve3(const float* h, float3 g) {
    const float3 m0 = make_float3(h[0], h[1], h[2]);
    const float3 m1 = make_float3(h[1], h[3], h[4]);
    const float3 m2 = make_float3(h[2], h[4], h[5]);
    const float det = det3(m0, m1, m2);
    if (fabsf(det) < 1e-30f) return make_float3(0.f, 0.f, 0.f);
    return make_float3(det3(g, m1, m2) / det, det3(m0, g, m2) / det, det3(m0, m1, g) / det);
}

// One pass's sums s (count, M, M^2, M e, M d, d, e d, d d' diagonal and off it, as rot_sums lays
// them out) taken in: the NCC, its gradient and Gauss-Newton matrix over the rotation
// (detector.wgsl:561-583), acceptance against the best so far, and unless `last` the next step.
__device__ __forceinline__ void gn_step(const RefArg& a, const float* s, bool last, Gn& g) {
    const float n = fmaxf(s[0], 1.f);
    const float mean = s[1] / n;
    const float var_n = s[2] - n * mean * mean;
    float ncc = -2.f;
    float3 grad = make_float3(0.f, 0.f, 0.f);
    float hess[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const float3 sd = make_float3(s[4], s[5], s[6]), sv = make_float3(s[7], s[8], s[9]), se = make_float3(s[10], s[11], s[12]);
    if (var_n > 1e-12f) {
        const float inv = 1.f / sqrtf(var_n);
        ncc = s[3] * inv;
        const float3 au = f3s(make_float3(sv.x - mean * sd.x, sv.y - mean * sd.y, sv.z - mean * sd.z), inv);
        grad = f3s(make_float3(se.x - ncc * au.x, se.y - ncc * au.y, se.z - ncc * au.z), inv);
        const float iv = inv * inv;
        hess[0] = (s[13] - sd.x * sd.x / n - au.x * au.x) * iv;
        hess[1] = (s[16] - sd.x * sd.y / n - au.x * au.y) * iv;
        hess[2] = (s[17] - sd.x * sd.z / n - au.x * au.z) * iv;
        hess[3] = (s[14] - sd.y * sd.y / n - au.y * au.y) * iv;
        hess[4] = (s[18] - sd.y * sd.z / n - au.y * au.z) * iv;
        hess[5] = (s[15] - sd.z * sd.z / n - au.z * au.z) * iv;
    }
    // accept against the best so far, rescaling the curvature by gain / promise
    if (ncc > g.best) {
        if (g.accepted > 0.5f && g.promised > 1e-6f) {
            const float rho = (ncc - g.best) / g.promised;
            g.mu = fminf(fmaxf(g.mu * (2.f - rho), g.mu / 3.f), g.mu * 3.f);
        }
        g.qbest = g.cur;
        g.best = ncc;
        g.gbest = grad;
#pragma unroll
        for (int i = 0; i < 6; ++i) g.hbest[i] = hess[i];
        g.last_step = g.step_size;
        g.accepted += 1.f;
    } else {
        g.mu = g.mu * 3.f;
    }
    g.mu = fminf(fmaxf(g.mu, a.scale_min), a.scale_max);
    if (last) return;
    float hh[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) hh[i] = g.hbest[i] * g.mu;
    const float tr = fmaxf(hh[0] + hh[3] + hh[5], 1e-20f);
    hh[0] += 1e-6f * tr;
    hh[3] += 1e-6f * tr;
    hh[5] += 1e-6f * tr;
    float3 st = solve3(hh, g.gbest);
    const float len = sqrtf(dot3(st, st));
    if (len > a.max_step) st = f3s(st, a.max_step / len);
    const float quad = hh[0] * st.x * st.x + hh[3] * st.y * st.y + hh[5] * st.z * st.z +
                       2.f * (hh[1] * st.x * st.y + hh[2] * st.x * st.z + hh[4] * st.y * st.z);
    g.promised = dot3(g.gbest, st) - 0.5f * quad;
    g.step_size = sqrtf(dot3(st, st));
    g.cur = qnormalize(qmul(qexp(st), g.qbest));
}

// What one pixel adds to a pass's sums: 0 count, 1 M, 2 M^2, 3 M e, 4 d, 7 M d, 10 e d, 13 d d'
// diagonal, 16 off it (d = c x grad M in the direction c, e the pattern's value).
__device__ __forceinline__ void add_pixel(float* s, float m, float3 d, float e) {
    s[0] += 1.f;
    s[1] += m;
    s[2] += m * m;
    s[3] += m * e;
    s[4] += d.x, s[5] += d.y, s[6] += d.z;
    s[7] += d.x * m, s[8] += d.y * m, s[9] += d.z * m;
    s[10] += d.x * e, s[11] += d.y * e, s[12] += d.z * e;
    s[13] += d.x * d.x, s[14] += d.y * d.y, s[15] += d.z * d.z;
    s[16] += d.x * d.y, s[17] += d.x * d.z, s[18] += d.y * d.z;
}

// One item's refinement, NMI and record (at records[out0 + b]) by the block's W waves, with the
// list of masked pixels or tiles already built and the histogram cleared.
// The Gauss-Newton passes read the half-precision gradient field (mgh: two adjacent 16-byte loads
// a lookup, each a texel and the one below it; half the vector-memory instructions of float32
// texels); the recorded NCC and the NMI are those of the float32 master (ms, the values the field
// holds in .w) at the best orientation, from the NMI's first pass (one 8-byte load per texel row
// pair). REF_HELD keeps its pixels' master values from that pass for the second, the others look
// them up again.
template <int W, int MODE>
__device__ __forceinline__ void refine_item(const RefArg& a, const float* __restrict__ ms, const uint2* __restrict__ mgh, const float* __restrict__ pats,
                                            const float4* __restrict__ items, const float* __restrict__ seeds, int seed_stride,
                                            float* __restrict__ records, int out0, unsigned* hist, const unsigned short* list, int n_px,
                                            Shared<W>& sh, int b, int wave, int lane) {
    const float inv_w = 1.f / (float)a.w;
    // the item's values are the same in every lane: held in scalar registers
    const float4 it = uniform4(items[b]);
    const float3 t = make_float3(it.x, it.y, it.z);
    const float* pat = pats + (size_t)(int)it.w * a.h * a.w;
    const Chunks ch = chunks_of<W>(MODE == REF_TILES ? 0 : n_px);
    // the wave's chunk of round `round`: its first step and its steps (0: none)
    auto chunk = [&](int round, int& id, int& step0) {
        id = round * W + wave;
        step0 = id * ch.size;
        return min(max(ch.steps - step0, 0), ch.size);
    };
    Held held;
    if constexpr (MODE == REF_HELD) {
#pragma unroll
        for (int r = 0; r < kHeld / kChunk; ++r) {
            int id, step0;
            const int cnt = r < ch.rounds ? chunk(r, id, step0) : 0;
#pragma unroll
            for (int i = 0; i < kChunk; ++i) {
                held.u[r * kChunk + i] = make_float3(0.f, 0.f, 1.f);
                held.e[r * kChunk + i] = 0.f;
                if (i < cnt)
                    held.u[r * kChunk + i] = list_pixel(a, list, 64 * (step0 + i) + lane, n_px, inv_w, t, pat, held.e[r * kChunk + i]);
            }
        }
    }
    if (wave == 0) {
        Gn g;
        const float* sd = seeds + (size_t)b * seed_stride;
        g.cur = make_float4(ufloat(sd[0]), ufloat(sd[1]), ufloat(sd[2]), ufloat(sd[3]));
        g.qbest = g.cur;
        g.best = -2.f;
        g.mu = a.scale0;
        g.gbest = make_float3(0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < 6; ++i) g.hbest[i] = 0.f;
        g.last_step = g.promised = g.step_size = g.accepted = 0.f;
        if (lane == 0) {
            sh.gn = g;
            sh.turn = 0;
            records[(size_t)(out0 + b) * 8 + 7] = a.stamp;  // (before the waits, which may take it away)
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t fh = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint2*>(mgh), (short)0, 2 * a.side * a.side * 16, 0x00020000);
    const __amdgpu_buffer_rsrc_t fm = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ms), (short)0, 2 * a.side * a.side * 4, 0x00020000);

    int base = 0;  // chunks of the passes before
    for (int itn = 0; itn <= a.iters; ++itn) {
        const Turn q = turn_of(uniform4(sh.gn.cur));
        float s[kPart];
#pragma unroll
        for (int i = 0; i < kPart; ++i) s[i] = 0.f;
        TapsH tp[kBatch];
        auto take_step = [&]() {
            Gn g = sh.gn;
            gn_step(a, s, itn == a.iters, g);
            if (lane == 0) sh.gn = g;
        };
        if constexpr (MODE != REF_TILES) {
            auto round = [&](int r, auto rc) {
                int id, step0;
                const int cnt = chunk(r, id, step0);
                if (id >= ch.count) return;
                float m[kChunk], e[kChunk];
                float3 d[kChunk];
                look_up<MODE, decltype(rc)::value>(
                    a, list, n_px, inv_w, t, pat, held, step0, cnt, lane,
                    [&](int p, float3 u) {
                        const float3 c = turn(q, u);
                        sheet_taps_h(fh, a.side, c, tp[p]);
                        return c;
                    },
                    [&](int i, int p, float3 c, float ev) {
                        const float4 v = taps_blend(tp[p]);
                        d[i] = cross3(c, make_float3(v.x, v.y, v.z));
                        m[i] = v.w;
                        e[i] = ev;
                    });
                wait_turn(sh, base + id, a.polls, records + (size_t)(out0 + b) * 8 + 7);
                if (id > 0) {
#pragma unroll
                    for (int j = 0; j < kPart / 4; ++j) {
                        const float4 x = sh.acc[j][lane];
                        s[4 * j] = x.x, s[4 * j + 1] = x.y, s[4 * j + 2] = x.z, s[4 * j + 3] = x.w;
                    }
                }
#pragma unroll
                for (int i = 0; i < kChunk; ++i)
                    if (i < cnt && 64 * (step0 + i) + lane < n_px) add_pixel(s, m[i], d[i], e[i]);
                if (id + 1 < ch.count) {
#pragma unroll
                    for (int j = 0; j < kPart / 4; ++j) sh.acc[j][lane] = make_float4(s[4 * j], s[4 * j + 1], s[4 * j + 2], s[4 * j + 3]);
                    pass_turn(&sh.turn, base + id, lane);
                } else {
                    // the pass's last chunk: the totals and the step
#pragma unroll
                    for (int i = 0; i < kPart - 1; ++i) s[i] = wave_sum(s[i]);
                    take_step();
                    pass_turn(&sh.turn, base + id, lane);
                }
            };
            if constexpr (MODE == REF_HELD) {
                round(0, Const<0>{});
                if (ch.rounds > 1) round(1, Const<1>{});
            } else {
                for (int r = 0; r < ch.rounds; ++r) round(r, Const<0>{});
            }
            base += ch.count;
        } else {
            float3 c[kBatch];
            float e[kBatch];
            walk_tiles<W>(
                a, list, n_px, t, wave, lane,
                [&](int p, float3 u, int pix) {
                    c[p] = turn(q, u);
                    sheet_taps_h(fh, a.side, c[p], tp[p]);
                    e[p] = pat[pix];
                },
                [&](int p) {
                    const float4 v = taps_blend(tp[p]);
                    add_pixel(s, v.w, cross3(c[p], make_float3(v.x, v.y, v.z)), e[p]);
                });
            float part[5];
            wave_sums20(s, part);
            if ((lane & 15) == 0) {
                const int r = lane >> 4, at = r == 1 ? 2 : r == 2 ? 1 : r;
#pragma unroll
                for (int j = 0; j < 5; ++j) sh.part[wave][4 * j + at] = part[j];
            }
            __syncthreads();
            if (wave == 0) {
                float v = 0.f;
                if (lane < kPart)
                    for (int w = 0; w < W; ++w) v += sh.part[w][lane];
#pragma unroll
                for (int i = 0; i < kPart; ++i) s[i] = lane_of(v, i);
                take_step();
            }
        }
        __syncthreads();
    }

    // normalized mutual information of the pattern and the master at the best orientation,
    // each binned between its own extremes under the mask (detector.wgsl:739-832)
    const Turn q = turn_of(uniform4(sh.gn.qbest));
    const int nb = a.nmi_bins;
    float emin = 3.4e38f, emax = -3.4e38f, smin = 3.4e38f, smax = -3.4e38f;
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);  // the NCC's sums there (float32 master): count, M, M^2, M e
    float simv[MODE == REF_HELD ? kHeld : 1];
    TapsM tp[kBatch];
    float e[kBatch];
    auto extremes = [&](float ev, float sim) {
        emin = fminf(emin, ev);
        emax = fmaxf(emax, ev);
        smin = fminf(smin, sim);
        smax = fmaxf(smax, sim);
    };
    auto ncc_sums = [&](float ev, float sim) {
        f.x += 1.f;
        f.y += sim;
        f.z += sim * sim;
        f.w += sim * ev;
    };
    auto tap_m = [&](int p, float3 u) {
        const float3 c = turn(q, u);
        sheet_taps_m(fm, a.side, c, tp[p]);
        return c;
    };
    auto tile_tap = [&](int p, float3 u, int pix) {
        tap_m(p, u);
        e[p] = pat[pix];
    };
    if constexpr (MODE != REF_TILES) {
        auto round = [&](int r, auto rc) {
            int id, step0;
            const int cnt = chunk(r, id, step0);
            if (id >= ch.count) return;
            float sv[kChunk], ev[kChunk];
            look_up<MODE, decltype(rc)::value>(a, list, n_px, inv_w, t, pat, held, step0, cnt, lane, tap_m, [&](int i, int p, float3, float x) {
                sv[i] = taps_blend(tp[p]);
                ev[i] = x;
            });
#pragma unroll
            for (int i = 0; i < kChunk; ++i) {
                if constexpr (MODE == REF_HELD) simv[decltype(rc)::value * kChunk + i] = sv[i];
                if (i < cnt && 64 * (step0 + i) + lane < n_px) extremes(ev[i], sv[i]);
            }
            wait_turn(sh, base + id, a.polls, records + (size_t)(out0 + b) * 8 + 7);
            if (id > 0) f = sh.acc[0][lane];
#pragma unroll
            for (int i = 0; i < kChunk; ++i)
                if (i < cnt && 64 * (step0 + i) + lane < n_px) ncc_sums(ev[i], sv[i]);
            sh.acc[0][lane] = f;
            pass_turn(&sh.turn, base + id, lane);
        };
        if constexpr (MODE == REF_HELD) {
            round(0, Const<0>{});
            if (ch.rounds > 1) round(1, Const<1>{});
        } else {
            for (int r = 0; r < ch.rounds; ++r) round(r, Const<0>{});
        }
    } else {
        walk_tiles<W>(a, list, n_px, t, wave, lane, tile_tap, [&](int p) {
            const float sim = taps_blend(tp[p]);
            extremes(e[p], sim);
            ncc_sums(e[p], sim);
        });
    }
    for (int o = 1; o < 64; o <<= 1) {
        emin = fminf(emin, __shfl_xor(emin, o, 64));
        emax = fmaxf(emax, __shfl_xor(emax, o, 64));
        smin = fminf(smin, __shfl_xor(smin, o, 64));
        smax = fmaxf(smax, __shfl_xor(smax, o, 64));
    }
    if constexpr (MODE == REF_TILES) f = make_float4(wave_sum(f.x), wave_sum(f.y), wave_sum(f.z), wave_sum(f.w));
    if (lane == 0) {
        float4* p = (float4*)sh.part[wave];
        p[0] = make_float4(emin, emax, smin, smax);
        p[1] = f;
    }
    __syncthreads();
    for (int w = 0; w < W; ++w) {
        const float4 x = ((const float4*)sh.part[w])[0];
        emin = fminf(emin, x.x), emax = fmaxf(emax, x.y), smin = fminf(smin, x.z), smax = fmaxf(smax, x.w);
    }
    const float ke = (float)nb / fmaxf(emax - emin, 1e-20f);
    const float ks = (float)nb / fmaxf(smax - smin, 1e-20f);
    auto bin = [&](float ev, float sim) {
        const int be = min((int)((ev - emin) * ke), nb - 1);
        const int bs = min((int)((sim - smin) * ks), nb - 1);
        atomicAdd(&hist[be * nb + bs], 1u);
    };
    if constexpr (MODE == REF_HELD) {
#pragma unroll
        for (int r = 0; r < kHeld / kChunk; ++r) {
            int id, step0;
            const int cnt = r < ch.rounds ? chunk(r, id, step0) : 0;
#pragma unroll
            for (int i = 0; i < kChunk; ++i)
                if (i < cnt && 64 * (step0 + i) + lane < n_px) bin(held.e[r * kChunk + i], simv[r * kChunk + i]);
        }
    } else if constexpr (MODE == REF_LIST) {
        for (int r = 0; r < ch.rounds; ++r) {
            int id, step0;
            const int cnt = chunk(r, id, step0);
            look_up<MODE, 0>(a, list, n_px, inv_w, t, pat, held, step0, cnt, lane, tap_m, [&](int i, int p, float3, float x) {
                if (i < cnt && 64 * (step0 + i) + lane < n_px) bin(x, taps_blend(tp[p]));
            });
        }
    } else {
        walk_tiles<W>(a, list, n_px, t, wave, lane, tile_tap, [&](int p) { bin(e[p], taps_blend(tp[p])); });
    }
    __syncthreads();
    if (wave != 0) return;
    float hj = 0.f, tot = 0.f, hm = 0.f;
    for (int i = lane; i < nb * nb; i += 64) {
        const float c = (float)hist[i];
        tot += c;
        if (c > 0.f) hj -= c * logf(c);
    }
    if (lane < nb) {
        float rs = 0.f, cs = 0.f;
        for (int k = 0; k < nb; ++k) {
            rs += (float)hist[lane * nb + k];
            cs += (float)hist[k * nb + lane];
        }
        if (rs > 0.f) hm -= rs * logf(rs);
        if (cs > 0.f) hm -= cs * logf(cs);
    }
    hj = wave_sum(hj);
    tot = wave_sum(tot);
    hm = wave_sum(hm);
    // the recorded NCC: that of the float32 master at the best orientation (the rule of the
    // Gauss-Newton passes)
    if constexpr (MODE == REF_TILES) {
        f = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int w = 0; w < W; ++w) {
            const float4 x = ((const float4*)sh.part[w])[1];
            f = make_float4(f.x + x.x, f.y + x.y, f.z + x.z, f.w + x.w);
        }
    } else {
        f = sh.acc[0][lane];
        f = make_float4(wave_sum(f.x), wave_sum(f.y), wave_sum(f.z), wave_sum(f.w));
    }
    float ncc_best = -2.f;
    {
        const float n = fmaxf(f.x, 1.f);
        const float mean = f.y / n;
        const float var_n = f.z - n * mean * mean;
        if (var_n > 1e-12f) ncc_best = f.w * (1.f / sqrtf(var_n));
    }
    if (lane == 0) {
        const float nn = fmaxf(tot, 1.f);
        const float h_joint = logf(nn) + hj / nn;
        const float h_marg = 2.f * logf(nn) + hm / nn;
        const float nmi = h_marg > 1e-12f ? 2.f * (h_marg - h_joint) / h_marg : 0.f;
        float* r = records + (size_t)(out0 + b) * 8;
        r[0] = sh.gn.qbest.x;
        r[1] = sh.gn.qbest.y;
        r[2] = sh.gn.qbest.z;
        r[3] = sh.gn.qbest.w;
        r[4] = ncc_best;
        r[5] = nmi;
        r[6] = sh.gn.last_step;
    }
}

// Several phases' refinements of one batch in one launch. The n_phases x n_items work items are
// taken phase-major (item k of phase p is p * n_items + k, in that phase's order; zb_refine_order's
// permutation sorts the items by the master region they look up).
// k_refine_grid: one block per work item, block i taking work item xcd_block(i), so that each XCD
// takes a contiguous run of the sequence (its items' gathers share that XCD's L2); the hardware
// deals blocks to CUs as others finish.
// k_refine_queue: a persistent grid (as many blocks as stay resident) pulling work items from
// device-side queues: the sequence cut into kQueues contiguous runs, one per XCD, each with its
// own counter; a block first drains its own XCD's run (block id mod 8, the round-robin dealing
// xcd_block assumes), then the other runs in turn, and leaves when all are empty, so that every
// block reaches that exit. Each block builds the list of masked pixels once for all its items.
// The phases' array pointers are separate restrict kernel arguments (so that the compiler knows
// them not to alias the records); their sides, seed strides and orders come as one more argument
// to the grid form, and for the queue form sit in a table in the work buffer after the queue
// counters, written with them by k_queue_setup on the same stream before the launch.
constexpr int kMaxRefinePhases = 4;
constexpr int kQueues = 8;
constexpr int kQueueStride = 16;
struct RefPhase {
    const int* order;
    int side, seed_stride;
};
struct RefPhases {
    RefPhase p[kMaxRefinePhases];
};
constexpr int kTableOffset = kQueues * kQueueStride * 4;
static_assert(kTableOffset + sizeof(RefPhases) <= ZB_REFINE_QUEUE_BYTES, "the counters and the phase table fit the work buffer");

// the phases' master, half-precision field, seeds and records, as restrict arguments
#define ZB_PHASE_ARGS(i) \
    const float *__restrict__ ms##i, const uint2 *__restrict__ mgh##i, const float *__restrict__ sd##i, float *__restrict__ rec##i
template <typename T>
__device__ __forceinline__ T pick(int p, T x0, T x1, T x2, T x3) {
    return p == 0 ? x0 : p == 1 ? x1 : p == 2 ? x2 : x3;
}

// Work item w of the sequence: phase p, item b (in that phase's order); then the item refined.
template <int W, int MODE>
__device__ __forceinline__ void refine_work(const RefArg& a, RefPhase e, int p, int i, ZB_PHASE_ARGS(0), ZB_PHASE_ARGS(1), ZB_PHASE_ARGS(2),
                                            ZB_PHASE_ARGS(3), const float* __restrict__ pats, const float4* __restrict__ items, unsigned* hist,
                                            const unsigned short* list, int n_px, Shared<W>& sh, int wave, int lane) {
    const int* order = e.order;
    const int b = order ? __builtin_amdgcn_readfirstlane(order[i]) : i;
    RefArg ap = a;
    ap.side = __builtin_amdgcn_readfirstlane(e.side);
    refine_item<W, MODE>(ap, pick(p, ms0, ms1, ms2, ms3), pick(p, mgh0, mgh1, mgh2, mgh3), pats, items, pick(p, sd0, sd1, sd2, sd3),
                         __builtin_amdgcn_readfirstlane(e.seed_stride), pick(p, rec0, rec1, rec2, rec3), a.out0, hist, list, n_px, sh, b, wave, lane);
}

// Work item w of the sequence: phase p and item i (in that phase's order).
__device__ __forceinline__ void work_item(unsigned w, int n_items, int& p, int& i) {
    p = __builtin_amdgcn_readfirstlane((int)(w / (unsigned)n_items));
    i = __builtin_amdgcn_readfirstlane((int)(w - (unsigned)p * (unsigned)n_items));
}

// The list of masked pixels or of tiles; how many (the tiles walked without a list).
template <int W, int MODE>
__device__ __forceinline__ int block_list(const RefArg& a, unsigned short* list, Shared<W>& sh, int wave, int lane) {
    if constexpr (MODE != REF_TILES) return build_list<W, false>(a, list, sh.cnt, wave, lane);
    if (a.tiles) return build_list<W, true>(a, list, sh.cnt, wave, lane);
    return ((a.w + 7) >> 3) * ((a.h + 7) >> 3);
}

template <int W, int MODE>
__global__ void __launch_bounds__(64 * W) k_refine_grid(RefArg a, ZB_PHASE_ARGS(0), ZB_PHASE_ARGS(1), ZB_PHASE_ARGS(2), ZB_PHASE_ARGS(3),
                                                        const float* __restrict__ pats, const float4* __restrict__ items, int n_items,
                                                        RefPhases ph) {
    extern __shared__ unsigned lds[];
    __shared__ Shared<W> sh;
    unsigned* hist = lds;
    unsigned short* list = (unsigned short*)(lds + a.nmi_bins * a.nmi_bins);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int j = threadIdx.x; j < a.nmi_bins * a.nmi_bins; j += 64 * W) hist[j] = 0u;
    const int n_px = block_list<W, MODE>(a, list, sh, wave, lane);
    int p, i;
    work_item((unsigned)xcd_block(blockIdx.x, gridDim.x), n_items, p, i);
    // the phase's entry picked from the argument (an index into it would place it in memory)
    const RefPhase e = pick(p, ph.p[0], ph.p[1], ph.p[2], ph.p[3]);
    refine_work<W, MODE>(a, e, p, i, ms0, mgh0, sd0, rec0, ms1, mgh1, sd1, rec1, ms2, mgh2, sd2, rec2, ms3, mgh3, sd3, rec3, pats, items, hist,
                         list, n_px, sh, wave, lane);
}

template <int W, int MODE>
__global__ void __launch_bounds__(64 * W) k_refine_queue(RefArg a, ZB_PHASE_ARGS(0), ZB_PHASE_ARGS(1), ZB_PHASE_ARGS(2), ZB_PHASE_ARGS(3),
                                                         int n_phases, const float* __restrict__ pats, const float4* __restrict__ items, int n_items,
                                                         unsigned* __restrict__ work) {
    extern __shared__ unsigned lds[];
    __shared__ Shared<W> sh;
    unsigned* hist = lds;
    unsigned short* list = (unsigned short*)(lds + a.nmi_bins * a.nmi_bins);
    const RefPhase* table = (const RefPhase*)((const char*)work + kTableOffset);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n_px = block_list<W, MODE>(a, list, sh, wave, lane);
    const unsigned total = (unsigned)n_items * (unsigned)n_phases;  // below 2^31 (the entry point's check)
    for (int r = 0; r < kQueues; ++r) {
        const unsigned x = (blockIdx.x + r) & (kQueues - 1);
        const unsigned lo = (unsigned)((unsigned long long)total * x / kQueues);
        const unsigned len = (unsigned)((unsigned long long)total * (x + 1) / kQueues) - lo;
        for (;;) {
            __syncthreads();  // every wave done with the last item's histogram and count
            if (threadIdx.x == 0) sh.cnt[0] = (int)atomicAdd(work + x * kQueueStride, 1u);
            for (int j = threadIdx.x; j < a.nmi_bins * a.nmi_bins; j += 64 * W) hist[j] = 0u;
            __syncthreads();
            const unsigned k = (unsigned)__builtin_amdgcn_readfirstlane(sh.cnt[0]);
            if (k >= len) break;
            int p, i;
            work_item(lo + k, n_items, p, i);
            refine_work<W, MODE>(a, table[p], p, i, ms0, mgh0, sd0, rec0, ms1, mgh1, sd1, rec1, ms2, mgh2, sd2, rec2, ms3, mgh3, sd3, rec3, pats,
                                 items, hist, list, n_px, sh, wave, lane);
        }
    }
}

// The queue counters cleared and the phase table written into the work buffer.
__global__ void k_queue_setup(RefPhases ph, int n_phases, unsigned* work) {
    const int t = threadIdx.x;
    if (t < kQueues) work[t * kQueueStride] = 0u;
    if (t < n_phases) ((RefPhase*)((char*)work + kTableOffset))[t] = ph.p[t];
}

// Cells of the refinement's order: each sheet of the master cut into 32 x 32 Lambert cells
constexpr int kOrderSide = 32;
constexpr int kOrderCells = 2 * kOrderSide * kOrderSide;

// The cell the detector centre's ray lands in on the master at orientation q (item position t),
// numbered by sheet and then along a Morton curve over the cell rows and columns, so that nearby
// cells get nearby numbers.
__device__ __forceinline__ int order_cell(const RefArg& a, float4 q, float3 t) {
    const float fr = 0.5f * (float)(a.h - 1), fc = 0.5f * (float)(a.w - 1);
    const float3 u = normalize3(make_float3(a.c0[0] * fr + a.c1[0] * fc + t.x, a.c0[1] * fr + a.c1[1] * fc + t.y,
                                            a.c0[2] * fr + a.c1[2] * fc + t.z));
    const float3 v = qrot(q, u);
    const float2 uv = sphere_to_square(v);
    const int col = min(max((int)((uv.x + 1.f) * (0.5f * kOrderSide)), 0), kOrderSide - 1);
    const int row = min(max((int)((uv.y + 1.f) * (0.5f * kOrderSide)), 0), kOrderSide - 1);
    int m = 0;
#pragma unroll
    for (int bit = 0; bit < 5; ++bit) m |= (((col >> bit) & 1) << (2 * bit)) | (((row >> bit) & 1) << (2 * bit + 1));
    return (v.z < 0.f ? kOrderSide * kOrderSide : 0) + m;
}

// A counting sort of the items by order_cell, one block: counts per cell in LDS, their exclusive
// prefix, then each item placed at its cell's next slot (the order within a cell is arbitrary;
// every item's record is the same whichever block computes it).
__global__ void __launch_bounds__(1024) k_order(RefArg a, const float4* __restrict__ items, int item_stride, const float* __restrict__ seeds,
                                                int seed_stride, int n_items, int* __restrict__ order) {
    __shared__ unsigned cnt[kOrderCells];
    __shared__ unsigned part[1024];
    const int tid = threadIdx.x;
    for (int i = tid; i < kOrderCells; i += 1024) cnt[i] = 0u;
    __syncthreads();
    auto cell_of = [&](int b) {
        const float* sd = seeds + (size_t)b * seed_stride;
        const float4 it = items[(size_t)b * item_stride];
        return order_cell(a, make_float4(sd[0], sd[1], sd[2], sd[3]), make_float3(it.x, it.y, it.z));
    };
    for (int b = tid; b < n_items; b += 1024) atomicAdd(&cnt[cell_of(b)], 1u);
    __syncthreads();
    // exclusive prefix over the cells: each thread sums its run of cells, a scan over the threads,
    // then the run's own offsets
    constexpr int per = kOrderCells / 1024;
    unsigned run = 0;
#pragma unroll
    for (int k = 0; k < per; ++k) run += cnt[tid * per + k];
    part[tid] = run;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const unsigned x = tid >= o ? part[tid - o] : 0u;
        __syncthreads();
        part[tid] += x;
        __syncthreads();
    }
    unsigned at = part[tid] - run;
#pragma unroll
    for (int k = 0; k < per; ++k) {
        const unsigned c = cnt[tid * per + k];
        cnt[tid * per + k] = at;
        at += c;
    }
    __syncthreads();
    for (int b = tid; b < n_items; b += 1024) order[atomicAdd(&cnt[cell_of(b)], 1u)] = b;
}

// The 43 sums of the six-direction fit for each item's pose (detector.wgsl:433-494 sums +
// sums_reduce): count, sum M, sum M^2, sum M e, then for d = (q^-1 grad M / |u|, c x grad M)
// (a shift of the rays' origin in pixels, a crystal rotation) sum d_i, sum M d_i, sum e d_i and
// the upper triangle of sum d_i d_j. One wave per item over the masked-pixel list; every lane
// ends with the same totals (xor butterflies) and the lanes write them out in parallel.
// rotation_only zeroes the shift's sums, as sums_reduce does for orientation refinement.
constexpr int kSums = 43;

// skip (or NULL): items whose entry is not 0 are left out (their sums untouched). LIST: the masked
// pixels as a list in LDS; else the whole frame walked with the mask tested a pixel. order (or
// NULL): block b takes item order[xcd_block(b)] rather than b, so the blocks of one XCD read one
// region of the field: with 4 000 poses of an 80 x 80 map in flight the field's 8 MB (float4 a texel)
// pass through every XCD's 4 MB of L2 in any order of the items (6.4 TB/s fetched past L2, the VALU
// a quarter busy). unit: the quaternion is brought to unit length (in 64 bits) and w >= 0 first.
template <bool LIST>
__global__ void __launch_bounds__(64) k_sums6(RefArg a, const float4* __restrict__ mg, const float* __restrict__ pats, const float* __restrict__ poses,
                                              int rotation_only, const int* __restrict__ skip, const int* __restrict__ order, int unit,
                                              float* __restrict__ out) {
    extern __shared__ unsigned lds[];
    unsigned short* list = (unsigned short*)lds;
    const int b = order ? __builtin_amdgcn_readfirstlane(order[xcd_block(blockIdx.x, gridDim.x)]) : blockIdx.x;
    if (skip && skip[b] != 0) return;
    const int lane = threadIdx.x;
    int n_px = a.h * a.w;
    if constexpr (LIST) n_px = build_list<1, false>(a, list, nullptr, 0, lane);
    const float inv_w = 1.f / (float)a.w;
    const float* ps = poses + (size_t)b * 8;
    const float3 t = make_float3(ps[0], ps[1], ps[2]);
    const float* pat = pats + (size_t)(int)ps[3] * a.h * a.w;
    float4 q = make_float4(ps[4], ps[5], ps[6], ps[7]);
    if (unit) {
        const double x = q.x, y = q.y, z = q.z, w = q.w;
        const double len = sqrt(x * x + y * y + z * z + w * w), f = x / len < 0.0 ? -1.0 : 1.0;
        q = make_float4((float)(f * (x / len)), (float)(f * (y / len)), (float)(f * (z / len)), (float)(f * (w / len)));
    }
    const float4 qi = make_float4(q.x, -q.y, -q.z, -q.w);
    float s[kSums];
#pragma unroll
    for (int i = 0; i < kSums; ++i) s[i] = 0.f;
    for (int k = lane; k < n_px; k += 64) {
        const int pix = LIST ? (int)list[k] : k;
        const int row = LIST ? (int)(((float)pix + 0.5f) * inv_w) : pix / a.w;
        if (!LIST && !under_mask(a, row, pix - row * a.w)) continue;
        const float fr = (float)row, fc = (float)(pix - row * a.w);
        const float3 u = make_float3(a.c0[0] * fr + a.c1[0] * fc + t.x, a.c0[1] * fr + a.c1[1] * fc + t.y, a.c0[2] * fr + a.c1[2] * fc + t.z);
        const float dist = sqrtf(dot3(u, u));
        const float id = 1.f / dist;
        const float3 c = qrot(q, make_float3(u.x * id, u.y * id, u.z * id));
        const float4 m = sheet_bilinear<float4>(mg, a.side, c);
        const float3 gm = make_float3(m.x, m.y, m.z);
        const float3 ac = cross3(c, gm);
        const float3 w = qrot(qi, gm);
        float d[6] = {w.x * id, w.y * id, w.z * id, ac.x, ac.y, ac.z};
        const float e = pat[pix];
        const float val = m.w;
        s[0] += 1.f;
        s[1] += val;
        s[2] += val * val;
        s[3] += val * e;
        int o = 22;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            s[4 + i] += d[i];
            s[10 + i] += val * d[i];
            s[16 + i] += e * d[i];
#pragma unroll
            for (int j = i; j < 6; ++j) s[o++] += d[i] * d[j];
        }
    }
#pragma unroll
    for (int i = 0; i < kSums; ++i) s[i] = wave_sum(s[i]);
    // lane i writes sum i (the shift's sums zero for orientation refinement), picked by value: a store a
    // sum under its lane's condition became a tree of some 900 branches, as long as 50 steps of the walk
    float x = s[0];
#pragma unroll
    for (int i = 1; i < kSums; ++i) x = lane == i ? s[i] : x;
    const bool shift = (lane >= 4 && lane < 7) || (lane >= 10 && lane < 13) || (lane >= 16 && lane < 19) || (lane >= 22 && lane < 37);
    if (lane < kSums) out[(size_t)b * kSums + lane] = (rotation_only && shift) ? 0.f : x;
}

}  // namespace zb

using namespace zb;

// The frame's geometry into `a`; returns its masked pixels, or an error (negative).
static int ref_frame(const zb_frame* frame, int side, RefArg& a, const char* who) {
    for (int i = 0; i < 3; ++i) {
        a.c0[i] = frame->c0[i];
        a.c1[i] = frame->c1[i];
        a.c2[i] = frame->c2[i];
        a.mask[i] = frame->mask[i];
    }
    a.h = frame->pat_h;
    a.w = frame->pat_w;
    a.side = side;
    if ((long)a.h * a.w > (1L << 26)) {
        set_error("%s: %d x %d pixels: at most 2^26", who, a.h, a.w);
        return ZB_EINVAL;
    }
    long n_px = 0;
    for (int r = 0; r < a.h; ++r)
        for (int c = 0; c < a.w; ++c) {
            const float dr = (float)r - a.mask[0], dc = (float)c - a.mask[1];
            n_px += (a.mask[2] <= 0.f || dr * dr + dc * dc <= a.mask[2]) ? 1 : 0;
        }
    return (int)n_px;
}

// Bytes of a list of n 16-bit entries in LDS.
static size_t list_bytes(long n) { return ((size_t)n * 2 + 15) / 16 * 16; }

extern "C" int32_t zb_sums(const float* mgrad, int32_t side, const zb_frame* frame, const float* pats, const float* poses, int32_t n_items,
                           int32_t flags, float* sums, void* stream) {
    return zb::sums_run(mgrad, side, frame, pats, poses, n_items, flags, nullptr, nullptr, 0, sums, stream);
}

extern "C" int32_t zb_sums_active(const float* mgrad, int32_t side, const zb_frame* frame, const float* pats, const float* poses,
                                  int32_t n_items, int32_t flags, const int32_t* state, float* sums, void* stream) {
    if (n_items > 0 && !state) {
        set_error("zb_sums_active: null state");
        return ZB_EINVAL;
    }
    return zb::sums_run(mgrad, side, frame, pats, poses, n_items, flags, state, nullptr, 0, sums, stream);
}

int32_t zb::sums_run(const float* mgrad, int32_t side, const zb_frame* frame, const float* pats, const float* poses, int32_t n_items, int32_t flags,
                     const int32_t* skip, const int32_t* order, int unit, float* sums, void* stream) {
    if (!frame || side < 2 || n_items < 0 || frame->pat_h < 2 || frame->pat_w < 2 || (flags & ~ZB_SUMS_ROTATION_ONLY)) {
        set_error("zb_sums: bad arguments");
        return ZB_EINVAL;
    }
    if (n_items == 0) return ZB_OK;
    if (!mgrad || !pats || !poses || !sums) {
        set_error("zb_sums: null pointer");
        return ZB_EINVAL;
    }
    RefArg a = {};
    const int n_px = ref_frame(frame, side, a, "zb_sums");
    if (n_px < 0) return n_px;
    // the masked pixels as a 16-bit list in LDS while their indices fit 16 bits and the list stays
    // within 60 KB; else the whole frame is walked with the mask tested per pixel
    const size_t lds = list_bytes(n_px);
    if ((long)a.h * a.w <= 65536 && lds <= 60 * 1024)
        ZB_LAUNCH("k_sums6", k_sums6<true>, dim3(n_items), dim3(64), lds, (hipStream_t)stream, a, (const float4*)mgrad, pats, poses,
                  (flags & ZB_SUMS_ROTATION_ONLY) ? 1 : 0, (const int*)skip, (const int*)order, unit, sums);
    else
        ZB_LAUNCH("k_sums6", k_sums6<false>, dim3(n_items), dim3(64), 0, (hipStream_t)stream, a, (const float4*)mgrad, pats, poses,
                  (flags & ZB_SUMS_ROTATION_ONLY) ? 1 : 0, (const int*)skip, (const int*)order, unit, sums);
    return check_launch("zb_sums");
}

static void ref_opts(RefArg& a, const zb_refine_opts* o, int out0) {
    a.iters = o->iters;
    a.nmi_bins = o->nmi_bins;
    a.polls = knob(KNOB_REFINE_POLLS);
    a.out0 = out0;
    a.max_step = o->max_step;
    a.scale0 = o->scale0;
    a.scale_min = o->scale_min;
    a.scale_max = o->scale_max;
    a.stamp = (float)o->stamp;
}

// The launch of a refinement: W waves a block, how its pixels are walked, and the LDS for the
// joint histogram and the list. The list forms' records do not depend on W, so it follows the
// speed (measured over frames of 8 x 8 to 180 x 180, 5 and 8 iterations):
//  - while a block's lanes hold all their pixels, as few waves as hold them (1 to 4): every
//    wave adds hand-overs and barriers (40 x 40, 8 000 items: 582 us with 2 waves, 788 with 4;
//    one wave an item, the list and the pattern read in each pass: 659), and holding beats reading
//    the list again (60 x 60, 4 500 items: 513 us against 613). One wave where it holds them: to 3 steps, and
//    past 4 items a CU (20 000 items of 8 x 8: 339 us, 530 with 2 waves; of 16 x 16: 513 and 650; 3 000 of 24 x 24:
//    162 and 175), where fewer leave the second wave room (30 items of 24 x 24: 55 us with one, 48 with 2);
//  - above that, more waves where the items are too few to fill the chip or a frame's list leaves
//    room for few blocks a CU: 8 up to one item a CU or past 256 steps (120 x 120, 8 items: 235 us
//    against 256 with 4 and 417 with 2; 180 x 180, 1 000 items: 1 208, 1 337 and 2 505), else 4 past
//    96 steps or up to two items a CU (120 x 120, 1 200 items: 798 us against 848 with 2 and 813
//    with 8; 80 x 80, 400 items: 238, 294 and 244), else 2 (80 x 80, 4 000 items: 1 233, 1 308 with
//    4, 1 392 with 8).
// (60 x 60 was measured at 4 500 and 16 000 items; what a few items of it gain from more waves was not.)
struct RefLaunch {
    int mode, waves;
    size_t lds;
};
static RefLaunch ref_launch(RefArg& a, int n_px, long total) {
    const size_t hist = (size_t)a.nmi_bins * a.nmi_bins * 4;
    RefLaunch l;
    if ((long)a.h * a.w <= 65536 && list_bytes(n_px) <= 60 * 1024) {
        const int steps = (n_px + 63) / 64;
        if (steps <= 4 * kHeld) {
            l.mode = REF_HELD;
            l.waves = steps <= 3 || (steps <= kHeld && total > 1024) ? 1 : std::max((steps + kHeld - 1) / kHeld, 2);
        } else {
            l.mode = REF_LIST;
            l.waves = total <= 256 || steps > 256 ? 8 : total <= 512 || steps > 96 ? 4 : 2;
        }
        l.lds = hist + list_bytes(n_px);
        return l;
    }
    const long tiles = (long)((a.h + 7) / 8) * ((a.w + 7) / 8);
    // the tiles' list within 48 KB of LDS; past that every tile is walked
    a.tiles = tiles <= 24 * 1024 ? (int)tiles : 0;
    l.mode = REF_TILES;
    l.waves = 16;
    l.lds = hist + list_bytes(a.tiles);
    return l;
}

// Blocks of k_refine_queue resident at once on the current device: CUs x blocks per CU, queried
// once per device, form and LDS size (host queries only, so that a call under stream capture
// records nothing else).
static int queue_blocks(const RefLaunch& l) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, size_t>, int> known;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> g(mu);
    const auto key = std::make_tuple(dev, l.mode * 64 + l.waves, l.lds);
    auto it = known.find(key);
    if (it != known.end()) return it->second;
    int cus = 0, per_cu = 0;
    const void* kern = nullptr;
#define ZB_KERN(W, MODE) \
    if (l.waves == W && l.mode == MODE) kern = (const void*)k_refine_queue<W, MODE>
    ZB_KERN(1, REF_HELD);
    ZB_KERN(3, REF_HELD);
    ZB_KERN(2, REF_HELD);
    ZB_KERN(2, REF_LIST);
    ZB_KERN(4, REF_HELD);
    ZB_KERN(4, REF_LIST);
    ZB_KERN(8, REF_LIST);
    ZB_KERN(16, REF_TILES);
#undef ZB_KERN
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 64 * l.waves, l.lds) != hipSuccess || per_cu < 1 || cus < 1)
        return 0;
    return known[key] = cus * per_cu;
}

// The refinement of n_phases phases launched (the arguments checked by the callers): block per
// work item, or with `work` the persistent form.
static int32_t refine_launch(const zb_refine_phase* phases, int n_phases, const zb_frame* frame, const float* pats, const float* items, int32_t n_items,
                             const zb_refine_opts* o, int32_t out0, unsigned* queues, hipStream_t st, const char* who) {
    RefArg a = {};
    const int n_px = ref_frame(frame, phases[0].side, a, who);
    if (n_px < 0) return n_px;
    ref_opts(a, o, out0);
    const long total = (long)n_items * n_phases;
    const RefLaunch l = ref_launch(a, n_px, total);
    // the phases' arrays as kernel arguments (phases past n_phases repeat the last: never read)
    RefPhases ph = {};
    const float* ms[kMaxRefinePhases];
    const uint2* mgh[kMaxRefinePhases];
    const float* sd[kMaxRefinePhases];
    float* rec[kMaxRefinePhases];
    for (int p = 0; p < kMaxRefinePhases; ++p) {
        const zb_refine_phase& q = phases[std::min(p, n_phases - 1)];
        ph.p[p] = RefPhase{q.order, q.side, q.seed_stride};
        ms[p] = q.master;
        mgh[p] = (const uint2*)q.mgrad_h;
        sd[p] = q.seeds;
        rec[p] = q.records;
    }
#define ZB_PHASES ms[0], mgh[0], sd[0], rec[0], ms[1], mgh[1], sd[1], rec[1], ms[2], mgh[2], sd[2], rec[2], ms[3], mgh[3], sd[3], rec[3]
#define ZB_REFINE1(KERNEL, GRID, W, MODE, ...) \
    if (l.waves == W && l.mode == MODE) ZB_LAUNCH("k_refine", (KERNEL<W, MODE>), dim3(GRID), dim3(64 * W), l.lds, st, a, ZB_PHASES, __VA_ARGS__)
#define ZB_REFINE(KERNEL, GRID, ...)                         \
    do {                                                     \
        ZB_REFINE1(KERNEL, GRID, 1, REF_HELD, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 2, REF_HELD, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 2, REF_LIST, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 3, REF_HELD, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 4, REF_HELD, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 4, REF_LIST, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 8, REF_LIST, __VA_ARGS__);  \
        ZB_REFINE1(KERNEL, GRID, 16, REF_TILES, __VA_ARGS__); \
    } while (0)
    if (queues) {
        // the queue counters cleared and the phase table written into the work buffer
        ZB_LAUNCH("k_queue_setup", k_queue_setup, dim3(1), dim3(64), 0, st, ph, n_phases, queues);
        if (int rc = check_launch("zb_refine_phases/setup")) return rc;
        // as many blocks as stay resident at once (more would only wait for the queues to empty)
        const int resident = queue_blocks(l);
        if (resident < 1) {
            set_error("%s: device or occupancy query failed", who);
            return ZB_ELAUNCH;
        }
        const int grid = (int)std::min<long>(total, resident);
        ZB_REFINE(k_refine_queue, grid, n_phases, pats, (const float4*)items, n_items, queues);
    } else {
        ZB_REFINE(k_refine_grid, total, pats, (const float4*)items, n_items, ph);
    }
#undef ZB_REFINE
#undef ZB_REFINE1
#undef ZB_PHASES
    return check_launch(who);
}

extern "C" int32_t zb_refine(const float* master, const uint16_t* mgrad_h, int32_t side, const zb_frame* frame, const float* pats, const float* items,
                             const float* seeds, int32_t seed_stride, int32_t n_items, const zb_refine_opts* o, float* records, int32_t out0,
                             void* stream) {
    if (!frame || !o || side < 2 || n_items < 0 || frame->pat_h < 2 || frame->pat_w < 2 || seed_stride < 4 || out0 < 0 || o->iters < 0 ||
        o->nmi_bins < 2 || o->nmi_bins > 32) {
        set_error("zb_refine: bad arguments");
        return ZB_EINVAL;
    }
    if (n_items == 0) return ZB_OK;
    if (!master || !mgrad_h || !pats || !items || !seeds || !records) {
        set_error("zb_refine: null pointer");
        return ZB_EINVAL;
    }
    const zb_refine_phase one = {master, mgrad_h, side, seeds, seed_stride, o->order, records};
    return refine_launch(&one, 1, frame, pats, items, n_items, o, out0, nullptr, (hipStream_t)stream, "zb_refine");
}

extern "C" int32_t zb_refine_phases(const zb_refine_phase* phases, int32_t n_phases, const zb_frame* frame, const float* pats, const float* items,
                                    int32_t n_items, const zb_refine_opts* o, int32_t out0, void* work, int64_t work_bytes, void* stream) {
    if (!frame || !o || n_phases < 1 || n_phases > kMaxRefinePhases || n_items < 0 || frame->pat_h < 2 || frame->pat_w < 2 || out0 < 0 ||
        o->iters < 0 || o->nmi_bins < 2 || o->nmi_bins > 32 || (long)n_items * n_phases >= (1L << 31)) {
        set_error("zb_refine_phases: bad arguments");
        return ZB_EINVAL;
    }
    if (!phases) {
        set_error("zb_refine_phases: null pointer");
        return ZB_EINVAL;
    }
    for (int p = 0; p < n_phases; ++p) {
        const zb_refine_phase& q = phases[p];
        if (q.side < 2 || q.seed_stride < 4) {
            set_error("zb_refine_phases: phase %d: bad arguments", p);
            return ZB_EINVAL;
        }
        if (n_items > 0 && (!q.master || !q.mgrad_h || !q.seeds || !q.records)) {
            set_error("zb_refine_phases: phase %d: null pointer", p);
            return ZB_EINVAL;
        }
    }
    if (n_items == 0) return ZB_OK;
    if (!pats || !items || !work) {
        set_error("zb_refine_phases: null pointer");
        return ZB_EINVAL;
    }
    if (work_bytes < ZB_REFINE_QUEUE_BYTES) {
        set_error("zb_refine_phases: work_bytes %lld below %d", (long long)work_bytes, ZB_REFINE_QUEUE_BYTES);
        return ZB_ESPACE;
    }
    if ((uintptr_t)work % 8) {
        set_error("zb_refine_phases: work not 8-byte aligned");
        return ZB_EINVAL;
    }
    return refine_launch(phases, n_phases, frame, pats, items, n_items, o, out0, knob(KNOB_REFINE_QUEUE) ? (unsigned*)work : nullptr,
                         (hipStream_t)stream, "zb_refine_phases");
}

extern "C" int32_t zb_refine_order(const zb_frame* frame, const float* items, const float* seeds, int32_t seed_stride, int32_t n_items,
                                   int32_t* order, void* stream) {
    if (!frame || n_items < 0 || seed_stride < 4 || frame->pat_h < 2 || frame->pat_w < 2) {
        set_error("zb_refine_order: bad arguments");
        return ZB_EINVAL;
    }
    if (n_items == 0) return ZB_OK;
    if (!items || !seeds || !order) {
        set_error("zb_refine_order: null pointer");
        return ZB_EINVAL;
    }
    return zb::order_run(frame, items, 1, seeds, seed_stride, n_items, order, stream);
}

int32_t zb::order_run(const zb_frame* frame, const float* items, int item_stride, const float* seeds, int32_t seed_stride, int32_t n_items,
                      int32_t* order, void* stream) {
    RefArg a = {};
    for (int i = 0; i < 3; ++i) {
        a.c0[i] = frame->c0[i];
        a.c1[i] = frame->c1[i];
        a.c2[i] = frame->c2[i];
        a.mask[i] = frame->mask[i];
    }
    a.h = frame->pat_h;
    a.w = frame->pat_w;
    ZB_LAUNCH("k_order", k_order, dim3(1), dim3(1024), 0, (hipStream_t)stream, a, (const float4*)items, item_stride, seeds, seed_stride,
              n_items, order);
    return check_launch("zb_refine_order");
}
