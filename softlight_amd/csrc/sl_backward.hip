// sl_backward.hip -- fixed-visibility adjoint of the draw path.
//
// The forward pass (k_raster_wave with a visibility attachment) leaves, for every
// pixel, the submitted-triangle number of the fragment that won the depth test
// and that fragment's perspective-correct weights b0, b1, b2 of the source
// triangle's vertices.  For an unclipped triangle the weights are bit-equal to
// the interpolation weights the forward used, so the backward rebuilds the
// fragment's varyings -- and with them the texture taps -- exactly as the
// forward computed them, then scatters
//   dL/d colour[v_k] += b_k * (dL/dC (.) texel)          (per channel)
//   dL/d texel[tap_j] += w_j * (dL/dC (.) colour)         (bilinear weight w_j)
// with float atomics, pre-aggregated per 16 x 16 pixel block in LDS.
//
// No reference counterpart: the reference renders forward only.
#include "sl_device.h"
#include "sl_stages.h"
#include "sl_backward.h"

namespace slg {

// Last draw whose first sequence number is below seq (draws ordered by seqBase).
__device__ __forceinline__ uint32_t seq_base(const GradDesc* D, uint32_t i) { return D[i].d.seqBase; }
__device__ __forceinline__ uint32_t seq_base(const uint32_t* D, uint32_t i) { return D[i]; }

template <class Bases>
__device__ __forceinline__ uint32_t find_grad_draw(Bases D, uint32_t n, uint32_t seq)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1)
    {
        const uint32_t mid = (lo + hi) >> 1;
        if (seq_base(D, mid) < seq) lo = mid;
        else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// Workgroup pre-aggregation (16 x 16 pixels): every destination (a vertex, a
// texel) is summed in LDS and added to HBM once.  A pixel contributes up to
// three vertex items and four texel items, each a weight times the pixel's
// vector (dL/d colour varying, or dL/dC (.) colour).  Items are sorted by
// destination with integer atomics and then summed by the lanes that own the
// destination:
//
//   1  each item finds its destination's slot in a hash table (texels by
//      groups of four neighbours, one 64 B line of the gradient image) and
//      takes its rank among the slot's items,
//   2  every used slot takes a range of the item array,
//   3  the items' products are written to their places,
//   4  16 lanes per texel group or vertex, 64 where their lists are long,
//      sum the products and add the sums to HBM.
//
// Why not add in LDS: a float LDS atomic takes 192 cycles a wave on this chip
// (three a lane, whatever the addresses) against 10 for an integer one and 25
// for a compare-and-swap, and a pixel made 25 of them.  Why groups: one HBM
// atomic instruction then covers four whole lines, not 64.  Measured per
// framebuffer of 2048x1024, against float LDS atomics into per-texel and
// per-vertex slots: eight views of a 20,480-triangle sphere 289 -> 133 us,
// eight views of eight spheres (minified texture, another draw per sphere)
// 507 -> 197; of four 128x128 views 24.8 -> 22.0.
//
// What is left is latency: 4 workgroups fit a CU by LDS (the vertex items take
// the texel items' storage, which made it 4 instead of 3: 152 -> 133 us), each
// a chain of dependent fetches (visibility, draw, indices, attributes,
// texels) and LDS round trips.
//
// A table serves one destination buffer (the first one a lane claims); items
// of other buffers, and items that find no free slot within the probes, add
// to HBM directly.
// ---------------------------------------------------------------------------
constexpr int kBwdTile = 16;
constexpr int kGroupBits = 9;         // 512 groups of four texels (about 430 where the texture is minified 2 x 4)
constexpr int kVertBits = 9;          // 512 vertices
constexpr int kGroups = 1 << kGroupBits, kVerts = 1 << kVertBits;
constexpr int kVertSlot0 = 4 * kGroups;            // slots: texels by group, then vertices
constexpr int kSlots = kVertSlot0 + kVerts;
constexpr int kMaxItems = 4 * kBwdTile * kBwdTile;  // texel items, then the vertex items in their place
constexpr int kLdsDraws = 64;        // draws whose sequence bases are searched in LDS
constexpr int kProbes = 16;
constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;

// Claims the table for buf (or finds it claimed for buf).
__device__ __forceinline__ bool claim(unsigned long long* owner, const float* buf)
{
    const unsigned long long mine = reinterpret_cast<unsigned long long>(buf);
    const unsigned long long prev = atomicCAS(owner, 0ull, mine);
    return prev == 0ull || prev == mine;
}

// Slot of `key` in an open-addressing table of 2^bits keys, or -1; a slot
// claimed by this call is appended to the list of used ones.
__device__ __forceinline__ int find_slot(uint32_t* keys, int bits, uint32_t key, uint16_t* used, uint32_t* numUsed)
{
    uint32_t h = (key * 2654435761u) >> (32 - bits);
    const uint32_t mask = (1u << bits) - 1u;
    for (int probe = 0; probe < kProbes; ++probe)
    {
        const uint32_t prev = atomicCAS(&keys[h], kEmptyKey, key);
        if (prev == kEmptyKey) used[atomicAdd(numUsed, 1u)] = (uint16_t)h;
        if (prev == kEmptyKey || prev == key) return (int)h;
        h = (h + 1u) & mask;
    }
    return -1;
}

__device__ __forceinline__ void add_global4(float* dst, uint64_t key, float w, float4 v)
{
    const float a[4] = {w * v.x, w * v.y, w * v.z, w * v.w};
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (a[c] != 0.f) unsafeAtomicAdd(dst + 4ull * key + c, a[c]);
}

// The used destinations' ranges of the item array: entry i of `range` (first
// item << 16 | items) for float 4 of the i-th used slot, `per` slots a key.
// Whole waves call it: a wave takes one range for all of its slots.
__device__ __forceinline__ void slot_ranges(int n, int per, const uint16_t* used, uint32_t* slots, uint32_t* numItems)
{
    const int lane = (int)threadIdx.x & 63;
    for (int i0 = (int)threadIdx.x - lane; i0 < n * per; i0 += 256)
    {
        const int i = i0 + lane;
        const int q = i < n * per ? per * (int)used[i / per] + (i & (per - 1)) : 0;
        const uint32_t num = i < n * per ? slots[q] : 0u;
        uint32_t sum = num;                            // inclusive prefix over the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1)
        {
            const uint32_t o = __shfl_up(sum, off, 64);
            if (lane >= off) sum += o;
        }
        uint32_t first = 0;
        if (lane == 63) first = atomicAdd(numItems, sum);
        first = __shfl(first, 63, 64) + sum - num;
        if (i < n * per) slots[q] = (first << 16) | num;
    }
}

// Sums the destinations of `n` used keys, each of `per` consecutive slots of
// four floats, with PARTS lanes per float, and adds them to dst (float
// 4 per * key on).
template <int PARTS>
__device__ __forceinline__ void sum_slots(float* dst, int n, int per, const uint16_t* used, const uint32_t* keys,
                                          const uint32_t* slots, const float4* items)
{
    const int lanes = 4 * per * PARTS;                  // per key: 4 .. 64, a power of two
    const int part = (int)threadIdx.x & (PARTS - 1);
    const int f = ((int)threadIdx.x & (lanes - 1)) / PARTS;
    for (int i = (int)threadIdx.x / lanes; i < n; i += 256 / lanes)
    {
        const int key = used[i];
        const uint32_t word = slots[per * key + (f >> 2)];
        const int first = (int)(word >> 16), num = (int)(word & 0xFFFFu);
        float acc = 0.f;
        int k = part;
        for (; k + 3 * PARTS < num; k += 4 * PARTS)
        {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const float*>(&items[first + k + u * PARTS])[f & 3];
            acc += (v[0] + v[1]) + (v[2] + v[3]);
        }
        for (; k < num; k += PARTS) acc += reinterpret_cast<const float*>(&items[first + k])[f & 3];
#pragma unroll
        for (int off = 1; off < PARTS; off <<= 1) acc += __shfl_xor(acc, off, 64);
        if (part == 0 && acc != 0.f) unsafeAtomicAdd(dst + (uint64_t)(4 * per) * keys[key] + f, acc);
    }
}

// One lane per pixel; a workgroup covers a 16 x 16 block (a wave 16 x 4).
__global__ __launch_bounds__(256) void k_backward(BackwardParams P)
{
    __shared__ uint32_t sGroupKey[kGroups], sVertKey[kVerts];
    __shared__ uint32_t sSlot[kSlots];                // items of the slot; then first item << 16 | items
    __shared__ uint16_t sGroupUsed[kGroups], sVertUsed[kVerts];
    __shared__ float4 sItem[kMaxItems];
    __shared__ uint32_t sSeqBase[kLdsDraws];
    __shared__ unsigned long long sVOwner, sTOwner;
    __shared__ uint32_t sNumGroups, sNumVerts, sNumItems[2];
    const int tid = threadIdx.x;

    const int bxN = (P.W + kBwdTile - 1) / kBwdTile;
    const int x = (int)(blockIdx.x % bxN) * kBwdTile + (tid & (kBwdTile - 1));
    const int y = (int)(blockIdx.x / bxN) * kBwdTile + (tid / kBwdTile);
    const bool inb = x < P.W && y < P.H;
    const uint64_t p = (uint64_t)y * P.W + x;

    float4 vis = make_float4(0.f, 0.f, 0.f, 0.f);
    if (inb) vis = P.vis[p];
    if (!__syncthreads_or(__float_as_uint(vis.x) != 0u)) return;     // background
    // the search for a pixel's draw reads its chain of keys from LDS
    const bool ldsDraws = P.numDraws <= (uint32_t)kLdsDraws;
    if (ldsDraws && tid < (int)P.numDraws) sSeqBase[tid] = P.draws[tid].d.seqBase;
    for (int i = tid; i < kGroups; i += 256) sGroupKey[i] = kEmptyKey;
    for (int i = tid; i < kVerts; i += 256) sVertKey[i] = kEmptyKey;
    for (int i = tid; i < kSlots; i += 256) sSlot[i] = 0u;
    if (tid == 0)
    {
        sVOwner = sTOwner = 0ull;
        sNumGroups = sNumVerts = sNumItems[0] = sNumItems[1] = 0u;
    }
    __syncthreads();

    const uint32_t seq = __float_as_uint(vis.x);
    bool live = inb && seq != 0u;
    uint32_t draw = 0;
    if (live) draw = ldsDraws ? find_grad_draw(sSeqBase, P.numDraws, seq) : find_grad_draw(P.draws, P.numDraws, seq);
    const float b[3] = {vis.y, vis.z, vis.w};
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live) g = P.gradImage[p];

    // varyings of the winning fragment, in the forward's operation order
    // (interpolate_tri_varyings, SL_FragmentProcessor.cpp:315-330).  A wave
    // takes its draws one after the other (mostly one), so that the draw's
    // descriptor is read into scalar registers.
    uint64_t vid[3] = {0, 0, 0};
    float4 col = make_float4(0.f, 0.f, 0.f, 0.f), tex = make_float4(1.f, 1.f, 1.f, 1.f);
    BilinearTaps taps{};
    bool textured = false, ct = false, nearest = false;
    float *gradCol = nullptr, *gradTex = nullptr;
    uint64_t gradColCount = 0, gradTexTexels = 0;
    for (uint64_t left = __ballot(live); left != 0;)
    {
        const uint32_t cur = (uint32_t)__builtin_amdgcn_readlane((int)draw, __ffsll((unsigned long long)left) - 1);
        const GradDesc& G = P.draws[cur];
        const DrawDesc& D = G.d;
        const bool mine = live && draw == cur;
        left &= ~__ballot(mine);
        if (!mine) continue;
        const uint64_t t = (uint64_t)(seq - 1u - D.seqBase);
        live = seq > D.seqBase && t < D.numTris;
        if (!live) continue;
        uint64_t ti;
        const uint64_t inst = split_instance(D, t, ti);
        const uint64_t e = D.elementBegin + 3u * ti;
        vid[0] = e; vid[1] = e + 1; vid[2] = e + 2;
        if (D.indexed)
        {
            uint32_t id[3];
            fetch_indices3(D, e, id);
            vid[0] = id[0];
            vid[1] = id[1];
            vid[2] = id[2];
        }
        gradCol = G.gradCol;
        gradColCount = G.gradColCount;
        gradTex = G.gradTex;
        gradTexTexels = G.gradTexTexels;
        ct = D.fsProg == SL_PROGRAM_COLOR_TEXTURED;
        nearest = D.nearest != 0;
        float4 a[3], uv[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            a[k] = read_attr(D, 1, vid[k], ct ? 0.f : 1.f);
            uv[k] = ct ? read_attr(D, 2, vid[k], 0.f) : f4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (ct) a[k].w = 1.f;    // varying0 = (rgb, 1)
        col = f4(((a[0].x * b[0]) + (a[1].x * b[1])) + (a[2].x * b[2]), ((a[0].y * b[0]) + (a[1].y * b[1])) + (a[2].y * b[2]),
                 ((a[0].z * b[0]) + (a[1].z * b[1])) + (a[2].z * b[2]), ((a[0].w * b[0]) + (a[1].w * b[1])) + (a[2].w * b[2]));
        if (ct && D.tex != nullptr && D.texType == SL_COLOR_RGBA_FLOAT)
        {
            const float u = ((uv[0].x * b[0]) + (uv[1].x * b[1])) + (uv[2].x * b[2]);
            const float v = ((uv[0].y * b[0]) + (uv[1].y * b[1])) + (uv[2].y * b[2]);
            if (nearest)
            {
                // one tap of weight 1 (SL_Sampler.hpp:122-148)
                taps = nearest_taps(D.texW, D.texH, u, v);
                tex = sample_nearest_rgbaf(D.tex, D.texW, D.texH, u, v);
            }
            else
            {
                taps = bilinear_taps(D.texW, D.texH, u, v);
                const auto px = gptr(reinterpret_cast<const float*>(D.tex));
                float o[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    o[c] = bilerp(taps, px[4 * taps.i0 + c], px[4 * taps.i1 + c], px[4 * taps.i2 + c], px[4 * taps.i3 + c]);
                tex = f4(o[0], o[1], o[2], o[3]);
            }
            textured = true;
        }
    }

    // dL/d colour varying = g (.) texel; colour attribute k gets b_k of it.
    // COLOR_TEXTURED's alpha varying is the constant 1: no gradient there.
    int slot[7];
    uint32_t rank[7];
    float weight[7];
    float4 gc = f4(0.f, 0.f, 0.f, 0.f), gt = f4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < 7; ++j) slot[j] = -1;
    if (live && gradCol != nullptr)
    {
        gc = f4(g.x * tex.x, g.y * tex.y, g.z * tex.z, ct ? 0.f : g.w * tex.w);
        const bool useTable = claim(&sVOwner, gradCol);
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            if (vid[k] >= gradColCount) continue;
            const int v = (useTable && vid[k] < kEmptyKey) ? find_slot(sVertKey, kVertBits, (uint32_t)vid[k], sVertUsed, &sNumVerts) : -1;
            if (v < 0)
            {
                add_global4(gradCol, vid[k], b[k], gc);
                continue;
            }
            slot[k] = kVertSlot0 + v;
            rank[k] = atomicAdd(&sSlot[slot[k]], 1u);
            weight[k] = b[k];
        }
    }

    // dL/d texel = w_j * (g (.) colour varying)
    if (live && textured && gradTex != nullptr)
    {
        gt = f4(g.x * col.x, g.y * col.y, g.z * col.z, g.w * col.w);
        const bool useTable = claim(&sTOwner, gradTex);
        const uint32_t ti[4] = {taps.i0, taps.i2, taps.i1, taps.i3};     // a row's neighbours follow each other
        const float tw[4] = {taps.omdx * taps.omdy, taps.dx * taps.omdy, taps.omdx * taps.dy, taps.dx * taps.dy};
        const int ntaps = nearest ? 1 : 4;
        uint32_t group = kEmptyKey;
        int gs = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            if (j >= ntaps || ti[j] >= gradTexTexels) continue;
            if (useTable && (ti[j] >> 2) != group)
            {
                group = ti[j] >> 2;
                gs = find_slot(sGroupKey, kGroupBits, group, sGroupUsed, &sNumGroups);
            }
            if (gs < 0)
            {
                add_global4(gradTex, ti[j], tw[j], gt);
                continue;
            }
            slot[3 + j] = 4 * gs + (int)(ti[j] & 3u);
            rank[3 + j] = atomicAdd(&sSlot[slot[3 + j]], 1u);
            weight[3 + j] = tw[j];
        }
    }
    __syncthreads();

    const int groups = (int)sNumGroups, verts = (int)sNumVerts;
    slot_ranges(groups, 4, sGroupUsed, sSlot, &sNumItems[0]);
    slot_ranges(verts, 1, sVertUsed, sSlot + kVertSlot0, &sNumItems[1]);
    __syncthreads();
    auto place = [&](int j, float4 v) {
        if (slot[j] >= 0)
            sItem[(sSlot[slot[j]] >> 16) + rank[j]] = make_float4(weight[j] * v.x, weight[j] * v.y, weight[j] * v.z, weight[j] * v.w);
    };
    // lanes by the mean list: a texel has a few items unless the texture is
    // magnified, a vertex a few dozen, or hundreds in a large triangle
#pragma unroll
    for (int j = 3; j < 7; ++j) place(j, gt);
    __syncthreads();
    float* tbuf = reinterpret_cast<float*>(sTOwner);
    if ((int)sNumItems[0] <= 64 * groups) sum_slots<1>(tbuf, groups, 4, sGroupUsed, sGroupKey, sSlot, sItem);
    else sum_slots<4>(tbuf, groups, 4, sGroupUsed, sGroupKey, sSlot, sItem);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 3; ++j) place(j, gc);
    __syncthreads();
    float* vbuf = reinterpret_cast<float*>(sVOwner);
    if ((int)sNumItems[1] <= 64 * verts) sum_slots<4>(vbuf, verts, 1, sVertUsed, sVertKey, sSlot + kVertSlot0, sItem);
    else sum_slots<16>(vbuf, verts, 1, sVertUsed, sVertKey, sSlot + kVertSlot0, sItem);
}

// grad = scale * 2 * (color - target), n RGBA32F texels
__global__ __launch_bounds__(256) void k_loss_l2_grad(const float4* __restrict__ color, const float4* __restrict__ target,
                                                      float4* __restrict__ grad, uint64_t n, float scale)
{
    const float s2 = scale * 2.f;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    {
        const float4 c = color[i], t = target[i];
        grad[i] = make_float4(s2 * (c.x - t.x), s2 * (c.y - t.y), s2 * (c.z - t.z), s2 * (c.w - t.w));
    }
}

hipError_t launch_backward(const BackwardParams& p, hipStream_t s)
{
    (void)hipGetLastError();   // drop a stale error from an earlier call
    if (p.W <= 0 || p.H <= 0 || p.numDraws == 0) return hipSuccess;
    const uint64_t blocks = (uint64_t)((p.W + kBwdTile - 1) / kBwdTile) * (uint64_t)((p.H + kBwdTile - 1) / kBwdTile);
    hipLaunchKernelGGL(k_backward, dim3((unsigned)blocks), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_loss_l2_grad(const float4* color, const float4* target, float4* grad, uint64_t n, float scale, hipStream_t s)
{
    (void)hipGetLastError();   // drop a stale error from an earlier call
    if (n == 0) return hipSuccess;
    uint64_t g = (n + 255) / 256;
    if (g > 8192) g = 8192;
    hipLaunchKernelGGL(k_loss_l2_grad, dim3((unsigned)g), dim3(256), 0, s, color, target, grad, n, scale);
    return hipGetLastError();
}

}  // namespace slg
