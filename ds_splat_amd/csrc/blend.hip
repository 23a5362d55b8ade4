// Stages 4 and 5a for gfx950: per-tile alpha blending, forward (front to back) and backward
// (back to front).
//
// What counts is how many vector instructions a (pixel, entry) pair costs and how many pairs are looked at that need not be: the forward has
// 0.99 to 1.30 of them under way in a SIMD every four clocks, the backward 0.74 to 0.93, and fewer have meant less time.  The backward
// also waits for its sums: timed without the adds to memory, and then with a place in LDS for each quad of lanes' own sums, one entry at a time,
// 1 M large Gaussians 300 -> 236 -> 209 us, 3 M 253 -> 252 -> 237, 2 M faint 1281 -> 1238 -> 1184.
// 1920x1080 unless noted, us within a whole pass (medians of a trace), four lists of entries per wavefront -> sixteen -> with the clamp of alpha where it
// is needed and plain zeros beside the forward, and two entries at a time in the backward, without spills:
//   forward   2 M faint Gaussians 881 -> 686 -> 639, 1.4 M at 1557x1038 309 -> 266 -> 254, 500 K opaque 127 -> 118 -> 115 (3 M: 149 -> 148 -> 125),
//             6 M at 3840x2160 509 -> 431 -> 380, 1 M large ones 123 -> 125 -> 109, 1 M at 1280x720 138 -> 120 -> 115
//   backward  2 M faint 1637 -> 1274 -> 1212, 1.4 M at 1557x1038 519 -> 457 -> 438, 500 K opaque 223 -> 216 -> 201 (3 M: 254 -> 253 -> 234),
//             1 M large ones 302 -> 306 -> 252 to 302, 300 K at 1237x822 244 -> 223 -> 206, 50 K at 512x512 77 -> 72 -> 61
#include "dsx_common.h"

#include <atomic>
#include <climits>
#include <cstddef>
#include <cstdlib>
#include <type_traits>

namespace dsx
{

// The exponent of a splat at a pixel is -sigma, sigma = 1/2 (a dx^2 + c dy^2) + b dx dy with d = pixel -
// mean, computed in ONE fixed sequence of roundings (explicit fused multiply-adds, no contraction
// left to the compiler): the forward and the backward kernel must get the same bits, because both
// decide on their own whether the splat's alpha reaches 1/255 at the pixel.  If they disagreed on a
// borderline entry, the backward would rebuild the transmittance of every entry in front of it from a
// final value that does (or does not) contain its factor: an error of alpha in all their gradients
// at that pixel.
//   ax = 1/2 a dx^2, bx = b dx; sigma = (c/2 dy + bx) dy + ax
// (the halves are exact scalings, taken once when the entry is staged; the forward stages -a/2 and takes
// -sigma = ax - (c/2 dy + bx) dy: the same bits but for the sign)
struct ExponentX
{
    float ax, bx;
};
__device__ __forceinline__ ExponentX exponent_x(float a_half, float b, float dx)
{
#pragma clang fp contract(off)
    ExponentX r;
    r.bx = b * dx;
    // (the same rounding as the plain product; a product that is zero becomes +0, never -0)
    r.ax = __builtin_fmaf(a_half * dx, dx, 0.0f);
    return r;
}

// alpha = opacity exp(-sigma) through the hardware base-2 exponential (the reference is built with fast-math), the
// opacity as a factor of it: as a term of the exponential's argument (one instruction less for each pixel and entry)
// a faint splat's alpha would be off by up to 1.7e-7 of itself, three to four times as much as it is.  log2(e) stays a
// factor of the finished exponent: folded into the conic when an entry is staged it would put one more rounding on
// every term of the quadratic form, and where the terms are large and cancel (thin, long splats far from their centre)
// the image would move 1.6 times as far from the reference's as it does.
constexpr float kLog2E = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kLog2Of255 = 7.994353436858858f;

// Largest sigma with alpha >= 1/255, about ln(255 opacity): the test of alpha is taken on sigma, before the
// exponential and with the same bits in both directions.  -infinity for an opacity that no pixel takes, whose entry is
// then not even staged; infinity for an infinite one; NaN for a NaN.
// The reach is the last float for which opacity * exp2(-sigma log2(e)), evaluated just so, passes: every decision is
// the one that comparing alpha itself would take (alpha falls with sigma).  It lies within 2.4e-7 of an estimate from
// the logarithm and one Newton step on that expression, or within four floats of it where those are further apart, and
// is found by bisection: three steps for a reach of a half and more, one more for every halving of it (opacities from
// 1/255 to 2/255, where ever more floats of sigma share one alpha).  All floats are bisected next to 1/255 and beyond
// 1e30, where the exponential underflows before alpha falls to 1/255.
__device__ __forceinline__ float reach_of(float opacity)
{
#pragma clang fp contract(off)
    const float guess = (__builtin_amdgcn_logf(opacity) + kLog2Of255) * kLn2;
    auto alpha_at = [&](float sigma) { return opacity * __builtin_amdgcn_exp2f(-sigma * kLog2E); };
    int bits = (int)(__float_as_uint(guess + __builtin_fmaf(alpha_at(guess), 255.0f, -1.0f)) - 4u);
    auto bisect = [&](int step) { bits += alpha_at(__int_as_float(bits + step)) >= 1.0f / 255.0f ? step : 0; };
    const bool few = opacity >= 1.0f / 255.0f && opacity < 2.0f / 255.0f, many = opacity > 1e30f;
    // (only wavefronts that stage such an entry take more than the three steps)
    if(__builtin_amdgcn_ballot_w64(few || many) != 0)
    {
        constexpr int kHalf = 0x3f000000, kLeast = 0x35800000; // 2^-20
        int step = 4;
        if(many || (few && bits < kLeast)) // (also where the estimate is below zero)
        {
            bits = 0;
            step = 1 << 30;
        }
        else if(few && bits < kHalf)
        {
            step = 4 << ((kHalf - bits + 0x7fffff) >> 23);
            bits -= step - 4;
        }
        while(__builtin_amdgcn_ballot_w64(step > 4) != 0)
            if(step > 4)
            {
                bisect(step);
                step >>= 1;
            }
    }
    bisect(4);
    bisect(2);
    bisect(1);
    // (masked and pruned Gaussians: zero, denormal and negative opacities)
    return opacity < 1.0f / 255.0f ? -__builtin_inff() : (opacity < __builtin_inff() ? __int_as_float(bits) : opacity);
}
// Both tests of an entry at a pixel, that sigma has the right sign and that it does not exceed the reach,
// in one integer compare: the bits of floats of one sign are ordered like their magnitudes.
// Forward (the reference drops sigma <= 0): the bits of -sigma as a signed number are below zero only if
// sigma > 0, and grow with it: they must not exceed those of -reach.  -sigma is never -0 (ax is not, and an
// exact cancellation gives +0).  A NaN of either sign lies above every limit.  (A NaN opacity gives alpha =
// 0.999 wherever sigma > 0, as in the reference, whose fminf drops the NaN; what is below 1/255, nowhere.)
__device__ __forceinline__ int reach_limit_fwd(float opacity, float reach)
{
    return reach > 0.0f ? __float_as_int(-reach) : (opacity != opacity ? __float_as_int(-__builtin_inff()) : INT_MIN);
}
// Backward (which drops sigma < 0 only): the bits of sigma as an unsigned number, up to those of reach.
__device__ __forceinline__ uint32_t reach_limit_bwd(float opacity, float reach)
{
    return reach >= 0.0f ? __float_as_uint(reach) : (opacity != opacity ? 0x7f800000u : 0u);
}

// Pixels per lane of the blend kernels: 4 (one wavefront per tile) when the image has enough tiles
// to occupy the chip, else 1 (a workgroup of four wavefronts per
// tile: more instructions in all, but four times as many wavefronts and shorter chains).  Measured on scenes of four
// kinds, us by which a whole forward (a whole training step) is longer with the workgroup form of that kernel:
//   forward, tiles                            3600  4590  5700  6370  7150  8160
//     opaque, 0.24 Gaussians a pixel           -12    -7    +2    +5    -4    +6   (of 177 to 243)
//     mixed, 0.9 a pixel                       -16   -23    +1    -9   +12   +21   (of 312 to 511)
//     faint, 0.6 a pixel                       -13    +5   +35   +53   +86  +108   (of 261 to 703)
//     large, 0.25 a pixel                       +1    +5    +9    -1   +14   +11   (of 202 to 301)
//   backward, tiles                           1200  1900  2170  3072  3600  4590
//     opaque                                   -42   -34   -22   +17   +26   +40   (of 213 to 409)
//     mixed                                    -93   -55   -27    -2   +70  +125   (of 312 to 919)
//     faint                                    -48   -35   -15    +9   +58  +122   (of 229 to 888)
//     large                                    -25   -13   -16   +10    +8   -31   (of 271 to 445)
//   the backward's kernel alone, since both take entries by pairs: 1920, 2170, 3072, 3600, 4590 tiles
//     opaque -37, -22, +3, +8, +15; mixed -65, -38, +2, +2, +32; faint -81, -41, -68, -24, +32; large +5, -13, +22, +26, +41
// The lines at 5500 and 3000 tiles lie within those crossings.
// dsx_set_blend_pixels_per_lane(1 | 4) overrides the choice for the whole process (tests run both
// forms); DSX_BLEND_PIXELS_PER_LANE=1|4 in the environment gives the override's initial value and is
// read once.  The forward's form of sixteen wavefronts per tile is the library's own choice only: either override switches it off.
static std::atomic<int> g_forced_pixels_per_lane{-1}; // -1: not yet read from the environment, 0: automatic

static int forced_pixels_per_lane()
{
    int v = g_forced_pixels_per_lane.load(std::memory_order_relaxed);
    if(v >= 0)
        return v;
    v = 0;
    if(const char* forced = getenv("DSX_BLEND_PIXELS_PER_LANE"))
        if((forced[0] == '1' || forced[0] == '4') && forced[1] == 0)
            v = forced[0] - '0';
    int expected = -1;
    g_forced_pixels_per_lane.compare_exchange_strong(expected, v, std::memory_order_relaxed);
    return g_forced_pixels_per_lane.load(std::memory_order_relaxed);
}

int set_blend_pixels_per_lane(int pixels)
{
    if(pixels != 0 && pixels != 1 && pixels != 4)
        return DSX_ERR_BAD_ARG;
    g_forced_pixels_per_lane.store(pixels, std::memory_order_relaxed);
    return DSX_OK;
}

static int blend_pixels_per_lane(int num_tiles, int four_from)
{
    const int forced = forced_pixels_per_lane();
    if(forced != 0)
        return forced;
    return num_tiles >= four_from ? 4 : 1;
}
// Binned tile lists (see ListGrid): what a blend kernel needs to find a tile's entries in its
// bin's list.  fine[t] .. fine[t + 1] is the tile's range in the reference's fully sorted key
// array: its length says how many entries of the bin list belong to the tile, and its start turns
// "the i-th entry of the tile" into the index that the reference's final_idx holds.
struct BinLists
{
    const int32_t* fine;      // int32[tiles + 1]
    const int32_t* last_tile; // highest occupied tile (-1: none)
    const int32_t* bins;      // int32[bins + 1]
    int32_t* walk;            // int32[tiles * 8]: per tile, where the forward's scan of the bin list stopped and how many of the tile's entries it had met by then
    int shift, nbx, nty;
};

// Where tile `tile` finds its entries.  The reference never records the end of the LAST run of
// its sorted keys (cpp/rasterizer_kernels.cu:313-322, cpp/rasterizer_torch.cu:31-39), so the pairs
// of the highest occupied tile are walked by the image's last tile instead, and by nobody if that
// is another tile; with no tile occupied at all, the last tile walks the pairs of negative depth
// (slot 0, positions [0, bins[0])), every one of them.  The per-tile ranges carry those rules;
// here they decide whose pairs (src) the tile takes out of which bin's list.
struct TileSource
{
    int start, end; // positions in sorted_ids to scan
    int count;      // entries among them that belong to the tile
    int fine_base;  // index of the tile's first entry in the fully sorted key array
    int sx, sy;     // the tile whose rectangle membership selects the entries; sx < 0: every entry belongs
};
__device__ __forceinline__ TileSource tile_source(const BinLists& L, int tile, int ntx)
{
    TileSource t;
    t.fine_base = L.fine[tile];
    t.count = L.fine[tile + 1] - t.fine_base;
    t.start = t.end = 0;
    t.sx = t.sy = 0;
    if(t.count <= 0)
        return t;
    int src = tile;
    if(tile == ntx * L.nty - 1)
        src = *L.last_tile;
    if(src < 0)
    {
        t.sx = -1;
        t.end = L.bins[0];
        return t;
    }
    t.sx = src % ntx;
    t.sy = src / ntx;
    const int bin = (t.sy >> L.shift) * L.nbx + (t.sx >> L.shift);
    t.start = L.bins[bin];
    t.end = L.bins[bin + 1];
    return t;
}

// Every pair of a bin list carries, in the high half of its key word, which tiles of the bin the
// Gaussian's rectangle covers: bit x for the columns, bit 8 + y for the rows (a rectangle is the
// product of a column range and a row range).  The two bits of the tile this wavefront takes its
// entries for; 0 when every entry belongs (the list of negative depths).
__device__ __forceinline__ uint32_t tile_bits_of(const TileSource& t, int shift)
{
    if(t.sx < 0)
        return 0u;
    const int side = (1 << shift) - 1;
    return (1u << (t.sx & side)) | (256u << (t.sy & side));
}

// number of set bits of a wavefront mask below this lane
__device__ __forceinline__ int bits_below_lane(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

constexpr int kFwdWideUpTo = 256;        // tiles (a workgroup of sixteen wavefronts for each compute unit)
constexpr int kWideSplitUpTo = 64;        // (a compute unit for each quadrant)
constexpr int kFwdFourPixelsFrom = 5500;
constexpr int kBwdFourPixelsFrom = 3000;
constexpr int kBwdBlocksUpTo = 256; // (lists per tile only, as kFwdWideUpTo)
constexpr int kBwdBlocksAlways = 100;
constexpr int64_t kBwdBlocksShared = 3700; // (beyond that many tiles: pairs times tiles, by Gaussian)

// -----------------------------------------------------------------------------------------
// what both directions share: the pixels, and the walk through the lists
// -----------------------------------------------------------------------------------------
// The pixels of the workgroup forms: wavefront w of a tile owns quadrant w, its rows of 16 lanes a 4 x 4 block each.  Blocks
// of a tile are numbered as in blocks_reached: row r of the wavefront owns block first_block_of(w) + block_of_row(r).
__host__ __device__ constexpr int first_block_of(int wave) { return 8 * (wave >> 1) + 2 * (wave & 1); }
__host__ __device__ constexpr int block_of_row(int row) { return 4 * (row >> 1) + (row & 1); }
struct Pixels
{
    int x, y;
    __device__ __forceinline__ Pixels(int tile, int wave, int ntx, int lane)
    {
        const int row = lane >> 4, i = lane & 15;
        x = (tile % ntx) * kTile + 8 * (wave & 1) + 4 * (row & 1) + (i & 3);
        y = (tile / ntx) * kTile + 8 * (wave >> 1) + 4 * (row >> 1) + i / 4;
    }
};

// word `i` of a device array (uniform base and a 32-bit byte offset: one address register; i < 2^30, so a scan of a
// list passes the place where it stands as the base)
__device__ __forceinline__ int word_at(const int32_t* base, uint32_t i)
{
    return *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(base) + 4u * i);
}

// a wavefront mask of the lanes below `count`
__device__ __forceinline__ uint64_t lanes_below(int count)
{
    return count >= DSX_WAVE ? ~0ull : (1ull << max(count, 0)) - 1;
}

// the lowest `count` set bits of a mask that has more
__device__ __forceinline__ uint64_t lowest_bits(uint64_t mask, int count)
{
    return __builtin_amdgcn_ballot_w64(bits_below_lane(mask) < count) & mask;
}

// the values of other lanes of each quad of lanes (quad_perm)
template <int kCtrl>
__device__ __forceinline__ float quad_lane(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true));
}

// A side job for the memory system, which the forward leaves idle: every workgroup prepares
// its share of the backward's gradient accumulator, twelve floats per Gaussian: the nine sums
// zeroed and, in the three spare places, the conic, which the per-Gaussian backward then has
// at hand with the sums instead of fetching the splat records for it.  At the end of the
// kernel, where nothing waits for the stores and the wavefronts arrive spread over time (at
// the start they would all come at once and hold up the first loads: 0.147 against 0.140 ms).
__device__ __forceinline__ void prepare_grads_share(const float4* splats, float4* prep, int64_t count, uint8_t* marks,
                                                    int part, int parts, int tid, int threads)
{
    static_assert(DSX_GRAD_FLOATS == 12, "three float4 per Gaussian");
    const int64_t share = (count + parts - 1) / parts;
    const int64_t g1 = min((part + 1) * share, count);
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    for(int64_t g = part * share + tid; g < g1; g += threads)
    {
        const float4 q1 = splats[3 * g + 1]; // conic a, b, c, opacity
        prep[3 * g] = zero;
        prep[3 * g + 1] = zero;
        prep[3 * g + 2] = make_float4(0.f, q1.x, q1.y, q1.z);
        if(marks)
            marks[g] = 0; // "no term added yet"
    }
}
// The same without the conics, records and bytes as one run of zeros: nothing is read, and what is written is written in order.
// (Figures at zeros_alone.  A few stores of each thread behind every round's loads, instead of all at the end: 3 M Gaussians the same,
// 2 M faint +3 us, the workgroup forms +5.  The tiles preparing the records of what they stage, and nobody the others': 3 M 124 us, but 2 M
// faint 764, whose every Gaussian seven tiles on different XCDs stage.)
__device__ __forceinline__ void zero_grads_share(float4* prep, int64_t count, int part, int parts, int tid, int threads)
{
    const int64_t all = 3 * count + (count + 15) / 16, share = (all + parts - 1) / parts;
    const int64_t end = min((part + 1) * share, all);
    for(int64_t i = part * share + tid; i < end; i += threads)
        prep[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// -----------------------------------------------------------------------------------------
// forward: cpp/rasterizer_kernels.cu:341-431
// -----------------------------------------------------------------------------------------
// No workgroup barrier anywhere: a workgroup is one wavefront.  A round takes entries of the tile's
// list, 64 at a time: what cannot reach the box around the blocks that still have a live pixel drops out (two words of its record
// and some forty instructions for 64 of them; two thirds of the faint Gaussians' rectangles touch tiles that they do not reach),
// and when 64 are left they are staged in LDS, each lane one, and the place of each goes into the list of every quad of
// lanes whose block it reaches.  Then the quads walk their lists side by side.
constexpr int kPix = 4; // pixels per lane of the wavefront forms
constexpr float kAlphaMax = 0.999f;       // the forward's clamp (the backward's is 0.99)
constexpr int kScanGroups = 4; // groups of 64 positions of a bin's list whose loads are in flight together

// The 16 blocks of a tile, 4 x 4 pixels each: bit 4 r + c of a mask is the block of the r-th four rows and c-th four
// columns.  A wavefront that works on a whole tile has a quad of lanes for each block (lane l: quad l >> 2, the column l & 15 of
// the tile and four pixels, one below the other), and each quad walks ITS OWN list of entries: sixteen entries are blended side by
// side.  An entry of a tile's list that touches the tile at all touches only part of it, so a wavefront that walks one list
// for all of its pixels spends most of its lanes on pixels that the entry cannot reach; skipping those on the
// scalar unit costs as much as it saves, while giving the lanes another entry costs two address instructions.  The quads
// wait for each other only once per round of staged entries.  Steps of the walk per tile, of four rows of lanes with a list for each
// 8 x 8 block and of sixteen quads (2 M faint Gaussians at 1920x1080, 1.4 M at 1557x1038, 1 M at 1280x720, 500 K opaque at 1920x1080):
// 713 -> 570, 258 -> 224, 195 -> 154, 86 -> 82; one list for all pixels takes 1056, 362, 300 and 120.
constexpr int kQuads = 16;

// which quads a wavefront mask has a lane of: bit q (uniform)
__device__ __forceinline__ uint32_t quads_of(uint64_t mask, int lane)
{
    return (uint32_t)__builtin_amdgcn_ballot_w64(((mask >> (4 * (lane & 15))) & 15u) != 0) & 0xffffu;
}

// The box of pixel centres around some blocks of a tile
struct LiveBox
{
    float x0, x1, y0, y1;
};
__device__ __forceinline__ LiveBox live_box(uint32_t blocks, float x, float y)
{
    const uint32_t columns = (blocks | blocks >> 4 | blocks >> 8 | blocks >> 12) & 15u;
    LiveBox box;
    box.x0 = x + (float)(4 * __builtin_ctz(columns | 16u));
    box.x1 = x + (float)(4 * (31 - __builtin_clz(columns | 1u)) + 3);
    box.y0 = y + (float)(__builtin_ctz(blocks | 0x10000u) & ~3);
    box.y1 = y + (float)(((31 - __builtin_clz(blocks | 1u)) & ~3) + 3);
    return box;
}

// Can this splat (the first two words of its record) reach a pixel of the box with alpha >= 1/255?
// The exponent's quadratic form q(d) = 1/2 (a dx^2 + c dy^2) + b dx dy is convex, so its minimum over the box is 0 if the
// splat's centre lies inside and otherwise sits on an edge that faces the centre, where it is a clamped one-dimensional
// parabola.  Taking the column and the row of the box that lie nearest to the centre covers both: they are the
// facing edges where there are any (and points of the box where not).  An entry is left out only if the minimum exceeds
// ln(255 opacity) by more than 0.01 (one percent of alpha) and what it may be off by where its terms are large and cancel; one
// with a degenerate conic or without a limit is kept.
// (That share of the terms, here and in blocks_reached, is two and a half times the largest difference between such a minimum and the
// exponents of the box's pixels, 1e-7 of the terms, among 1.3 M splats of 50 to 2000 pixels' length and 0.55 to 0.77 width; it
// exceeds 0.01 from 300 pixels on.)
constexpr float kOfTerms = 2.5e-7f;
__device__ __forceinline__ bool box_reached(const LiveBox& box, const float4 q0, const float4 q1)
{
    const float a = q1.x, b = q1.y, c = q1.z, opacity = q1.w;
    const float half_a = 0.5f * a, half_c = 0.5f * c;
    const float u0 = box.x0 - q0.x, u1 = box.x1 - q0.x, v0 = box.y0 - q0.y, v1 = box.y1 - q0.y;
    const float u_far = fmaxf(fabsf(u0), fabsf(u1)), v_far = fmaxf(fabsf(v0), fabsf(v1));
    const float limit = __builtin_fmaf(__builtin_amdgcn_logf(opacity) + kLog2Of255, kLn2, 0.01f) +
                        kOfTerms * (a * u_far * u_far + c * v_far * v_far);
    const float un = __builtin_amdgcn_fmed3f(0.0f, u0, u1), vn = __builtin_amdgcn_fmed3f(0.0f, v0, v1);
    // along the nearest column, and along the nearest row
    const float v = __builtin_amdgcn_fmed3f(-b * __builtin_amdgcn_rcpf(c) * un, v0, v1);
    const float u = __builtin_amdgcn_fmed3f(-b * __builtin_amdgcn_rcpf(a) * vn, u0, u1);
    const float qmin = fminf(v * (half_c * v + b * un) + half_a * un * un, u * (half_a * u + b * vn) + half_c * vn * vn);
    // (below 1/255: no pixel takes it; a NaN opacity is kept)
    return !(opacity < 1.0f / 255.0f) && !(a > 0.0f && c > 0.0f && qmin > limit);
}

// Which of a tile's blocks can this entry reach?  For each four rows of pixels the ellipse q <= limit takes up a range of
// columns: its right and left extremes lie at v = -+ (b/c) umax (umax: the ellipse's half width) where those rows hold them and
// at the nearest row otherwise.  The limit is the reach plus 0.01 and plus what q may be off by where its
// terms are large and cancel (the determinant, too, is one rounding off its value, not off its terms); the range is
// widened by 1/16 pixel.  All blocks for a degenerate conic or an entry without a limit.
// (x0, y0: the tile's first pixel centre)
__device__ __forceinline__ uint32_t blocks_reached(float mx, float my, float a, float b, float c, float reach, float x0, float y0)
{
    constexpr float kSlack = 1.0f / 64.0f; // in blocks
    float det;
    {
#pragma clang fp contract(off)
        const float bb = b * b;
        det = __builtin_fmaf(a, c, -bb) - __builtin_fmaf(b, b, -bb);
    }
    const float u_first = x0 - mx, v_first = y0 - my;
    const float u_far = fmaxf(fabsf(u_first), fabsf(u_first + (kTile - 1))), v_far = fmaxf(fabsf(v_first), fabsf(v_first + (kTile - 1)));
    const float limit = reach + 0.01f + kOfTerms * (a * u_far * u_far + c * v_far * v_far);
    const bool all = !(a > 0.0f && c > 0.0f && det > 1e-30f && limit < 1e30f);
    const float two = 2.0f * limit, inv_a = __builtin_amdgcn_rcpf(a), per_det = two * __builtin_amdgcn_rcpf(det);
    const float vmax = __builtin_amdgcn_sqrtf(a * per_det);
    const float v_left = b * __builtin_amdgcn_rcpf(c) * __builtin_amdgcn_sqrtf(c * per_det); // (the right extreme: -v_left)
    const float from = (u_first + 3.0f) * -0.25f - kSlack, to = u_first * -0.25f + (1.0f + kSlack);
    const float quarter = 0.25f * inv_a;
    uint32_t reached = 0;
#pragma unroll
    for(int r = 0; r < 4; ++r)
    {
        const float v0 = fmaxf(v_first + (float)(4 * r), -vmax), v1 = fminf(v_first + (float)(4 * r + 3), vmax);
        const float vl = __builtin_amdgcn_fmed3f(v_left, v0, v1), vr = __builtin_amdgcn_fmed3f(-v_left, v0, v1);
        const float left = __builtin_amdgcn_sqrtf(fmaxf(a * two - det * vl * vl, 0.0f)) + b * vl;
        const float right = __builtin_amdgcn_sqrtf(fmaxf(a * two - det * vr * vr, 0.0f)) - b * vr;
        // the first block that ends behind the left extreme, the first one that begins behind the right
        const int first = (int)__builtin_amdgcn_fmed3f(ceilf(from - left * quarter), 0.0f, 4.0f);
        const int behind = v0 <= v1 ? (int)__builtin_amdgcn_fmed3f(floorf(to + right * quarter), 0.0f, 4.0f) : 0;
        reached |= ((1u << max(behind - first, 0)) - 1u) << (first + 4 * r);
    }
    return all ? 0xffffu : (reach >= 0.0f ? reached : 0u);
}

// The lists of a round, from which blocks the entry of every lane reaches: the places of the entries of each quad, in order, in
// bytes that held kPlaces, nobody's place.  Returns the longest list's length.
constexpr int kBatch = DSX_WAVE; // staged entries of a round
template <int kPlaces>
__device__ __forceinline__ int quad_lists(uint8_t* bytes, uint32_t reached, int lane)
{
    int longest = 0;
#pragma unroll
    for(int q = 0; q < kQuads; ++q)
    {
        const uint64_t m = __builtin_amdgcn_ballot_w64((reached & (1u << q)) != 0);
        if(__builtin_amdgcn_inverse_ballot_w64(m))
            bytes[__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, q * kPlaces))] = (uint8_t)lane;
        longest = max(longest, (int)__popcll(m));
    }
    return longest;
}

// a pixel's colour: interleaved, or channel-first with the background composited
__device__ __forceinline__ void store_pixel(float* image, int64_t pix, int64_t plane, float red, float green, float blue, float T,
                                            bool broken, const float* bg, int planar)
{
    if(broken)
        red = green = blue = __builtin_nanf("");
    if(planar)
    {
        image[pix] = broken ? red : __builtin_fmaf(T, bg[0], red);
        image[pix + plane] = broken ? green : __builtin_fmaf(T, bg[1], green);
        image[pix + 2 * plane] = broken ? blue : __builtin_fmaf(T, bg[2], blue);
    }
    else
    {
        image[3 * pix] = red;
        image[3 * pix + 1] = green;
        image[3 * pix + 2] = blue;
    }
}

// kBinned: the entries come out of the list of the tile's bin (BinLists).  The wavefront first
// FILTERS the bin's list: 64 positions at a time it reads the pair's id and key word (two coalesced
// 4-byte loads, those of four groups in flight together), tests the two bits of its tile in the key's mask,
// and queues the ids of its own entries, one per lane, until 64 are there or the list ends.  Only those
// are then gathered and tested for reach, so a tile pays a dozen instructions per 64
// entries of its bin's list instead of a gather and a rectangle test per entry; a scene whose
// pixels do not saturate early, where every tile reads its bin's whole list, costs a few percent
// more than with per-tile lists instead of twice as much.  final_idx still receives the
// reference's index: the tile's range start plus the entry's rank among the tile's own entries.
// (seven wavefronts per SIMD: 72 registers; with eight and 64 the walk waits for reloads, 500 K opaque 135 against 130 us, 6 M
// at 4K 461 against 446; with six the last tiles of a 1080p image start late, 2 M faint 748 against 706)
template <bool kBinned>
__global__ __launch_bounds__(DSX_WAVE) __attribute__((amdgpu_waves_per_eu(7, 7))) void blend_fwd_kernel(const int32_t* __restrict__ ranges,
                                                             const int32_t* __restrict__ ids,
                                                             const float4* __restrict__ splats,
                                                             float* __restrict__ image, float* __restrict__ final_T,
                                                             int32_t* __restrict__ final_idx, int W, int H, int ntx,
                                                             uint32_t last_id, int k,
                                                             const int32_t* __restrict__ header, int header_shift,
                                                             const uint32_t* __restrict__ sort_flag_a,
                                                             const uint32_t* __restrict__ sort_flag_b,
                                                             float4* __restrict__ prep, int64_t prep_count,
                                                             uint8_t* __restrict__ prep_marks, int prep_zeros,
                                                             const float* __restrict__ bg, int planar,
                                                             const BinLists lists)
{
    // the last place is nobody's entry (no exponent passes): quads whose list has ended point at it
    __shared__ float4 s_a[kBatch + 1]; // pixel x, pixel y, conic -a/2, conic b
    __shared__ float4 s_b[kBatch + 1]; // conic c/2, opacity, limit of the exponent's bits, index in the sorted key array
    __shared__ float4 s_c[kBatch + 1]; // red, green, blue
    __shared__ uint4 s_list[kQuads * kBatch / 16 + 1]; // a byte per entry and quad: its place (one word more than is used: read ahead)
    __shared__ int2 s_left[kBatch]; // candidates (id, index) that did not fit the round
    // while a round is staged, in the records' memory: the candidates, and ids of the tile's own entries on their way from
    // the scan to the gather (the last place stays as it is)
    int2* const s_cand = reinterpret_cast<int2*>(s_a);
    int* const s_queue = reinterpret_cast<int*>(s_b);
    static_assert(2 * kBatch * sizeof(int2) <= kBatch * sizeof(float4), "candidates fit the records' memory");

    const int lane = threadIdx.x;
    const int tile = blockIdx.x;
    const int x0 = (tile % ntx) * kTile, y0 = (tile / ntx) * kTile;
    const int x = x0 + (lane & 15), y = y0 + kPix * (lane >> 4); // this lane's column of four pixels
    const float pxf = (float)x + 0.5f;

    // The lists are data from the device: positions are taken for what they are only inside
    // sorted_ids[0, k), and a `ranges` buffer that was built for another bin size (its header word,
    // which every layout has in the same place, says which) is not read any further; the image is
    // then NaN, like after a sort that gave up.
    const bool layout_ok = header == nullptr || *header == header_shift;
    int start = 0, end = 0;
    TileSource src = {};
    if(kBinned)
    {
        if(layout_ok)
            src = tile_source(lists, tile, ntx);
        start = src.start;
        end = src.end;
    }
    else if(layout_ok)
    {
        start = ranges[tile];
        end = ranges[tile + 1];
    }
    start = min(max(start, 0), k);
    end = min(max(end, 0), k);

    // A pixel that has stopped (or lies outside the image) gets NaN as its row coordinate: its
    // exponent is then NaN, the test of it fails whatever the entry holds, and the loop
    // needs no per-pixel flag.  `alive` counts the wavefront's live pixels (a scalar: it is kept
    // from ballots, on the scalar unit, and costs the vector unit nothing).
    float pyf[kPix], T[kPix], red[kPix], green[kPix], blue[kPix];
    int last[kPix];
    int alive = 0;
#pragma unroll
    for(int p = 0; p < kPix; ++p)
    {
        const bool inside = x < W && y + p < H;
        pyf[p] = inside ? (float)(y + p) + 0.5f : __builtin_nanf("");
        alive += __popcll(__builtin_amdgcn_ballot_w64(inside));
        T[p] = 1.0f;
        red[p] = green[p] = blue[p] = 0.0f;
        last[p] = 0;
    }
    if(lane == 0)
    {
        s_a[kBatch] = s_c[kBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kBatch] = make_float4(0.f, 0.f, __int_as_float(INT_MIN), 0.f);
    }

    // binned lists: the scan of the bin's list
    const uint32_t tile_bits = kBinned ? tile_bits_of(src, lists.shift) << 16 : 0u; // (in the key word's high half)
    const int32_t* const keys = ids + k; // the pairs' key words lie behind the ids (binned lists)
    int scan = start;  // next position of the list to look at
    int seen = 0;      // entries of the tile's own list found so far
    int index_next = kBinned ? src.fine_base : start; // what final_idx records for the next entry
    int left = 0;      // candidates that the last round left
    while(alive != 0 && (left > 0 || (scan < end && (!kBinned || seen < src.count))))
    {
        // blocks with a live pixel, and the box around them
        uint64_t live = 0;
#pragma unroll
        for(int p = 0; p < kPix; ++p)
            live |= __builtin_amdgcn_ballot_w64(pyf[p] == pyf[p]);
        const uint32_t live_blocks = quads_of(live, lane);
        const LiveBox box = live_box(live_blocks, (float)x0 + 0.5f, (float)y0 + 0.5f);

        __syncthreads(); // single wavefront: orders the LDS reads of the last round before these writes
        constexpr uint32_t kNobodies = 0x01010101u * kBatch;
        s_list[lane] = make_uint4(kNobodies, kNobodies, kNobodies, kNobodies);
        int found = left;
        if(lane < left)
            s_cand[lane] = s_left[lane];
        while(found < kBatch && scan < end && (!kBinned || seen < src.count))
        {
            int id = 0;
            int batch; // entries in this gather
            if(kBinned)
            {
                batch = 0;
                do
                {
                    // the loads of four groups of positions are issued together: the scan is bound by
                    // their latency, not by its dozen instructions per group
                    int gid[kScanGroups], key[kScanGroups];
                    const int32_t* const ids_here = ids + scan;
                    const int32_t* const keys_here = keys + scan;
#pragma unroll
                    for(int j = 0; j < kScanGroups; ++j)
                    {
                        const uint32_t e = (uint32_t)min(j * DSX_WAVE + lane, end - 1 - scan);
                        gid[j] = word_at(ids_here, e);
                        key[j] = word_at(keys_here, e);
                    }
#pragma unroll
                    for(int j = 0; j < kScanGroups; ++j)
                    {
                        // (uniform; a group that lies behind the end has no members, and moves nothing)
                        uint64_t m = __builtin_amdgcn_ballot_w64(((uint32_t)key[j] & tile_bits) == tile_bits) &
                                     lanes_below(end - scan);
                        int taken = min(end - scan, DSX_WAVE);
                        const int room = DSX_WAVE - batch;
                        if(__popcll(m) > room)
                        {
                            // not all of the group's members fit: it is taken up to the last one that does
                            m = lowest_bits(m, room);
                            taken = room > 0 ? DSX_WAVE - __builtin_clzll(m) : 0;
                        }
                        if(m != 0)
                        {
                            if(__builtin_amdgcn_inverse_ballot_w64(m))
                                s_queue[batch + bits_below_lane(m)] = gid[j];
                            batch += __popcll(m);
                        }
                        scan += taken;
                        if(taken < DSX_WAVE)
                            break;
                    }
                } while(batch < DSX_WAVE && scan < end && seen + batch < src.count);
                seen += batch;
                __syncthreads();
                id = s_queue[lane];
                __syncthreads();
            }
            else
            {
                batch = min(end - scan, DSX_WAVE);
                if(lane < batch)
                    id = ids[scan + lane];
                scan += batch;
            }
            bool reaches = false;
            if(lane < batch)
            {
                // (an id is taken for what it is only up to the last Gaussian: lists that a failed sort or a
                // caller's mix-up left in disorder then give a wrong image, not a fetch outside the records)
                id = (int)min((uint32_t)id, last_id);
                const float4* const rec = splats + 3 * (int64_t)id;
                reaches = box_reached(box, rec[0], rec[1]);
            }
            const uint64_t m = __builtin_amdgcn_ballot_w64(reaches);
            if(reaches)
                s_cand[found + bits_below_lane(m)] = make_int2(id, index_next + lane);
            found += __popcll(m);
            index_next += batch;
        }
        __syncthreads();
        const int staged = min(found, kBatch);
        const int2 mine = s_cand[lane], spare = s_cand[kBatch + lane];
        left = found - staged;
        __syncthreads();
        if(lane < left)
            s_left[lane] = spare;
        uint32_t reached = 0;
        bool clamp = false; // (does its alpha reach the clamp anywhere?)
        if(lane < staged)
        {
            const float4* const rec = splats + 3 * (int64_t)mine.x;
            const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];
            const float reach = reach_of(q1.w);
            clamp = !(q1.w <= kAlphaMax);
            reached = live_blocks & blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, (float)x0 + 0.5f, (float)y0 + 0.5f);
            s_a[lane] = make_float4(q0.x, q0.y, q1.x * -0.5f, q1.y);
            s_b[lane] = make_float4(q1.z * 0.5f, q1.w, __int_as_float(reach_limit_fwd(q1.w, reach)), __int_as_float(mine.y));
            s_c[lane] = q2;
        }
        const int rounds = quad_lists<kBatch>(reinterpret_cast<uint8_t*>(s_list), reached, lane);
        const bool clamps = __builtin_amdgcn_ballot_w64(clamp) != 0;
        __syncthreads();

        // Two entries at a time, the transmittance going from T to U and back: a pixel that an entry makes opaque keeps the
        // former (its copy costs nothing where, as nearly always, no pixel stops).
        const uint16_t* my_list = reinterpret_cast<const uint16_t*>(s_list) + (lane >> 2) * (kBatch / 2);
        int places = *my_list;
        for(int i = 0; i < rounds; i += 2)
        {
            if(alive == 0)
                break;
            const int here = places;
            places = *++my_list;
            float U[kPix];
            auto blend = [&](int place, const float (&before)[kPix], float (&after)[kPix]) {
                const float4 A = s_a[place];
                const float4 B = s_b[place];
                const float4 C = s_c[place];
                const int limit = __float_as_int(B.z);
                // what final_idx records for this entry: its position in the sorted key array (binned
                // lists: the tile's range start plus the entry's rank among the tile's own entries)
                const int entry_index = __float_as_int(B.w);
                const ExponentX ex = exponent_x(A.z, A.w, pxf - A.x);
                float alpha[kPix], weight[kPix];
                uint64_t m_pass[kPix];
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
#pragma clang fp contract(off)
                    const float dy = pyf[p] - A.y;
                    const float power = __builtin_fmaf(-__builtin_fmaf(B.x, dy, ex.bx), dy, ex.ax);
                    // the decisions as wavefront masks (each is its compare's own result register),
                    // combined on the scalar unit and handed back to the lanes as conditions
                    m_pass[p] = __builtin_amdgcn_ballot_w64(__float_as_int(power) <= limit);
                    alpha[p] = B.y * __builtin_amdgcn_exp2f(power * kLog2E);
                }
                // (only where an entry of the round can reach the clamp: four of some 66 instructions an entry.  A branch costs less here than
                // a second walk without the clamp, which does not fit the registers; 6 M Gaussians at 3840x2160 401 -> 381 us, 1.4 M at
                // 1557x1038 266 -> 257, 500 K opaque 122 -> 117, 2 M faint 671 -> 660.  Where nearly every round has one, against a clamp without the
                // branch: 500 K of which half reach beyond 0.99 91 -> 94, all 82 -> 84, 6 M 182 -> 188, 1.4 M 79 -> 82)
                if(__builtin_expect(clamps, 0))
                {
                    // (a NaN opacity gives 0.999, as in the reference: fminf drops the NaN)
#pragma unroll
                    for(int p = 0; p < kPix; ++p)
                        alpha[p] = fminf(kAlphaMax, alpha[p]);
                }
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
                    const float taken = __builtin_amdgcn_inverse_ballot_w64(m_pass[p]) ? alpha[p] : 0.0f;
                    weight[p] = taken * before[p];
                    after[p] = __builtin_fmaf(-taken, before[p], before[p]); // (1 - alpha) T in one rounding
                }
                // (one compare for the least of the four: three instructions an entry instead of four, and four mask words less; whole
                // passes of 2 M faint Gaussians 2294 -> 2276 us, 1.4 M 973 -> 966, 6 M at 3840x2160 965 -> 958)
                static_assert(kPix == 4, "the least of four");
                if(__builtin_amdgcn_ballot_w64(fminf(fminf(fminf(after[0], after[1]), after[2]), after[3]) < 0.0001f) != 0)
                {
                    // pixels that this entry would make opaque stop without it
#pragma unroll
                    for(int p = 0; p < kPix; ++p)
                    {
                        const uint64_t m_low = __builtin_amdgcn_ballot_w64(after[p] < 0.0001f);
                        const bool stop = __builtin_amdgcn_inverse_ballot_w64(m_low);
                        weight[p] = stop ? 0.0f : weight[p];
                        after[p] = stop ? before[p] : after[p];
                        pyf[p] = stop ? __builtin_nanf("") : pyf[p];
                        m_pass[p] &= ~m_low;
                        alive -= __popcll(m_low);
                    }
                }
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
                    red[p] = __builtin_fmaf(weight[p], C.x, red[p]);
                    green[p] = __builtin_fmaf(weight[p], C.y, green[p]);
                    blue[p] = __builtin_fmaf(weight[p], C.z, blue[p]);
                    last[p] = __builtin_amdgcn_inverse_ballot_w64(m_pass[p]) ? entry_index : last[p];
                }
            };
            blend(here & 0xff, T, U);
            blend(here >> 8, U, T);
        }
    }

    // A sort pass that gave up waiting on its predecessor (bounded wait, never seen to happen)
    // leaves its flag set and the tile lists wrong: make that loud instead of plausible.
    const bool broken = !layout_ok || (sort_flag_a && *sort_flag_a) || (sort_flag_b && *sort_flag_b);
#pragma unroll
    for(int p = 0; p < kPix; ++p)
        if(x < W && y + p < H)
        {
            const int64_t pix = (int64_t)(y + p) * W + x;
            final_T[pix] = T[p];
            final_idx[pix] = last[p];
            store_pixel(image, pix, (int64_t)W * H, red[p], green[p], blue[p], T[p], broken, bg, planar);
        }
    if(kBinned && layout_ok)
    {
        // for the backward: where this wavefront's scan of the bin's list stopped and how many of the
        // tile's entries it had met by then (everything that any of its pixels blended lies below).
        // The tile's other six words are marked as empty.
        int32_t* w = lists.walk + (int64_t)tile * 8;
        const int stopped = min(scan, end);
        if(lane < 8)
            w[lane] = lane == 0 ? stopped : (lane == 1 ? seen : (lane & 1 ? 0 : -1));
    }
    if(prep_zeros)
        zero_grads_share(prep, prep_count, blockIdx.x, gridDim.x, lane, DSX_WAVE);
    else
        prepare_grads_share(splats, prep, prep_count, prep_marks, blockIdx.x, gridDim.x, lane, DSX_WAVE);
}

// -----------------------------------------------------------------------------------------
// the same for images of few tiles: a workgroup of four wavefronts per tile
// -----------------------------------------------------------------------------------------
// When the tiles are too few to fill the chip, a wavefront per tile leaves much of it idle and takes as
// long as its longest dependency chain.  Here four wavefronts share a tile: each owns a quadrant (its
// rows of lanes the quadrant's four 4x4 blocks, one pixel per lane), the four stage a round
// of up to kTileBatch entries together (each thread gathers and tests one candidate, against
// all sixteen blocks), and every wavefront then builds and walks its own rows' lists.  The smaller blocks leave
// a row a third to a half of the tile's entries, and entries are taken four (backward: two) at a time, with their
// LDS reads and exponentials in flight together.
constexpr int kTileBatch = 248;   // (places are bytes; a multiple of 8)
constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / DSX_WAVE;

// The scan of a bin's list by a workgroup: positions `at`, `at + step`, ... of which `left` lie inside
// the list; queues up to kTileBatch ids of the entries whose key word has `bits`, after the first `skip` of
// them.  Returns the number queued; `left` becomes the number of positions that remain, `skip` what remains of it.
struct TileScan
{
    int counts[kScanGroups * kTileWaves]; // members per group of positions and wavefront
    int taken;                            // positions up to the last accepted member
};
template <int kStep>
__device__ __forceinline__ int tile_scan(TileScan& s, int* queue, const int32_t* ids, const int32_t* keys, int& at, int& left,
                                         int& skip, uint32_t bits, int wanted)
{
    const int tid = threadIdx.x, wave = tid / DSX_WAVE;
    int batch = 0;
    while(left > 0 && batch < kTileBatch && batch < wanted)
    {
        int id[kScanGroups];
        uint64_t m[kScanGroups];
        uint32_t key[kScanGroups];
        const int most = min(left, kScanGroups * kTileThreads) - 1;
        const int32_t* const ids_here = ids + (kStep > 0 ? at : at - most);
        const int32_t* const keys_here = keys + (kStep > 0 ? at : at - most);
#pragma unroll
        for(int j = 0; j < kScanGroups; ++j)
        {
            const int o = min(j * kTileThreads + tid, most);
            const uint32_t e = (uint32_t)(kStep > 0 ? o : most - o);
            id[j] = word_at(ids_here, e);
            key[j] = (uint32_t)word_at(keys_here, e);
        }
#pragma unroll
        for(int j = 0; j < kScanGroups; ++j)
        {
            m[j] = __builtin_amdgcn_ballot_w64((key[j] & bits) == bits) &
                   lanes_below(left - j * kTileThreads - wave * DSX_WAVE);
            if((tid & (DSX_WAVE - 1)) == 0)
                s.counts[j * kTileWaves + wave] = __popcll(m[j]);
        }
        if(tid == 0)
            s.taken = kScanGroups * kTileThreads;
        __syncthreads();
        int before = 0, first[kScanGroups] = {};
#pragma unroll
        for(int i = 0; i < kScanGroups * kTileWaves; ++i)
        {
            const int c = s.counts[i];
#pragma unroll
            for(int j = 0; j < kScanGroups; ++j)
                first[j] += i < j * kTileWaves + wave ? c : 0;
            before += c;
        }
        const int total = __builtin_amdgcn_readfirstlane(before);
        const int room = kTileBatch - batch;
#pragma unroll
        for(int j = 0; j < kScanGroups; ++j)
        {
            const int rank = first[j] + bits_below_lane(m[j]) - skip; // among the accepted
            if(__builtin_amdgcn_inverse_ballot_w64(m[j]) && rank >= 0 && rank < room)
            {
                queue[batch + rank] = id[j];
                if(rank == room - 1)
                    s.taken = j * kTileThreads + tid + 1;
            }
        }
        __syncthreads();
        const int taken = min(left, __builtin_amdgcn_readfirstlane(s.taken));
        at += kStep > 0 ? taken : -taken;
        left -= taken;
        batch += min(max(total - skip, 0), room);
        skip = max(skip - total, 0);
        __syncthreads(); // s is written again
    }
    return batch;
}

// A wavefront's lists of one round: the places of the staged entries that reach each of its four blocks,
// padded with the place that is nobody's.  Returns the longest list's length.
__device__ __forceinline__ int build_lists(uint32_t* list_words, const uint16_t* reach, int staged, int wave, int first_block, int lane)
{
    uint8_t* const bytes = reinterpret_cast<uint8_t*>(list_words + wave * kTileBatch);
    for(int i = lane; i < kTileBatch; i += DSX_WAVE)
        list_words[wave * kTileBatch + i] = 0x01010101u * kTileBatch;
    int length[4] = {0, 0, 0, 0};
    for(int first = 0; first < staged; first += DSX_WAVE)
    {
        const int place = first + lane;
        const uint32_t mine = place < staged ? (uint32_t)reach[place] >> first_block : 0u;
#pragma unroll
        for(int r = 0; r < 4; ++r)
        {
            const uint64_t m = __builtin_amdgcn_ballot_w64((mine >> block_of_row(r)) & 1);
            if(__builtin_amdgcn_inverse_ballot_w64(m))
                bytes[r * kTileBatch + length[r] + bits_below_lane(m)] = (uint8_t)place;
            length[r] += __popcll(m);
        }
    }
    return max(max(length[0], length[1]), max(length[2], length[3]));
}

// this thread's place among the threads of the workgroup whose `m` (a mask per wavefront) is set, and their number
__device__ __forceinline__ int tile_place(int* counts, uint64_t m, int& total)
{
    const int wave = threadIdx.x / DSX_WAVE;
    if((threadIdx.x & (DSX_WAVE - 1)) == 0)
        counts[wave] = __popcll(m);
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for(int w = 0; w < kTileWaves; ++w)
    {
        const int c = counts[w];
        before += w < wave ? c : 0;
        all += c;
    }
    total = __builtin_amdgcn_readfirstlane(all);
    return before + bits_below_lane(m);
}

constexpr int kFwdAtOnce = 4; // entries that a row takes at a time
static_assert(kFwdAtOnce == 4 && kTileBatch % 4 == 0, "a word of the list holds four places");

// (six wavefronts per SIMD: 79 registers instead of the 92 that the scan's loads in flight take; whole passes of 1 M at 1280x720
// 254 -> 248 us, 300 K at 1237x822 430 -> 423; with seven and 72 the walk reloads, 251 and 426)
template <bool kBinned>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(6))) void blend_fwd_tile_kernel(const int32_t* __restrict__ ranges, const int32_t* __restrict__ ids,
                                                                      const float4* __restrict__ splats, float* __restrict__ image,
                                                                      float* __restrict__ final_T, int32_t* __restrict__ final_idx, int W,
                                                                      int H, int ntx, uint32_t last_id, int k,
                                                                      const int32_t* __restrict__ header, int header_shift,
                                                                      const uint32_t* __restrict__ sort_flag_a,
                                                                      const uint32_t* __restrict__ sort_flag_b, float4* __restrict__ prep,
                                                                      int64_t prep_count, uint8_t* __restrict__ prep_marks, int prep_zeros,
                                                                      const float* __restrict__ bg, int planar,
                                                                      const BinLists lists)
{
    // (arrays as in the wavefront form)
    __shared__ float4 s_a[kTileBatch + 1], s_b[kTileBatch + 1], s_c[kTileBatch + 1];
    __shared__ uint16_t s_reach[kTileBatch]; // which of the tile's 16 blocks an entry reaches
    __shared__ uint32_t s_list[kTileWaves * kTileBatch];
    __shared__ int s_queue[kTileBatch];
    __shared__ TileScan s_scan;
    __shared__ int s_counts[kTileWaves];
    __shared__ uint32_t s_live[kTileWaves];

    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), row = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / DSX_WAVE);
    const int tile = blockIdx.x;
    const int first_block = first_block_of(wave);
    const Pixels px(tile, wave, ntx, lane);
    const float pxf = (float)px.x + 0.5f;
    const float tile_x = (float)(tile % ntx * kTile) + 0.5f, tile_y = (float)(tile / ntx * kTile) + 0.5f;

    // (positions and layout are taken for what they are as in the wavefront form)
    const bool layout_ok = header == nullptr || *header == header_shift;
    int start = 0, end = 0;
    TileSource src = {};
    if(kBinned)
    {
        if(layout_ok)
            src = tile_source(lists, tile, ntx);
        start = src.start;
        end = src.end;
    }
    else if(layout_ok)
    {
        start = ranges[tile];
        end = ranges[tile + 1];
    }
    start = min(max(start, 0), k);
    end = min(max(end, 0), k);

    const bool inside = px.x < W && px.y < H;
    float pyf = inside ? (float)px.y + 0.5f : __builtin_nanf(""); // (NaN: stopped)
    float T = 1.0f;
    float red = 0.f, green = 0.f, blue = 0.f;
    int last = 0;
    if(tid == 0)
    {
        s_a[kTileBatch] = s_c[kTileBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kTileBatch] = make_float4(0.f, 0.f, __int_as_float(INT_MIN), 0.f);
    }

    const uint32_t tile_bits = kBinned ? tile_bits_of(src, lists.shift) << 16 : 0u;
    const int32_t* const keys = ids + k;
    int scan = start, left = end - start, seen = 0, no_skip = 0;
    int index_next = kBinned ? src.fine_base : start;
    int id_ahead = 0;
    if(!kBinned && tid < min(left, kTileBatch))
        id_ahead = ids[scan + tid];
    while(true)
    {
        // blocks with a live pixel
        const uint64_t live = __builtin_amdgcn_ballot_w64(pyf == pyf);
        uint32_t live_rows = 0;
#pragma unroll
        for(int r = 0; r < 4; ++r)
            live_rows |= (live >> (16 * r)) & 0xffffull ? 1u << block_of_row(r) : 0u;
        if(lane == 0)
            s_live[wave] = live_rows << first_block;
        __syncthreads(); // (and the last round's entries have been walked)
        const uint32_t live_blocks = __builtin_amdgcn_readfirstlane(s_live[0] | s_live[1] | s_live[2] | s_live[3]);
        if(live_blocks == 0 || left <= 0 || (kBinned && seen >= src.count))
            break;
        int id, batch;
        if(kBinned)
        {
            batch = tile_scan<1>(s_scan, s_queue, ids, keys, scan, left, no_skip, tile_bits, src.count - seen);
            seen += batch;
            id = tid < batch ? s_queue[tid] : 0;
        }
        else
        {
            batch = min(left, kTileBatch);
            id = id_ahead;
            scan += batch;
            left -= batch;
            if(tid < min(left, kTileBatch))
                id_ahead = ids[scan + tid]; // the next round's: in flight meanwhile
        }
        uint32_t reached = 0;
        float4 q0, q1, q2;
        float reach = 0.0f;
        if(tid < batch)
        {
            const float4* const rec = splats + 3 * (int64_t)min((uint32_t)id, last_id);
            q0 = rec[0], q1 = rec[1], q2 = rec[2];
            reach = reach_of(q1.w);
            reached = live_blocks & blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, tile_x, tile_y);
        }
        int staged;
        const int place = tile_place(s_counts, __builtin_amdgcn_ballot_w64(reached != 0), staged);
        if(reached != 0)
        {
            s_a[place] = make_float4(q0.x, q0.y, q1.x * -0.5f, q1.y);
            s_b[place] = make_float4(q1.z * 0.5f, q1.w,
                                     __int_as_float(reach_limit_fwd(q1.w, reach)), __int_as_float(index_next + tid));
            s_c[place] = q2;
            s_reach[place] = (uint16_t)reached;
        }
        index_next += batch;
        __syncthreads();
        if(live_rows == 0)
            continue; // (nothing left in this quadrant: the others' barriers are met)

        const int rounds = (build_lists(s_list, s_reach, staged, wave, first_block, lane) + kFwdAtOnce - 1) / kFwdAtOnce;
        const uint32_t* my_list = s_list + wave * kTileBatch + row * (kTileBatch / 4);
        for(int i = 0; i < rounds; ++i)
        {
            const uint32_t places = my_list[i];
            float4 A[kFwdAtOnce], B[kFwdAtOnce], C[kFwdAtOnce];
            float alpha[kFwdAtOnce], weight[kFwdAtOnce];
            uint64_t m_pass[kFwdAtOnce];
#pragma unroll
            for(int u = 0; u < kFwdAtOnce; ++u)
            {
                const uint32_t p = (places >> (8 * u)) & 0xffu;
                A[u] = s_a[p];
                B[u] = s_b[p];
                C[u] = s_c[p];
            }
            float Tn = T;
#pragma unroll
            for(int u = 0; u < kFwdAtOnce; ++u)
            {
#pragma clang fp contract(off)
                const ExponentX ex = exponent_x(A[u].z, A[u].w, pxf - A[u].x);
                const float dy = pyf - A[u].y;
                const float power = __builtin_fmaf(-__builtin_fmaf(B[u].x, dy, ex.bx), dy, ex.ax);
                m_pass[u] = __builtin_amdgcn_ballot_w64(__float_as_int(power) <= __float_as_int(B[u].z));
                const float full = fminf(kAlphaMax, B[u].y * __builtin_amdgcn_exp2f(power * kLog2E));
                alpha[u] = __builtin_amdgcn_inverse_ballot_w64(m_pass[u]) ? full : 0.0f;
            }
#pragma unroll
            for(int u = 0; u < kFwdAtOnce; ++u)
            {
                weight[u] = alpha[u] * Tn;
                Tn = __builtin_fmaf(-alpha[u], Tn, Tn);
            }
            if(__builtin_amdgcn_ballot_w64(Tn < 0.0001f) != 0)
            {
                // some pixel becomes opaque within these entries: once more, one entry after the other
                Tn = T;
#pragma unroll
                for(int u = 0; u < kFwdAtOnce; ++u)
                {
                    const float taken = pyf == pyf ? alpha[u] : 0.0f;
                    weight[u] = taken * Tn;
                    const float next = __builtin_fmaf(-taken, Tn, Tn);
                    const uint64_t m_low = __builtin_amdgcn_ballot_w64(next < 0.0001f);
                    const bool stop = __builtin_amdgcn_inverse_ballot_w64(m_low);
                    m_pass[u] &= __builtin_amdgcn_ballot_w64(pyf == pyf) & ~m_low;
                    weight[u] = stop ? 0.0f : weight[u];
                    Tn = stop ? Tn : next;
                    pyf = stop ? __builtin_nanf("") : pyf;
                }
                if(__builtin_amdgcn_ballot_w64(pyf == pyf) == 0)
                    i = rounds; // no pixel left
            }
            T = Tn;
#pragma unroll
            for(int u = 0; u < kFwdAtOnce; ++u)
            {
                red = __builtin_fmaf(weight[u], C[u].x, red);
                green = __builtin_fmaf(weight[u], C[u].y, green);
                blue = __builtin_fmaf(weight[u], C[u].z, blue);
                last = __builtin_amdgcn_inverse_ballot_w64(m_pass[u]) ? __float_as_int(B[u].w) : last;
            }
        }
    }

    const bool broken = !layout_ok || (sort_flag_a && *sort_flag_a) || (sort_flag_b && *sort_flag_b);
    if(inside)
    {
        const int64_t pix = (int64_t)px.y * W + px.x;
        final_T[pix] = T;
        final_idx[pix] = last;
        store_pixel(image, pix, (int64_t)W * H, red, green, blue, T, broken, bg, planar);
    }
    if(kBinned && layout_ok && tid < 8)
    {
        // (as in the wavefront form, which speaks for the whole tile too)
        lists.walk[(int64_t)tile * 8 + tid] = tid == 0 ? scan : (tid == 1 ? seen : (tid & 1 ? 0 : -1));
    }
    if(prep_zeros)
        zero_grads_share(prep, prep_count, blockIdx.x, gridDim.x, tid, kTileThreads);
    else
        prepare_grads_share(splats, prep, prep_count, prep_marks, blockIdx.x, gridDim.x, tid, kTileThreads);
}

// -----------------------------------------------------------------------------------------
// the same for images of very few tiles: a workgroup of sixteen wavefronts per tile
// -----------------------------------------------------------------------------------------
// Up to a few hundred tiles the chip holds every wavefront of the form above with slots to spare, and a launch lasts as long
// as its longest tile: 72000 cycles at 256 tiles of 325 entries, 40000 of them the walk (190 an entry, of
// which a pixel's transmittance needs one multiply-add), the rest four rounds of 248 entries, each with its gather's
// latency and its barriers.  Here each 4x4 block has a wavefront, each of its pixels a quad of lanes: the
// four lanes work out four entries' alphas side by side, hand them to each other, take the same four steps of
// the transmittance (the bits of one lane that takes one entry after the other), and each adds its own entry's colour; and up to
// 960 entries are staged in one round.  us of the kernel, four wavefronts -> sixteen: 2 K Gaussians at 64x64 23.6 -> 13.6, 16 K at
// 256x256 35.5 -> 21.2 (1024 tiles of 50 K at 512x512: 32.7 -> 51.1).  Whole forwards of the four kinds of scenes above, and of a mixed one
// that is nearer:
//   64 tiles    46 -> 45, 67 -> 60, 57 -> 53, 66 -> 57, 84 -> 71
//   169 tiles   56 -> 54, 95 -> 92, 92 -> 89, 76 -> 68, 116 -> 102
//   256 tiles   68 -> 66, 107 -> 102, 99 -> 96, 90 -> 85, 140 -> 121
//   400 tiles   85 -> 85, 118 -> 116, 103 -> 105, 124 -> 132
// and at 169 and 256 tiles 40 more of 2 K to 1 M Gaussians, opaque, mixed, faint (322 -> 241) and large (248 -> 246): none is slower
// by more than its runs differ.
// The line lies at 256, a tile for each compute unit; beyond it some units get two.
// Up to 64 tiles a workgroup for each quadrant, sixteen wavefronts to find and stage its entries and four to walk, one to a SIMD.  us of the
// kernel, a workgroup for each tile -> four: 16 tiles of 60 K faint Gaussians 258 -> 176, of 400 K mixed ones 94 -> 52, 36 tiles 150 -> 104 and 62 -> 38, 64
// tiles 100 -> 70 and 45 -> 31.
// Lists per tile only (images of so few tiles have no others unless the caller asks).
constexpr int kWideBatch = 960; // (two workgroups' records and lists fit a compute unit's LDS)
constexpr int kWideThreads = 1024;
constexpr int kWideWaves = kWideThreads / DSX_WAVE;
static_assert(kWideWaves == kQuads, "a wavefront for each block");

// Lists that nobody made: a forward without a backward, of few tiles and not too many Gaussians, needs none but each tile's own
// entries in order, and a workgroup finds them faster than a depth order, pairs and their partition can bring them (and the
// host need not wait for the pairs' number): it looks at all rectangles, takes those that cover its tile, sorts them
// by depth and index in LDS, and blends them.  Where more than kOwnMost do, it takes them in windows, nearest first, each found by
// counting the rest into bins.  Each colour is then a sum in other parts; all else has the same bits.  Up to 960 entries (a round) take the
// short way: a thread for each fetches its record and its depth together, drops it if it reaches no block of the workgroup's, and puts it where it belongs
// among the others.  us of a forward, found, sorted and then staged -> this -> and by quadrants up to 64 tiles: 2 K Gaussians at 64x64 25.5 -> 22.7 -> 18.7, 2 K
// at 128x128 19.8 -> 17.2 -> 16.2, 6 K at 128x128 27.0 -> 23.8 -> 21.2, 10 K at 208x208 29.1 -> 26.9, 16 K at 256x256 37.4 -> 35.1.
struct OwnLists
{
    const uint32_t* depth_keys; // by Gaussian, as the projection leaves them
    const uint2* rects;
    int n;
    int last_tile; // of the image
};
// us of a whole forward, 64x64 / 128x128 / 208x208 / 256x256, four kinds of scenes (small, mixed, faint, large), with lists -> without:
//   6 K Gaussians   62, 63, 57, 63 -> 47, 48, 42, 46 / 43, 45, 42, 55 -> 25, 28, 23, 36 / 41, 44, 40, 53 -> 22, 24, 21, 34 / 45, 48, 45, 61 -> 21, 23, 20, 33
//   10 K            81, 84, 72, 66 -> 69, 73, 61, 57 / 52, 55, 49, 56 -> 36, 38, 33, 40 / 45, 49, 43, 57 -> 27, 30, 26, 37 / 48, 54, 49, 67 -> 25, 29, 24, 36
//   16 K            89, 112, 97, 62 -> 103, 144, 111, 61 / 61, 68, 57, 56 -> 45, 53, 42, 50 / 51, 58, 50, 58 -> 33, 40, 32, 38 / 54, 63, 52, 66 -> 30, 37, 28, 37
//   24 K            (slower) / 74, 86, 69, 58 -> 59, 72, 56, 59 / 62, 71, 57, 61 -> 45, 53, 40, 60 / 64, 75, 61, 72 -> 40, 49, 37, 58
//   32 K            (slower) / 77, 90, 81, 60 -> 65, 120, 71, 68 / 68, 81, 65, 63 -> 53, 66, 50, 68 / 72, 85, 68, 73 -> 49, 60, 44, 66
// Without, since a round's entries are tested and placed in one go and quadrants have workgroups:
//   6 K             39, 41, 36, 33 / 21, 22, 21, 28 / 21, 24, 21, 33 / 20, 22, 20, 33
//   10 K            53, 53, 54, 42 / 32, 36, 32, 41 / 27, 32, 27, 44 / 25, 30, 26, 36
//   16 K            70, 68, 85, 60 / 56, 60, 56, 55 / 39, 42, 39, 51 / 32, 41, 37, 51
// 2 K at 64x64 40 -> 24 -> 18.  What ends it are the windows, each of which costs another three or four looks at everything: the line of
// 9000 Gaussians and a hundred more for each tile lies below where the first kind of scene loses.
constexpr int kOwnGaussians = 9000, kOwnGaussiansPerTile = 100;
constexpr int kOwnMost = 4096; // entries of a window
constexpr int kOwnBins = 4096;
constexpr int kOwnBinBits = 12;
static_assert(kOwnBins == 4 * kWideThreads && kOwnMost == 4 * kWideThreads, "what the threads take");
constexpr int kOwnGroupMost = 64; // entries in one bin that are compared with each other one by one
// The same on the short way, where a thread has one entry.  Beyond, all are sorted.  us of a forward, compared whatever their number -> sorted
// beyond 64 / 128 / 256: equal depths, 1200 Gaussians at 64x64 19.1 -> 22.4 / 19.0 / 19.0, 3500 at 64x64 31.2 -> 27.0 / 27.1 / 31.4, 12 K at
// 176x160 58.1 -> 37.9 / 37.9 / 40.6, 16 K at 256x256 57.3 -> 40.0 / 39.8 / 42.0; two planes, 12 K 53.8 -> 39.9 / 40.0 / 44.3.
constexpr int kOwnCrowd = 128;

// The entries of one tile (sx >= 0), or, one copy for each tile that they touch, all those of negative depth (see TileSource)
struct OwnSource
{
    int sx, sy;
    __device__ __forceinline__ int copies(uint2 r) const
    {
        const uint32_t w = r.y & 0xffffu, h = (r.y >> 16) & 0x7fffu;
        if(sx < 0)
            return (int)r.y < 0 ? (int)(w * h) : 0;
        return (int)r.y >= 0 && (uint32_t)sx - (r.x & 0xffffu) < w && (uint32_t)sy - (r.x >> 16) < h ? 1 : 0;
    }
};

// What finding and sorting a window's entries takes of the LDS
struct OwnScratch
{
    uint64_t numbers[kOwnMost]; // depth key, index
    uint64_t binned[kOwnMost];
    uint32_t hist[kOwnBins];
};
struct OwnShared
{
    uint32_t tot[kWideWaves];
    uint32_t found[3];
    uint32_t taken, most, nearest, farthest;
    uint32_t reaching, reaching_near, reaching_far; // of the short way: how many, and their extreme keys (the nearest one's complement)
    uint32_t crowded;                               // and does a bin hold more than kOwnCrowd of them?
    int highest;
};

// f(first index, this thread's eight rectangles, source) for all of them, eight thousand at a time (the next ones asked for meanwhile: the
// registers spill, and forwards of 12 K to 30 K Gaussians whose tiles have more than a round's entries take 39.6 -> 38.5 us at 176x160,
// 42.5 -> 40.6, 41.4 -> 39.7 and 43.2 -> 41.3 at 256x256 without)
template <typename F>
__device__ __forceinline__ void own_for_all(const OwnLists& L, const OwnSource& src, F f)
{
    for(int i0 = 0; i0 < L.n; i0 += 8 * kWideThreads)
    {
        uint2 r[8];
#pragma unroll
        for(int b = 0; b < 8; ++b)
        {
            const int i = i0 + b * kWideThreads + (int)threadIdx.x;
            r[b] = i < L.n ? L.rects[i] : make_uint2(0u, 0u);
        }
        f(i0, r, src);
    }
}

// The source's entries with numbers in [low, high): their indices (as far as there is room), in any order, where own_found has them;
// returns how many there are.
__device__ __forceinline__ const uint32_t* own_found(const OwnScratch& S) { return reinterpret_cast<const uint32_t*>(S.binned); }
__device__ __forceinline__ int own_find(const OwnLists& L, const OwnSource& src, OwnScratch& S, OwnShared& sh, uint64_t low, uint64_t high,
                                        bool everything)
{
    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1);
    __syncthreads();
    if(tid == 0)
    {
        sh.taken = 0;
        sh.nearest = 0xffffffffu;
        sh.farthest = 0;
        sh.reaching = sh.reaching_near = sh.reaching_far = sh.crowded = 0;
    }
    __syncthreads();
    int highest = 0;
    uint32_t* const ids = reinterpret_cast<uint32_t*>(S.binned);
    own_for_all(L, src, [&](int i0, const uint2 (&r)[8], const OwnSource& from) {
        uint32_t mine = 0, copies[8];
#pragma unroll
        for(int b = 0; b < 8; ++b)
        {
            // (columns and rows behind the rectangle's last ones, packed: the largest is the highest tile's; below zero behind the camera)
            highest = max(highest, (int)(r[b].x + r[b].y));
            copies[b] = (uint32_t)from.copies(r[b]);
            if(!everything && copies[b])
            {
                const uint64_t number = (uint64_t)L.depth_keys[i0 + b * kWideThreads + tid] << 32 | (uint32_t)(i0 + b * kWideThreads + tid);
                copies[b] = number >= low && number < high ? copies[b] : 0u;
            }
            mine += copies[b];
        }
        if(__builtin_amdgcn_ballot_w64(mine != 0) == 0)
            return;
        const uint32_t incl = wave_incl_scan_u32(mine);
        uint32_t at = 0;
        if(lane == DSX_WAVE - 1)
            at = atomicAdd(&sh.taken, incl);
        at = (uint32_t)__builtin_amdgcn_readlane((int)at, DSX_WAVE - 1) + incl - mine;
#pragma unroll
        for(int b = 0; b < 8; ++b)
            for(uint32_t c = 0; c < copies[b]; ++c, ++at)
                if(at < (uint32_t)kOwnMost)
                    ids[at] = (uint32_t)(i0 + b * kWideThreads + tid);
    });
    if(everything)
    {
        highest = (int)wave_incl_max_scan((uint32_t)highest); // (it begins with zero)
        if(lane == DSX_WAVE - 1)
            atomicMax(&sh.highest, highest);
    }
    __syncthreads();
    return (int)__builtin_amdgcn_readfirstlane((int)sh.taken);
}

// the numbers of `total` found entries, and their nearest and farthest depth keys
__device__ __forceinline__ void own_numbers(const OwnLists& L, OwnScratch& S, OwnShared& sh, int total)
{
    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), count = min(total, kOwnMost);
    const uint32_t* const ids = own_found(S);
    uint32_t nearest = 0, farthest = 0; // (the nearest one's complement)
#pragma unroll
    for(int b = 0; b < kOwnMost / kWideThreads; ++b)
    {
        const int at = b * kWideThreads + tid;
        if(at < count)
        {
            const uint32_t id = ids[at], key = L.depth_keys[id];
            S.numbers[at] = (uint64_t)key << 32 | id;
            nearest = max(nearest, ~key);
            farthest = max(farthest, key);
        }
    }
    nearest = wave_incl_max_scan(nearest);
    farthest = wave_incl_max_scan(farthest);
    if(lane == DSX_WAVE - 1)
    {
        atomicMin(&sh.nearest, ~nearest);
        atomicMax(&sh.farthest, farthest);
    }
    __syncthreads();
}

__device__ __forceinline__ int number_bits(uint64_t v)
{
    return v ? 64 - __builtin_clzll(v) : 0;
}

// exclusive sums of the histogram's bins in place of their counts
__device__ __forceinline__ void own_scan(uint32_t* hist, OwnShared& sh)
{
    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), wave = tid / DSX_WAVE;
    __syncthreads();
    uint4* const mine = reinterpret_cast<uint4*>(hist) + tid;
    const uint4 c = *mine;
    const uint32_t sum = c.x + c.y + c.z + c.w, incl = wave_incl_scan_u32(sum);
    if(lane == DSX_WAVE - 1)
        sh.tot[wave] = incl;
    __syncthreads();
    const uint32_t at = sum_of_waves_before<kWideWaves>(sh.tot, wave) + incl - sum;
    *mine = make_uint4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
    __syncthreads();
}

// where a number's bin begins to matter: the range of keys in 2^kOwnBinBits bins
struct OwnBinning
{
    uint64_t from;
    int shift;
    __device__ __forceinline__ OwnBinning(uint32_t nearest, uint32_t farthest)
        : from((uint64_t)nearest << 32),
          shift(max(number_bits(((uint64_t)(farthest - nearest) << 32) | 0xffffffffull) - kOwnBinBits, 0))
    {
    }
    __device__ __forceinline__ uint32_t operator()(uint64_t number) const { return (uint32_t)((number - from) >> shift); }
};

// scratch.numbers [0, count), of depth keys nearest to farthest, in order: their indices into `ids`
__device__ __forceinline__ void own_sort(OwnScratch& S, OwnShared& sh, int count, uint32_t* ids)
{
    constexpr int kItems = kOwnMost / kWideThreads;
    const int tid = threadIdx.x;
    const OwnBinning bin_of(sh.nearest, sh.farthest);
    reinterpret_cast<uint4*>(S.hist)[tid] = make_uint4(0u, 0u, 0u, 0u);
    if(tid == 0)
        sh.most = 0;
    __syncthreads();
    uint64_t mine[kItems];
    uint32_t bin[kItems], nth[kItems], most = 0;
#pragma unroll
    for(int b = 0; b < kItems; ++b)
    {
        const int at = b * kWideThreads + tid;
        bin[b] = nth[b] = 0;
        mine[b] = ~0ull;
        if(at < count)
        {
            mine[b] = S.numbers[at];
            bin[b] = bin_of(mine[b]);
            nth[b] = atomicAdd(&S.hist[bin[b]], 1u);
            most = max(most, nth[b]);
        }
    }
    if(__builtin_amdgcn_ballot_w64(most >= kOwnGroupMost) != 0 && (tid & (DSX_WAVE - 1)) == 0)
        sh.most = 1;
    own_scan(S.hist, sh);
    if(__builtin_amdgcn_readfirstlane((int)sh.most) == 0)
    {
        uint32_t start[kItems], end[kItems];
#pragma unroll
        for(int b = 0; b < kItems; ++b)
            if(b * kWideThreads + tid < count)
            {
                start[b] = S.hist[bin[b]];
                end[b] = bin[b] + 1 < kOwnBins ? S.hist[bin[b] + 1] : (uint32_t)count;
                S.binned[start[b] + nth[b]] = mine[b];
            }
        __syncthreads();
#pragma unroll
        for(int b = 0; b < kItems; ++b)
            if(b * kWideThreads + tid < count)
            {
                uint32_t r = start[b];
                for(uint32_t j = start[b]; j < end[b]; ++j) // (copies of one entry among them)
                    r += S.binned[j] < mine[b] || (S.binned[j] == mine[b] && j < start[b] + nth[b]) ? 1u : 0u;
                ids[r] = (uint32_t)mine[b];
            }
    }
    else
    {
        // many depths alike: a bitonic sort
        int size = kWideThreads;
        while(size < count)
            size *= 2;
        for(int at = tid; at < size; at += kWideThreads)
            S.binned[at] = at < count ? S.numbers[at] : ~0ull;
        for(int k = 2; k <= size; k *= 2)
            for(int j = k / 2; j > 0; j /= 2)
            {
                __syncthreads();
                for(int e = tid; e < size / 2; e += kWideThreads)
                {
                    const int i = 2 * e - (e & (j - 1)), l = i + j;
                    const uint64_t u = S.binned[i], v = S.binned[l];
                    if((u > v) == ((i & k) == 0))
                    {
                        S.binned[i] = v;
                        S.binned[l] = u;
                    }
                }
            }
        __syncthreads();
        for(int at = tid; at < count; at += kWideThreads)
            ids[at] = (uint32_t)S.binned[at];
    }
    __syncthreads();
}

// Where each thread's word stands among all of them, which differ (or are ~0: their places are nobody's) and hold their thread's number in
// the last ten bits: for depths that are alike.  A bitonic sort whose steps within a wavefront need no barrier, 8 us.
__device__ __forceinline__ uint32_t own_places(uint64_t word, uint64_t* words, uint32_t* places)
{
    static_assert(kWideThreads == 1 << 10 && kOwnGaussians + kOwnGaussiansPerTile * kFwdWideUpTo < 1 << 22, "index and thread in 32 bits");
    const int tid = threadIdx.x;
#pragma unroll 1
    for(int k = 2; k <= kWideThreads; k *= 2)
#pragma unroll 1
        for(int j = k / 2; j > 0; j /= 2)
        {
            uint64_t other;
            if(j >= DSX_WAVE)
            {
                __syncthreads();
                words[tid] = word;
                __syncthreads();
                other = words[tid ^ j];
            }
            else
                other = (uint64_t)__shfl_xor((unsigned long long)word, j, DSX_WAVE);
            const bool smaller = ((tid & j) == 0) == ((tid & k) == 0);
            word = (word < other) == smaller ? word : other;
        }
    if(word != ~0ull)
        places[(uint32_t)word & (kWideThreads - 1)] = (uint32_t)tid;
    __syncthreads();
    return places[tid];
}

// Of the source's numbers from `low` on, more than kOwnMost: a border that leaves half as many to kOwnMost of them in front.
__device__ __forceinline__ uint64_t own_border(const OwnLists& L, const OwnSource& src, OwnScratch& S, OwnShared& sh, uint64_t low)
{
    constexpr uint32_t kWanted = kOwnMost / 2;
    const int tid = threadIdx.x;
    uint64_t base = low;
    uint32_t before = 0; // numbers in [low, base)
    int wide = number_bits(~low), shift = max(wide - kOwnBinBits, 0);
    while(true)
    {
        __syncthreads();
        reinterpret_cast<uint4*>(S.hist)[tid] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        own_for_all(L, src, [&](int i0, const uint2 (&r)[8], const OwnSource& from) {
#pragma unroll
            for(int b = 0; b < 8; ++b)
            {
                const int copies = from.copies(r[b]), i = i0 + b * kWideThreads + tid;
                if(copies)
                {
                    const uint64_t number = (uint64_t)L.depth_keys[i] << 32 | (uint32_t)i, d = number - base;
                    if(number >= base && (wide >= 64 || (d >> wide) == 0))
                        atomicAdd(&S.hist[(uint32_t)(d >> shift)], (uint32_t)copies);
                }
            }
        });
        __syncthreads();
        const uint4 c = reinterpret_cast<const uint4*>(S.hist)[tid];
        const uint32_t count[4] = {c.x, c.y, c.z, c.w};
        own_scan(S.hist, sh);
        // the first bin border with kWanted numbers or more in front
#pragma unroll
        for(int u = 0; u < 4; ++u)
        {
            const uint32_t at = before + S.hist[4 * tid + u];
            if(at < kWanted && kWanted <= at + count[u])
            {
                sh.found[0] = 4 * tid + u;
                sh.found[1] = at;
                sh.found[2] = at + count[u];
            }
        }
        __syncthreads();
        const uint32_t bin = __builtin_amdgcn_readfirstlane((int)sh.found[0]);
        const uint32_t front = __builtin_amdgcn_readfirstlane((int)sh.found[1]), behind = __builtin_amdgcn_readfirstlane((int)sh.found[2]);
        if(behind <= (uint32_t)kOwnMost || shift == 0) // (copies of one entry: a tile each of an image of few)
            return base + ((uint64_t)(bin + 1) << shift);
        base += (uint64_t)bin << shift;
        before = front;
        wide = shift;
        shift = max(wide - kOwnBinBits, 0);
    }
}

template <bool kOwn>
__global__ __launch_bounds__(kWideThreads) void blend_fwd_wide_kernel(const int32_t* __restrict__ ranges, const int32_t* __restrict__ ids,
                                                                      const float4* __restrict__ splats,
                                                                      float* __restrict__ image, float* __restrict__ final_T,
                                                                      int32_t* __restrict__ final_idx, int W, int H, int ntx,
                                                                      uint32_t last_id, int k,
                                                                      const int32_t* __restrict__ header, int header_shift,
                                                                      const uint32_t* __restrict__ sort_flag_a,
                                                                      const uint32_t* __restrict__ sort_flag_b,
                                                                      float4* __restrict__ prep, int64_t prep_count,
                                                                      uint8_t* __restrict__ prep_marks, int prep_zeros,
                                                                      const float* __restrict__ bg, int planar, int split, const OwnLists own)
{
    // (arrays as in the other forms; eight places more than an entry has blocks: the lists' ends name nobody's place, read ahead)
    struct Staged
    {
        float4 a[kWideBatch + 1], b[kWideBatch + 1], c[kWideBatch + 1];
        uint16_t list[kWideWaves][kWideBatch + 8];
        uint16_t reach[kWideBatch];
    };
    union Memory // (own lists: a window's entries are found and sorted before they are staged)
    {
        Staged staged;
        OwnScratch scratch;
    };
    __shared__ __attribute__((aligned(16))) char s_memory[kOwn ? sizeof(Memory) : sizeof(Staged)];
    __shared__ uint32_t s_own_ids[kOwn ? kOwnMost : 1];
    __shared__ __attribute__((aligned(16))) OwnShared s_own;
    Staged& staged_lds = *reinterpret_cast<Staged*>(s_memory);
    float4 *const s_a = staged_lds.a, *const s_b = staged_lds.b, *const s_c = staged_lds.c;
    uint16_t* const s_reach = staged_lds.reach;
    uint16_t (*const s_list)[kWideBatch + 8] = staged_lds.list;
    __shared__ int s_counts[kWideWaves];
    __shared__ uint32_t s_live[kWideWaves];

    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), slot = lane & 3, pixel = lane >> 2;
    const int wave = __builtin_amdgcn_readfirstlane(tid / DSX_WAVE);
    // (split: a workgroup for each quadrant of a tile, of which four wavefronts have a block and the others help to find and stage)
    const int tile = split ? blockIdx.x / 4 : blockIdx.x, quadrant = blockIdx.x % 4;
    const bool has_block = !split || wave < 4;
    const int block = split ? first_block_of(quadrant) + block_of_row(wave & 3) : wave;
    const int x0 = (tile % ntx) * kTile, y0 = (tile / ntx) * kTile;
    const int x = x0 + 4 * (block & 3) + (pixel & 3), y = y0 + 4 * (block >> 2) + (pixel >> 2);
    const float pxf = (float)x + 0.5f;

    // (positions and layout are taken for what they are as in the wavefront form)
    const bool layout_ok = kOwn || header == nullptr || *header == header_shift;
    int scan = 0, end = 0;
    if(!kOwn && layout_ok)
    {
        scan = min(max(ranges[tile], 0), k);
        end = min(max(ranges[tile + 1], 0), k);
    }
    int left = end - scan;

    const bool inside = has_block && x < W && y < H;
    float pyf = inside ? (float)y + 0.5f : __builtin_nanf(""); // (NaN: stopped)
    float T = 1.0f, red = 0.f, green = 0.f, blue = 0.f;        // (the colours of this lane's entries)
    int last = 0;

    // this wavefront's list of what is staged, and its walk
    auto blend_staged = [&](int staged) {
        uint16_t* const list = s_list[wave];
        int length = 0;
        for(int first = 0; first < staged; first += DSX_WAVE)
        {
            const int at = first + lane;
            const uint64_t mine = __builtin_amdgcn_ballot_w64(at < staged && ((uint32_t)s_reach[min(at, kWideBatch - 1)] >> block & 1) != 0);
            if(__builtin_amdgcn_inverse_ballot_w64(mine))
                list[length + bits_below_lane(mine)] = (uint16_t)at;
            length += __popcll(mine);
        }
        if(lane < 8)
            list[length + lane] = kWideBatch;

        struct Entry
        {
            float4 A, B, C;
        };
        auto fetch = [&](int at) { return Entry{s_a[at], s_b[at], s_c[at]}; };
        Entry next = fetch(list[slot]);
        int after = list[4 + slot];
        for(int i = 0; i < length; i += 4)
        {
            const Entry e = next;
            next = fetch(after);
            after = list[min(i + 8, length + 4) + slot];
            float alpha;
            uint64_t m_pass;
            {
#pragma clang fp contract(off)
                const ExponentX ex = exponent_x(e.A.z, e.A.w, pxf - e.A.x);
                const float dy = pyf - e.A.y;
                const float power = __builtin_fmaf(-__builtin_fmaf(e.B.x, dy, ex.bx), dy, ex.ax);
                m_pass = __builtin_amdgcn_ballot_w64(__float_as_int(power) <= __float_as_int(e.B.z));
                const float full = fminf(kAlphaMax, e.B.y * __builtin_amdgcn_exp2f(power * kLog2E));
                alpha = __builtin_amdgcn_inverse_ballot_w64(m_pass) ? full : 0.0f;
            }
            const float alphas[4] = {quad_lane<0x00>(alpha), quad_lane<0x55>(alpha), quad_lane<0xAA>(alpha), quad_lane<0xFF>(alpha)};
            const float T1 = __builtin_fmaf(-alphas[0], T, T), T2 = __builtin_fmaf(-alphas[1], T1, T1);
            const float T3 = __builtin_fmaf(-alphas[2], T2, T2), T4 = __builtin_fmaf(-alphas[3], T3, T3);
            float before = slot & 2 ? (slot & 1 ? T3 : T2) : (slot & 1 ? T1 : T);
            float Tn = T4;
            if(__builtin_amdgcn_ballot_w64(T4 < 0.0001f) != 0)
            {
                // some pixel becomes opaque within these entries: once more, each lane up to where its pixel stops
                Tn = T;
                bool stopped = pyf != pyf, counts = !stopped;
#pragma unroll
                for(int u = 0; u < 4; ++u)
                {
                    before = slot == u ? Tn : before;
                    const float further = __builtin_fmaf(-alphas[u], Tn, Tn);
                    stopped = stopped || further < 0.0001f;
                    Tn = stopped ? Tn : further;
                    counts = slot == u ? !stopped : counts;
                }
                pyf = stopped ? __builtin_nanf("") : pyf;
                m_pass &= __builtin_amdgcn_ballot_w64(counts);
                alpha = counts ? alpha : 0.0f;
                if(__builtin_amdgcn_ballot_w64(pyf == pyf) == 0)
                    i = length; // no pixel left
            }
            T = Tn;
            const float weight = alpha * before;
            red = __builtin_fmaf(weight, e.C.x, red);
            green = __builtin_fmaf(weight, e.C.y, green);
            blue = __builtin_fmaf(weight, e.C.z, blue);
            last = __builtin_amdgcn_inverse_ballot_w64(m_pass) ? __float_as_int(e.B.w) : last;
        }
    };

    if(tid < kWideWaves)
        s_live[tid] = 0;
    if(!kOwn) // (own lists: there are barriers before it is written)
        __syncthreads();
    // own lists: whose entries (as tile_source has it), all of them if they fit a window
    OwnSource src = {tile % ntx, tile / ntx};
    OwnScratch& scratch = *reinterpret_cast<OwnScratch*>(s_memory);
    uint64_t low = 0;
    int remaining = 0;
    if(kOwn)
    {
        if(tid == 0)
            s_own.highest = 0;
        remaining = own_find(own, src, scratch, s_own, 0, 0, true);
        const int highest = __builtin_amdgcn_readfirstlane(s_own.highest); // (0: no tile is occupied)
        const int last_x = (highest & 0xffff) - 1, last_y = (highest >> 16) - 1;
        const bool occupied = highest > 0, mine = occupied && src.sx == last_x && src.sy == last_y;
        if(tile == own.last_tile)
        {
            if(!mine)
            {
                src.sx = occupied ? last_x : -1;
                src.sy = occupied ? last_y : -1;
                remaining = own_find(own, src, scratch, s_own, 0, 0, true);
            }
        }
        else if(mine)
            remaining = 0;
    }
    if(kOwn && remaining > 0 && remaining <= kWideBatch)
    {
        // A thread for each: what reaches no block is dropped before it is sorted, and the rest goes to its place at once.  (In the
        // lists' memory: the bins, and the numbers by bin.)
        uint32_t* const hist = reinterpret_cast<uint32_t*>(s_list);
        uint64_t* const binned = reinterpret_cast<uint64_t*>(hist + kOwnBins);
        static_assert(kOwnBins * 4 + kWideThreads * 8 <= sizeof(staged_lds.list) && offsetof(Staged, list) % 16 == 0, "room");
        static_assert(offsetof(OwnScratch, binned) + kWideThreads * 4 <= offsetof(Staged, list), "the bins leave the found indices alone");
        uint32_t reached = 0, key = 0;
        uint64_t number = 0;
        float4 q0, q1, q2;
        float reach = 0.0f;
        if(tid < remaining)
        {
            const uint32_t id = own_found(scratch)[tid];
            const float4* const rec = splats + 3 * (int64_t)id;
            q0 = rec[0], q1 = rec[1], q2 = rec[2];
            key = own.depth_keys[id];
            reach = reach_of(q1.w);
            reached = blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, (float)x0 + 0.5f, (float)y0 + 0.5f);
            if(split)
                reached &= 0x33u << first_block_of(quadrant);
            number = (uint64_t)key << 32 | id;
        }
        reinterpret_cast<uint4*>(hist)[tid] = make_uint4(0u, 0u, 0u, 0u);
        const uint32_t near = wave_incl_max_scan(reached ? ~key : 0u), far = wave_incl_max_scan(reached ? key : 0u);
        const int reaching = __popcll(__builtin_amdgcn_ballot_w64(reached != 0));
        if(lane == DSX_WAVE - 1 && reaching)
        {
            atomicAdd(&s_own.reaching, (uint32_t)reaching);
            atomicMax(&s_own.reaching_near, near);
            atomicMax(&s_own.reaching_far, far);
        }
        __syncthreads();
        const int count = __builtin_amdgcn_readfirstlane((int)s_own.reaching);
        const OwnBinning bin_of(~s_own.reaching_near, s_own.reaching_far);
        uint32_t bin = 0, nth = 0;
        if(reached)
        {
            bin = bin_of(number);
            nth = atomicAdd(&hist[bin], 1u);
            if(nth >= (uint32_t)kOwnCrowd)
                s_own.crowded = 1;
        }
        own_scan(hist, s_own);
        uint32_t place = 0;
        if(__builtin_amdgcn_readfirstlane((int)s_own.crowded) == 0)
        {
            uint32_t start = 0, end = 0;
            if(reached)
            {
                start = hist[bin];
                end = bin + 1 < kOwnBins ? hist[bin + 1] : (uint32_t)count;
                binned[start + nth] = number;
            }
            __syncthreads();
            place = start;
            for(uint32_t j = start; j < end; ++j) // (copies of one entry among them)
                place += binned[j] < number || (binned[j] == number && j < start + nth) ? 1u : 0u;
        }
        else
            place = own_places(reached ? (uint64_t)key << 32 | (uint32_t)number << 10 | (uint32_t)tid : ~0ull, binned, hist);
        if(reached)
        {
            s_a[place] = make_float4(q0.x, q0.y, q1.x * -0.5f, q1.y);
            s_b[place] = make_float4(q1.z * 0.5f, q1.w, __int_as_float(reach_limit_fwd(q1.w, reach)), 0.0f);
            s_c[place] = q2;
            s_reach[place] = (uint16_t)reached;
        }
        if(tid == 0)
        {
            s_a[kWideBatch] = s_c[kWideBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
            s_b[kWideBatch] = make_float4(0.f, 0.f, __int_as_float(INT_MIN), 0.f);
        }
        __syncthreads();
        if(has_block)
            blend_staged(count);
        remaining = 0;
    }
    bool first_window = true;
    while(true) // (windows; one of lists that are there)
    {
        if(kOwn)
        {
            if(remaining <= 0)
                break;
            int count = remaining;
            if(!first_window || remaining > kOwnMost)
            {
                const uint64_t high = remaining > kOwnMost ? own_border(own, src, scratch, s_own, low) : ~0ull;
                count = min(own_find(own, src, scratch, s_own, low, high, false), kOwnMost);
                low = high;
            }
            own_numbers(own, scratch, s_own, count);
            own_sort(scratch, s_own, count, s_own_ids);
            remaining -= count;
            first_window = false;
            scan = 0;
            left = count;
        }
        if(tid == 0)
        {
            s_a[kWideBatch] = s_c[kWideBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
            s_b[kWideBatch] = make_float4(0.f, 0.f, __int_as_float(INT_MIN), 0.f);
        }
        const int32_t* const list_ids = kOwn ? reinterpret_cast<const int32_t*>(s_own_ids) : ids;
        int id_ahead = 0;
        if(tid < min(left, kWideBatch))
            id_ahead = list_ids[scan + tid];
        while(true)
        {
            const bool live = __builtin_amdgcn_ballot_w64(pyf == pyf) != 0;
            if(lane == 0 && has_block)
                s_live[block] = live;
            __syncthreads(); // (and the last round's entries have been walked)
            const uint32_t live_blocks = (uint32_t)__builtin_amdgcn_ballot_w64(lane < kWideWaves && s_live[lane & (kWideWaves - 1)] != 0);
            if(live_blocks == 0)
                remaining = 0;
            if(live_blocks == 0 || left <= 0)
                break;
            const int batch = min(left, kWideBatch), id = id_ahead, index_next = scan;
            scan += batch;
            left -= batch;
            if(tid < min(left, kWideBatch))
                id_ahead = list_ids[scan + tid]; // the next round's: in flight meanwhile
            uint32_t reached = 0;
            float4 q0, q1, q2;
            float reach = 0.0f;
            if(tid < batch)
            {
                const float4* const rec = splats + 3 * (int64_t)min((uint32_t)id, last_id);
                q0 = rec[0], q1 = rec[1], q2 = rec[2];
                reach = reach_of(q1.w);
                reached = live_blocks & blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, (float)x0 + 0.5f, (float)y0 + 0.5f);
            }
            const uint64_t m = __builtin_amdgcn_ballot_w64(reached != 0);
            if(lane == 0)
                s_counts[wave] = __popcll(m);
            __syncthreads();
            int staged = 0, place = bits_below_lane(m);
#pragma unroll
            for(int w = 0; w < kWideWaves; ++w)
            {
                const int c = s_counts[w];
                place += w < wave ? c : 0;
                staged += c;
            }
            staged = __builtin_amdgcn_readfirstlane(staged);
            if(reached != 0)
            {
                s_a[place] = make_float4(q0.x, q0.y, q1.x * -0.5f, q1.y);
                s_b[place] = make_float4(q1.z * 0.5f, q1.w, __int_as_float(reach_limit_fwd(q1.w, reach)),
                                         __int_as_float(index_next + tid));
                s_c[place] = q2;
                s_reach[place] = (uint16_t)reached;
            }
            __syncthreads();
            if(!live)
                continue; // (nothing left in this block: the others' barriers are met)

            blend_staged(staged);
        }
        if(!kOwn)
            break;
    }

    const bool broken = !layout_ok || (sort_flag_a && *sort_flag_a) || (sort_flag_b && *sort_flag_b);
    // the quad's four parts of the colour, and the last of its last entries
    auto sum = [](float v) {
        v += quad_lane<0xB1>(v);
        return v + quad_lane<0x4E>(v);
    };
    red = sum(red), green = sum(green), blue = sum(blue);
    last = max(last, __float_as_int(quad_lane<0xB1>(__int_as_float(last))));
    last = max(last, __float_as_int(quad_lane<0x4E>(__int_as_float(last))));
    if(inside && slot == 0)
    {
        const int64_t pix = (int64_t)y * W + x;
        if(!kOwn)
        {
            final_T[pix] = T;
            final_idx[pix] = last;
        }
        store_pixel(image, pix, (int64_t)W * H, red, green, blue, T, broken, bg, planar);
    }
    if(!kOwn && prep_zeros)
        zero_grads_share(prep, prep_count, blockIdx.x, gridDim.x, tid, kWideThreads);
    else if(!kOwn)
        prepare_grads_share(splats, prep, prep_count, prep_marks, blockIdx.x, gridDim.x, tid, kWideThreads);
}

// Does a forward without a backward find its lists itself?
bool blends_own_lists(int64_t n, const ListGrid& lg)
{
    return n > 0 && lg.shift == 0 && lg.tiles() > 0 && lg.tiles() <= kFwdWideUpTo &&
           n <= kOwnGaussians + (int64_t)kOwnGaussiansPerTile * lg.tiles() && forced_pixels_per_lane() == 0;
}

int launch_blend_fwd_own(const dsx_camera& cam, int64_t n, const uint32_t* depth_keys, const uint2* rects, const float* splats, float* image,
                         hipStream_t stream)
{
    const ListGrid lg = list_grid(cam);
    if(!blends_own_lists(n, lg))
        return DSX_ERR_BAD_ARG;
    {
        DSX_TIMED("blend_fwd_kernel", stream);
        const int split = lg.tiles() <= kWideSplitUpTo;
        hipLaunchKernelGGL(blend_fwd_wide_kernel<true>, dim3(split ? 4 * lg.tiles() : lg.tiles()), dim3(kWideThreads), 0, stream, nullptr, nullptr,
                           reinterpret_cast<const float4*>(splats), image, nullptr, nullptr, cam.image_width, cam.image_height, lg.ntx,
                           (uint32_t)(n - 1), 0, nullptr, 0, nullptr, nullptr, nullptr, (int64_t)0, nullptr, 0, cam.bg,
                           camera_flag(cam, DSX_PLANAR_IMAGE), split, OwnLists{depth_keys, rects, (int)n, lg.tiles() - 1});
    }
    DSX_LAUNCH_CHECK();
    return DSX_OK;
}

// The BinLists view of a `ranges` buffer in ranges_layout(lg) (lists per bin: lg.shift > 0)
static BinLists bin_lists(const ListGrid& lg, int32_t* ranges)
{
    BinLists L = {};
    if(lg.shift)
    {
        const RangesLayout rl = ranges_layout(lg);
        L.fine = ranges + rl.fine;
        L.last_tile = ranges + rl.last_tile;
        L.bins = ranges + rl.bins;
        L.walk = ranges + rl.walk;
        L.shift = lg.shift;
        L.nbx = lg.nbx;
        L.nty = lg.nty;
    }
    return L;
}

// ranges: the `ranges` buffer in ranges_layout(list_grid(cam)) (the kernel also writes its `walk` part
// when the lists are per bin).  check_header: the buffer has its header word, which must name the
// bin size of this call (always so for binned lists; per-tile lists may come as the tiles + 1 words
// of launch_tile_ranges, which have none).  n, k: Gaussians and entries of sorted_ids; ids and list
// positions beyond them are not followed.
int launch_blend_fwd(const dsx_camera& cam, int64_t n, int64_t k, int32_t* ranges, const int32_t* sorted_ids,
                     const float* splats, float* image, float* final_T, int32_t* final_idx, hipStream_t stream,
                     bool check_header, const uint32_t* sort_flag_a, const uint32_t* sort_flag_b,
                     float* prepare_grads, bool prepare_marks)
{
    const ListGrid lg = list_grid(cam);
    const int ntx = lg.ntx, nty = lg.nty;
    if(ntx * nty == 0)
        return prepare_grads ? DSX_ERR_BAD_ARG : DSX_OK; // (no image, no kernel, nothing prepared)
    if(prepare_grads && (((uintptr_t)prepare_grads & 15) != 0 || splats == nullptr))
        return DSX_ERR_BAD_ARG;
    if(n < 0 || k < 0 || k > 0x7fffffffll || (k > 0 && (sorted_ids == nullptr || splats == nullptr || n == 0)))
        return DSX_ERR_BAD_ARG;
    float4* prep = reinterpret_cast<float4*>(prepare_grads);
    const int64_t prep_count = prepare_grads ? n : 0;
    uint8_t* prep_marks = prepare_grads && prepare_marks ? grad_marks(prepare_grads, n) : nullptr;
    const BinLists L = bin_lists(lg, ranges);
    const int32_t* header = (lg.shift || check_header) ? ranges + ranges_layout(lg).header : nullptr;
    // the largest id that the kernel takes from the lists
    const uint32_t last_id = n > 0 ? (uint32_t)(n - 1) : 0u;
    {
        DSX_TIMED("blend_fwd_kernel", stream);
        const bool four = blend_pixels_per_lane(ntx * nty, kFwdFourPixelsFrom) == 4;
        const bool wide = forced_pixels_per_lane() == 0 && lg.shift == 0 && ntx * nty <= kFwdWideUpTo;
        const dim3 grid(ntx * nty);
        const float4* sp = reinterpret_cast<const float4*>(splats);
        const int prep_zeros = prep_marks != nullptr && zeros_alone(cam, n);
        const int split = lg.tiles() <= kWideSplitUpTo;
        if(wide)
            hipLaunchKernelGGL(blend_fwd_wide_kernel<false>, dim3(split ? 4 * lg.tiles() : lg.tiles()), dim3(kWideThreads), 0, stream, ranges, sorted_ids, sp, image, final_T,
                               final_idx, cam.image_width, cam.image_height, ntx, last_id, (int)k, header, lg.shift, sort_flag_a,
                               sort_flag_b, prep, prep_count, prep_marks, prep_zeros, cam.bg, camera_flag(cam, DSX_PLANAR_IMAGE), split, OwnLists{});
#define DSX_LAUNCH_FWD(KERNEL, THREADS)                                                                          \
    hipLaunchKernelGGL((KERNEL), grid, dim3(THREADS), 0, stream, ranges, sorted_ids, sp, image, final_T, final_idx,  \
                       cam.image_width, cam.image_height, ntx, last_id, (int)k, header, lg.shift, sort_flag_a,     \
                       sort_flag_b, prep, prep_count, prep_marks, prep_zeros, cam.bg, camera_flag(cam, DSX_PLANAR_IMAGE), L)
        else if(four && lg.shift)
            DSX_LAUNCH_FWD(blend_fwd_kernel<true>, DSX_WAVE);
        else if(four)
            DSX_LAUNCH_FWD(blend_fwd_kernel<false>, DSX_WAVE);
        else if(lg.shift)
            DSX_LAUNCH_FWD(blend_fwd_tile_kernel<true>, kTileThreads);
        else
            DSX_LAUNCH_FWD(blend_fwd_tile_kernel<false>, kTileThreads);
#undef DSX_LAUNCH_FWD
    }
    DSX_LAUNCH_CHECK();
    return DSX_OK;
}

// -----------------------------------------------------------------------------------------
// backward: cpp/gsplat/backward.cu:25-202
// -----------------------------------------------------------------------------------------

template <int kCtrl, bool kZeroOutside = false>
__device__ __forceinline__ float dpp_move(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, kZeroOutside));
}
template <int kCtrl>
__device__ __forceinline__ float dpp_add(float v)
{
    return v + dpp_move<kCtrl>(v);
}

// Sums over the 16 lanes of a row, the four rows at once (their lanes hold four entries' terms), with
// data-parallel-primitive adds only: no LDS traffic.
__device__ __forceinline__ float row_sum(float v)
{
    v = dpp_add<0xB1>(v);  // quad_perm [1,0,3,2]
    v = dpp_add<0x4E>(v);  // quad_perm [2,3,0,1]
    v = dpp_add<0x124>(v); // row_ror:4
    v = dpp_add<0x128>(v); // row_ror:8
    return v;
}

__host__ __device__ constexpr int block_lane(int block) { return 16 * (block / 4) + block % 4; } // (the first one)

// Sums of eight values over the four lanes of a block (lanes four apart in a row), as a reduce-scatter with the DPP's bank masks, which
// choose the lanes of an add for free: 12 instructions.  Lane l gets the sums of v[2 * bit 2 of l + bit 3 of l] and of the one four further.
// (s_nop: as in row_sum8_scatter.)
__device__ __forceinline__ void bank_sum8_scatter(const float (&v)[8], float& first, float& second)
{
    float s0, s1, s2, s3;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %1, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %2, %8, %8 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %3, %10, %10 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc"
        : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3)
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %2, %2 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %4, %4 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %0, %3, %3 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %1, %5, %5 row_shr:4 row_mask:0xf bank_mask:0xa"
        : "=&v"(first), "=&v"(second)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3));
}

// The same for one value of each of two entries: lanes 0 to 3 of a row get the first's sums, lanes 8 to 11 the second's.
__device__ __forceinline__ float bank_sum2(float a, float b)
{
    float s, sum;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %2, %2 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %1, %0, %0 row_shl:4 row_mask:0xf bank_mask:0x5"
        : "=&v"(s), "=&v"(sum)
        : "v"(a), "v"(b));
    return sum;
}

// Eight values at once as a reduce-scatter.  A step takes two registers into one: the lanes of one half
// keep the first value and add their partner's share of it, the other half the second.  The
// DPP bank mask (banks of four lanes) chooses the lanes of an add for free where the halves are whole banks,
// so the first two steps (lanes 8 apart: 8 -> 4 registers; lanes 7 - l of a half row: 4 -> 2) take two
// instructions per pair; the last pair trades between neighbouring lanes by selects, and one add over lanes
// two apart finishes: 16 instructions for the eight sums of four entries.
// Lane l ends up with the total of v[4 * (l & 1) + 2 * ((l >> 2) & 1) + ((l >> 3) & 1)].
// (In the asm a VALU result may be read through DPP only two wait states after it was written, which the
// compiler cannot see to inside: hence the s_nop in front; no later instruction of a block reads another's result.)
__device__ __forceinline__ float row_sum8_scatter(const float (&v)[8], int lane)
{
    float s0, s1, s2, s3;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %1, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %2, %8, %8 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %3, %10, %10 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc"
        : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3)
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
    float t0, t1;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %2, %2 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %4, %4 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %0, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %1, %5, %5 row_half_mirror row_mask:0xf bank_mask:0xa"
        : "=&v"(t0), "=&v"(t1)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3));
    // the half mirror pairs lane l with 7 - l: after it a bank's four lanes hold four partial sums of one value
    const bool odd = lane & 1;
    const float keep = odd ? t1 : t0;
    const float send = odd ? t0 : t1;
    const float o = keep + dpp_move<0xB1>(send); // quad_perm [1,0,3,2]: the neighbour's share
    return dpp_add<0x4E>(o);                     // quad_perm [2,3,0,1]: lanes that differ in bit 1
}

// The same for two entries' eight values each and a ninth of each: `one` is the sum of a[l & 7] for lanes 0 to 7 of a row, of b[l & 7] for
// lanes 8 to 15, `ninth` that of a8 and b8.  Lanes 8 apart take the two entries apart, half rows mirrored the values four apart, and
// neighbours and lanes two apart trade by selects: 33 + 5 instructions instead of 2 x 22.
__device__ __forceinline__ void row_sum16_scatter(const float (&a)[8], const float (&b)[8], float a8, float b8, int lane, float& one,
                                                  float& ninth)
{
    float s[8], t[4], n;
#pragma unroll
    for(int h = 0; h < 8; h += 4)
        asm("s_nop 1\n\t"
            "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %1, %5, %5 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %2, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %3, %7, %7 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc"
            : "=&v"(s[h]), "=&v"(s[h + 1]), "=&v"(s[h + 2]), "=&v"(s[h + 3])
            : "v"(a[h]), "v"(a[h + 1]), "v"(a[h + 2]), "v"(a[h + 3]), "v"(b[h]), "v"(b[h + 1]), "v"(b[h + 2]), "v"(b[h + 3]));
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %4, %13, %13 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %4, %14, %14 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %0, %5, %5 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %6, %6 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %2, %7, %7 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %3, %8, %8 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %0, %9, %9 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %1, %10, %10 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %2, %11, %11 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %3, %12, %12 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %4, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xf"
        : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(n)
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(s[4]), "v"(s[5]), "v"(s[6]), "v"(s[7]), "v"(a8), "v"(b8));
    const bool odd = lane & 1, upper = lane & 2;
    const float x = (odd ? t[1] : t[0]) + dpp_move<0xB1, true>(odd ? t[0] : t[1]); // quad_perm [1,0,3,2]
    const float y = (odd ? t[3] : t[2]) + dpp_move<0xB1, true>(odd ? t[2] : t[3]);
    one = (upper ? y : x) + dpp_move<0x4E, true>(upper ? x : y);                   // quad_perm [2,3,0,1]
    n += dpp_move<0xB1, true>(n);
    ninth = n + dpp_move<0x4E, true>(n);
}

// The nine sums of a staged entry, added up in LDS over the rows of lanes: as doubles, because the LDS adds a double
// in a third of a cycle per lane where a float takes three (36 lanes: 11 cycles against 109, of a unit
// that the compute unit's wavefronts share).
constexpr int kSums = 9;
constexpr float kAlphaMaxBwd = 0.99f;
// Where the sums of a place lie: four and four of each place side by side, then the ninths.  An add serves 16 lanes at a time
// over 16 doubles: four rows' or blocks' lots of four meet only where their places are the same or a multiple of four apart (nine
// doubles side by side: with 7 of 16 of all other places).  Blocks that are at the same entry do meet, and where entries
// reach every block nearly all are: 2.6 to 3.5 conflict cycles an LDS instruction.  The backward's wavefront form without its adds to memory, us,
// as it is / with a place for each quad's own sums / without adds in LDS: 1 M large Gaussians 236 / 209 / 205, 3 M 252 / 237 / 234, 2 M
// faint 1238 / 1184 / 1151.
template <int kPlaces>
__host__ __device__ constexpr int sum_at(int place, int slot)
{
    return slot == 8 ? 8 * kPlaces + place : 4 * (slot & 4 ? kPlaces + place : place) + (slot & 3);
}
// staged entries of a round: 7.5 KB of LDS with their sums, 20 wavefronts per compute unit (64 entries and 16 wavefronts: 2 M
// faint Gaussians 1353 -> 1430 us; 12: 1545, 8: 1815)
constexpr int kBwdBatch = 56;

// An entry's sums in LDS, from the moments of w = vis v_alpha over its pixels (vis = exp(-sigma), and v_sigma =
// -opacity w) to the gradients: v_x = sum of v_sigma (a dx + b dy) with d = mean - pixel (v_sigma and d both change
// sign), ...; v_opacity is the sum of w itself.  times_opacity: they are moments of opacity w (an opacity from 1/255 to the clamp)
template <int kPlaces>
__device__ __forceinline__ void moments_to_gradients(double* sums, int place, const float4 A, const float4 B, bool times_opacity,
                                                     uint8_t* mark)
{
    double* const m = sums + 4 * place;
    double* const n = m + 4 * kPlaces;
    const float half_a = A.z, b = A.w, half_c = B.x;
    const double opacity = (double)B.y;
    // (a sum that is zero stays so whatever the opacity: an infinite or NaN one of an entry that no pixel took)
    const double factor = times_opacity ? 1.0 : opacity;
    auto scaled = [&](double v) { return v != 0.0 ? factor * v : 0.0; };
    const double w = m[0], wx = m[1], wxx = m[2], wy = m[3], wxy = n[0], wyy = n[1];
    const bool any = w != 0.0 || n[2] != 0.0 || n[3] != 0.0 || sums[8 * kPlaces + place] != 0.0 || wx != 0.0 || wxx != 0.0 ||
                     wy != 0.0 || wxy != 0.0 || wyy != 0.0;
    if(any && mark)
        *mark = 1;
    m[0] = scaled((double)(2.0f * half_a) * wx + (double)b * wy);
    m[1] = scaled((double)b * wx + (double)(2.0f * half_c) * wy);
    m[2] = scaled(-0.5 * wxx);
    m[3] = scaled(-wxy);
    n[0] = scaled(-0.5 * wyy);
    n[1] = times_opacity ? w / opacity : w;
}
// One set of hardware float atomics per entry and round, and none where no pixel was valid: nine threads for each entry (those
// that are over sit out: a record's adds leave in one instruction, which takes the memory one or two requests; requests to a
// line that every tile adds to wait 13 ns for each other; all adds together: 64 of 300 us for 1 M large Gaussians, 43 of 1281 for 2 M faint
// ones, 1 of 253 for 3 M).
// A load that is issued behind these adds waits for them too, so a round's are issued once the next round's records have arrived, and
// end during its walk (right after their own walk: 1 M wide Gaussians 306 -> 284 us, 1.4 M at 1557x1038 494 -> 486, 500 K 239 -> 236;
// tile form: 50 K at 512x512 74.0 -> 71.8, 100 K at 979x546 104.2 -> 103.1).
template <int kPlaces>
__device__ __forceinline__ void flush_sums(const double* sums, const int* ids, int staged, float* grads, int tid, int threads)
{
    const int at_once = threads / kSums, slot = tid % kSums;
    if(tid < at_once * kSums)
        for(int e = tid / kSums; e < staged; e += at_once)
        {
            const float v = (float)sums[sum_at<kPlaces>(e, slot)];
            if(v != 0.0f)
                unsafeAtomicAdd(grads + (int64_t)ids[e] * DSX_GRAD_FLOATS + slot, v);
        }
}

// Colours and upstream gradients below this keep all products of theirs finite.
constexpr float kTame = 1e12f;
// the largest magnitude, infinite if one is NaN
__device__ __forceinline__ float largest(float a, float b, float c)
{
    const float m = fmaxf(fabsf(a), fmaxf(fabsf(b), fabsf(c)));
    return a == a && b == b && c == c ? m : __builtin_inff();
}

// What is worked out anew in every round of the backward: kept over the rounds it would be spilled, and the wait for its reload is
// one for the last round's adds to memory too.  (Two vectors of constants and the list's place so; us of the kernel: 1920x1080, 500 K mixed
// Gaussians 256 -> 248, 3 M 242 -> 235, 3 M faint 1899 -> 1848, 500 K that reach the clamp 160 -> 156; 1557x1038, 1.4 M mixed 211 -> 206.)
__device__ __forceinline__ uint32_t made_here(uint32_t v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// What an entry asks of the walk: may its product with an alpha of zero be anything but zero (kAnyEntry), does its alpha reach the
// clamp (kClampedEntry), or neither (0)?  An opacity beyond 2, which no training gives, is left to the general walk: its moments are
// not taken times the opacity before they are summed.
constexpr uint32_t kClampedEntry = 1, kAnyEntry = 2;
__device__ __forceinline__ uint32_t entry_kind(const float4 q0, const float4 q1, const float4 q2)
{
    const bool tame = q1.w <= 2.0f && largest(q0.x, q0.y, 0.0f) < kTame && largest(q2.x, q2.y, q2.z) < kTame;
    return !tame ? kAnyEntry : (q1.w <= kAlphaMaxBwd ? 0 : kClampedEntry);
}

// How an entry's gradient at a pixel follows from what lies behind it: with T the transmittance in front of the
// entry, the reference's v_alpha = T (rgb . v_out) - B / (1 - alpha), B the sum over the entries behind of alpha T (rgb . v_out) and
// the background's T_final (bg . v_out).  Let `behind` be B over the transmittance behind the entry, T (1 - alpha); then
//   v_alpha = T (rgb . v_out - behind), and for the next entry in front: behind += alpha (rgb . v_out - behind).
// The weight alpha T is the colours' too, and where alpha is opacity * vis (no clamp) alpha T (rgb . v_out - behind) is opacity w, whose
// moments are then summed.  19 instructions a pixel and entry instead of 21 with B; 2 M faint Gaussians 1269 -> 1240 us, 1.4 M at
// 1557x1038 468 -> 460, 1 M large ones 277 -> 272.  `behind` is a mean of what is seen, B a sum of ever smaller terms: the distance of
// the gradients from a 64-bit evaluation of the same records (relative 2-norm, scenes of 700 Gaussians; means, conics, opacities, 1e-7):
// ordinary 2.9, 3.8, 3.0 -> 2.1, 2.5, 2.2; opacity 0.9 3.2, 4.5, 3.1 -> 2.5, 3.2, 2.2; large 9.9, 7.8, 5.4 -> 6.6, 6.5, 4.7; faint 3.4,
// 5.9, 3.7 -> 2.6, 3.0, 2.8.  (An infinite colour makes the gradients of what lies in front of it infinite or NaN, with B infinite.)
// Same shape as the forward: sixteen quads of lanes, each with its block of pixels and its own list of the
// entries that reach it, back to front from the last entry that any pixel blended.
// The per-Gaussian gradients are first summed over a lane's four pixels, then over the quad's four lanes, all
// sixteen quads' entries at once, then in LDS over the quads.
// kBinned: the entries come out of the list of the tile's bin, filtered into a queue as in the forward
// but downwards; the forward left, per tile, the bin-list position where its scan stopped and
// the number of the tile's entries it had met by then, from which every entry met on the way down
// gets its index in the sorted key array (final_idx is compared with those).
template <bool kBinned>
__global__ __launch_bounds__(DSX_WAVE) __attribute__((amdgpu_waves_per_eu(5, 5))) void blend_bwd_kernel(
    const int32_t* __restrict__ ranges, const int32_t* __restrict__ ids, const float4* __restrict__ splats,
    const float* __restrict__ final_T, const int32_t* __restrict__ final_idx, const float* __restrict__ v_image,
    const float* __restrict__ bg, float* grads, uint8_t* marks, int W, int H, int ntx, uint32_t last_id, int k,
    const int32_t* __restrict__ header, int header_shift, int planar, const BinLists lists, const ZeroJobs zeros)
{
    // (one place more: nobody's entry, as in the forward.  Side by side, because with what the compiler puts between them the 7672
    // bytes would not fit 7680, the most of 20 wavefronts per compute unit)
    __shared__ struct
    {
        float4 c[kBwdBatch + 1];              // red, green, blue
        float4 a[kBwdBatch + 1];              // pixel x, pixel y, conic a/2, conic b
        float4 b[kBwdBatch + 1];              // conic c/2, opacity, limit of sigma's bits, index in the sorted key array
        uint4 list[kQuads * kBwdBatch / 16];  // (what follows is read ahead)
        double sum[kBwdBatch * kSums + 1];    // (nobody's zeros are added to others' sums)
    } s;
    static_assert(sizeof(s) <= 7680, "20 wavefronts per compute unit");
    float4* const s_c = s.c;
    float4* const s_a = s.a;
    float4* const s_b = s.b;
    uint4* const s_list = s.list;
    double* const s_sum = s.sum;
    // while a round is staged, in the records' memory: candidates and the scan's queue, as in the forward (nobody's colour, which they
    // overwrite, is written again for each round)
    int2* const s_cand = reinterpret_cast<int2*>(&s);
    int* const s_queue = reinterpret_cast<int*>(&s.a[DSX_WAVE - kBwdBatch - 1]);
    static_assert(DSX_WAVE + DSX_WAVE / 4 <= 2 * kBwdBatch && kBwdBatch % 2 == 0 && (kQuads * kBwdBatch) % 16 == 0 &&
                      kQuads * kBwdBatch / 16 <= DSX_WAVE, "what the records' memory holds; lists of pairs of bytes, cleared by words");

    const int lane = threadIdx.x;
    const int tile = blockIdx.x;
    const int x0 = (tile % ntx) * kTile, y0 = (tile / ntx) * kTile;
    // this lane's column of four pixels: a row of lanes has a row of four blocks, lanes four apart the columns of a block
    const int block = 4 * (lane >> 4) + (lane & 3);
    const int x = x0 + 4 * (lane & 3) + ((lane >> 2) & 3), y = y0 + kPix * (lane >> 4);
    const float pxf = (float)x + 0.5f;
    const float bg0 = bg[0], bg1 = bg[1], bg2 = bg[2];

    // behind = v_out . (the colour that the entries behind and the background would give this pixel if nothing lay in front of
    // them), see above: the three per-channel colour buffers of cpp/gsplat/backward.cu:156-168 only ever appear dotted with
    // v_out, so one scalar carries them
    const int64_t step = planar ? 1 : 3, plane = planar ? (int64_t)W * H : 1; // of v_image: between pixels, between channels
    float pyf[kPix], T[kPix], vo0[kPix], vo1[kPix], vo2[kPix], behind[kPix];
    int bin_final[kPix];
    int m_quad = -1;
#pragma unroll
    for(int p = 0; p < kPix; ++p)
    {
        const bool inside = x < W && y + p < H;
        const int64_t pix = inside ? (int64_t)(y + p) * W + x : 0;
        pyf[p] = (float)(y + p) + 0.5f;
        const float Tf = inside ? final_T[pix] : 0.0f;
        T[p] = Tf;
        bin_final[p] = inside ? final_idx[pix] : -1;
        vo0[p] = inside ? v_image[step * pix] : 0.f;
        vo1[p] = inside ? v_image[step * pix + plane] : 0.f;
        vo2[p] = inside ? v_image[step * pix + 2 * plane] : 0.f;
        behind[p] = bg0 * vo0[p] + bg1 * vo1[p] + bg2 * vo2[p];
        m_quad = max(m_quad, bin_final[p]);
    }

    // last entry (as an index in the sorted key array) that any pixel of each block, of the wavefront, blended
    m_quad = max(m_quad, __shfl_xor(m_quad, 4, DSX_WAVE));
    m_quad = max(m_quad, __shfl_xor(m_quad, 8, DSX_WAVE));
    int m = m_quad;
#pragma unroll
    for(int o = 1; o < DSX_WAVE; o = o == 2 ? 16 : 2 * o)
        m = max(m, __shfl_xor(m, o, DSX_WAVE));
    m = __builtin_amdgcn_readfirstlane(m);
    if(lane == 0)
    {
        // (its sigma is NaN: no pixel takes it.  Its centre is finite, or a pixel's zeros times the distance to it would not be zero)
        s_a[kBwdBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kBwdBatch] = make_float4(__builtin_nanf(""), 0.f, 0.f, __int_as_float(INT_MAX));
    }

    // lists that were built for another bin size than this launch assumes are not read (see the forward)
    const bool layout_ok = header == nullptr || *header == header_shift;
    int start = 0;
    int pos = -1;       // next position of the list to look at
    int left = 0;       // entries of the tile's own list that are still to be found (binned lists)
    int skip = 0;       // those among the next ones that lie behind everything that was blended (binned lists)
    int idx_next = 0;   // index (in the sorted key array) of the next entry that is handed to the blend
    TileSource src = {};
    uint32_t my_bits = 0u; // the two bits of this wavefront's tile in a pair's key word (high half)
    if(kBinned && layout_ok)
    {
        // The forward's scan of the bin's list stopped at position w[0] after meeting w[1] of the
        // tile's entries (the largest of the four pairs of words, of which three are empty); everything
        // that was blended lies below, and the entries are taken from there downwards.  An entry's
        // index is the tile's range start plus its rank; those above the last blended one (m) are
        // not even queued, so the entries that are handed on have consecutive indices.
        src = tile_source(lists, tile, ntx);
        my_bits = tile_bits_of(src, lists.shift) << 16;
        start = max(src.start, 0);
        const int32_t* w = lists.walk + (int64_t)tile * 8;
        const int stopped = max(max(w[0], w[2]), max(w[4], w[6]));
        const int seen = max(max(w[1], w[3]), max(w[5], w[7]));
        // (positions outside sorted_ids are not followed, as in the forward)
        pos = min(stopped, min(src.end, k)) - 1;
        const int last = src.fine_base + min(seen, src.count) - 1;
        idx_next = min(m, last);
        skip = last - idx_next;
        left = idx_next - src.fine_base + 1;
        if(src.count <= 0 || left <= 0) // nothing of this tile was blended
            pos = start - 1;
    }
    else if(layout_ok)
    {
        start = max(ranges[tile], 0);
        const int end = min(ranges[tile + 1], k);
        pos = min(end - 1, m);
        idx_next = pos;
    }

    double* const my_sums = s_sum + 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1); // (see bank_sum8_scatter)
    // Entries up to the smallest last one are behind no pixel's.  (A pixel that blended nothing at all takes no part: its
    // transmittance is zero where only that counts, and every index lies behind its last one's.)
    const int first_index = kBinned ? src.fine_base : start;
    int m_least = INT_MAX;
    bool tame = true;
#pragma unroll
    for(int p = 0; p < kPix; ++p)
    {
        const bool none = bin_final[p] < first_index;
        T[p] = none ? 0.0f : T[p];
        bin_final[p] = none ? INT_MIN : bin_final[p];
        tame = tame && largest(vo0[p], vo1[p], vo2[p]) < kTame && fabsf(behind[p]) < kTame;
        m_least = none ? m_least : min(m_least, bin_final[p]);
    }
#pragma unroll
    for(int o = 1; o < DSX_WAVE; o <<= 1)
        m_least = min(m_least, __shfl_xor(m_least, o, DSX_WAVE));
    m_least = __builtin_amdgcn_readfirstlane(m_least);
    bool wild = __builtin_amdgcn_ballot_w64(!tame) != 0;

    const LiveBox box = {(float)x0 + 0.5f, (float)x0 + 15.5f, (float)y0 + 0.5f, (float)y0 + 15.5f};
    const int32_t* const keys = ids + k; // the pairs' key words lie behind the ids (binned lists)
    int2 spare = make_int2(0, 0);        // candidates that the last round left, and their number
    int spares = 0;
    int* const s_ids = reinterpret_cast<int*>(s_list); // between two rounds: the ids of the last one's entries,
    int summed = 0;                                    // whose sums are still to be added to memory
    while(spares > 0 || (pos >= start && (!kBinned || left > 0)))
    {
        __syncthreads(); // single wavefront: orders the LDS reads of the last round before these writes
        int found = spares;
        if(lane < spares)
            s_cand[lane] = spare;
        while(found < kBwdBatch && pos >= start && (!kBinned || left > 0))
        {
            int id = 0;
            int batch; // entries in this gather
            if(kBinned)
            {
                // (four groups of 64 positions in flight at a time, as in the forward)
                batch = 0;
                do
                {
                    int gid[kScanGroups], key[kScanGroups];
                    const int most = min(pos - start, kScanGroups * DSX_WAVE - 1);
                    const int32_t* const ids_here = ids + (pos - most);
                    const int32_t* const keys_here = keys + (pos - most);
#pragma unroll
                    for(int j = 0; j < kScanGroups; ++j)
                    {
                        const uint32_t e = (uint32_t)max(most - j * DSX_WAVE - lane, 0);
                        gid[j] = word_at(ids_here, e);
                        key[j] = word_at(keys_here, e);
                    }
#pragma unroll
                    for(int j = 0; j < kScanGroups; ++j)
                    {
                        // lower lanes hold higher positions
                        uint64_t m = __builtin_amdgcn_ballot_w64(((uint32_t)key[j] & my_bits) == my_bits) &
                                     lanes_below(pos - start + 1);
                        int taken = min(pos - start + 1, DSX_WAVE);
                        if(skip > 0)
                        {
                            const uint64_t skipped = __popcll(m) > skip ? lowest_bits(m, skip) : m;
                            skip -= __popcll(skipped);
                            m &= ~skipped;
                        }
                        const int room = DSX_WAVE - batch;
                        if(__popcll(m) > room)
                        {
                            // not all of the group's members fit: it is taken down to the last one that does
                            m = lowest_bits(m, room);
                            taken = room > 0 ? DSX_WAVE - __builtin_clzll(m) : 0;
                        }
                        if(m != 0)
                        {
                            if(__builtin_amdgcn_inverse_ballot_w64(m))
                                s_queue[batch + bits_below_lane(m)] = gid[j];
                            batch += __popcll(m);
                        }
                        pos -= taken;
                        if(taken < DSX_WAVE)
                            break;
                    }
                } while(batch < DSX_WAVE && pos >= start && batch < left);
                left -= batch;
                __syncthreads();
                id = s_queue[lane];
                __syncthreads();
            }
            else
            {
                batch = min(pos - start + 1, DSX_WAVE);
                if(lane < batch)
                    id = ids[pos - lane];
                pos -= batch;
            }
            bool reaches = false;
            if(lane < batch)
            {
                id = (int)min((uint32_t)id, last_id); // (as in the forward)
                const float4* const rec = splats + 3 * (int64_t)id;
                reaches = box_reached(box, rec[0], rec[1]);
            }
            const uint64_t m = __builtin_amdgcn_ballot_w64(reaches);
            if(reaches)
                s_cand[found + bits_below_lane(m)] = make_int2(id, idx_next - lane);
            found += __popcll(m);
            idx_next -= batch;
        }
        __syncthreads();
        const int staged = min(found, kBwdBatch);
        const int2 mine = s_cand[lane];
        spare = s_cand[kBwdBatch + lane];
        spares = found - staged;
        __syncthreads();
        uint32_t reached = 0;
        uint32_t kind = 0;
        bool last_here = false;
        if(lane < staged)
        {
            const float4* const rec = splats + 3 * (int64_t)mine.x;
            const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];
            const float reach = reach_of(q1.w);
            last_here = mine.y > m_least;
            kind = entry_kind(q0, q1, q2);
            reached = blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, (float)x0 + 0.5f, (float)y0 + 0.5f);
            s_a[lane] = make_float4(q0.x, q0.y, q1.x * 0.5f, q1.y);
            s_b[lane] = make_float4(q1.z * 0.5f, q1.w, __uint_as_float(reach_limit_bwd(q1.w, reach)), __int_as_float(mine.y));
            s_c[lane] = q2;
        }
        if(lane == kBwdBatch)
        {
            const float zero = __uint_as_float(made_here(0u));
            s_c[made_here(kBwdBatch)] = make_float4(zero, zero, zero, zero);
        }
        // (entries behind everything that a quad's pixels blended are not in its list)
#pragma unroll
        for(int q = 0; q < kQuads; ++q)
            if(mine.y > __builtin_amdgcn_readlane(m_quad, block_lane(q)))
                reached &= ~(1u << q);
        flush_sums<kBwdBatch>(s_sum, s_ids, summed, grads, lane, DSX_WAVE);
        __syncthreads();
        if(lane < kQuads * kBwdBatch / 16)
        {
            const uint32_t nobodies = made_here(0x01010101u * kBwdBatch);
            s_list[lane] = make_uint4(nobodies, nobodies, nobodies, nobodies);
        }
        __syncthreads();
        const int rounds = quad_lists<kBwdBatch>(reinterpret_cast<uint8_t*>(s_list), reached, lane);
        const int zero = (int)made_here(0u);
        for(int i = lane; i < kBwdBatch * kSums; i += DSX_WAVE)
            s_sum[i] = __hiloint2double(zero, zero);
        __syncthreads();

        // Two entries at a time, without branches: a pixel that does not take an entry gives it the alpha zero.  Both
        // transmittances come from one reciprocal, and the moments over a lane's four rows from those of two rows each that count
        // from the upper one, eleven operations instead of sixteen (all four counted from one row: nine, but terms that cancel where a
        // splat is hardly wider than a pixel: 1.3 times the error there).  A pair's sums are added when the next one's records have been
        // asked for: the LDS serves a wavefront in order, and behind the adds the reads would wait for them.  117 vector instructions
        // an entry instead of 132 (of which a seventh was jumped over where no lane took a row).  us, one entry after the other -> pairs, of
        // which without the late adds: 2 M faint Gaussians 1253 -> 1236 (1235), 1.4 M at 1557x1038 468 -> 451 (457), 500 K 217 -> 205 (210), 3 M 258 -> 243
        // (255), 300 K at 1237x822 225 -> 215 (221).  Distance of the gradients from a 64-bit evaluation (scenes of 700 records; means, conics,
        // opacities, 1e-7): ordinary 3.1, 3.0, 3.0 -> 2.9, 2.8, 2.8; opacity 0.9 3.6, 3.5, 3.3 -> 3.2, 3.2, 2.9; large 5.1, 5.4, 6.5 -> 4.6, 3.5, 4.9;
        // faint 2.1, 2.2, 2.0 -> 2.0, 2.1, 1.9; hardly wider than a pixel 1.2, 1.3, 1.1 -> 1.2, 1.4, 1.1.
        // clamps: some entry's alpha may reach the clamp, which the moments do not see: three instructions more a pixel and entry.  One such
        // entry in a round is the rule where a scene has been trained for long; us, the general walk for these rounds (one entry at
        // a time) -> this, half of the opacities beyond the clamp: 1.4 M at 1557x1038 143 -> 123, 500 K 157 -> 145, 3 M 215 -> 200, 300 K at 1237x822 142 ->
        // 132.  (The distance from 64 bits: as before for conics, opacities and colours, 0 to 15 % less for means.)
        auto walk_pairs = [&](auto ends, auto clamps) {
        const uint16_t* my_list = reinterpret_cast<const uint16_t*>(s_list) + made_here(block) * (kBwdBatch / 2);
        int places = *my_list;
        // (zeros at first, for each quad elsewhere)
        const int fresh = made_here(lane);
        int summed_places = (fresh >> 2 & 12) | (fresh & 3);
        summed_places |= summed_places << 8;
        float sums8[2][2] = {}, sums_blue = 0.0f;
        auto add_sums = [&]() {
#pragma unroll
            for(int u = 0; u < 2; ++u)
            {
                double* const sums = my_sums + 4 * (u == 0 ? summed_places & 0xff : summed_places >> 8);
                unsafeAtomicAdd(sums, (double)sums8[u][0]);
                unsafeAtomicAdd(sums + 4 * kBwdBatch, (double)sums8[u][1]);
            }
            if((lane & 4) == 0)
                unsafeAtomicAdd(s_sum + 8 * kBwdBatch + ((summed_places >> (lane & 8)) & 0xff), (double)sums_blue);
        };
        for(int i = 0; i < rounds; i += 2)
        {
            const int here = places;
            places = *++my_list;
            const float4 A[2] = {s_a[here & 0xff], s_a[here >> 8]};
            const float4 B[2] = {s_b[here & 0xff], s_b[here >> 8]};
            const float4 C[2] = {s_c[here & 0xff], s_c[here >> 8]};
            asm volatile("" ::: "memory");
            add_sums();
            summed_places = here;
            float unclamped[2][kPix], dx[2], dy0[2];
            auto clamped = [&](float alpha) { return clamps ? fminf(kAlphaMaxBwd, alpha) : alpha; };
#pragma unroll
            for(int u = 0; u < 2; ++u)
            {
                dx[u] = pxf - A[u].x;
                const ExponentX ex = exponent_x(A[u].z, A[u].w, dx[u]);
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
#pragma clang fp contract(off)
                    // sigma exactly as the forward computed it
                    const float dy = pyf[p] - A[u].y;
                    const float sigma = __builtin_fmaf(__builtin_fmaf(B[u].x, dy, ex.bx), dy, ex.ax);
                    uint64_t m_valid = __builtin_amdgcn_ballot_w64(__float_as_uint(sigma) <= __float_as_uint(B[u].z));
                    if(ends)
                        m_valid &= __builtin_amdgcn_ballot_w64(__float_as_int(B[u].w) <= bin_final[p]);
                    const float full = B[u].y * __builtin_amdgcn_exp2f(-sigma * kLog2E);
                    unclamped[u][p] = __builtin_amdgcn_inverse_ballot_w64(m_valid) ? full : 0.0f;
                    if(p == 0)
                        dy0[u] = dy;
                }
            }
            float between[kPix]; // the transmittance in front of the first, T becomes that in front of both
#pragma unroll
            for(int p = 0; p < kPix; ++p)
            {
                const float alpha1 = clamped(unclamped[1][p]), through = 1.0f - clamped(unclamped[0][p]);
                T[p] *= __builtin_amdgcn_rcpf(__builtin_fmaf(-alpha1, through, through));
                between[p] = __builtin_fmaf(-alpha1, T[p], T[p]);
            }
            float blue[2];
#pragma unroll
            for(int u = 0; u < 2; ++u)
            {
                // per lane, over its pixels (which share dx): the weights of the colour's gradient, and w of every pixel
                // (opacity * w: alpha holds the opacity)
                float v_red = 0.f, v_green = 0.f, v_blue = 0.f, w[kPix];
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
                    const float alpha = clamped(unclamped[u][p]), T_here = u == 0 ? between[p] : T[p], fac = alpha * T_here;
                    v_red = p == 0 ? fac * vo0[p] : v_red + fac * vo0[p];
                    v_green = p == 0 ? fac * vo1[p] : v_green + fac * vo1[p];
                    v_blue = p == 0 ? fac * vo2[p] : v_blue + fac * vo2[p];
                    const float ahead = C[u].x * vo0[p] + (C[u].y * vo1[p] + (C[u].z * vo2[p] - behind[p]));
                    behind[p] += alpha * ahead;
                    w[p] = (clamps ? unclamped[u][p] * T_here : fac) * ahead;
                }
                // 1 | dy | dy^2
                static_assert(kPix == 4, "two times two rows");
                float of0[2], of1[2], of2[2];
#pragma unroll
                for(int h = 0; h < 2; ++h)
                {
                    const float dy = dy0[u] + (float)(2 * h), lower = w[2 * h + 1];
                    of0[h] = w[2 * h] + lower;
                    of1[h] = __builtin_fmaf(dy, of0[h], lower);
                    of2[h] = __builtin_fmaf(dy, of1[h] + lower, lower);
                }
                const float S0 = of0[0] + of0[1], S1 = of1[0] + of1[1], S2 = of2[0] + of2[1];
                const float S0x = S0 * dx[u];
                const float sum8[8] = {S0, S0x, S0x * dx[u], S1, S1 * dx[u], S2, v_red, v_green};
                bank_sum8_scatter(sum8, sums8[u][0], sums8[u][1]);
                blue[u] = v_blue;
            }
            sums_blue = bank_sum2(blue[0], blue[1]);
        }
        add_sums();
        };
        // what the walk above leaves out: values so large that a product with zero is not zero
        auto walk_any = [&]() {
        const uint16_t* my_list = reinterpret_cast<const uint16_t*>(s_list) + made_here(block) * (kBwdBatch / 2);
        int places = *my_list;
        for(int i = 0; i < rounds; i += 2)
        {
            const int here = places;
            places = *++my_list;
#pragma unroll
            for(int u = 0; u < 2; ++u)
            {
                const int place = u == 0 ? here & 0xff : here >> 8;
                const float4 A = s_a[place];
                const float4 B = s_b[place];
                const float4 C = s_c[place];
                const uint32_t limit = __float_as_uint(B.z);
                const int idx = __float_as_int(B.w);
                // sigma exactly as the forward computed it
                const float dx = pxf - A.x;
                const ExponentX ex = exponent_x(A.z, A.w, dx);
                float vis[kPix], alpha[kPix], dy[kPix]; // dy = pixel - mean
                // which lanes' pixel p takes part: wavefront masks (each compare's own result register),
                // combined on the scalar unit
                uint64_t m_valid[kPix];
                uint64_t m_any = 0;
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
#pragma clang fp contract(off)
                    dy[p] = pyf[p] - A.y;
                    const float sigma = __builtin_fmaf(__builtin_fmaf(B.x, dy[p], ex.bx), dy[p], ex.ax);
                    m_valid[p] = __builtin_amdgcn_ballot_w64(__float_as_uint(sigma) <= limit) &
                                 __builtin_amdgcn_ballot_w64(idx <= bin_final[p]);
                    m_any |= m_valid[p];
                    vis[p] = __builtin_amdgcn_exp2f(-sigma * kLog2E);
                    alpha[p] = fminf(kAlphaMaxBwd, B.y * vis[p]);
                }
                if(m_any == 0)
                    continue;
                // Per lane, over its pixels (which share dx): the weights of the colour's gradient, and three
                // moments over dy of w = vis * v_alpha
                float v_red = 0.f, v_green = 0.f, v_blue = 0.f, S0 = 0.f, S1 = 0.f, S2 = 0.f;
#pragma unroll
                for(int p = 0; p < kPix; ++p)
                {
                    if(__builtin_amdgcn_inverse_ballot_w64(m_valid[p]))
                    {
                        T[p] *= __builtin_amdgcn_rcpf(1.0f - alpha[p]);
                        const float fac = alpha[p] * T[p];
                        v_red += fac * vo0[p];
                        v_green += fac * vo1[p];
                        v_blue += fac * vo2[p];
                        const float ahead = C.x * vo0[p] + (C.y * vo1[p] + (C.z * vo2[p] - behind[p]));
                        behind[p] += alpha[p] * ahead;
                        const float w = vis[p] * T[p] * ahead;
                        const float wdy = w * dy[p];
                        S0 += w;
                        S1 += wdy;
                        S2 += wdy * dy[p];
                    }
                }
                // what is summed over the pixels: the moments of w, 1 | dx | dx^2 | dy | dx dy | dy^2, and the colour's three
                const float S0x = S0 * dx;
                const float sum8[8] = {S0, S0x, S0x * dx, S1, S1 * dx, S2, v_red, v_green};
                float first, second;
                bank_sum8_scatter(sum8, first, second);
                v_blue = dpp_add<0x128>(v_blue); // row_ror:8
                v_blue += dpp_move<0x104, true>(v_blue); // row_shl:4 (the sum in every row's first four lanes)
                double* const sums = my_sums + 4 * place;
                unsafeAtomicAdd(sums, (double)first);
                unsafeAtomicAdd(sums + 4 * kBwdBatch, (double)second);
                if((lane & 12) == 0)
                    unsafeAtomicAdd(s_sum + 8 * kBwdBatch + place, (double)v_blue);
            }
        }
        };
        const bool in_pairs = !wild && __builtin_amdgcn_ballot_w64((kind & kAnyEntry) != 0) == 0;
        if(!in_pairs)
        {
            walk_any();
            bool still = true;
#pragma unroll
            for(int p = 0; p < kPix; ++p)
                still = still && fabsf(behind[p]) < kTame;
            wild = wild || __builtin_amdgcn_ballot_w64(!still) != 0; // (an infinite colour stays behind all entries in front)
        }
        else if(__builtin_amdgcn_ballot_w64((kind & kClampedEntry) != 0) != 0)
            walk_pairs(std::true_type(), std::true_type());
        else if(__builtin_amdgcn_ballot_w64(last_here) != 0) // (some pixel's last entry lies among these: one compare a pixel and entry more)
            walk_pairs(std::true_type(), std::false_type());
        else
            walk_pairs(std::false_type(), std::false_type());
        __syncthreads();
        if(lane < staged)
        {
            s_ids[lane] = mine.x;
            moments_to_gradients<kBwdBatch>(s_sum, lane, s_a[lane], s_b[lane], in_pairs, marks ? marks + mine.x : nullptr);
        }
        summed = staged;
    }
    __syncthreads();
    flush_sums<kBwdBatch>(s_sum, s_ids, summed, grads, lane, DSX_WAVE);
    // A side job for the memory system, as in the forward: the zeros of the per-Gaussian backward's
    // outputs (that kernel writes only the Gaussians that received a term here), every wavefront a
    // share, at its end, where nothing waits for the stores (3 M Gaussians, 780 MB: the kernel takes
    // 0.275 ms instead of 0.250; a few stores in every round of the walk instead: no better).
    if(zeros.any)
        zero_share(zeros, blockIdx.x, gridDim.x, lane, DSX_WAVE);
}

// the workgroup form (see the forward's): the sums of a round's entries are shared by the four wavefronts
constexpr int kBwdAtOnce = 2; // entries that a row takes at a time
template <bool kBinned>
__global__ __launch_bounds__(kTileThreads) void blend_bwd_tile_kernel(
    const int32_t* __restrict__ ranges, const int32_t* __restrict__ ids, const float4* __restrict__ splats,
    const float* __restrict__ final_T, const int32_t* __restrict__ final_idx, const float* __restrict__ v_image,
    const float* __restrict__ bg, float* grads, uint8_t* marks, int W, int H, int ntx, uint32_t last_id, int k,
    const int32_t* __restrict__ header, int header_shift, int planar, const BinLists lists, const ZeroJobs zeros)
{
    __shared__ float4 s_a[kTileBatch + 1], s_b[kTileBatch + 1], s_c[kTileBatch + 1];
    __shared__ int s_id[kTileBatch];
    __shared__ double s_sum[(kTileBatch + 1) * kSums];
    __shared__ uint16_t s_reach[kTileBatch];
    __shared__ uint32_t s_list[kTileWaves * kTileBatch + 1]; // (one word more: read ahead)
    __shared__ TileScan s_scan;
    __shared__ int s_counts[kTileWaves];
    __shared__ uint32_t s_special[kTileWaves]; // per wavefront: the kinds of its entries (entry_kind)
    __shared__ int s_last[4 * kTileWaves]; // per block: the last entry that any of its pixels blended
    int* const s_queue = reinterpret_cast<int*>(s_list); // (free while a round is staged)

    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), row = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / DSX_WAVE);
    const int tile = blockIdx.x;
    const int first_block = first_block_of(wave);
    const Pixels px(tile, wave, ntx, lane);
    const float pxf = (float)px.x + 0.5f, pyf = (float)px.y + 0.5f;
    const float tile_x = (float)(tile % ntx * kTile) + 0.5f, tile_y = (float)(tile / ntx * kTile) + 0.5f;

    const bool inside = px.x < W && px.y < H;
    const int64_t pix = inside ? (int64_t)px.y * W + px.x : 0;
    const float Tf = inside ? final_T[pix] : 0.0f;
    float T = Tf;
    const int bin_final = inside ? final_idx[pix] : -1;
    const int64_t step = planar ? 1 : 3, plane = planar ? (int64_t)W * H : 1; // (between pixels, between channels)
    const float vo0 = inside ? v_image[step * pix] : 0.f, vo1 = inside ? v_image[step * pix + plane] : 0.f,
                vo2 = inside ? v_image[step * pix + 2 * plane] : 0.f;
    float behind = bg[0] * vo0 + bg[1] * vo1 + bg[2] * vo2;
    const bool tame = largest(vo0, vo1, vo2) < kTame && fabsf(behind) < kTame;
    bool wild = __builtin_amdgcn_ballot_w64(!tame) != 0; // (of this wavefront's pixels)
    int m = bin_final;
#pragma unroll
    for(int o = 8; o > 0; o >>= 1)
        m = max(m, __shfl_xor(m, o, DSX_WAVE));
    if((lane & 15) == 0)
        s_last[first_block + block_of_row(row)] = m;
    if(tid == 0)
    {
        s_a[kTileBatch] = s_c[kTileBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kTileBatch] = make_float4(0.f, 0.f, 0.f, __int_as_float(INT_MAX));
    }
    __syncthreads();
    m = s_last[0];
#pragma unroll
    for(int b = 1; b < 4 * kTileWaves; ++b)
        m = max(m, s_last[b]);
    m = __builtin_amdgcn_readfirstlane(m);

    // (where the lists start: as in the wavefront form)
    const bool layout_ok = header == nullptr || *header == header_shift;
    int pos = -1, left = 0, skip = 0, idx_next = 0, wanted = 0;
    TileSource src = {};
    uint32_t my_bits = 0u;
    if(kBinned && layout_ok)
    {
        src = tile_source(lists, tile, ntx);
        my_bits = tile_bits_of(src, lists.shift) << 16;
        const int start = max(src.start, 0);
        const int32_t* w = lists.walk + (int64_t)tile * 8;
        const int stopped = max(max(w[0], w[2]), max(w[4], w[6]));
        const int seen = max(max(w[1], w[3]), max(w[5], w[7]));
        pos = min(stopped, min(src.end, k)) - 1;
        const int last = src.fine_base + min(seen, src.count) - 1;
        idx_next = min(m, last);
        skip = last - idx_next;
        wanted = idx_next - src.fine_base + 1;
        left = src.count <= 0 || wanted <= 0 ? 0 : pos - start + 1;
    }
    else if(layout_ok)
    {
        const int start = max(ranges[tile], 0);
        pos = min(min(ranges[tile + 1], k) - 1, m);
        idx_next = pos;
        left = pos - start + 1;
    }
    left = __builtin_amdgcn_readfirstlane(left);

    const bool carries_blue = (lane & 15) == 2;
    const bool carries = (lane & 2) == 0 || carries_blue;
    const int sum_slot = carries_blue ? 8 : 4 * (lane & 1) + 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1);
    double* const my_sums = s_sum + sum_at<kTileBatch + 1>(0, sum_slot);
    const int sum_step = carries_blue ? 1 : 4;
    double* const my_sum = s_sum + sum_at<kTileBatch + 1>(0, lane & 7); // (see row_sum16_scatter)

    const int32_t* const keys = ids + k;
    int id_ahead = 0;
    int summed = 0; // entries of the last round, whose sums are still to be added to memory
    if(!kBinned && tid < min(left, kTileBatch))
        id_ahead = ids[pos - tid];
    while(left > 0 && (!kBinned || wanted > 0))
    {
        int id, batch;
        if(kBinned)
        {
            batch = tile_scan<-1>(s_scan, s_queue, ids, keys, pos, left, skip, my_bits, wanted);
            wanted -= batch;
            id = tid < batch ? s_queue[tid] : 0;
        }
        else
        {
            batch = min(left, kTileBatch);
            id = id_ahead;
            pos -= batch;
            left -= batch;
            if(tid < min(left, kTileBatch))
                id_ahead = ids[pos - tid];
        }
        uint32_t reached = 0;
        uint32_t kind = wild ? kAnyEntry : 0;
        float4 q0, q1, q2;
        float reach = 0.0f;
        const int idx = idx_next - tid;
        if(tid < batch)
        {
            id = (int)min((uint32_t)id, last_id);
            const float4* const rec = splats + 3 * (int64_t)id;
            q0 = rec[0], q1 = rec[1], q2 = rec[2];
            reach = reach_of(q1.w);
            reached = blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, tile_x, tile_y);
#pragma unroll
            for(int b = 0; b < 4 * kTileWaves; ++b)
                if(idx > s_last[b])
                    reached &= ~(1u << b);
            kind |= reached != 0 ? entry_kind(q0, q1, q2) : 0;
        }
        if(tid < batch) // (the loads end here: behind the adds they would wait for those)
            asm volatile("" : "+v"(q2.x), "+v"(q2.y), "+v"(q2.z), "+v"(q2.w));
        flush_sums<kTileBatch + 1>(s_sum, s_id, summed, grads, tid, kTileThreads);
        const uint32_t kinds = (__builtin_amdgcn_ballot_w64((kind & kClampedEntry) != 0) != 0 ? kClampedEntry : 0) |
                               (__builtin_amdgcn_ballot_w64((kind & kAnyEntry) != 0) != 0 ? kAnyEntry : 0);
        if(lane == 0)
            s_special[wave] = kinds;
        int staged;
        const int place = tile_place(s_counts, __builtin_amdgcn_ballot_w64(reached != 0), staged);
        // (the barrier inside: the queue has been read, the last round's sums have been taken)
        for(int i = tid; i < 4 * staged; i += kTileThreads)
            s_sum[i] = s_sum[sum_at<kTileBatch + 1>(0, 4) + i] = 0.0;
        if(tid < staged)
            s_sum[sum_at<kTileBatch + 1>(tid, 8)] = 0.0;
        if(reached != 0)
        {
            s_a[place] = make_float4(q0.x, q0.y, q1.x * 0.5f, q1.y);
            s_b[place] = make_float4(q1.z * 0.5f, q1.w, __uint_as_float(reach_limit_bwd(q1.w, reach)),
                                     __int_as_float(idx));
            s_c[place] = q2;
            s_id[place] = id;
            s_reach[place] = (uint16_t)reached;
        }
        idx_next -= batch;
        __syncthreads();

        const int rounds = (build_lists(s_list, s_reach, staged, wave, first_block, lane) + kBwdAtOnce - 1) / kBwdAtOnce;
        const uint16_t* my_list = reinterpret_cast<const uint16_t*>(s_list + wave * kTileBatch + row * (kTileBatch / 4));
        // (one walk for all wavefronts: the sums' unit depends on it)
        const uint32_t all_kinds = __builtin_amdgcn_readfirstlane(s_special[0] | s_special[1] | s_special[2] | s_special[3]);
        const bool in_pairs = all_kinds < kAnyEntry;
        auto walk_pairs = [&](auto clamps) {
            // Two entries at a time as in the wavefront form.  Of the sixteen sums of their moments and colours each lane gets one: one add
            // to LDS of all lanes for two entries instead of two of nine lanes of a row.  us: 50 K at 512x512 71 -> 62, 100 K at
            // 979x546 98 -> 88; the gradients' distance from a 64-bit evaluation 3 to 30 % less (hardly wider than a pixel: the same).
            // Where alphas may reach the clamp (general walk -> this, half of the opacities beyond it): 50 K at 512x512 39 -> 35, 200 K
            // 70 -> 62, 100 K at 979x546 88 -> 78, 400 K 92 -> 80.
            int places = *my_list;
            int summed_places = 4 * row | 4 * row << 8; // (zeros at first, elsewhere for each row)
            float sums_one = 0.0f, sums_blue = 0.0f;
            auto add_sums = [&]() {
                const int place = (summed_places >> (lane & 8)) & 0xff;
                unsafeAtomicAdd(my_sum + 4 * place, (double)sums_one);
                if((lane & 7) == 0)
                    unsafeAtomicAdd(s_sum + sum_at<kTileBatch + 1>(0, 8) + place, (double)sums_blue);
            };
            for(int i = 0; i < rounds; ++i)
            {
                const int here = places;
                places = *++my_list;
                const float4 A[2] = {s_a[here & 0xff], s_a[here >> 8]};
                const float4 B[2] = {s_b[here & 0xff], s_b[here >> 8]};
                const float4 C[2] = {s_c[here & 0xff], s_c[here >> 8]};
                asm volatile("" ::: "memory");
                add_sums();
                summed_places = here;
                float reached_alpha[2], alpha[2], dx[2], dy[2]; // (before and after the clamp)
#pragma unroll
                for(int u = 0; u < 2; ++u)
                {
#pragma clang fp contract(off)
                    dx[u] = pxf - A[u].x;
                    dy[u] = pyf - A[u].y;
                    const ExponentX ex = exponent_x(A[u].z, A[u].w, dx[u]);
                    const float sigma = __builtin_fmaf(__builtin_fmaf(B[u].x, dy[u], ex.bx), dy[u], ex.ax);
                    const uint64_t m_valid = __builtin_amdgcn_ballot_w64(__float_as_int(B[u].w) <= bin_final) &
                                             __builtin_amdgcn_ballot_w64(__float_as_uint(sigma) <= __float_as_uint(B[u].z));
                    const float full = B[u].y * __builtin_amdgcn_exp2f(-sigma * kLog2E);
                    reached_alpha[u] = __builtin_amdgcn_inverse_ballot_w64(m_valid) ? full : 0.0f;
                    alpha[u] = clamps ? fminf(kAlphaMaxBwd, reached_alpha[u]) : reached_alpha[u];
                }
                const float through = 1.0f - alpha[0];
                T *= __builtin_amdgcn_rcpf(__builtin_fmaf(-alpha[1], through, through));
                float v[2][8], blue[2];
#pragma unroll
                for(int u = 0; u < 2; ++u)
                {
                    const float T_here = u == 0 ? __builtin_fmaf(-alpha[1], T, T) : T;
                    const float fac = alpha[u] * T_here;
                    const float ahead = C[u].x * vo0 + (C[u].y * vo1 + (C[u].z * vo2 - behind));
                    behind += alpha[u] * ahead;
                    // (of the unclamped alpha: the opacity times vis)
                    const float w = (clamps ? reached_alpha[u] * T_here : fac) * ahead, wx = w * dx[u], wy = w * dy[u];
                    v[u][0] = w, v[u][1] = wx, v[u][2] = wx * dx[u], v[u][3] = wy;
                    v[u][4] = wy * dx[u], v[u][5] = wy * dy[u], v[u][6] = fac * vo0, v[u][7] = fac * vo1;
                    blue[u] = fac * vo2;
                }
                row_sum16_scatter(v[0], v[1], blue[0], blue[1], lane, sums_one, sums_blue);
            }
            add_sums();
        };
        if(all_kinds == 0)
            walk_pairs(std::false_type());
        else if(in_pairs)
            walk_pairs(std::true_type());
        else
        {
            for(int i = 0; i < rounds; ++i)
            {
                const uint32_t places = my_list[i];
                float4 A[kBwdAtOnce], B[kBwdAtOnce];
                float dx[kBwdAtOnce], dy[kBwdAtOnce], vis[kBwdAtOnce], alpha[kBwdAtOnce], ra[kBwdAtOnce], rv[kBwdAtOnce];
                double* sums[kBwdAtOnce];
                uint64_t m_valid[kBwdAtOnce];
                uint64_t m_any = 0;
#pragma unroll
                for(int u = 0; u < kBwdAtOnce; ++u)
                {
                    const uint32_t p = (places >> (8 * u)) & 0xffu;
                    A[u] = s_a[p];
                    B[u] = s_b[p];
                    const float4 C = s_c[p];
                    rv[u] = C.x * vo0 + C.y * vo1 + C.z * vo2;
                    sums[u] = my_sums + p * sum_step;
                }
#pragma unroll
                for(int u = 0; u < kBwdAtOnce; ++u)
                {
#pragma clang fp contract(off)
                    dx[u] = pxf - A[u].x;
                    dy[u] = pyf - A[u].y;
                    const ExponentX ex = exponent_x(A[u].z, A[u].w, dx[u]);
                    const float sigma = __builtin_fmaf(__builtin_fmaf(B[u].x, dy[u], ex.bx), dy[u], ex.ax);
                    m_valid[u] = __builtin_amdgcn_ballot_w64(__float_as_int(B[u].w) <= bin_final) &
                                 __builtin_amdgcn_ballot_w64(__float_as_uint(sigma) <= __float_as_uint(B[u].z));
                    m_any |= m_valid[u];
                    vis[u] = __builtin_amdgcn_exp2f(-sigma * kLog2E);
                    alpha[u] = fminf(0.99f, B[u].y * vis[u]);
                    ra[u] = __builtin_amdgcn_rcpf(1.0f - alpha[u]);
                }
                if(m_any == 0)
                    continue;
#pragma unroll
                for(int u = 0; u < kBwdAtOnce; ++u)
                {
                    float w = 0.f, v_red = 0.f, v_green = 0.f, v_blue = 0.f;
                    if(__builtin_amdgcn_inverse_ballot_w64(m_valid[u]))
                    {
                        T *= ra[u];
                        const float fac = alpha[u] * T;
                        v_red = fac * vo0;
                        v_green = fac * vo1;
                        v_blue = fac * vo2;
                        const float ahead = rv[u] - behind;
                        behind += alpha[u] * ahead;
                        w = vis[u] * T * ahead;
                    }
                    const float wx = w * dx[u], wy = w * dy[u];
                    const float sum8[8] = {w, wx, wx * dx[u], wy, wy * dx[u], wy * dy[u], v_red, v_green};
                    const float total = row_sum8_scatter(sum8, lane);
                    v_blue = row_sum(v_blue);
                    if(carries)
                        unsafeAtomicAdd(sums[u], (double)(carries_blue ? v_blue : total));
                }
            }
            // (an infinite colour stays behind all entries in front)
            wild = wild || __builtin_amdgcn_ballot_w64(!(fabsf(behind) < kTame)) != 0;
        }
        __syncthreads();
        for(int e = tid; e < staged; e += kTileThreads)
            moments_to_gradients<kTileBatch + 1>(s_sum, e, s_a[e], s_b[e], in_pairs, marks ? marks + s_id[e] : nullptr);
        __syncthreads();
        summed = staged;
    }
    flush_sums<kTileBatch + 1>(s_sum, s_id, summed, grads, tid, kTileThreads);
    if(zeros.any)
        zero_share(zeros, blockIdx.x, gridDim.x, tid, kTileThreads);
}

// -----------------------------------------------------------------------------------------
// the same for images of very few tiles: four workgroups per tile, a wavefront for each block
// -----------------------------------------------------------------------------------------
// Up to 256 tiles the workgroup form leaves a SIMD one wavefront or none, and the kernel lasts as long as its longest chain: 55
// instructions an entry, each waiting for the one before.  Here each 4x4 block has a wavefront and each of its pixels a quad of lanes,
// which work on four entries at a time: they hand each other alphas and colours, each takes the same steps of what they let through and of
// what lies behind, and keeps its own entry's; sums over the sixteen pixels by twelve DPP adds and two swaps, one add to
// LDS for all four entries.  86 instructions for four.  A tile's four quadrants are workgroups of their own, so that 64 tiles reach every
// compute unit; each stages what reaches its quadrant.  What it costs are four times the adds to memory, which wait for each other where many tiles share
// a Gaussian.  us of the kernel, workgroup form -> this, 20 K Gaussians, opaque / mixed / faint, by the tiles that one covers:
//    64 tiles   13  17 -> 14, 44 -> 26, 196 -> 105   28  16 -> 14, 31 -> 21, 181 -> 96
//   100          9  23 -> 16, 52 -> 34, 146 -> 88    19  17 -> 16, 43 -> 33, 170 -> 104   41  16 -> 15, 28 -> 22, 167 -> 99
//   144         12  22 -> 19, 50 -> 36, 135 -> 86    25  17 -> 19, 43 -> 36, 163 -> 105   58  15 -> 20, 27 -> 29, 160 -> 111
//   196         15  22 -> 21, 46 -> 41, 126 -> 80    33  17 -> 23, 41 -> 38, 163 -> 121   77  15 -> 24, 28 -> 35, 152 -> 150
//   256          8  27 -> 24, 67 -> 48, 57 -> 43     18  22 -> 24, 46 -> 46, 123 -> 90    42  17 -> 27, 39 -> 43, 154 -> 134
//   324          9  27 -> 26, 63 -> 47, 53 -> 41     22  22 -> 33, 51 -> 58, 115 -> 85    52  19 -> 32, 43 -> 57, 162 -> 157
//   100 K of 18 at 256 tiles 21 -> 27, 41 -> 51, 183 -> 160; 400 K of 9 at 324 33 -> 37, 63 -> 67, 239 -> 239
// Up to 100 tiles it is taken always; up to 256, a compute unit for each tile, where pairs times tiles are at most 3700 a Gaussian (14 tiles
// covered of 256, 26 of 144), between the second and the third column.
// the two lower halves and the two upper halves of two registers side by side (v_permlane32_swap), and their rows of 16 lanes: the
// even rows of both and the odd rows of both (v_permlane16_swap)
__device__ __forceinline__ float add_halves(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_rows(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
constexpr int kBlockThreads = 256;
constexpr int kBlockAtOnce = 4; // entries that a wavefront takes at a time: one for each lane of a pixel's quad
__global__ __launch_bounds__(kBlockThreads) void blend_bwd_block_kernel(
    const int32_t* __restrict__ ranges, const int32_t* __restrict__ ids, const float4* __restrict__ splats,
    const float* __restrict__ final_T, const int32_t* __restrict__ final_idx, const float* __restrict__ v_image,
    const float* __restrict__ bg, float* grads, uint8_t* marks, int W, int H, int ntx, uint32_t last_id, int k,
    const int32_t* __restrict__ header, int header_shift, int planar, const ZeroJobs zeros)
{
    static_assert(kBlockThreads == kTileThreads && kTileBatch % kBlockAtOnce == 0, "rounds as in the tile's form");
    __shared__ float4 s_a[kTileBatch + 1], s_b[kTileBatch + 1], s_c[kTileBatch + 1];
    __shared__ int s_id[kTileBatch];
    __shared__ double s_sum[(kTileBatch + 1) * kSums];
    __shared__ uint16_t s_reach[kTileBatch];
    __shared__ uint32_t s_list[kTileWaves][kTileBatch / 4 + 1]; // (a word more: read ahead)
    __shared__ int s_counts[kTileWaves];
    __shared__ uint32_t s_special[kTileWaves];
    __shared__ int s_last[kTileWaves]; // per block: the last entry that any of its pixels blended

    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), slot = lane & 3, pixel = lane >> 2;
    const int wave = __builtin_amdgcn_readfirstlane(tid / DSX_WAVE);
    const int tile = blockIdx.x / 4, quadrant = blockIdx.x % 4;
    const int first_block = first_block_of(quadrant), block = first_block + block_of_row(wave);
    const int x = tile % ntx * kTile + 4 * (block & 3) + (pixel & 3), y = tile / ntx * kTile + 4 * (block >> 2) + (pixel >> 2);
    const float pxf = (float)x + 0.5f, pyf = (float)y + 0.5f;
    const float tile_x = (float)(tile % ntx * kTile) + 0.5f, tile_y = (float)(tile / ntx * kTile) + 0.5f;

    const bool inside = x < W && y < H;
    const int64_t pix = inside ? (int64_t)y * W + x : 0;
    float T = inside ? final_T[pix] : 0.0f;
    const int bin_final = inside ? final_idx[pix] : -1;
    const int64_t step = planar ? 1 : 3, plane = planar ? (int64_t)W * H : 1; // (between pixels, between channels)
    const float vo0 = inside ? v_image[step * pix] : 0.f, vo1 = inside ? v_image[step * pix + plane] : 0.f,
                vo2 = inside ? v_image[step * pix + 2 * plane] : 0.f;
    float behind = bg[0] * vo0 + bg[1] * vo1 + bg[2] * vo2;
    const bool tame = largest(vo0, vo1, vo2) < kTame && fabsf(behind) < kTame;
    bool wild = __builtin_amdgcn_ballot_w64(!tame) != 0; // (of this wavefront's pixels)
    int m = bin_final;
#pragma unroll
    for(int o = 4; o < DSX_WAVE; o <<= 1)
        m = max(m, __shfl_xor(m, o, DSX_WAVE));
    if(lane == 0)
        s_last[wave] = m;
    if(tid == 0)
    {
        s_a[kTileBatch] = s_c[kTileBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kTileBatch] = make_float4(0.f, 0.f, 0.f, __int_as_float(INT_MAX));
    }
    __syncthreads();
    m = s_last[0];
#pragma unroll
    for(int w = 1; w < kTileWaves; ++w)
        m = max(m, s_last[w]);
    m = __builtin_amdgcn_readfirstlane(m);

    // (where the lists start: as in the wavefront form)
    int pos = -1, left = 0, idx_next = 0;
    if(header == nullptr || *header == header_shift)
    {
        pos = min(min(ranges[tile + 1], k) - 1, m);
        idx_next = pos;
        left = pos - max(ranges[tile], 0) + 1;
    }
    left = __builtin_amdgcn_readfirstlane(left);

    // which of an entry's sums this lane adds, and where: rows 0 and 2 the eight that bank_sum8_scatter leaves, the odd rows' first
    // four lanes halves of the ninth
    const int row = lane >> 4;
    const bool carries = (row & 1) == 0 || (lane & 12) == 0;
    const int sum_shift = row & 1 ? 3 : 5;
    char* const my_sums = reinterpret_cast<char*>(
        s_sum + sum_at<kTileBatch + 1>(0, row & 1 ? 8 : 2 * row + 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1)));

    int id_ahead = 0;
    int summed = 0; // entries of the last round, whose sums are still to be added to memory
    if(tid < min(left, kTileBatch))
        id_ahead = ids[pos - tid];
    while(left > 0)
    {
        const int batch = min(left, kTileBatch);
        int id = id_ahead;
        pos -= batch;
        left -= batch;
        if(tid < min(left, kTileBatch))
            id_ahead = ids[pos - tid];
        uint32_t reached = 0;
        bool special = wild;
        float4 q0, q1, q2;
        float reach = 0.0f;
        const int idx = idx_next - tid;
        if(tid < batch)
        {
            id = (int)min((uint32_t)id, last_id);
            const float4* const rec = splats + 3 * (int64_t)id;
            q0 = rec[0], q1 = rec[1], q2 = rec[2];
            reach = reach_of(q1.w);
            const uint32_t blocks = blocks_reached(q0.x, q0.y, q1.x, q1.y, q1.z, reach, tile_x, tile_y) >> first_block;
#pragma unroll
            for(int w = 0; w < kTileWaves; ++w)
                if(idx <= s_last[w])
                    reached |= blocks & (1u << block_of_row(w));
            special = special || (reached != 0 && entry_kind(q0, q1, q2) != 0);
        }
        if(tid < batch) // (the loads end here: behind the adds they would wait for those)
            asm volatile("" : "+v"(q2.x), "+v"(q2.y), "+v"(q2.z), "+v"(q2.w));
        flush_sums<kTileBatch + 1>(s_sum, s_id, summed, grads, tid, kBlockThreads);
        const bool mine_special = __builtin_amdgcn_ballot_w64(special) != 0;
        if(lane == 0)
            s_special[wave] = mine_special;
        int staged;
        const int place = tile_place(s_counts, __builtin_amdgcn_ballot_w64(reached != 0), staged);
        // (the barrier inside: the last round's sums have been taken)
        for(int i = tid; i < 4 * staged; i += kBlockThreads)
            s_sum[i] = s_sum[sum_at<kTileBatch + 1>(0, 4) + i] = 0.0;
        if(tid < staged)
            s_sum[sum_at<kTileBatch + 1>(tid, 8)] = 0.0;
        if(reached != 0)
        {
            s_a[place] = make_float4(q0.x, q0.y, q1.x * 0.5f, q1.y);
            s_b[place] = make_float4(q1.z * 0.5f, q1.w, __uint_as_float(reach_limit_bwd(q1.w, reach)), __int_as_float(idx));
            s_c[place] = q2;
            s_id[place] = id;
            s_reach[place] = (uint16_t)reached;
        }
        idx_next -= batch;
        __syncthreads();

        // this wavefront's list: the places of the entries that reach its block, and nobody's at the end
        uint8_t* const bytes = reinterpret_cast<uint8_t*>(s_list[wave]);
        if(lane < kTileBatch / 4)
            s_list[wave][lane] = 0x01010101u * kTileBatch;
        int length = 0;
        for(int first = 0; first < staged; first += DSX_WAVE)
        {
            const int mine = first + lane;
            const uint64_t reaches = __builtin_amdgcn_ballot_w64(mine < staged && ((s_reach[min(mine, kTileBatch - 1)] >> block_of_row(wave)) & 1));
            if(__builtin_amdgcn_inverse_ballot_w64(reaches))
                bytes[length + bits_below_lane(reaches)] = (uint8_t)mine;
            length += __popcll(reaches);
        }
        // (one walk for all wavefronts: the sums' unit depends on it)
        const bool all_plain = __builtin_amdgcn_readfirstlane(s_special[0] | s_special[1] | s_special[2] | s_special[3]) == 0;
        auto walk = [&](auto plain) {
            const int rounds = (length + kBlockAtOnce - 1) / kBlockAtOnce;
            const uint32_t* my_list = s_list[wave];
            uint32_t places = *my_list;
            for(int i = 0; i < rounds; ++i)
            {
                const uint32_t here = __builtin_amdgcn_ubfe(places, 8 * slot, 8);
                places = *++my_list;
                const float4 A = s_a[here], B = s_b[here], C = s_c[here];
                float alpha, vis;
                const float dx = pxf - A.x, dy = pyf - A.y;
                uint64_t m_valid;
                {
#pragma clang fp contract(off)
                    // sigma exactly as the forward computed it
                    const ExponentX ex = exponent_x(A.z, A.w, dx);
                    const float sigma = __builtin_fmaf(__builtin_fmaf(B.x, dy, ex.bx), dy, ex.ax);
                    m_valid = __builtin_amdgcn_ballot_w64(__float_as_int(B.w) <= bin_final) &
                              __builtin_amdgcn_ballot_w64(__float_as_uint(sigma) <= __float_as_uint(B.z));
                    vis = __builtin_amdgcn_exp2f(-sigma * kLog2E);
                    const float full = plain ? B.y * vis : fminf(kAlphaMaxBwd, B.y * vis);
                    alpha = __builtin_amdgcn_inverse_ballot_w64(m_valid) ? full : 0.0f;
                }
                const float colour = C.x * vo0 + (C.y * vo1 + C.z * vo2);
                // the quad's four entries from the farthest one on: what they let through, and what lies behind each
                const float a[4] = {quad_lane<0x00>(alpha), quad_lane<0x55>(alpha), quad_lane<0xaa>(alpha), quad_lane<0xff>(alpha)};
                const float q[4] = {quad_lane<0x00>(colour), quad_lane<0x55>(colour), quad_lane<0xaa>(colour), quad_lane<0xff>(colour)};
                const float through0 = 1.0f - a[0], through1 = __builtin_fmaf(-a[1], through0, through0);
                const float through2 = __builtin_fmaf(-a[2], through1, through1), through3 = __builtin_fmaf(-a[3], through2, through2);
                const float T_here =
                    T * __builtin_amdgcn_rcpf(slot == 0 ? through0 : (slot == 1 ? through1 : (slot == 2 ? through2 : through3)));
                T = quad_lane<0xff>(T_here); // in front of all four
                float behind_here = behind;
#pragma unroll
                for(int u = 0; u < 4; ++u)
                {
                    behind_here = slot == u ? behind : behind_here;
                    const float next = behind + a[u] * (q[u] - behind);
                    behind = plain || a[u] != 0.0f ? next : behind; // (zero times infinity)
                }
                const float fac = alpha * T_here, ahead = colour - behind_here;
                float w = (plain ? fac : vis * T_here) * ahead;
                float v_red = fac * vo0, v_green = fac * vo1, v_blue = fac * vo2;
                if(!plain)
                {
                    // (a pixel that does not take the entry adds nothing, whatever its gradient: zero times infinity again)
                    const bool takes = __builtin_amdgcn_inverse_ballot_w64(m_valid);
                    w = takes ? w : 0.0f;
                    v_red = takes ? v_red : 0.0f;
                    v_green = takes ? v_green : 0.0f;
                    v_blue = takes ? v_blue : 0.0f;
                }
                const float wx = w * dx, wy = w * dy;
                const float sum8[8] = {w, wx, wx * dx, wy, wy * dx, wy * dy, v_red, v_green};
                float first, second;
                bank_sum8_scatter(sum8, first, second);
                v_blue = dpp_add<0x128>(v_blue);         // row_ror:8
                v_blue += dpp_move<0x104, true>(v_blue);  // row_shl:4 (the sum in every row's first four lanes)
                // (v_blue's two upper rows are the lower ones' other halves)
                const float halves = add_halves(first, second);
                const float total = add_rows(halves, v_blue);
                if(carries)
                    unsafeAtomicAdd(reinterpret_cast<double*>(my_sums + (here << sum_shift)), (double)total);
            }
        };
        if(all_plain)
            walk(std::true_type());
        else
        {
            walk(std::false_type());
            // (an infinite colour stays behind all entries in front)
            wild = wild || __builtin_amdgcn_ballot_w64(!(fabsf(behind) < kTame)) != 0;
        }
        __syncthreads();
        for(int e = tid; e < staged; e += kBlockThreads)
            moments_to_gradients<kTileBatch + 1>(s_sum, e, s_a[e], s_b[e], all_plain, marks ? marks + s_id[e] : nullptr);
        __syncthreads();
        summed = staged;
    }
    flush_sums<kTileBatch + 1>(s_sum, s_id, summed, grads, tid, kBlockThreads);
    if(zeros.any)
        zero_share(zeros, blockIdx.x, gridDim.x, tid, kBlockThreads);
}

// ranges, check_header, n, k: as for launch_blend_fwd (the kernel reads the `walk` part that the forward wrote)
int launch_blend_bwd(const dsx_camera& cam, int64_t n, int64_t k, const int32_t* ranges, const int32_t* sorted_ids,
                     const float* splats, const float* final_T, const int32_t* final_idx, const float* v_image,
                     float* grads, hipStream_t stream, bool check_header, bool grads_prepared, bool with_marks,
                     const ZeroJobs* zeros)
{
    if(k < 0 || k > 0x7fffffffll || (k > 0 && sorted_ids == nullptr))
        return DSX_ERR_BAD_ARG;
    // (the marks lie right behind the records, padded to whole words: one fill covers both)
    if(!grads_prepared)
        if(int rc = launch_fill_u32(reinterpret_cast<uint32_t*>(grads),
                                    with_marks ? (int64_t)(grads_bytes(n) / 4) : n * DSX_GRAD_FLOATS, 0u, stream))
            return rc;
    const ListGrid lg = list_grid(cam);
    const int ntx = lg.ntx, nty = lg.nty;
    if(ntx * nty == 0 || n == 0)
        return zeros ? launch_zero_outputs(*zeros, stream) : DSX_OK; // (no tile, no wavefront to store them)
    ZeroJobs Z = {};
    if(zeros)
        Z = *zeros;
    const BinLists L = bin_lists(lg, const_cast<int32_t*>(ranges));
    const int32_t* header = (lg.shift || check_header) ? ranges + ranges_layout(lg).header : nullptr;
    const uint32_t last_id = (uint32_t)(n - 1);
    {
        DSX_TIMED("blend_bwd_kernel", stream);
        const bool four = blend_pixels_per_lane(ntx * nty, kBwdFourPixelsFrom) == 4;
        const dim3 grid(ntx * nty);
        const float4* sp = reinterpret_cast<const float4*>(splats);
#define DSX_LAUNCH_BWD(KERNEL, THREADS)                                                                          \
    hipLaunchKernelGGL((KERNEL), grid, dim3(THREADS), 0, stream, ranges, sorted_ids, sp, final_T, final_idx, v_image, \
                       cam.bg, grads, with_marks ? grad_marks(grads, n) : nullptr, cam.image_width,                 \
                       cam.image_height, ntx, last_id, (int)k, header, lg.shift, camera_flag(cam, DSX_PLANAR_IMAGE), L, Z)
        const int tiles = ntx * nty;
        const bool blocks = forced_pixels_per_lane() == 0 && lg.shift == 0 && tiles <= kBwdBlocksUpTo &&
                            (tiles <= kBwdBlocksAlways || k * tiles <= kBwdBlocksShared * n);
        if(blocks)
            hipLaunchKernelGGL(blend_bwd_block_kernel, dim3(4 * ntx * nty), dim3(kBlockThreads), 0, stream, ranges, sorted_ids, sp, final_T,
                               final_idx, v_image, cam.bg, grads, with_marks ? grad_marks(grads, n) : nullptr, cam.image_width,
                               cam.image_height, ntx, last_id, (int)k, header, lg.shift, camera_flag(cam, DSX_PLANAR_IMAGE), Z);
        else if(four && lg.shift)
            DSX_LAUNCH_BWD(blend_bwd_kernel<true>, DSX_WAVE);
        else if(four)
            DSX_LAUNCH_BWD(blend_bwd_kernel<false>, DSX_WAVE);
        else if(lg.shift)
            DSX_LAUNCH_BWD(blend_bwd_tile_kernel<true>, kTileThreads);
        else
            DSX_LAUNCH_BWD(blend_bwd_tile_kernel<false>, kTileThreads);
#undef DSX_LAUNCH_BWD
    }
    DSX_LAUNCH_CHECK();
    return DSX_OK;
}

} // namespace dsx
