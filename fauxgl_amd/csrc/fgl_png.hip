// fgl_png.hip -- the context's color buffer as a PNG file, the way
// SavePNG (util.go:56-63) writes an *image.NRGBA through Go's image/png:
// RGB when every alpha is 255 (NRGBA.Opaque), RGBA otherwise; 8 bits per
// sample, no interlace; each row filtered with the filter image/png picks
// (the smallest sum of |byte| taken as signed, candidates in the order Up,
// Paeth, None, Sub, Average, the first minimum kept); one zlib stream.
//
// The compressed bytes are this build's own: the filtered stream is cut
// into PNG_CHUNK-byte pieces that one workgroup each deflates (runs of a
// repeated byte as distance-1 matches, the piece's own dynamic Huffman code
// or the fixed one, whichever is shorter) and ends with an empty stored
// block, so the pieces are byte-aligned and concatenate into one valid
// deflate stream.  The stream's Adler-32 and the pieces' part of the IDAT
// CRC are combined on the device too, so one small read tells the host the
// file's size and checksums.  Decoding gives back the same filtered bytes
// and the same pixels as Go's file.
#include "fgl_internal.h"

namespace fgl {

// any alpha below 255: flag[0] = 1 (every writer stores the same value)
__global__ __launch_bounds__(256) void k_png_opaque(const uint32_t *color, int64_t n, uint32_t *flag) {
    bool seen = false;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        seen |= (color[i] >> 24) != 255u;
    if (__ballot(seen) != 0 && (threadIdx.x & 63) == 0) flag[0] = 1u;
}

FGL_D int abs8(uint32_t d) { return d < 128u ? (int)d : 256 - (int)d; }
FGL_D uint32_t paeth(uint32_t a, uint32_t b, uint32_t c) {
    int pc = (int)c;
    int pa = (int)b - pc, pb = (int)a - pc;
    pc = abs(pa + pb);
    pa = abs(pa);
    pb = abs(pb);
    if (pa <= pb && pa <= pc) return a;
    if (pb <= pc) return b;
    return c;
}

// byte x under filter f (PNG types 0 None, 1 Sub, 2 Up, 3 Average, 4 Paeth)
// with its left, upper and upper left neighbours
FGL_D uint32_t png_filtered(int f, uint32_t x, uint32_t a, uint32_t b, uint32_t c) {
    switch (f) {
    case 0: return x;
    case 1: return (x - a) & 255u;
    case 2: return (x - b) & 255u;
    case 3: return (x - ((a + b) >> 1)) & 255u;
    default: return (x - paeth(a, b, c)) & 255u;
    }
}

// One workgroup per row, one pixel per lane: four word loads give all of a
// pixel's bytes and their neighbours (loading byte by byte, with a division
// for the pixel of an RGB byte, took 27 us for 1023x767; now 11).
// The five sums, the choice, the filtered row; neighbours outside the image
// are zero.
template <int BPP>
FGL_D void png_filter_row(const uint32_t *color, int32_t W, uint8_t *out, int (*part)[4], int *chosen) {
    const int y = blockIdx.x;
    const uint32_t *cur = color + (int64_t)y * W;
    int sum[5] = {0, 0, 0, 0, 0};
    for (int x = threadIdx.x; x < W; x += 256) {
        const uint32_t px = cur[x], pa = x > 0 ? cur[x - 1] : 0u;
        const uint32_t pb = y > 0 ? cur[x - W] : 0u, pc = (x > 0 && y > 0) ? cur[x - W - 1] : 0u;
#pragma unroll
        for (int ch = 0; ch < BPP; ch++) {
            const int sh = 8 * ch;
#pragma unroll
            for (int f = 0; f < 5; f++)
                sum[f] += abs8(png_filtered(f, (px >> sh) & 255u, (pa >> sh) & 255u, (pb >> sh) & 255u, (pc >> sh) & 255u));
        }
    }
#pragma unroll
    for (int f = 0; f < 5; f++) {
        int v = sum[f];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if ((threadIdx.x & 63) == 0) part[f][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot[5];
        for (int f = 0; f < 5; f++) tot[f] = part[f][0] + part[f][1] + part[f][2] + part[f][3];
        static const int order[5] = {2, 4, 0, 1, 3};  // Up, Paeth, None, Sub, Average
        int best = tot[2], pick = 2;
        for (int k = 1; k < 5; k++)
            if (tot[order[k]] < best) {
                best = tot[order[k]];
                pick = order[k];
            }
        *chosen = pick;
    }
    __syncthreads();
    const int f = *chosen;
    uint8_t *o = out + (int64_t)y * ((int64_t)W * BPP + 1);
    if (threadIdx.x == 0) o[0] = (uint8_t)f;
    for (int x = threadIdx.x; x < W; x += 256) {
        const uint32_t px = cur[x], pa = x > 0 ? cur[x - 1] : 0u;
        const uint32_t pb = y > 0 ? cur[x - W] : 0u, pc = (x > 0 && y > 0) ? cur[x - W - 1] : 0u;
#pragma unroll
        for (int ch = 0; ch < BPP; ch++) {
            const int sh = 8 * ch;
            o[1 + (int64_t)x * BPP + ch] =
                (uint8_t)png_filtered(f, (px >> sh) & 255u, (pa >> sh) & 255u, (pb >> sh) & 255u, (pc >> sh) & 255u);
        }
    }
}

__global__ __launch_bounds__(256) void k_png_filter(const uint32_t *color, int32_t W, const PngResult *res,
                                                    uint8_t *out) {
    __shared__ int part[5][4];
    __shared__ int chosen;
    if (res->translucent) png_filter_row<4>(color, W, out, part, &chosen);
    else png_filter_row<3>(color, W, out, part, &chosen);
}

// ---------------------------------------------------------------------------
// CRC-32 (ISO 3309, reflected) as polynomials over GF(2): bit 31 - k is the
// coefficient of x^k.  The register after a block B that follows state s is
// s * x^(8 |B|) + raw(B), raw(B) the register B leaves from 0.

constexpr uint32_t CRC_POLY = 0xEDB88320u;

__host__ __device__ constexpr uint32_t crc_mul(uint32_t a, uint32_t b) {
    uint32_t r = 0;
    for (int k = 0; k < 32; k++) {
        if (b & 0x80000000u) r ^= a;
        b <<= 1;
        a = (a >> 1) ^ ((a & 1u) ? CRC_POLY : 0u);
    }
    return r;
}
// x^(8 n)
__host__ __device__ constexpr uint32_t crc_shift(uint64_t n) {
    uint32_t r = 0x80000000u, q = 0x00800000u;  // 1, x^8
    for (; n; n >>= 1) {
        if (n & 1) r = crc_mul(r, q);
        q = crc_mul(q, q);
    }
    return r;
}
uint32_t png_crc_append(uint32_t state, uint32_t raw, uint64_t n) { return crc_mul(state, crc_shift(n)) ^ raw; }

// ---------------------------------------------------------------------------
// deflate (RFC 1951), one workgroup per piece

constexpr int PD_THREADS = 256, PD_WAVES = PD_THREADS / 64;
constexpr int PD_BYTES = PNG_CHUNK / PD_THREADS;  // bytes a thread owns
static_assert(PD_BYTES == 16, "a thread's bytes are one 16-byte load");
constexpr int NLIT = 286;  // literal/length symbols
constexpr int NCL = 19;    // code-length symbols
constexpr int PD_SYM = 288;  // table size (a multiple of 4 above NLIT + 1)
// bytes of the finished piece a thread's CRC slice covers (all slices equal,
// the piece padded in front with zeros, which leave the register at 0)
constexpr int PD_CRC = 20;
static_assert(PD_CRC * PD_THREADS >= PNG_CAP_WORDS * 4, "the slices cover the longest piece");

__constant__ uint16_t c_len_base[29] = {3,  4,  5,  6,  7,  8,  9,  10, 11,  13,  15,  17,  19,  23, 27,
                                        31, 35, 43, 51, 59, 67, 83, 99, 115, 131, 163, 195, 227, 258};
__constant__ uint8_t c_len_extra[29] = {0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 3, 3, 4, 4, 4, 4, 5, 5, 5, 5, 0};
// order in which the code-length code lengths are sent (RFC 1951 3.2.7)
__constant__ uint8_t c_cl_order[NCL] = {16, 17, 18, 0, 8, 7, 9, 6, 10, 5, 11, 4, 12, 3, 13, 2, 14, 1, 15};

FGL_D int len_sym(int len) {  // match length 3..258 -> index into the length tables
    int k = 28;
    while (c_len_base[k] > len) k--;
    return k;
}
FGL_D int fixed_len(int s) { return s < 144 ? 8 : s < 256 ? 9 : s < 280 ? 7 : 8; }
FGL_D uint32_t fixed_code(int s) {  // RFC 1951 3.2.6, most significant bit first
    return s < 144 ? 0x30u + s : s < 256 ? 0x190u + (s - 144) : s < 280 ? s - 256 : 0xC0u + (s - 280);
}

// The tokens of a run of r equal bytes: a literal, then distance-1 matches
// of up to 258 (none leaving a remainder of 1 or 2), then what is left as
// literals.  g(match length) per match; returns the literals.
template <typename Match>
FGL_D int run_tokens(int r, Match g) {
    int rest = r - 1;
    while (rest >= 3) {
        int m = rest < 258 ? rest : 258;
        if (rest - m > 0 && rest - m < 3) m -= 3;
        g(m);
        rest -= m;
    }
    return 1 + rest;
}

// The symbols a run of r equal code lengths v is sent as (RFC 1951 3.2.7):
// f(symbol, extra bits' value) per symbol.
template <typename F>
FGL_D void cl_tokens(int v, int r, F f) {
    int left = r;
    if (v == 0) {
        while (left >= 11) {
            const int k = left < 138 ? left : 138;
            f(18, k - 11);
            left -= k;
        }
        if (left >= 3) {
            f(17, left - 3);
            left = 0;
        }
    } else {
        f(v, 0);
        left--;
        while (left >= 3) {
            const int k = left < 6 ? left : 6;
            f(16, k - 3);
            left -= k;
        }
    }
    for (; left > 0; left--) f(v, 0);
}
FGL_D int cl_extra(int s) { return s == 16 ? 2 : s == 17 ? 3 : s == 18 ? 7 : 0; }

struct PdShared {
    uint32_t out[PNG_CAP_WORDS];
    __align__(16) uint8_t bytes[PNG_CHUNK];
    uint32_t freq[PD_SYM];
    __align__(16) uint32_t key[PD_SYM];  // sort keys, then internal nodes per depth
    uint32_t w[PD_SYM];                  // leaf weights in ascending order, then leaf depths
    uint32_t inner[PD_SYM];              // internal node weights
    uint16_t parent[PD_SYM];             // parent of each internal node
    uint16_t sym[PD_SYM];                // symbols in ascending frequency
    uint16_t code[PD_SYM];
    uint8_t len[PD_SYM];
    uint16_t rle[PD_SYM];                // code-length symbol | extra << 5
    uint32_t starts[PD_SYM / 32];        // runs of equal code lengths
    uint32_t clfreq[32];
    uint16_t clcode[32];
    uint8_t cllen[32];
    uint32_t count[16];
    uint32_t wsum[PD_WAVES];
    uint32_t first[PD_WAVES];            // first run start of each wave's bytes
    uint32_t red[PD_WAVES][4];
    uint32_t table[256];                 // CRC of one byte
    int32_t ok, hlit;
};

// Exclusive prefix of v over the workgroup; *total = the sum.
FGL_D uint32_t pd_scan(PdShared &h, uint32_t v, uint32_t *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) h.wsum[wave] = x;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < PD_WAVES; w++) {
        if (w < wave) base += h.wsum[w];
        tot += h.wsum[w];
    }
    __syncthreads();
    *total = tot;
    return base + x - v;
}

// Sums of up to four values over the workgroup, in every thread.
template <int N>
FGL_D void pd_sum(PdShared &h, uint32_t (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k++) {
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off);
        if ((threadIdx.x & 63) == 0) h.red[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        v[k] = 0;
        for (int w = 0; w < PD_WAVES; w++) v[k] += h.red[w][k];
    }
    __syncthreads();
}

// ORs bit fields into the zeroed output words, least significant bit first.
struct BitOr {
    uint32_t *w;
    uint64_t acc;
    int nbits;
    FGL_D BitOr(uint32_t *out, uint32_t at) : w(out + (at >> 5)), acc(0), nbits((int)(at & 31u)) {}
    FGL_D void put(uint32_t v, int n) {  // n <= 24
        acc |= (uint64_t)v << nbits;
        nbits += n;
        if (nbits >= 32) {
            atomicOr(w++, (uint32_t)acc);
            acc >>= 32;
            nbits -= 32;
        }
    }
    FGL_D void flush() {
        if (nbits) atomicOr(w, (uint32_t)acc);
    }
};

// Code lengths of a Huffman code for freq[0..n) (symbols with freq 0 get
// length 0), no longer than limit: minimum-redundancy lengths by Moffat and
// Katajainen's two-queue method ("In-place calculation of
// minimum-redundancy codes", 1995) on the used symbols sorted by frequency
// (ties by symbol); if the longest exceeds limit, the frequencies are halved
// (rounding up) and the code is built again, which keeps it a complete
// prefix code.  At least two symbols are used: a piece has a literal and the
// end of block, and the lengths sent are not all equal (the distance code's
// is 1).  The workgroup sorts by counting smaller keys and walks each
// internal node's depth in parallel; only the merge of the two queues, a
// chain of at most 284 steps, is one thread's work.
FGL_D void pd_huff_lengths(PdShared &h, const uint32_t *freq, int n, int limit, uint8_t *len) {
    const int tid = threadIdx.x;
    for (int i = tid; i < PD_SYM; i += PD_THREADS) {
        const uint32_t f = i < n ? freq[i] : 0u;
        h.key[i] = f ? (f << 9) | (uint32_t)i : ~0u;
        if (i < n) len[i] = 0;
    }
    __syncthreads();
    uint32_t used = 0;
    for (int i = tid; i < n; i += PD_THREADS) {
        const uint32_t k = h.key[i];
        if (k == ~0u) continue;
        used++;
        uint32_t rank = 0;
        for (int j = 0; j < n; j += 4) {
            const uint4 q = *reinterpret_cast<const uint4 *>(&h.key[j]);
            rank += (q.x < k) + (q.y < k) + (q.z < k) + (q.w < k);
        }
        h.sym[rank] = (uint16_t)i;
    }
    uint32_t tot;
    (void)pd_scan(h, used, &tot);
    const int m = (int)tot;
    for (int shift = 0;; shift++) {
        for (int i = tid; i < PD_SYM; i += PD_THREADS) {
            h.w[i] = i < m ? ((freq[h.sym[i]] - 1) >> shift) + 1 : ~0u;
            h.key[i] = 0;
        }
        __syncthreads();
        if (tid == 0) {
            // the two queues: leaves w[leaf ..] (the next two held in
            // registers) and internal nodes inner[root .. next)
            uint32_t l0 = h.w[2], l1 = h.w[3];  // ~0 past the last leaf
            int leaf = 2, root = 0;
            uint32_t r0 = h.w[0] + h.w[1];  // inner[root] when root < next
            h.inner[0] = r0;
            for (int next = 1; next < m - 1; next++) {
                uint32_t s = 0;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    if (root < next && r0 < l0) {
                        s += r0;
                        h.parent[root] = (uint16_t)next;
                        root++;
                        r0 = h.inner[root < next ? root : 0];
                    } else {
                        s += l0;
                        l0 = l1;
                        leaf++;
                        l1 = h.w[leaf + 1 < PD_SYM ? leaf + 1 : PD_SYM - 1];
                    }
                }
                h.inner[next] = s;
                if (root == next) r0 = s;
            }
        }
        __syncthreads();
        // depth of each internal node (the root is node m - 2), counted
        for (int i = tid; i < m - 1; i += PD_THREADS) {
            int d = 0;
            for (int q = i; q != m - 2; q = h.parent[q]) d++;
            atomicAdd(&h.key[d], 1u);
        }
        __syncthreads();
        if (tid == 0) {
            // leaves per depth, the most frequent symbols first
            int avail = 1, depth = 0, at = m - 1;
            while (avail > 0) {
                const int used_d = (int)h.key[depth];
                for (int q = avail - used_d; q > 0; q--) h.w[at--] = (uint32_t)depth;
                avail = 2 * used_d;
                depth++;
            }
            h.ok = (int)h.w[0] <= limit;  // the rarest symbol has the longest code
        }
        __syncthreads();
        if (h.ok) break;
        __syncthreads();
    }
    for (int i = tid; i < m; i += PD_THREADS) len[h.sym[i]] = (uint8_t)h.w[i];
    __syncthreads();
}

// canonical codes (RFC 1951 3.2.2), bit-reversed for LSB-first output, by
// the first wave: 64 symbols at a time, equal lengths ranked by ballots
FGL_D void pd_huff_codes(PdShared &h, const uint8_t *len, int n, uint16_t *code) {
    const int tid = threadIdx.x;
    if (tid < 16) h.count[tid] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += PD_THREADS)
        if (len[i]) atomicAdd(&h.count[len[i]], 1u);
    __syncthreads();
    uint32_t first = 0;  // first code of length tid
    if (tid < 16) {
        uint32_t c = 0;
        for (int b = 1; b <= tid; b++) c = (c + (b > 1 ? h.count[b - 1] : 0u)) << 1;
        first = c;
    }
    __syncthreads();
    if (tid < 16) h.count[tid] = first;
    __syncthreads();
    if (tid < 64) {
        for (int i0 = 0; i0 < n; i0 += 64) {
            const int i = i0 + tid;
            const uint32_t l = i < n ? len[i] : 0u;
            uint64_t peers = __ballot(l != 0);
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const bool bit = (l >> b) & 1u;
                const uint64_t mm = __ballot(bit);
                peers &= bit ? mm : ~mm;
            }
            const uint32_t rank = (uint32_t)__popcll(peers & ((1ull << tid) - 1ull));
            const uint32_t base = l ? h.count[l] : 0u;
            __builtin_amdgcn_wave_barrier();
            if (l && rank == 0) h.count[l] = base + (uint32_t)__popcll(peers);
            __builtin_amdgcn_wave_barrier();
            if (i < n) code[i] = l ? (uint16_t)(__brev(base + rank) >> (32 - l)) : (uint16_t)0;
        }
    }
    __syncthreads();
}

// Piece c covers bytes [c * PNG_CHUNK, min(n, (c + 1) * PNG_CHUNK)) of the
// filtered stream; its words go to out + c * PNG_CAP_WORDS.  The block uses
// fixed or dynamic codes, whichever is shorter, so a piece never exceeds the
// fixed-code bound PNG_CAP_WORDS is sized for.
//
// What bounds it: the latency of one piece's chain (loads, histogram, the
// serial queue merge, the prefix sums), six pieces to a CU at a time.  One
// thread per piece (16 to a workgroup), the earlier form, ran the whole piece
// as a chain of byte loads and LDS scratch accesses: 13.3 ms for the 576
// pieces of a 1023x767 image, on 36 of the 256 CUs; now 0.119 ms.
__global__ __launch_bounds__(PD_THREADS) void k_png_deflate(const uint8_t *s, int32_t W, int32_t H,
                                                            const PngResult *res, uint32_t *out, PngPiece *pieces) {
    __shared__ PdShared h;
    const int64_t n = (int64_t)H * ((int64_t)W * (res->translucent ? 4 : 3) + 1);
    const int64_t b0 = (int64_t)blockIdx.x * PNG_CHUNK;
    if (b0 >= n) return;
    const int len = (int)((n - b0) < PNG_CHUNK ? (n - b0) : PNG_CHUNK);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int p0 = tid * PD_BYTES;
    const int mine = len - p0 < 0 ? 0 : (len - p0 < PD_BYTES ? len - p0 : PD_BYTES);

    // the thread's bytes (the stream buffer is a whole number of pieces)
    const uint4 v4 = *reinterpret_cast<const uint4 *>(s + b0 + p0);
    *reinterpret_cast<uint4 *>(&h.bytes[p0]) = v4;
    for (int i = tid; i < PNG_CAP_WORDS; i += PD_THREADS) h.out[i] = 0;
    for (int i = tid; i < PD_SYM; i += PD_THREADS) h.freq[i] = i == 256 ? 1u : 0u;
    if (tid < 32) h.clfreq[tid] = 0;
    if (tid < PD_SYM / 32) h.starts[tid] = 0;
    {
        uint32_t c = (uint32_t)tid;
#pragma unroll
        for (int k = 0; k < 8; k++) c = (c >> 1) ^ ((c & 1u) ? CRC_POLY : 0u);
        h.table[tid] = c;
    }
    if (tid == 0) h.hlit = 257;
    __syncthreads();
    const uint32_t vw[4] = {v4.x, v4.y, v4.z, v4.w};
    auto byte = [&](int k) { return (vw[k >> 2] >> (8 * (k & 3))) & 255u; };

    // run starts among the thread's bytes, and the first start after them
    uint32_t starts = 0;
    uint32_t sums[2] = {0, 0};  // Adler-32 parts: sum of bytes, sum of (len - i) * byte i (below 2^32 for a piece)
    {
        uint32_t prev = p0 > 0 ? h.bytes[p0 - 1] : 256u;
#pragma unroll
        for (int k = 0; k < PD_BYTES; k++) {
            if (k < mine) {
                const uint32_t b = byte(k);
                if (b != prev) starts |= 1u << k;
                prev = b;
                sums[0] += b;
                sums[1] += (uint32_t)(len - p0 - k) * b;
            }
        }
    }
    const uint64_t any = __ballot(starts != 0);
    const uint32_t my_first = (uint32_t)p0 + (uint32_t)(starts ? __builtin_ctz(starts) : 0);
    if (any ? lane == __builtin_ctzll(any) : lane == 0) h.first[wave] = any ? my_first : (uint32_t)len;
    const uint64_t later = lane == 63 ? 0 : any >> (lane + 1);
    const uint32_t in_wave = __shfl(my_first, later ? lane + 1 + __builtin_ctzll(later) : lane);
    __syncthreads();
    int next_start = len;
    if (later) {
        next_start = (int)in_wave;
    } else {
        for (int w = PD_WAVES - 1; w > wave; w--)
            if (h.first[w] < (uint32_t)next_start) next_start = (int)h.first[w];
    }
    // f(first byte's position in the thread's bytes, run length) per run
    auto runs = [&](auto f) {
        for (uint32_t rest = starts; rest;) {
            const int k = __builtin_ctz(rest);
            rest &= rest - 1;
            f(k, (rest ? p0 + __builtin_ctz(rest) : next_start) - (p0 + k));
        }
    };

    // symbol frequencies, the lengths' extra bits, the matches
    uint32_t bits[4] = {0, 0, sums[0], sums[1]};
    runs([&](int k, int r) {
        const int lits = run_tokens(r, [&](int m) {
            const int q = len_sym(m);
            atomicAdd(&h.freq[257 + q], 1u);
            bits[0] += c_len_extra[q];
            bits[1]++;
        });
        atomicAdd(&h.freq[h.bytes[p0 + k]], (uint32_t)lits);
    });
    pd_sum(h, bits);
    const uint32_t extra_bits = bits[0], nmatch = bits[1], sa = bits[2], sb = bits[3];

    // dynamic code: literal/length lengths, the run-length coded length
    // sequence, the code-length code
    pd_huff_lengths(h, h.freq, NLIT, 15, h.len);
    for (int i = tid; i < NLIT; i += PD_THREADS)
        if (h.len[i]) atomicMax(&h.hlit, i + 1);
    __syncthreads();
    const int hlit = h.hlit, nlen = hlit + 1;
    if (tid == 0) h.len[hlit] = 1;  // the one distance code (distance 1), one bit
    __syncthreads();
    for (int i = tid; i < nlen; i += PD_THREADS)
        if (i == 0 || h.len[i] != h.len[i - 1]) atomicOr(&h.starts[i >> 5], 1u << (i & 31));
    __syncthreads();
    // two entries a thread; a run is its first entry's
    int run_of[2] = {0, 0};
    uint32_t nsym = 0;
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int i = 2 * tid + e;
        if (i >= nlen || !((h.starts[i >> 5] >> (i & 31)) & 1u)) continue;
        int j = i + 1;
        while (j < nlen) {
            const uint32_t rest = h.starts[j >> 5] >> (j & 31);
            if (rest) {
                j += __builtin_ctz(rest);
                break;
            }
            j = (j | 31) + 1;
        }
        run_of[e] = (j < nlen ? j : nlen) - i;
        cl_tokens(h.len[i], run_of[e], [&](int, int) { nsym++; });
    }
    uint32_t nrle;
    uint32_t at = pd_scan(h, nsym, &nrle);
#pragma unroll
    for (int e = 0; e < 2; e++) {
        if (!run_of[e]) continue;
        cl_tokens(h.len[2 * tid + e], run_of[e], [&](int sy, int ex) {
            h.rle[at++] = (uint16_t)(sy | (ex << 5));
            atomicAdd(&h.clfreq[sy], 1u);
        });
    }
    __syncthreads();
    pd_huff_lengths(h, h.clfreq, NCL, 7, h.cllen);
    int hclen = NCL;
    while (hclen > 4 && h.cllen[c_cl_order[hclen - 1]] == 0) hclen--;
    // bits of the code lengths' symbols (two a thread, in order), of the
    // tokens under the dynamic and under the fixed code
    uint32_t cl_bits = 0;
    uint32_t cost[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const uint32_t i = 2 * tid + e;
        if (i < nrle) cl_bits += h.cllen[h.rle[i] & 31] + cl_extra(h.rle[i] & 31);
    }
    for (int i = tid; i < NLIT; i += PD_THREADS) {
        cost[1] += h.freq[i] * h.len[i] * (i < hlit ? 1u : 0u);
        cost[2] += h.freq[i] * (uint32_t)fixed_len(i);
    }
    cost[0] = cl_bits;
    pd_sum(h, cost);
    const uint32_t dyn_bits = 3 + 5 + 5 + 4 + 3u * hclen + cost[0] + cost[1] + extra_bits + nmatch;
    const uint32_t fixed_bits = 3 + cost[2] + extra_bits + 5 * nmatch;
    const bool dyn = dyn_bits < fixed_bits;

    uint32_t pos;  // bits before the tokens
    if (dyn) {
        pd_huff_codes(h, h.len, hlit, h.code);
        pd_huff_codes(h, h.cllen, NCL, h.clcode);
        uint32_t total;
        const uint32_t before = pd_scan(h, cl_bits, &total);
        if (tid == 0) {
            BitOr bo(h.out, 0);
            bo.put(0u | (2u << 1), 3);  // BFINAL 0, BTYPE 10: dynamic codes
            bo.put((uint32_t)(hlit - 257), 5);
            bo.put(0u, 5);  // HDIST - 1: one distance code
            bo.put((uint32_t)(hclen - 4), 4);
            for (int i = 0; i < hclen; i++) bo.put(h.cllen[c_cl_order[i]], 3);
            bo.flush();
        }
        BitOr bo(h.out, 17u + 3u * hclen + before);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint32_t i = 2 * tid + e;
            if (i >= nrle) continue;
            const int cs = h.rle[i] & 31;
            bo.put(h.clcode[cs], h.cllen[cs]);
            if (cl_extra(cs)) bo.put((uint32_t)(h.rle[i] >> 5), cl_extra(cs));
        }
        if (2u * tid < nrle) bo.flush();
        pos = 17u + 3u * hclen + total;
    } else {
        for (int i = tid; i < NLIT; i += PD_THREADS) {
            h.len[i] = (uint8_t)fixed_len(i);
            h.code[i] = (uint16_t)(__brev(fixed_code(i)) >> (32 - fixed_len(i)));
        }
        if (tid == 0) atomicOr(&h.out[0], 1u << 1);  // BFINAL 0, BTYPE 01: fixed codes
        pos = 3;
        __syncthreads();
    }
    const int dist_bits = dyn ? 1 : 5;  // distance code 0 (distance 1) is all zeros
    uint32_t tok_bits = 0;
    runs([&](int k, int r) {
        const int lits = run_tokens(r, [&](int m) {
            const int q = len_sym(m);
            tok_bits += h.len[257 + q] + c_len_extra[q] + dist_bits;
        });
        tok_bits += (uint32_t)lits * h.len[h.bytes[p0 + k]];
    });
    uint32_t all_tok;
    const uint32_t before = pd_scan(h, tok_bits, &all_tok);
    if (tok_bits) {
        BitOr bo(h.out, pos + before);
        runs([&](int k, int r) {
            const uint32_t v = h.bytes[p0 + k];
            const uint32_t code = h.code[v];
            const int cl = h.len[v];
            bo.put(code, cl);
            int lits = run_tokens(r, [&](int m) {
                const int q = len_sym(m);
                bo.put(h.code[257 + q], h.len[257 + q]);
                if (c_len_extra[q]) bo.put((uint32_t)(m - c_len_base[q]), c_len_extra[q]);
                bo.put(0u, dist_bits);
            });
            for (; lits > 1; lits--) bo.put(code, cl);
        });
        bo.flush();
    }
    pos += all_tok;
    // end of block, then an empty stored block, which brings the piece to a
    // byte boundary
    const uint32_t eob_bits = h.len[256];
    const uint32_t stored = (pos + eob_bits + 3 + 7) & ~7u;  // where LEN and NLEN start
    if (tid == 0) {
        BitOr bo(h.out, pos);
        bo.put(h.code[256], (int)eob_bits);
        bo.flush();
        BitOr be(h.out, stored);
        be.put(0x0000u, 16);
        be.put(0xFFFFu, 16);
        be.flush();
    }
    __syncthreads();
    const int size = (int)(stored / 8) + 4;
    uint32_t *dst = out + (int64_t)blockIdx.x * PNG_CAP_WORDS;
    for (int i = tid; 4 * i < size; i += PD_THREADS) dst[i] = h.out[i];

    // raw CRC of the piece: PD_CRC bytes a thread, combined pairwise
    const uint8_t *ob = reinterpret_cast<const uint8_t *>(h.out);
    uint32_t crc = 0;
    for (int k = 0; k < PD_CRC; k++) {
        const int i = size - PD_CRC * PD_THREADS + PD_CRC * tid + k;
        if (i >= 0) crc = h.table[(crc ^ ob[i]) & 255u] ^ (crc >> 8);
    }
    constexpr uint32_t sh[8] = {crc_shift(PD_CRC),      crc_shift(PD_CRC * 2),  crc_shift(PD_CRC * 4),
                                crc_shift(PD_CRC * 8),  crc_shift(PD_CRC * 16), crc_shift(PD_CRC * 32),
                                crc_shift(PD_CRC * 64), crc_shift(PD_CRC * 128)};
#pragma unroll
    for (int l = 0; l < 6; l++) {
        const uint32_t right = __shfl_down(crc, 1 << l);
        crc = crc_mul(crc, sh[l]) ^ right;  // lanes that are no left partner keep a value nobody reads
    }
    if (lane == 0) h.wsum[wave] = crc;
    __syncthreads();
    if (tid == 0) {
        const uint32_t left = crc_mul(h.wsum[0], sh[6]) ^ h.wsum[1], right = crc_mul(h.wsum[2], sh[6]) ^ h.wsum[3];
        PngPiece &pc = pieces[blockIdx.x];
        pc.size = (uint32_t)size;
        pc.sa = sa % 65521u;
        pc.sb = sb % 65521u;
        pc.crc = crc_mul(left, sh[7]) ^ right;
    }
}

// One workgroup: the pieces' offsets (exclusive prefix of their sizes), the
// size of the stream and its Adler-32: from a = 1 + all bytes before a piece
// and b, a piece of p bytes makes b + p * a + sb.
constexpr int PS_THREADS = 1024;
__global__ __launch_bounds__(PS_THREADS) void k_png_scan(const PngPiece *pieces, int32_t W, int32_t H, PngResult *res,
                                                         uint64_t *offs) {
    __shared__ uint64_t ws[PS_THREADS / 64][2];
    __shared__ uint32_t wb[PS_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n = (int64_t)H * ((int64_t)W * (res->translucent ? 4 : 3) + 1);
    const int64_t np = (n + PNG_CHUNK - 1) / PNG_CHUNK;
    uint64_t size0 = 0, a0 = 1;
    uint32_t b = 0;
    for (int64_t k0 = 0; k0 < np; k0 += PS_THREADS) {
        const int64_t k = k0 + tid;
        const PngPiece pc = k < np ? pieces[k] : PngPiece{0, 0, 0, 0};
        uint64_t x = pc.size, y = pc.sa;
        for (int off = 1; off < 64; off <<= 1) {
            const uint64_t u = __shfl_up(x, off), v = __shfl_up(y, off);
            if (lane >= off) {
                x += u;
                y += v;
            }
        }
        if (lane == 63) {
            ws[wave][0] = x;
            ws[wave][1] = y;
        }
        __syncthreads();
        uint64_t xb = size0, yb = a0;
        for (int w = 0; w < PS_THREADS / 64; w++) {
            if (w < wave) {
                xb += ws[w][0];
                yb += ws[w][1];
            }
            size0 += ws[w][0];
            a0 += ws[w][1];
        }
        if (k < np) {
            offs[k] = xb + x - pc.size;
            const uint64_t plen = (uint64_t)((n - k * PNG_CHUNK) < PNG_CHUNK ? (n - k * PNG_CHUNK) : PNG_CHUNK);
            b = (uint32_t)((b + plen * ((yb + y - pc.sa) % 65521u) + pc.sb) % 65521u);
        }
        __syncthreads();
    }
    for (int off = 32; off > 0; off >>= 1) b += __shfl_xor(b, off);  // 64 values below 65521
    if (lane == 0) wb[wave] = b;
    __syncthreads();
    if (tid == 0) {
        uint32_t s = 0;
        for (int w = 0; w < PS_THREADS / 64; w++) s += wb[w];
        res->total = size0;
        res->adler = ((s % 65521u) << 16) | (uint32_t)(a0 % 65521u);
    }
}

// x^(8 * 2^k)
struct CrcPow {
    uint32_t v[40];
};
constexpr CrcPow crc_pow_table() {
    CrcPow t{};
    uint32_t q = 0x00800000u;
    for (int k = 0; k < 40; k++) {
        t.v[k] = q;
        q = crc_mul(q, q);
    }
    return t;
}
__constant__ CrcPow c_crc_pow = crc_pow_table();

// Pieces packed back to back at their offsets, four bytes a lane where the
// destination is aligned (the source is read from LDS at any byte); each
// piece's CRC moved to its place in the stream's.
__global__ __launch_bounds__(256) void k_png_pack(const uint32_t *words, const PngPiece *pieces, const uint64_t *offs,
                                                  int32_t W, int32_t H, PngResult *res, uint8_t *dst) {
    __shared__ uint32_t w[PNG_CAP_WORDS + 1];
    const int64_t c = blockIdx.x;
    const int64_t n = (int64_t)H * ((int64_t)W * (res->translucent ? 4 : 3) + 1);
    if (c * PNG_CHUNK >= n) return;
    const int size = (int)pieces[c].size, tid = threadIdx.x;
    const uint32_t *src = words + c * PNG_CAP_WORDS;
    for (int i = tid; 4 * i < size; i += 256) w[i] = src[i];
    __syncthreads();
    const uint8_t *sb = reinterpret_cast<const uint8_t *>(w);
    uint8_t *d = dst + offs[c];
    const int lead = (int)((4 - (offs[c] & 3)) & 3);  // bytes before the first aligned word (dst is aligned)
    const int nw = size > lead ? (size - lead) / 4 : 0;
    if (tid < lead && tid < size) d[tid] = sb[tid];
    uint32_t *dw = reinterpret_cast<uint32_t *>(d + lead);
    for (int i = tid; i < nw; i += 256) dw[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], (uint32_t)lead);
    const int tail = lead + 4 * nw;
    if (tid < size - tail) d[tail + tid] = sb[tail + tid];
    if (tid < 64) {
        // x^(8 after), after = the stream's bytes behind the piece: lane k
        // holds the factor of bit k, multiplied pairwise
        const uint64_t after = res->total - offs[c] - (uint64_t)size;
        uint32_t f = tid < 40 && ((after >> tid) & 1) ? c_crc_pow.v[tid < 40 ? tid : 0] : 0x80000000u;
#pragma unroll
        for (int l = 0; l < 6; l++) f = crc_mul(f, __shfl_xor(f, 1 << l));
        if (tid == 0) atomicXor(&res->crc, crc_mul(pieces[c].crc, f));
    }
}

hipError_t launch_png_opaque(const uint32_t *color, int64_t n, PngResult *res, hipStream_t s) {
    int64_t b = (n + 255) / 256;
    hipLaunchKernelGGL(k_png_opaque, dim3((unsigned)(b < 1 ? 1 : (b > 4096 ? 4096 : b))), dim3(256), 0, s, color, n,
                       &res->translucent);
    return hipGetLastError();
}
hipError_t launch_png_filter(const uint32_t *color, int32_t W, int32_t H, const PngResult *res, uint8_t *out,
                             hipStream_t s) {
    hipLaunchKernelGGL(k_png_filter, dim3(H), dim3(256), 0, s, color, W, res, out);
    return hipGetLastError();
}
hipError_t launch_png_deflate(const uint8_t *stream, int32_t W, int32_t H, const PngResult *res, int64_t npieces,
                              uint32_t *out, PngPiece *pieces, hipStream_t s) {
    hipLaunchKernelGGL(k_png_deflate, dim3((unsigned)npieces), dim3(PD_THREADS), 0, s, stream, W, H, res, out, pieces);
    return hipGetLastError();
}
hipError_t launch_png_scan(const PngPiece *pieces, int32_t W, int32_t H, PngResult *res, uint64_t *offs,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_png_scan, dim3(1), dim3(PS_THREADS), 0, s, pieces, W, H, res, offs);
    return hipGetLastError();
}
hipError_t launch_png_pack(const uint32_t *words, const PngPiece *pieces, const uint64_t *offs, int32_t W, int32_t H,
                           int64_t npieces, PngResult *res, uint8_t *dst, hipStream_t s) {
    hipLaunchKernelGGL(k_png_pack, dim3((unsigned)npieces), dim3(256), 0, s, words, pieces, offs, W, H, res, dst);
    return hipGetLastError();
}

}  // namespace fgl
