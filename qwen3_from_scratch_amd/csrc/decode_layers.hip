// All decoder layers of a step of single tokens in one launch: pre-norm layers of softmax attention with grouped heads of 128 and a
// gated unit, bfloat16, up to 32 rows, of some shapes 24 or 16, or 3 to 8 of a wide one. What gemm.hip's few-row products and attention.hip's decoding attention do layer by layer.
//
// A kernel that waits for its predecessor costs 2 us inside a graph if it does nothing and 4 to 4.5 if it loads, reduces and stores a
// row, and a step of the 0.6B shape was 145 of them: 1,011 us where its bytes take 240. Here a block per compute unit stays for all
// layers and blocks exchange rows through memory past the chiplets' own caches. What is exchanged says itself that it is there: the
// exchange is filled with words of ones (ABSENT) beforehand, a block stores its results and nobody anything else, and a reader asks for
// what it needs until no word of ones is among it. So a product's rows reach the next one in a store's way to memory and a load's
// back, some 1.2 us, where flags behind the data took 3.8 and a barrier of all blocks alone 2.6 (256 blocks, 2,048 numbers a
// block). The weights of a product's first steps are asked for while the last one's results are on their way, so memory is not idle
// meanwhile.
//
// What it measured (us a step in a graph, the layers' kernels one by one / this): the 0.6B shape, one request over 100 keys 973 / 504,
// over 1,100 1,013 / 563, over 8,000 1,137 / 758, over 30,000 1,531 / 1,138, four over 1,100 1,145 / 623, eight over 2,000 1,412 / 876,
// sixteen 1,921 / 1,273, 20 over 770 1,433 / 990, 32 over 2,000 2,410 / 1,916; the 8B shape, one over 2,060 3,382 / 2,769, eight
// 3,923 / 3,157, sixteen 4,843 / 3,799, eight over 8,000 5,179 / 4,166, sixteen 6,773 / 5,802. With rows in one piece each (`place_of`) it was
// faster at each of 39 sizes of these two from 1 to 32 rows (16) and 100 to 30,000 keys, all contexts alike, by 3 percent (32 over 8,000)
// to 93; uneven ones: `share_out`; other shapes: `rows_most`.
//
// What bounds it: one request of the small shape the chain of five or six exchanges a layer; a look that fails costs a second one behind
// the first, a store holds up the wavefront's next look (they come back in order), and a wavefront alone on its SIMD takes 4 to 5 cycles
// an instruction, 20 for a number that goes from a vector's lane into scalar arithmetic. So what is between two exchanges is kept short:
// offsets that are constants of an instruction, steps of K in one stretch, bounds by the descriptors (500 instructions a product less:
// 801 -> 779), the next weights asked for behind the results (779 -> 749; 8B 2,990 -> 2,860) and behind all wavefronts' results, with
// the shares of K read together (749 -> 701; 2,860 -> 2,820), blocks of their own for the products into the stream of a small model (701 -> 597),
// weights in registers that nothing copies (585 -> 576; 2,820 -> 2,760), lane sums in the vector unit (575 -> 563). The large shape is bound by its weights (5.5 of the
// 5.8 TB/s that a plain read reaches, the whole step through) and the attention's part, where few weights move.
// What did not help: the block split into wavefronts that multiply and wavefronts that look, prepare and store, with the weights in a
// ring in shared memory (0.6B 905: more handovers a product), asking for the sums of squares together with the rows (lines that many blocks
// write and all ask for again and again are slow to change: 915; in the rows' own lines, 80 bytes for 32 numbers, 600 for 576), copies of what all read (nothing), the first keys asked for ahead of
// the [q | k | v] product's end (937: a second copy of the product, 61 KB of code beyond what the instruction caches keep).
#include "common.h"
#include "attention_tiles.h"
#include "gates.h"

namespace {

typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2_t;

constexpr int WAVES = 8;                      // of a block
constexpr int THREADS = 64 * WAVES;
constexpr int HEAD = 128;                     // the head size
constexpr int MOST_SLABS = 8;                 // slabs of 16 weight rows that a block multiplies between two barriers
constexpr int RESULTS = 128;                  // of them times rows, at most
constexpr int CHUNKS = 16;                    // steps of K, times groups of sixteen rows, that a wavefront has in registers
constexpr unsigned ABSENT = 0xffffffffu;      // a word of the exchange that nobody has written yet
constexpr unsigned CLOSED = 0x80000000u;
enum { CAME, CLOSED_AT, GAVE_UP, CONTROL_WORDS };
constexpr int THROUGH = 16;                   // cache policy of what blocks exchange: past the chiplets' own caches (sc1)
constexpr int MOST_PARTS = 32;                // of a sequence's keys
constexpr int ITEMS_MOST = 512;               // pieces of attention, where sequences are in parts
constexpr int ROUND = 256;                    // of them that run side by side (not the launch's blocks: their number changes no bit)
constexpr int PIECE = 3;                      // steps of a wavefront's walk over tiles that the start of a piece is counted as
constexpr int MOST_ROWS = 32;                 // in two groups of sixteen
constexpr int MOST_LAYERS = 128;
constexpr int CLOSING = 1 << 18;               // looks for how many blocks there are, once their number is closed
constexpr int NOWHERE = 1 << 30;              // an offset behind the end of every buffer: reads of it are zero

// One layer as the host gives it and as the launch's table holds it.
struct Layer {
  const void* w[4];            // tile-ordered: [q | k | v], the attention's output, gate and up interleaved, down
  const void *q_norm, *k_norm, *entry_norm, *middle_norm;
  void *keys, *values;
  float entry_eps, middle_eps;
};
constexpr int LAYERS_A_LAUNCH = 40;           // as many as the preparing kernel's arguments hold
struct LayerPack {
  Layer layer[LAYERS_A_LAUNCH];
};

struct ShareArgs {
  const int* kv_lens;
  int rows, kv_heads, parts_most, items_most;
};
struct Args {
  const Layer* layers;
  unsigned* control;
  char* exchange;
  float* residual;
  const float* table;
  const int* block_table;
  long per_layer;              // bytes of exchange
  int at_part, at_att, at_mid, at_mid_sums, at_hid, at_out, at_out_sums;
  int at_ml;
  ShareArgs shares;
  int count, rows, width, heads, kv_heads, group, inner, norm_f32, max_pos, table_width, page, page_bits, num_pages, patience, limit;
  float qk_eps, scale_log2;
};

// The step's attention as pieces: a sequence's keys for one key head, in `parts` parts. Sequence b's are FIRST and those behind it,
// the parts of a key head side by side; those of sequences in many parts come first, and a block takes every so many-th.
struct Shares {
  __attribute__((aligned(16))) float tiles[MOST_ROWS];
  int first[MOST_ROWS], parts[MOST_ROWS], kv_len[MOST_ROWS];
  int items, in_parts;
};
struct AttentionShared {
  float k[HEAD], v[HEAD];                     // the token's own, as the caches hold them
  __attribute__((aligned(16))) bf16_t q[16][HEAD + 8];
  float m[WAVES + 1][16], l[WAVES][16];
  __attribute__((aligned(16))) float acc[WAVES][16][HEAD + 4];
};
struct Shared {
  // the wavefronts' shares of K of a product: [slab][wavefront][four columns of sixteen][row], 16 bytes each
  __attribute__((aligned(16))) char red[RESULTS * WAVES * 4 * 16];
  AttentionShared attention;
  __attribute__((aligned(16))) uint64_t layers[MOST_LAYERS * sizeof(Layer) / 8];
  uint64_t first_at[THREADS][2];              // where a thread's first keys and values of the block's first item lie in each layer's caches
  float scale[MOST_ROWS];
  int rank, blocks, gave_up;
  Shares shares;
};

// Sixteen bytes, or eight, of memory through a pointer out of the launch's table (an access through a plain pointer is one to
// either kind of memory, which waits for whatever is on its way in both).
typedef const __attribute__((address_space(1))) u32x4_t* memory16;
typedef const __attribute__((address_space(1))) u32x2_t* memory8;
__device__ __forceinline__ uint4 load16(const void* p) {
  const u32x4_t v = *(memory16)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 load_four(const float* p) {
  const u32x4_t v = *(memory16)p;
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}
__device__ __forceinline__ void store16(void* p, const u32x4_t& v) { *(__attribute__((address_space(1))) u32x4_t*)p = v; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u32x4_t peek16(__amdgpu_buffer_rsrc_t r, int at, int base = 0) { return __builtin_amdgcn_raw_buffer_load_b128(r, at, base, THROUGH); }
__device__ __forceinline__ bool there(const u32x4_t& v) { return v.x != ABSENT && v.y != ABSENT && v.z != ABSENT && v.w != ABSENT; }
// A word of results that happens to be the mark (not a number, either way) becomes another one.
__device__ __forceinline__ unsigned marked(unsigned w, unsigned instead) { return w == ABSENT ? instead : w; }
__device__ __forceinline__ void put8(__amdgpu_buffer_rsrc_t r, int at, uint2 v) {
  const u32x2_t p = {marked(v.x, 0x7fc07fc0u), marked(v.y, 0x7fc07fc0u)};
  __builtin_amdgcn_raw_buffer_store_b64(p, r, at, 0, THROUGH);
}
__device__ __forceinline__ void put4(__amdgpu_buffer_rsrc_t r, int at, unsigned v, unsigned instead) {
  __builtin_amdgcn_raw_buffer_store_b32(marked(v, instead), r, at, 0, THROUGH);
}
__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }

// Lane ^ N's value, N 1 or 2
template <int N>
__device__ __forceinline__ float quad_xor(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), N == 1 ? 0xb1 : 0x4e, 0xf, 0xf, true));
}

// Lane ^ 32's value
__device__ __forceinline__ float other_half(float v, int lane) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(lane < 32 ? a[1] : a[0]);
}

// Where numbers k .. of row `row`, of `width`, lie among what a product multiplies with, in bytes: `turned` rows (1, 2, 4, 8, 16, as many
// as hold the step's or 16) side by side, a row's eight numbers followed by the next row's, as the lanes of a matrix instruction take
// them. Neighbouring lanes then look at neighbouring places, where with each row in one piece a look cost a CU's address path up to four
// times as long, and lines of memory by rows. Rows in one piece each / side by side, us a step: the 0.6B shape over 1,000 keys, two 592 / 577,
// four 637 / 615, eight 746 / 690, sixteen 919 / 829, 20 1,214 / 1,058, 32 over 2,000 1,953 / 1,726; the 8B shape, four over 1,000
// 2,888 / 2,842, eight over 2,000 3,179 / 3,005, sixteen over 1,000 3,591 / 3,202.
__host__ __device__ __forceinline__ int place_of(int turned, int row, int k, int width) {
  if (turned == 1) return (row * width + k) * 2;
  const unsigned rest = (unsigned)row % (unsigned)turned;
  return (row - (int)rest) * width * 2 + (k >> 3) * (16 * turned) + (int)rest * 16 + (k & 7) * 2;
}

// Until shared memory holds what the block's wavefronts have written (and nothing about memory)
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- which slabs of 16 weight rows a block multiplies, and which steps of 32 of K a wavefront ----

// What a wavefront knows of a product, each number in a lane of one register (lane 16 product + number): numbers that are computed
// where they are needed, over and over, are what the compiler moves ahead of loops, 500 instructions a product on the way from one
// exchange to the next. A block has COUNT slabs, SLAB and every STEP-th behind it: neighbours where products have blocks for themselves
// (whose results lie in the same lines; the 0.6B shape 596 -> 585 us), else one beside the other blocks' (all blocks then read
// one stretch of memory; the 8B shape 2,841 -> 2,819).
enum { OWN, FIRST_STEP, START, STRIDE, COUNT, SLAB, STEP, SRC, SUMS, DST, DST_SUMS, ROW_BYTES, OUT_WIDTH };
// Who does what. Where a quarter of the blocks has a slab for each of the two products that add into the stream, those have the
// last quarter for themselves, and the other two products the rest: of two products that follow one another each finds its block
// waiting, its weights there and nothing of its own on the way to memory.
struct Roles {
  int apart;                   // how many blocks the products into the stream have for themselves, or none
  __device__ __forceinline__ Roles(const Args& a, int blocks) : apart(4 * (a.width / 16) <= blocks ? a.width / 16 : 0) {}
  // a block's place among those that share product `which` out, and how many they are; its first item of the attention and its first pair of
  // row and key head whose parts it joins
  __device__ __forceinline__ int place(int which, int rank, int blocks) const {
    if (apart) return which & 1 ? rank - (blocks - apart) : rank;
    return !(which & 1) ? rank : rank >= blocks / 2 ? rank - blocks / 2 : rank + blocks - blocks / 2;
  }
  __device__ __forceinline__ int places(int which, int blocks) const { return !apart ? blocks : which & 1 ? apart : blocks - apart; }
  // the first pieces of attention are the stream's blocks', whose keys come while the first product is multiplied
  __device__ __forceinline__ int item(int rank, int blocks) const {
    return !apart ? rank : rank >= blocks - apart ? rank - (blocks - apart) : rank + apart;
  }
  __device__ __forceinline__ int pair(int rank, int blocks) const {
    const int all = blocks - apart, middle = apart ? all / 2 : blocks / 4;
    return rank >= all ? 1 << 24 : rank >= middle ? rank - middle : rank + all - middle;
  }
};
__device__ __forceinline__ int numbers_of(const Args& a, int rank, int blocks, int wave, int lane) {
  const int which = lane >> 4, qkv = (a.heads + 2 * a.kv_heads) * HEAD;
  const int K = which == 1 ? a.heads * HEAD : which == 3 ? a.inner : a.width, steps = K / 32;
  const int slabs = (which == 0 ? qkv : which == 2 ? 2 * a.inner : a.width) / 16;
  const Roles roles(a, blocks);
  const int place = roles.place(which, rank, blocks), places = roles.places(which, blocks);
  const int share = slabs / places, extra = slabs % places, count = place >= 0 && place < places ? share + (place < extra ? 1 : 0) : 0;
  const int slab = roles.apart ? place * share + min(place, extra) : place, step = roles.apart ? 1 : places;
  const int each = steps / WAVES, more = steps % WAVES, first = wave * each + min(wave, more);
  switch (lane & 15) {
    case OWN: return each + (wave < more ? 1 : 0);
    case FIRST_STEP: return first;
    case START: return slab * steps + first;                  // in kilobytes of the tile-ordered matrix
    case STRIDE: return step * steps;
    case COUNT: return count;
    case SLAB: return slab;
    case STEP: return step;
    case SRC: return which == 0 ? a.at_out : which == 1 ? a.at_att : which == 2 ? a.at_mid : a.at_hid;
    case SUMS: return which == 0 ? a.at_out_sums : a.at_mid_sums;
    case DST: return which == 0 ? 0 : which == 1 ? a.at_mid : which == 2 ? a.at_hid : a.at_out;
    case DST_SUMS: return which == 1 ? a.at_mid_sums : a.at_out_sums;
    case ROW_BYTES: return 2 * K;
    case OUT_WIDTH: return which == 0 ? qkv : which == 2 ? a.inner : a.width;
  }
  return 0;
}

// How the keys are shared out (one wavefront; every block comes to the same). A sequence gets as many parts as its tiles ask for where the
// longest one has `s`, and s is the number for which the rounds of pieces cost least: per round a piece's start (PIECE steps of a wavefront's walk) and
// the longest piece's steps, and half a step for every eight parts that have to be joined. It is their lengths that count, not the bound that a
// captured step has for them, and not their number alone: 24 requests of the 0.6B shape of which one holds 30,000 keys and the others 500 took 9,700 us a
// step with a part a sequence (2,738 kernel by kernel), and take 1,782; one of 8,000 3,153 (1,906), 1,279; sixteen with one of 8,000 1,898 (1,803), 1,012;
// of the 8B shape eight with one of 30,000 5,768 (5,079), 3,737, sixteen 8,964 (5,645), 4,241. With a PIECE of 2 sixteen over 2,000 take 1,318 us
// and not 1,286, with 6 the first of these 2,052.
// (Straight code, and sums and maxima in the vector unit: it runs beside the gathering of the blocks, which takes 2.6 us.)
__device__ __forceinline__ float parts_of(float tiles, float per_tile, float s) { return fminf(fmaxf(ceilf(tiles * per_tile), 1.f), s); }
__device__ __forceinline__ void share_out(const ShareArgs& a, Shares& sh, int lane) {
  const bool row = lane < a.rows;
  const int kv_len = row ? max(a.kv_lens[lane], 0) : 0;
  const float tiles = (float)((max(kv_len - 1, 0) + FAST_TILE - 1) / FAST_TILE);
  if (lane < MOST_ROWS) sh.tiles[lane] = tiles, sh.kv_len[lane] = kv_len;
  const float longest = wave_max(tiles);
  float s = 1.f;
  if (a.parts_most > 1 && longest > WAVES) {
    const float tried = (float)(lane + 1), per_tile = tried / longest;            // (a lane tries a number)
    float items = (float)(a.rows - MOST_ROWS);     // (rows that are none count as a part here)
#pragma unroll
    for (int r = 0; r < MOST_ROWS; r += 4) {
      const float4 t = *reinterpret_cast<const float4*>(&sh.tiles[r]);
      items += (parts_of(t.x, per_tile, tried) + parts_of(t.y, per_tile, tried)) + (parts_of(t.z, per_tile, tried) + parts_of(t.w, per_tile, tried));
    }
    items *= (float)a.kv_heads;
    const float steps = ceilf(longest / (WAVES * tried)), rounds = ceilf(items * (1.f / ROUND));
    const float cost = fminf(2.f * rounds * (PIECE + steps) + (lane > 0 ? (float)((lane + 8) / 8) : 0.f), 131071.f);
    const bool fits = lane == 0 || (lane < a.parts_most && items <= (float)a.items_most && (float)(WAVES * lane) < longest);
    // (of equal ones the most parts: 8B shape, four over 2,060 keys 2,896 us, in five parts 2,961)
    const int best = (int)-wave_max(fits ? -(cost * 64.f + (float)(63 - lane)) : -INFINITY);
    s = (float)(64 - (best & 63));
  }
  const int parts = row ? (int)parts_of(tiles, s / fmaxf(longest, 1.f), s) : 0, key = parts * 64 + 63 - lane;
  int first = 0, all = 0;
#pragma unroll
  for (int r = 0; r < MOST_ROWS; ++r) {
    const int other = __builtin_amdgcn_readlane(key, r);
    first += other > key ? other >> 6 : 0;
    all += other >> 6;
  }
  if (lane < MOST_ROWS) sh.first[lane] = first * a.kv_heads, sh.parts[lane] = parts;
  if (lane == 0) sh.items = all * a.kv_heads, sh.in_parts = s > 1.f;
}

typedef const __attribute__((address_space(4))) int* entries_ptr;
constexpr int LAYER_WORDS = sizeof(Layer) / 8;
enum { Q_NORM = 4, K_NORM, ENTRY_NORM, MIDDLE_NORM, KEYS, VALUES, EPS };    // words of an entry behind its four matrices

// A wait has been given up: nobody's result stands (`Block::layers`, at its end).
__device__ __forceinline__ void gave_up(const Args& a) {
  __hip_atomic_store(a.control + GAVE_UP, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_s_waitcnt(0);
  compiler_fence();
}

template <typename QKW, int GROUPS, int TURNED>
struct Block {
  Shared& sh;
  const Args& a;
  const int rank, blocks;
  int wave, lane, tid;
  int numbers;                 // of the products
  int pass;                    // slabs between two barriers
  int most;                    // looks at the exchange before a wait is given up
  int alive;
  unsigned rows_inverse;
  int held;                    // the product whose first weights are on their way: four times its layer, and which
  static constexpr int STEPS = CHUNKS / GROUPS;          // kilobytes of weights that a wavefront has on their way
  static constexpr int STEP_BYTES = 64 * TURNED;            // from a lane's numbers of one step of K to those of the next
  u32x4_t w[STEPS];            // they

  // (as a number of its own: what is computed from it is not kept in registers over the whole launch)
  __device__ __forceinline__ static int anew(int v) {
    asm volatile("" : "+v"(v));
    return v;
  }
  // Between two looks at the exchange: whether to look again. Every wait ends: after so many looks this wavefront waits for nothing
  // any more. That is in the control words before anything that it passes on afterwards (and in shared memory, for its own block's token).
  __device__ __forceinline__ bool again(int n) {
    if (__builtin_expect(n >= most, 0)) {
      alive = 0;
      gave_up(a);
      sh.gave_up = 1;
    }
    alive = __builtin_amdgcn_readfirstlane(alive);
    return alive != 0;
  }

  // ---- products ----

  __device__ __forceinline__ int number(int which, int k) const { return __builtin_amdgcn_readlane(numbers, 16 * which + k); }
  // A pointer, or the two norms' eps, out of a layer's entry
  __device__ __forceinline__ uint64_t entry(int layer, int which) const { return word(layer * LAYER_WORDS + which); }
  __device__ __forceinline__ uint64_t word(int at) const {
    const uint64_t v = sh.layers[at];
    return (uint64_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | (unsigned)__builtin_amdgcn_readfirstlane((int)v);
  }
  // What the registers of weights hold is of no use any more (a load that is left out would otherwise keep it where registers are scarce)
  __device__ __forceinline__ void forget() {
    u32x4_t nothing;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
      asm volatile("" : "=v"(nothing));
      w[j] = nothing;
    }
  }
  // The wavefront's steps of a slab; what is behind them reads as zeros
  __device__ __forceinline__ static __amdgpu_buffer_rsrc_t slab_of(uint64_t matrix, int kilobytes, int own) {
    return buffer_of((const char*)matrix + ((uint64_t)(unsigned)kilobytes << 10), own << 10);
  }
  __device__ __forceinline__ static u32x4_t load(__amdgpu_buffer_rsrc_t r, int at) { return __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0); }
  __device__ __forceinline__ static f32x4_t dot(const u32x4_t& w, const u32x4_t& x, const f32x4_t& acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
  }
  // STEPS kilobytes of `left` slabs: as many steps of one, or where K has no more for a wavefront, eight of two or four of four. (One
  // sequence for all: registers that several may have loaded are copied behind each, and so waited for.)
  __device__ __forceinline__ void ask(uint64_t matrix, int at, int stride, int left, int own) {
    const int off = anew(lane) * 16, bits = own <= 4 ? 0 : STEPS == 8 || own <= 8 ? 1 : 2;
#pragma unroll
    for (int quarter = 0; quarter < STEPS / 4; ++quarter) {
      const int s = quarter >> bits;
      if (quarter == 0 || s < left) {
        const auto r = slab_of(matrix, at + s * stride, own);
        const int from = off + ((quarter - (s << bits)) << 12);
#pragma unroll
        for (int j = 0; j < 4; ++j) w[4 * quarter + j] = load(r, from + 1024 * j);
      }
    }
  }
  __device__ __forceinline__ void begin(int layer, int which, int done) {
    const int stride = number(which, STRIDE);
    ask(entry(layer, which), number(which, START) + done * stride, stride, number(which, COUNT) - done, number(which, OWN));
  }
  // The first weights of product `which`, or the first one behind it that this block has part in, asked for as early as their registers are free
  __device__ __forceinline__ void look_ahead(int layer, int which) {
    for (;; ++which) {
      if (which == 4) which = 0, ++layer;
      if (layer >= a.count) return;
      if (number(which, COUNT)) break;
    }
    held = 4 * layer + which;
    begin(layer, which, 0);
  }

  // What a product multiplies with: K numbers a row at `src` of the exchange, their squares' partial sums at `sums`
  struct Rows {
    __amdgpu_buffer_rsrc_t ex;
    int src, sums;
    int at[GROUPS];              // the lane's first eight numbers, row lane % 16 (and 16 behind it) and eight k of 32; nowhere for a row that is none
    float eps;
  };
  // N steps of rows, `left` of which there are, from step `i` on; of a second group behind those of the first
  template <int N>
  __device__ __forceinline__ static void look(u32x4_t (&x)[CHUNKS], const Rows& r, int i, int left) {
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      const int at = anew(r.at[g] + STEP_BYTES * i);
#pragma unroll
      for (int quarter = 0; quarter < N / 4; ++quarter) {
        const int from = (N < STEPS || quarter == 0 || left > 4 * quarter ? at : NOWHERE) + 4 * STEP_BYTES * quarter;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[N * g + 4 * quarter + j] = peek16(r.ex, from + STEP_BYTES * j, r.src);
      }
      if (left < N && (left == 0 || left & 3)) {
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (j >= left) x[N * g + j] = u32x4_t{0, 0, 0, 0};
      }
    }
  }
  template <int N>
  __device__ __forceinline__ static bool all_there(const u32x4_t (&x)[CHUNKS]) {
    unsigned least = 0;                                  // (the mark is the largest word)
#pragma unroll
    for (int j = 0; j < N * GROUPS; ++j) least = max(max(least, max(x[j].x, x[j].y)), max(x[j].z, x[j].w));
    return least != ABSENT;
  }
  // The look at the exchange is the wait: a word without the mark is there. With many rows, a lane that has all of its numbers asks no
  // more (24 rows of the 0.6B shape 1,146 -> 1,122 us, sixteen 849 -> 837; one row 574 -> 582, and so not with few).
  template <int N>
  __device__ __forceinline__ void fetch(u32x4_t (&x)[CHUNKS], const Rows& r, int i, int left) {
    // One look at one place first: so many rows asked for again and again hold up those that write them. From four rows on (the 0.6B shape,
    // four over 1,100 keys 638 us, without 663, six over 500 649 and 694; the 8B shape, two 2,829 with it, 2,819 without).
    if (i == 0 && a.rows >= 4 && left > 0) {
      const int place = __builtin_amdgcn_readfirstlane(r.at[0]) + STEP_BYTES * (min(left, N) - 1);
      for (int n = 0;; ++n) {
        compiler_fence();
        const u32x4_t v = peek16(r.ex, place, r.src);
        if (__builtin_amdgcn_readfirstlane((int)there(v)) || !again(n)) break;
      }
    }
    bool have = false;
    for (int n = 0;; ++n) {
      compiler_fence();
      if (TURNED < 8 || !have) {
        look<N>(x, r, i, left);
        have = all_there<N>(x);
      }
      if (__all(have) || !again(n)) break;
    }
  }
  // Four of a norm's weights among the sixteen bytes around them, and as numbers
  __device__ __forceinline__ u32x4_t raw_norm(const void* n, int at) const {
    return *(memory16)(static_cast<const char*>(n) + (a.norm_f32 ? 4 * at : 2 * (at & ~7)));
  }
  __device__ __forceinline__ float4 norm_of(const u32x4_t& v, int at) const {
    if (a.norm_f32) return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    const unsigned x = at & 4 ? v.z : v.x, y = at & 4 ? v.w : v.y;
    return make_float4(__uint_as_float(x << 16), __uint_as_float(x & 0xffff0000u), __uint_as_float(y << 16), __uint_as_float(y & 0xffff0000u));
  }

  // A slab's sums of this wavefront's steps into shared memory
  __device__ __forceinline__ void leave(const f32x4_t& acc, int slab, int group) {
    const int col = (lane & 15) + 16 * group, grp = lane >> 4;
    if (col < a.rows) *reinterpret_cast<f32x4_t*>(sh.red + (unsigned)(((slab * WAVES + wave) * 4 + grp) * a.rows + col) * 16) = acc;
  }

  // `slabs` slabs from `done` on, whose first group's weights have been asked for. With `scaled`, the first look at the rows' sums is
  // asked for between the rows and the multiplications.
  struct Sums {
    u32x4_t v[2 * GROUPS];       // of every eighth row, from the wavefront's number on
  };
  __device__ __forceinline__ Sums multiply(const Rows& r, int layer, int which, int done, int slabs, bool scaled) {
    const uint64_t matrix = entry(layer, which);
    const int own = number(which, OWN), stride = number(which, STRIDE), off = lane * 16;
    int at = number(which, START) + done * stride;
    Sums sums;
    u32x4_t x[CHUNKS];
    if (own > STEPS / 2) {
      const bool sections = own > STEPS;                 // (whose rows are asked for with every slab)
      if (!sections) {
        fetch<STEPS>(x, r, 0, own);
        if (scaled) sums = first_sums(r);
      }
#pragma unroll 1
      for (int s = 0; s < slabs; ++s, at += stride) {
        const auto here = slab_of(matrix, at, own), after = slab_of(matrix, at + stride, own);
        f32x4_t acc[2][GROUPS];
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) acc[0][g] = acc[1][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int i = 0; i < own; i += STEPS) {
          if (sections) {
            fetch<STEPS>(x, r, i, own - i);
            if (scaled && i == 0 && s == 0) sums = first_sums(r);
          }
          const bool ends = i + STEPS >= own;
          if (!ends || s + 1 < slabs) {
            const auto next = ends ? after : here;
            const int from = anew(ends ? off : off + ((i + STEPS) << 10));
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
#pragma unroll
              for (int g = 0; g < GROUPS; ++g) acc[j & 1][g] = dot(w[j], x[STEPS * g + j], acc[j & 1][g]);
              w[j] = load(next, from + 1024 * j);
            }
          } else {
#pragma unroll
            for (int j = 0; j < STEPS; ++j)
#pragma unroll
              for (int g = 0; g < GROUPS; ++g) acc[j & 1][g] = dot(w[j], x[STEPS * g + j], acc[j & 1][g]);
          }
        }
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) leave(acc[0][g] + acc[1][g], s, g);
      }
    } else if (STEPS > 8 && own > 4) {
      fetch<8>(x, r, 0, own);
      if (scaled) sums = first_sums(r);
#pragma unroll 1
      for (int s = 0; s < slabs; s += 2) {
        f32x4_t acc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < STEPS; ++j) acc[j >> 2] = dot(w[j], x[j & 7], acc[j >> 2]);
        if (s + 2 < slabs) ask(matrix, at += 2 * stride, stride, slabs - s - 2, own);
        leave(acc[0] + acc[1], s, 0);
        if (s + 1 < slabs) leave(acc[2] + acc[3], s + 1, 0);
      }
    } else {
      constexpr int EACH = STEPS / 4;
      fetch<4>(x, r, 0, own);
      if (scaled) sums = first_sums(r);
#pragma unroll 1
      for (int s = 0; s < slabs; s += EACH) {
        f32x4_t acc[EACH][GROUPS];
#pragma unroll
        for (int q = 0; q < EACH; ++q)
#pragma unroll
          for (int g = 0; g < GROUPS; ++g) acc[q][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
#pragma unroll
          for (int g = 0; g < GROUPS; ++g) acc[j >> 2][g] = dot(w[j], x[4 * g + (j & 3)], acc[j >> 2][g]);
        if (s + EACH < slabs) ask(matrix, at += EACH * stride, stride, slabs - s - EACH, own);
#pragma unroll
        for (int q = 0; q < EACH; ++q)
#pragma unroll
          for (int g = 0; g < GROUPS; ++g)
            if (s + q < slabs) leave(acc[q][g], s + q, g);
      }
    }
    return sums;
  }

  // The rows' scales from the partial sums of squares, [row][slab]; `first`: the first of them, as they were when the rows had come
  __device__ __forceinline__ Sums first_sums(const Rows& r) const {
    const int lane = anew(this->lane), slabs = a.width / 16;
    Sums first;
#pragma unroll
    for (int i = 0; i < 2 * GROUPS; ++i) {
      const int row = wave + WAVES * i;
      first.v[i] = peek16(r.ex, row < a.rows && lane * 4 < slabs ? (row * slabs + lane * 4) * 4 : NOWHERE, r.sums);
    }
    return first;
  }
  __device__ __forceinline__ void scales(const Rows& r, Sums first) {
    const int slabs = a.width / 16;
#pragma unroll
    for (int i = 0; i < 2 * GROUPS; ++i) {
      const int row = wave + WAVES * i;
      if (row >= a.rows) break;
      u32x4_t v = first.v[i];
      bool asked = true;
      float s = 0.f;
#pragma unroll 1
      for (int k = lane * 4; __builtin_amdgcn_readfirstlane(k) < slabs; k += 256) {
        const int at = k < slabs ? (row * slabs + k) * 4 : NOWHERE;
        for (int n = 0;; ++n) {
          if (!asked) v = peek16(r.ex, at, r.sums);
          asked = false;
          if (__all(there(v)) || !again(n)) break;
          compiler_fence();
        }
        s += (__uint_as_float(v.x) + __uint_as_float(v.y)) + (__uint_as_float(v.z) + __uint_as_float(v.w));
      }
      s = wave_sum(s);
      if (lane == 0) sh.scale[row] = rsqrtf(s * (1.f / (float)a.width) + r.eps);
    }
  }

  // The wavefronts' shares of K of one pass, added in a fixed order, and what follows the product. `res`, `raw`: the stream and the
  // norm's weights at the lane's first four results.
  __device__ __forceinline__ int over_rows(int n) const { return (unsigned)n * rows_inverse >> 20; }    // n / a.rows, n below 4,096
  struct Follow {
    float4 res;
    u32x4_t raw;
  };
  __device__ __forceinline__ Follow follow(int which, int done, int slabs, const void* norm) const {
    const int tid = anew(this->tid), q = tid >> 2, s = over_rows(q), row = q - s * a.rows, n = (number(which, SLAB) + (done + s) * number(which, STEP)) * 16 + 4 * (tid & 3);
    Follow f;
    f.res = make_float4(0.f, 0.f, 0.f, 0.f);
    f.raw = u32x4_t{0, 0, 0, 0};
    if (s < slabs) {
      f.res = load_four(a.residual + (size_t)row * a.width + n);
      if (norm) f.raw = raw_norm(norm, n);
    }
    return f;
  }
  __device__ __forceinline__ void finish(__amdgpu_buffer_rsrc_t ex, int which, int done, int slabs, const void* norm, Follow f) {
    const bool stream = which & 1;
    const int tid = anew(this->tid), entries = slabs * 4 * a.rows, grp = tid & 3;
    const int width = number(which, OUT_WIDTH), dst = number(which, DST), step = number(which, STEP), first = number(which, SLAB) + done * step;
    if (tid < entries) {         // (a thread has one at most)
      const int q = tid >> 2, s = over_rows(q), row = q - s * a.rows, slab = first + s * step, n = slab * 16 + 4 * grp;
      const char* part = sh.red + (unsigned)((s * WAVES * 4 + grp) * a.rows + row) * 16;
      f32x4_t share[WAVES];
#pragma unroll
      for (int v = 0; v < WAVES; ++v) share[v] = *reinterpret_cast<const f32x4_t*>(part + (unsigned)(v * 4 * a.rows) * 16);
#pragma unroll
      for (int v = 0; v < WAVES; ++v) asm volatile("" : "+v"(share[v]));       // (all of them asked for, then added)
      f32x4_t acc = share[0];
#pragma unroll
      for (int v = 1; v < WAVES; ++v) acc += share[v];
      union {
        uint2 u;
        __bf16 e[4];
      } pk;
      if (stream) {
        const float x[4] = {f.res.x + (float)(__bf16)acc[0], f.res.y + (float)(__bf16)acc[1], f.res.z + (float)(__bf16)acc[2],
                            f.res.w + (float)(__bf16)acc[3]};
        if (norm) {
          const float4 nw = norm_of(f.raw, n);
          const float w4[4] = {nw.x, nw.y, nw.z, nw.w};
          float ss = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            ss += x[e] * x[e];
            pk.e[e] = (__bf16)(x[e] * w4[e]);
          }
          put8(ex, dst + place_of(TURNED, row, n, width), pk.u);
          ss += quad_xor<1>(ss);
          ss += quad_xor<2>(ss);
          if (grp == 0) put4(ex, number(which, DST_SUMS) + (row * (width / 16) + slab) * 4, __float_as_uint(ss), 0x7fc00000u);
        }
        store16(a.residual + (size_t)row * a.width + n,
                u32x4_t{__float_as_uint(x[0]), __float_as_uint(x[1]), __float_as_uint(x[2]), __float_as_uint(x[3])});
      } else {
        acc *= sh.scale[row];
        if (which == 2) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float g = (float)(__bf16)acc[2 * e], u = (float)(__bf16)acc[2 * e + 1];
            pk.e[e] = (__bf16)(gate_value<0>(g) * u);
          }
          put4(ex, dst + place_of(TURNED, row, n / 2, width), pk.u.x, 0x7fc07fc0u);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) pk.e[e] = (__bf16)acc[e];
          put8(ex, dst + (row * width + n) * 2, pk.u);
        }
      }
    }
  }

  __device__ __forceinline__ void product_of(const Rows& r, __amdgpu_buffer_rsrc_t ex, int layer, int which, int count, const void* norm) {
#pragma unroll 1
    for (int done = 0; done < count; done += pass) {
      const int slabs = min(pass, count - done);
      if (done || held != 4 * layer + which) begin(layer, which, done);
      Follow f;
      if (which & 1) f = follow(which, done, slabs, norm);
      const bool scaled = done == 0 && !(which & 1);
      const Sums sums = multiply(r, layer, which, done, slabs, scaled);
      if (scaled) scales(r, sums);
      forget();
      meet();
      finish(ex, which, done, slabs, norm, f);
      meet();                    // (the results on their way ahead of the other wavefronts' loads: 8B shape, one request, 3 us a product otherwise)
      if (done + slabs >= count && which != 0) look_ahead(layer, which + 1);
    }
  }

  // ---- attention ----

  // A piece of the attention, and what all layers have of it in common.
  struct Item {
    int n, part, parts, g_kv, b, kv_len, there;
    TilePages second;            // of this wavefront's second tile
    uint64_t keys, values;       // where the lane's parts of its first one lie
  };
  __device__ __forceinline__ TilePages pages_of(int b, int tile) const {
    const entries_ptr row = (entries_ptr)(uintptr_t)(a.block_table + (size_t)b * a.table_width);
    TilePages p;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int entry = (tile * FAST_TILE + 16 * h) >> a.page_bits;
      p.pg[h] = entry < a.table_width ? row[entry] : -1;
    }
    return p;
  }
  // attention_tiles.h's tile_addr over again, with the lane as a number of its own: what follows from it is not kept over the launch. (As an
  // argument of that function the lane changes the registers of all of attention.hip's kernels.)
  __device__ __forceinline__ TileAddr addr_of(const TilePages& p, const bf16_t* keys, const bf16_t* values, int g_kv, int tile) const {
    const int lane = anew(this->lane), col = lane & 15, grp = lane >> 4;
    long kh[2], vh[2];
    TileAddr t;
    t.there = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool there = p.pg[h] >= 0 && p.pg[h] < a.num_pages;
      const long head = (long)(there ? p.pg[h] : 0) * a.kv_heads + g_kv;
      const int slot = (tile * FAST_TILE + 16 * h) & (a.page - 1);
      kh[h] = (head * a.page + slot) * HEAD;
      vh[h] = head * HEAD * a.page + slot;
      t.there |= there ? 1 << h : 0;
    }
    t.k = keys + (col >> 3 ? kh[1] : kh[0]) + (unsigned)((8 * ((col >> 2) & 1) + (col & 3)) * HEAD + 8 * grp);
    t.v = values + (grp >> 1 ? vh[1] : vh[0]) + (unsigned)(col * a.page + 8 * (grp & 1));
    return t;
  }
  __device__ __forceinline__ Item item_of(int n) const {
    Item it;
    const int row = min(lane, a.rows - 1), from = sh.shares.first[row], parts = sh.shares.parts[row], kv_len = sh.shares.kv_len[row];
    it.b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(n >= from && n < from + parts * a.kv_heads));
    it.n = n;
    it.parts = __builtin_amdgcn_readlane(parts, it.b);
    it.kv_len = __builtin_amdgcn_readlane(kv_len, it.b);
    const int within = n - __builtin_amdgcn_readlane(from, it.b);
    it.g_kv = within / it.parts;
    it.part = within - it.g_kv * it.parts;
    const int first = it.part * WAVES + wave;
    const TileAddr t = addr_of(pages_of(it.b, first), nullptr, nullptr, it.g_kv, first);
    it.there = t.there;
    it.keys = (uint64_t)t.k;
    it.values = (uint64_t)t.v;
    it.second = pages_of(it.b, first + WAVES * it.parts);
    return it;
  }

  // What attention.hip's decoding block does, from and to the exchange. The heads' norms and rotations are shared out: a wavefront
  // prepares one query row, the next ones the token's key and value. A wavefront asks for its next tile's keys when this one's have been
  // multiplied, and for the values likewise.
  __device__ __forceinline__ void attend(__amdgpu_buffer_rsrc_t ex, int layer, const Item& it) {
    constexpr int D = HEAD;
    AttentionShared& s = sh.attention;
    const bf16_t *keys = (const bf16_t*)entry(layer, KEYS), *values = (const bf16_t*)entry(layer, VALUES);
    const char *q_norm = (const char*)entry(layer, Q_NORM), *k_norm = (const char*)entry(layer, K_NORM);
    const int g_kv = it.g_kv, b = it.b;
    const int lane = anew(this->lane), col = lane & 15, grp = lane >> 4;
    const int G = a.group, joined = (a.heads + 2 * a.kv_heads) * D;
    const int first = it.part * WAVES + wave, step = WAVES * it.parts;
    const bool brings_new = it.part == it.parts - 1;
    const int pos = it.kv_len - 1;                    // the token's own position; the cache is read up to the one before
    const bool turned = a.table != nullptr && pos >= 0 && pos < a.max_pos;
    const int kv_seen = max(pos, 0), row_pos = col < G ? pos - 1 : -1;
    const int last = (kv_seen + FAST_TILE - 1) / FAST_TILE;
    TileRegs<D, D> r;
    auto ask_keys = [&](const TileAddr& to) {
      r.at = to;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < D / 32; ++j) r.k[kb][j].u = load16(to.k + 4 * D * kb + 32 * j);
    };
    auto ask_values = [&]() {
#pragma unroll
      for (int nb = 0; nb < D / 16; ++nb) r.v[nb].u = load16(r.at.v + (size_t)(16 * nb) * a.page);
    };
    TilePages next = it.second;
    if (first < last) {
      ask_keys(TileAddr{(const bf16_t*)((uint64_t)keys + it.keys), (const bf16_t*)((uint64_t)values + it.values), it.there});
      ask_values();
    }
    // the token's rows: lane n has elements 2 n and 2 n + 1, its pair's other half is lane n ^ 32. qk_prepare.h's steps, each product and sum rounded where
    // it is there, but the squares summed over all 64 lanes at once and not in eights: a key may differ in its last bit from the one
    // that another kernel makes of the same row (and does anyway by the row itself, a product whose K is added up in another order).
    for (int row = wave; row < G + (brings_new ? 2 : 0); row += WAVES) {
      const int head = row < G ? g_kv * G + row : a.heads + (row == G ? 0 : a.kv_heads) + g_kv;
      const bool prepared = row <= G;                 // (values are taken as they are)
      unsigned norm[2] = {0, 0};                      // as they lie in memory
      float2 cs = make_float2(1.f, 1.f), sn = make_float2(0.f, 0.f);
      if (prepared && q_norm != nullptr) {
        const char* weights = row < G ? q_norm : k_norm;
        if constexpr (sizeof(QKW) == 4) {
          const u32x2_t v = *(memory8)(weights + 8 * lane);
          norm[0] = v.x;
          norm[1] = v.y;
        } else {
          norm[0] = *(const __attribute__((address_space(1))) unsigned*)(weights + 4 * lane);
        }
      }
      if (prepared && turned) {
        const float* at = a.table + (size_t)pos * D + 2 * (lane & 31);
        const u32x2_t c = *(memory8)at, n = *(memory8)(at + D / 2);
        cs = make_float2(__uint_as_float(c.x), __uint_as_float(c.y));
        sn = make_float2(__uint_as_float(n.x), __uint_as_float(n.y));
      }
      unsigned v;
      for (int n = 0;; ++n) {
        compiler_fence();
        v = __builtin_amdgcn_raw_buffer_load_b32(ex, (b * joined + head * D) * 2 + lane * 4, 0, THROUGH);
        if (__all(v != ABSENT) || !again(n)) break;
      }
      float x0 = __uint_as_float(v << 16), x1 = __uint_as_float(v & 0xffff0000u);
      if (prepared && q_norm != nullptr) {
        const float scale = head_norm_scale(wave_sum(__fmaf_rn(x0, x0, __fmul_rn(x1, x1))), D, a.qk_eps);
        x0 = __fmul_rn(__fmul_rn(x0, scale), __uint_as_float(sizeof(QKW) == 4 ? norm[0] : norm[0] << 16));
        x1 = __fmul_rn(__fmul_rn(x1, scale), __uint_as_float(sizeof(QKW) == 4 ? norm[1] : norm[0] & 0xffff0000u));
      }
      if (prepared && turned) {
        const float y0 = other_half(x0, lane), y1 = other_half(x1, lane);
        const float sign = lane < 32 ? -1.f : 1.f;
        x0 = __fmaf_rn(x0, cs.x, __fmul_rn(sign * y0, sn.x));
        x1 = __fmaf_rn(x1, cs.y, __fmul_rn(sign * y1, sn.y));
      }
      union {
        unsigned u;
        __bf16 e[2];
      } pk;
      pk.e[0] = (__bf16)x0;
      pk.e[1] = (__bf16)x1;
      if (row < G)
        *reinterpret_cast<unsigned*>(&s.q[row][2 * lane]) = pk.u;
      else
        *reinterpret_cast<float2*>((row == G ? s.k : s.v) + 2 * lane) = make_float2((float)pk.e[0], (float)pk.e[1]);
    }
    meet();
    const int failed = sh.gave_up;                    // (the token's rows may not have come)
    Pack16 q[D / 32];
#pragma unroll
    for (int j = 0; j < D / 32; ++j) {
      q[j].u = make_uint4(0, 0, 0, 0);
      if (col < G) q[j].u = *reinterpret_cast<const uint4*>(&s.q[col][32 * j + 8 * grp]);
    }
    if (brings_new) {                                 // the new key's scores: the rows shared out once more
      for (int row = WAVES - 1 - wave; row < G; row += WAVES) {      // (by wavefronts that may have no tile: the first ones have)
        const bf16_t* mine = &s.q[row][2 * lane];
        const float dot = wave_sum(fmaf(bf16_to_float(mine[0]), s.k[2 * lane], bf16_to_float(mine[1]) * s.k[2 * lane + 1]));
        if (lane == 0) s.m[WAVES][row] = pos >= 0 ? dot * a.scale_log2 : -INFINITY;
      }
    } else if (wave == 0 && lane < 16) {
      s.m[WAVES][lane] = -INFINITY;
    }
    f32x4_t acc[D / 16];
#pragma unroll
    for (int nb = 0; nb < D / 16; ++nb) acc[nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (int t = first; t < last; t += step) {
      const bool more = t + step < last;
      const int have = r.at.there, key0 = t * FAST_TILE;
      if (have != 3 && !((have >> (col >> 3)) & 1)) {          // a half without a page counts as zeros
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int j = 0; j < D / 32; ++j) r.k[kb][j].u = make_uint4(0, 0, 0, 0);
      }
      f32x4_t sc[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        sc[kb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < D / 32; ++j) sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.k[kb][j].v, q[j].v, sc[kb], 0, 0, 0);
      }
      if (more) {
        ask_keys(addr_of(next, keys, values, g_kv, t + step));
        next = pages_of(b, t + 2 * step);
      }
      const Pack16 p = softmax_step<D / 16>(sc, false, key0, grp, row_pos, 0, a.scale_log2, m_run, l_run, acc);
      if (have != 3 && !((have >> (grp >> 1)) & 1)) {
#pragma unroll
        for (int nb = 0; nb < D / 16; ++nb) r.v[nb].u = make_uint4(0, 0, 0, 0);
      }
      if (key0 + FAST_TILE > kv_seen) {  // slots past the sequence's end hold anything: zero them, 0 * NaN is NaN
#pragma unroll
        for (int nb = 0; nb < D / 16; ++nb)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (key0 + 8 * grp + e >= kv_seen) r.v[nb].e[e] = (__bf16)0.f;
      }
#pragma unroll
      for (int nb = 0; nb < D / 16; ++nb) acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.v[nb].v, p.v, acc[nb], 0, 0, 0);
      if (more) ask_values();
    }
    const float l_all = quad_rows_sum(l_run);
    if (grp == 0) {
      s.m[wave][col] = m_run;
      s.l[wave][col] = l_all;
    }
    if (col < G) {
#pragma unroll
      for (int nb = 0; nb < D / 16; ++nb) *reinterpret_cast<f32x4_t*>(&s.acc[wave][col][16 * nb + 4 * grp]) = acc[nb];
    }
    meet();
    const int tid = anew(this->tid);
    for (int idx = tid; idx < G * (D / 4); idx += THREADS) {
      const int row = idx / (D / 4), d = idx % (D / 4) * 4;
      float m[WAVES + 1], mr = -INFINITY, lr = 0.f;
#pragma unroll
      for (int v = 0; v <= WAVES; ++v) mr = fmaxf(mr, m[v] = s.m[v][row]);
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        const float weight = m[v] > -INFINITY ? fast_exp2(m[v] - mr) : 0.f;
        lr += s.l[v][row] * weight;
        o += *reinterpret_cast<const f32x4_t*>(&s.acc[v][row][d]) * weight;
      }
      if (m[WAVES] > -INFINITY) {
        const float weight = fast_exp2(m[WAVES] - mr);
        lr += weight;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += s.v[d + e] * weight;
      }
      if (it.parts == 1) {
        const float inv = lr > 0.f ? 1.f / lr : lr;      // (a row that sees nothing, a sequence without a length, is zero)
        union {
          uint2 u;
          __bf16 e[4];
        } pk;
#pragma unroll
        for (int e = 0; e < 4; ++e) pk.e[e] = (__bf16)(o[e] * inv);
        put8(ex, a.at_att + place_of(TURNED, b, (g_kv * G + row) * D + d, a.heads * D), pk.u);
      } else {
        const int slot = it.n * G + row;
        u32x4_t p;
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = marked(__float_as_uint(o[e]), 0x7fc00000u);
        __builtin_amdgcn_raw_buffer_store_b128(p, ex, a.at_part + (slot * D + d) * 4, 0, THROUGH);
        if (d == 0) {
          const u32x2_t ml = {marked(__float_as_uint(mr), 0x7fc00000u), marked(__float_as_uint(lr), 0x7fc00000u)};
          __builtin_amdgcn_raw_buffer_store_b64(ml, ex, a.at_ml + slot * 8, 0, THROUGH);
        }
      }
    }
    if (brings_new && pos >= 0 && tid >= THREADS - 2 * HEAD && !failed) {       // the token's key and value into the caches, for later steps
      const int d = tid & (HEAD - 1), blk = pos >> a.page_bits, at = pos & (a.page - 1);
      const int pg = blk < a.table_width ? ((entries_ptr)(uintptr_t)(a.block_table + (size_t)b * a.table_width))[blk] : -1;
      if (pg >= 0 && pg < a.num_pages) {
        const size_t head = (size_t)pg * a.kv_heads + g_kv;
        const bool value = tid >= THREADS - HEAD;
        auto dst = (__attribute__((address_space(1))) uint16_t*)(value ? values : keys) + head * D * a.page;
        dst[value ? (size_t)d * a.page + at : (size_t)at * D + d] = float_to_bf16(value ? s.v[d] : s.k[d]).bits;
      }
    }
    meet();      // (whoever writes here next)
  }

  // The parts of sequence `b` and key head `g_kv`, pieces `first` to `first` + `parts` - 1, joined
  __device__ __forceinline__ void merge(__amdgpu_buffer_rsrc_t ex, int g_kv, int b, int first, int parts) {
    constexpr int D = HEAD, N = 8;
    const int tid = anew(this->tid), G = a.group;
    for (int idx = tid; idx < ((G * (D / 4) + 63) & ~63); idx += THREADS) {
      const int r = min(idx / (D / 4), G - 1), d = idx % (D / 4) * 4;
      float m = -INFINITY, sum = 0.f;
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < parts; s0 += N) {
        u32x4_t p[N];
        u32x2_t ml[N];
        for (int n = 0;; ++n) {
          compiler_fence();
          bool ok = true;
#pragma unroll
          for (int s = 0; s < N; ++s) {
            const int slot = (first + min(s0 + s, parts - 1)) * G + r;
            p[s] = peek16(ex, a.at_part + (slot * D + d) * 4);
            ml[s] = __builtin_amdgcn_raw_buffer_load_b64(ex, a.at_ml + slot * 8, 0, THROUGH);
          }
#pragma unroll
          for (int s = 0; s < N; ++s) ok = ok && there(p[s]) && ml[s].x != ABSENT && ml[s].y != ABSENT;
          if (__all(ok) || !again(n)) break;
        }
        float m_all = m;
#pragma unroll
        for (int s = 0; s < N; ++s)
          if (s0 + s < parts) m_all = fmaxf(m_all, __uint_as_float(ml[s].x));
        const float kept = m > -INFINITY ? fast_exp2(m - m_all) : 0.f;
        sum *= kept;
        o *= kept;
#pragma unroll
        for (int s = 0; s < N; ++s)
          if (s0 + s < parts && __uint_as_float(ml[s].x) > -INFINITY) {
            const float weight = fast_exp2(__uint_as_float(ml[s].x) - m_all);
            sum += __uint_as_float(ml[s].y) * weight;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += __uint_as_float(p[s][e]) * weight;
          }
        m = m_all;
      }
      const float inv = sum > 0.f ? 1.f / sum : sum;
      union {
        uint2 u;
        __bf16 e[4];
      } pk;
#pragma unroll
      for (int e = 0; e < 4; ++e) pk.e[e] = (__bf16)(o[e] * inv);
      if (idx < G * (D / 4)) put8(ex, a.at_att + place_of(TURNED, b, (g_kv * G + r) * D + d, a.heads * D), pk.u);
    }
  }

  __device__ __forceinline__ void layers() {
    const int items = __builtin_amdgcn_readfirstlane(sh.shares.items), pairs = a.rows * a.kv_heads;
    const Roles roles(a, blocks);
    const int my_item = roles.item(rank, blocks), my_pair = roles.pair(rank, blocks), pair_step = blocks - roles.apart;
    Item mine = item_of(min(my_item, items - 1));
    sh.first_at[tid][0] = mine.keys;
    sh.first_at[tid][1] = mine.values;
    struct Pair {
      int b, g, first, parts;
    };
    auto pair_of = [&](int n) {
      Pair p;
      p.b = n / a.kv_heads;
      p.g = n - p.b * a.kv_heads;
      const int row = min(p.b, a.rows - 1);
      p.parts = __builtin_amdgcn_readfirstlane(sh.shares.parts[row]);
      p.first = __builtin_amdgcn_readfirstlane(sh.shares.first[row]) + p.g * p.parts;
      return p;
    };
    const Pair my = pair_of(my_pair);
    look_ahead(0, 0);
#pragma unroll 1
    for (int n = 0; n < a.count; ++n) {
      const auto ex = buffer_of(a.exchange + n * a.per_layer, a.per_layer);
#pragma unroll 1
      for (int which = 0; which < 4; ++which) {
        // (new numbers to the compiler: it would otherwise work out every product's addresses ahead of all of them, and has no registers for those)
        asm volatile("" : "+v"(lane), "+v"(tid));
        if (which == 1) {
#pragma unroll 1
          for (int n_item = my_item; n_item < items; n_item += blocks) {
            Item it = mine;
            it.keys = sh.first_at[tid][0];
            it.values = sh.first_at[tid][1];
            if (n_item != my_item) it = item_of(n_item);
            attend(ex, n, it);
          }
          if (a.shares.parts_most > 1)  // (its loads would come behind the next weights')
#pragma unroll 1
            for (int pair = my_pair; pair < pairs; pair += pair_step) {
              const Pair p = pair == my_pair ? my : pair_of(pair);
              if (p.parts > 1) merge(ex, p.g, p.b, p.first, p.parts);
            }
          look_ahead(n, 1);
        }
        const int count = number(which, COUNT);
        if (count == 0) continue;
        const int col = lane & 15;
        Rows r;
        r.ex = which == 0 ? buffer_of(a.exchange + (n - 1) * a.per_layer, a.per_layer) : ex;
        r.src = number(which, SRC);
        r.sums = number(which, SUMS);
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
          r.at[g] = col + 16 * g >= a.rows ? NOWHERE
                    : g * 16 * number(which, ROW_BYTES) + STEP_BYTES * number(which, FIRST_STEP) + 16 * (TURNED * (lane >> 4) + col);
        const uint64_t eps = entry(n, EPS);
        r.eps = __uint_as_float((unsigned)(which == 0 ? eps : eps >> 32));
        // (the last layer's down product prepares no rows: its norm is the one behind the layers, of another kernel)
        const int at = which == 1 ? n * LAYER_WORDS + MIDDLE_NORM : which == 3 && n + 1 < a.count ? (n + 1) * LAYER_WORDS + ENTRY_NORM : -1;
        const void* norm = at >= 0 ? (const void*)word(at) : nullptr;
        product_of(r, ex, n, which, count, norm);
      }
    }
    // A wait that was given up, in whatever block: no number of the result stands. Every block with a part in the last product has multiplied with
    // numbers that come, over however many blocks, from each of those that had work before it, and these say that they gave up
    // before they pass anything on. One that gives up in the last product itself may be too late for the others: its own columns of every row are
    // no numbers, and so the norm behind the layers and all logits. (A thread stores what `finish` had it store.)
    const int count = number(3, COUNT);
    if (count && __hip_atomic_load(a.control + GAVE_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      const unsigned nan = 0x7fc00000u;
      for (int done = 0; done < count; done += pass) {
        const int q = tid >> 2, s = over_rows(q), row = q - s * a.rows, n = (number(3, SLAB) + (done + s) * number(3, STEP)) * 16 + 4 * (tid & 3);
        if (s < min(pass, count - done)) store16(a.residual + (size_t)row * a.width + n, u32x4_t{nan, nan, nan, nan});
      }
    }
  }
};

// The blocks that are here when the launch begins share its work; one that only finds room later has none. Nothing is assumed
// about how many run at once, so two such launches on two streams, or a kernel that keeps some of the processors, cannot wait
// for each other without end. CAME: how many have come, and CLOSED; CLOSED_AT: how many there are, if not all came in time.
__device__ __forceinline__ void gather(const Args& a, int& rank, int& blocks) {
  unsigned* came = a.control + CAME;
  const unsigned ticket = __hip_atomic_fetch_add(came, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  rank = blocks = 0;
  if (ticket & CLOSED) return;
  for (int n = 0;; ++n) {
    unsigned now = __hip_atomic_load(came, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (now == gridDim.x) {
      rank = blockIdx.x;
      blocks = gridDim.x;
      return;
    }
    if (!(now & CLOSED) && n >= a.patience) {
      const unsigned seen = now;
      if (__hip_atomic_compare_exchange_strong(came, &now, seen | CLOSED, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        __hip_atomic_store(a.control + CLOSED_AT, seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      continue;
    }
    if (now & CLOSED) {
      const unsigned closed_at = __hip_atomic_load(a.control + CLOSED_AT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (closed_at) {
        rank = ticket;
        blocks = closed_at;
        return;
      }
      if (n >= a.patience + CLOSING) {
        gave_up(a);
        return;
      }
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

template <typename QKW, int GROUPS, int TURNED>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void decode_layers_kernel(Args a) {
  __shared__ Shared sh;
  if (threadIdx.x == 0) {
    sh.gave_up = 0;
    gather(a, sh.rank, sh.blocks);
  }
  if (threadIdx.x >> 6 == 1) share_out(a.shares, sh.shares, threadIdx.x & 63);
  __syncthreads();
  const int rank = __builtin_amdgcn_readfirstlane(sh.rank), blocks = __builtin_amdgcn_readfirstlane(sh.blocks);
  if (blocks == 0) return;
  for (int i = threadIdx.x; i < a.count * LAYER_WORDS; i += THREADS) sh.layers[i] = reinterpret_cast<const uint64_t*>(a.layers)[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Block<QKW, GROUPS, TURNED> b{sh, a, rank, blocks, wave, (int)threadIdx.x & 63, (int)threadIdx.x, numbers_of(a, rank, blocks, wave, threadIdx.x & 63),
                  min(MOST_SLABS, RESULTS / a.rows), a.limit, 1, (1u << 20) / a.rows + 1, -1};
  b.layers();
}

// The launch's table, its control words, an exchange without a word in it (a row of blocks fills a layer's), and before its first
// layer's part the stream's rows as a last product would leave them there. What parts of sequences there are room for but none of, stays
// as it is (24 rows of the 0.6B shape over 770 keys: 15 MB, 1,184 us a step and 1,169 without); where there are few a layer, asking how many
// there are takes longer.
struct Entry {
  const float* residual;
  const void* norm;
  int rows, width, norm_f32, turned;
  char *out, *sums;
};
struct Blank {
  char* exchange;
  long per_layer;
  int at_part, at_ml, at_att, group;
  ShareArgs shares;
};
constexpr int ITEMS_BLANKED = 256;
__device__ __forceinline__ void blank(char* from, long bytes) {
  const long each = (long)gridDim.x * 256;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < bytes / 16; i += each)
    reinterpret_cast<uint4*>(from)[i] = make_uint4(ABSENT, ABSENT, ABSENT, ABSENT);
}
__global__ __launch_bounds__(256) void decode_layers_begin_kernel(LayerPack pack, int first, int count, Layer* layers, unsigned* control, Blank to_blank,
                                                                  Entry entry) {
  if (blockIdx.x == 0 && blockIdx.y == 0) {
    const unsigned* from = reinterpret_cast<const unsigned*>(&pack);
    unsigned* to = reinterpret_cast<unsigned*>(layers + first);
    for (int i = threadIdx.x; i < count * (int)(sizeof(Layer) / 4); i += 256) to[i] = from[i];
    if (threadIdx.x < CONTROL_WORDS) control[threadIdx.x] = 0;
  }
  if (to_blank.exchange) {
    char* mine = to_blank.exchange + blockIdx.y * to_blank.per_layer;
    if (to_blank.shares.items_most <= ITEMS_BLANKED) {
      blank(mine, to_blank.per_layer);
    } else {
      __shared__ Shares shares;
      if (threadIdx.x < 64) share_out(to_blank.shares, shares, threadIdx.x);
      blank(mine, to_blank.at_part);
      blank(mine + to_blank.at_att, to_blank.per_layer - to_blank.at_att);
      __syncthreads();
      const long rows = shares.in_parts ? (long)shares.items * to_blank.group : 0;
      blank(mine + to_blank.at_part, rows * HEAD * 4);
      blank(mine + to_blank.at_ml, (rows * 8 + 15) & ~15l);
    }
  }
  const long each = (long)gridDim.x * gridDim.y * 256, me = ((long)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
  for (long i = me; i < (long)entry.rows * entry.width / 4; i += each) {       // (sixteen columns are four neighbouring lanes')
    const float4 x = reinterpret_cast<const float4*>(entry.residual)[i];
    const int n = (int)(i * 4 % entry.width);
    float4 w;
    if (entry.norm_f32) {
      w = *reinterpret_cast<const float4*>(static_cast<const float*>(entry.norm) + n);
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(entry.norm) + n);
      w = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
    }
    union {
      uint2 u;
      __bf16 e[4];
    } pk;
    pk.e[0] = (__bf16)(x.x * w.x), pk.e[1] = (__bf16)(x.y * w.y), pk.e[2] = (__bf16)(x.z * w.z), pk.e[3] = (__bf16)(x.w * w.w);
    const int to = place_of(entry.turned, (int)(i * 4 / entry.width), n, entry.width);
    *reinterpret_cast<uint2*>(entry.out + to) = make_uint2(marked(pk.u.x, 0x7fc07fc0u), marked(pk.u.y, 0x7fc07fc0u));
    float ss = x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    if ((i & 3) == 0) reinterpret_cast<unsigned*>(entry.sums)[i / 4] = marked(__float_as_uint(ss), 0x7fc00000u);
  }
}

__global__ void decode_layers_shares_kernel(ShareArgs args, int* out) {
  __shared__ Shares shares;
  share_out(args, shares, threadIdx.x);
  __syncthreads();
  if ((int)threadIdx.x < args.rows) out[2 * threadIdx.x] = shares.first[threadIdx.x], out[2 * threadIdx.x + 1] = shares.parts[threadIdx.x];
}

inline long up(long n) { return (n + 255) & ~255l; }

// How many rows lie side by side in what a product multiplies with (`place_of`), and for how many there is room.
inline int turned(int rows) { return rows > 8 ? 16 : rows > 4 ? 8 : rows > 2 ? 4 : rows; }
inline long rows_held(int rows) { return (long)(rows + turned(rows) - 1) / turned(rows) * turned(rows); }

struct Layout {
  long part, ml, att, mid, mid_sums, hid, out, out_sums, size;
};
inline Layout layout_of(long rows, long width, long heads, long kv_heads, long inner, long items) {
  Layout l;
  l.part = up(rows * (heads + 2 * kv_heads) * HEAD * 2);
  l.ml = l.part + items * (heads / kv_heads) * HEAD * 4;
  l.att = l.ml + up(items * (heads / kv_heads) * 8);
  const long held = rows_held(rows);
  l.mid = l.att + up(held * heads * HEAD * 2);
  l.mid_sums = l.mid + up(held * width * 2);
  l.hid = l.mid_sums + up(rows * (width / 16) * 4);
  l.out = l.hid + up(held * inner * 2);
  l.out_sums = l.out + up(held * width * 2);
  l.size = l.out_sums + up(rows * (width / 16) * 4);
  return l;
}

// Into how many parts a sequence may go, up to `parts`, and how many pieces that are in parts there may be
inline int parts_taken(long pairs, int parts) { return pairs < ITEMS_MOST ? parts : 1; }
inline long items_taken(long pairs, int parts) {
  if (parts_taken(pairs, parts) == 1) return 0;
  return pairs * parts < ITEMS_MOST ? pairs * parts : ITEMS_MOST;
}

// Up to how many rows this launch is the faster way (what is slower it does not take). Rows of more than 4,096 numbers, of two groups of
// sixteen more than 2,048, do not stay in registers from slab to slab and are asked for with each, rows / 16 of what its weights
// are; a width of that size is where a block has many slabs. The kernels one by one / this, us a step:
// - two groups, up to a width of 1,024 (14 layers): the 0.6B shape 17 rows over 300 keys 601 / 399, 32 over 2,000 1,170 / 948; an inner size of
//   8,192 17 over 300 712 / 525, 24 over 2,000 1,106 / 893. Longer sums, and widths up to 1,536: sixteen rows, and for more the kernels one by one;
// - two groups from 1,536 to 4,096, inner sizes to 18,944 (with rows in one piece each, `place_of`, the 8B shape took 20 over 1,000 in 4,327 / 5,229):
//   1,536 and 8,960 (12 layers) 17 over 300 807 / 571, 32 over 8,000 1,339 / 1,060; 2,048 and 6,144 (14) 17 over 300 833 / 591, 32 over
//   8,000 3,219 / 2,845; 2,560 and 9,728 (12) 17 over 300 1,032 / 916, 32 over 8,000 3,105 / 2,881; the 8B shape 17 over 1,000 4,244 / 3,886,
//   24 over 2,000 4,937 / 4,430, 32 over 500 4,312 / 4,008, over 2,000 5,210 / 4,892, 10 of its layers 17 over 100 1,061 / 969, 32 1,095 / 1,046, 32 over 8,000
//   2,833 / 2,656, one over 30,000 and 31 over 500 1,658 / 1,383; 4,096 and 18,944 (8) 17 over 300 1,349 / 1,107, 32 1,295 / 1,195; faster at each of 92 sizes;
// - one group, up to 4,096: 12 shapes from 512 to 4,096 wide, inner sizes to 18,944, 1 to 16 rows over 300 to 8,000 keys, all the faster
//   here, by 10 (the 8B shape, sixteen over 8,000) to 80 percent;
// - wider ones by how evenly the blocks have the slabs of the products into the stream. A last round half full or more: 6,144
//   (8 layers), one row 1,392 / 1,220, 8 1,541 / 1,501, 16 1,860 / 1,945; 8,192 (6 layers), one 1,954 / 1,783, 8 2,101 / 2,026, 16 2,373 / 2,441.
//   Less than that: 5,120 with an inner size of 17,408 (12 layers), 3 rows 2,007 / 1,987, 4 1,988 / 1,995, 5 2,105 / 2,164, 16 2,584 / 2,766; with
//   25,600 (10 layers) 3 rows 2,297 / 2,230, 5 2,395 / 2,411, 16 2,951 / 3,120; 4,608, 3 rows 1,052 / 1,028, 6 1,089 / 1,118.
inline int rows_most(int width, int heads, int inner) {
  if (width > 4096) return width / 16 % 256 == 0 || width / 16 % 256 >= 128 ? 8 : 3;
  const int longest = inner > heads * HEAD ? inner : heads * HEAD;
  if (width >= 1536) return longest <= 18944 ? MOST_ROWS : 16;
  return width > 1024 || longest > 8192 ? 16 : longest > 4096 ? 24 : MOST_ROWS;
}
// Every wavefront of a block has a step of 32 of each product's K at least: the smallest K is 256, from two heads on.
inline bool sizes_fit(int rows, int width, int heads, int kv_heads, int dim, int inner) {
  return rows >= 1 && dim == HEAD && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0 && heads / kv_heads <= 16 &&
         width >= 32 * WAVES && width % 128 == 0 && inner >= 32 * WAVES && inner % 128 == 0 && heads * HEAD >= 32 * WAVES &&
         width <= (1 << 16) && inner <= (1 << 18) && heads <= 512 && rows <= rows_most(width, heads, inner);
}

// The kernel for as many rows: two groups of sixteen of them, and how many lie side by side.
template <typename QKW>
void (*kernel_of(int rows))(Args) {
  if (rows > 16) return decode_layers_kernel<QKW, 2, 16>;
  switch (turned(rows)) {
    case 1: return decode_layers_kernel<QKW, 1, 1>;
    case 2: return decode_layers_kernel<QKW, 1, 2>;
    case 4: return decode_layers_kernel<QKW, 1, 4>;
    case 8: return decode_layers_kernel<QKW, 1, 8>;
    default: return decode_layers_kernel<QKW, 1, 16>;
  }
}

}  // namespace

extern "C" {

// Bytes of workspace for a step of `rows` single tokens over `count` layers: the layers' table, the control words, the exchange;
// 0 for sizes that are not taken.
long q3_decode_layers_workspace(int count, int rows, int width, int heads, int kv_heads, int dim, int inner, int parts) {
  if (count < 1 || count > MOST_LAYERS || !sizes_fit(rows, width, heads, kv_heads, dim, inner) || parts < 1 || parts > MOST_PARTS) return 0;
  const Layout l = layout_of(rows, width, heads, kv_heads, inner, items_taken((long)rows * kv_heads, parts));
  if (l.size > (1l << 30)) return 0;
  return up((long)count * sizeof(Layer)) + 256 + (count + 1) * l.size;
}

// How a step of `rows` sequences shares out their keys: per row its first piece and its parts, `out` (rows, 2).
int q3_decode_layers_shares(const int* kv_lens, int rows, int kv_heads, int parts, int* out, hipStream_t stream) {
  if (!kv_lens || !out || rows < 1 || rows > MOST_ROWS || kv_heads < 1 || kv_heads > 512 || parts < 1 || parts > MOST_PARTS) return Q3_ERR_BAD_ARGUMENT;
  const long pairs = (long)rows * kv_heads;
  const ShareArgs shares{kv_lens, rows, kv_heads, parts_taken(pairs, parts), (int)items_taken(pairs, parts)};
  hipLaunchKernelGGL(decode_layers_shares_kernel, dim3(1), dim3(64), 0, stream, shares, out);
  return q3_launch_status();
}

// Row b is the one token of sequence b, at position kv_lens[b] - 1, whose key and value are written to the caches; `residual` (rows,
// width) float32 is the stream, which the layers add to in place. `parts`: of a sequence's keys, at most. `blocks`: of the launch (0: one per processor); `patience`, `limit`: looks
// before the launch goes on with the blocks it has, and before a wait gives up (the stream is then not numbers, all of it, or some columns of
// every row: `Block::layers`, at its end).
int q3_decode_layers(const Layer* layers, int count, float* residual, int rows, int width, int heads, int kv_heads, int dim, int inner,
                     int norm_dtype, int qk_dtype, float qk_eps, float scale, const float* table, int rotary_dim, int max_pos,
                     const int* block_table, int table_width, const int* kv_lens, int max_kv_len, int page, int num_pages, int parts,
                     void* workspace, int blocks, int patience, int limit, hipStream_t stream) {
  if (!layers || !residual || !block_table || !kv_lens || !workspace || count < 1 || count > MOST_LAYERS || page < 16 || (page & (page - 1)) || num_pages < 1)
    return Q3_ERR_BAD_ARGUMENT;
  if (!sizes_fit(rows, width, heads, kv_heads, dim, inner) || parts < 1 || parts > MOST_PARTS || (table && rotary_dim != dim))
    return Q3_ERR_UNSUPPORTED;
  if ((table && max_kv_len > max_pos) || (long)table_width * page < max_kv_len || max_kv_len < 1 || patience < 1 || limit < 1 || blocks < 0)
    return Q3_ERR_BAD_ARGUMENT;
  if ((norm_dtype != Q3_F32 && norm_dtype != Q3_BF16) || (qk_dtype != Q3_F32 && qk_dtype != Q3_BF16)) return Q3_ERR_BAD_ARGUMENT;
  for (int i = 0; i < count; ++i) {
    const Layer& l = layers[i];
    if (!l.w[0] || !l.w[1] || !l.w[2] || !l.w[3] || !l.entry_norm || !l.middle_norm || !l.keys || !l.values ||
        (l.q_norm == nullptr) != (l.k_norm == nullptr))
      return Q3_ERR_BAD_ARGUMENT;
  }
  if (blocks == 0) {
    int device = 0;
    hipError_t status = hipGetDevice(&device);
    if (status == hipSuccess) status = hipDeviceGetAttribute(&blocks, hipDeviceAttributeMultiprocessorCount, device);
    if (status != hipSuccess) return (int)status;
  }
  const long items = items_taken((long)rows * kv_heads, parts);
  const Layout l = layout_of(rows, width, heads, kv_heads, inner, items);
  if (l.size > (1l << 30)) return Q3_ERR_UNSUPPORTED;
  Layer* held = (Layer*)workspace;
  unsigned* control = (unsigned*)((char*)workspace + up((long)count * sizeof(Layer)));
  char *entry_part = (char*)control + 256, *exchange = entry_part + l.size;
  const ShareArgs shares{kv_lens, rows, kv_heads, parts_taken((long)rows * kv_heads, parts), (int)items};
  const Blank to_blank{exchange, l.size, (int)l.part, (int)l.ml, (int)l.att, heads / kv_heads, shares};
  const Entry entry{residual, layers[0].entry_norm, rows, width, norm_dtype == Q3_F32, turned(rows), entry_part + l.out, entry_part + l.out_sums};
  for (int first = 0; first < count; first += LAYERS_A_LAUNCH) {
    const int n = count - first < LAYERS_A_LAUNCH ? count - first : LAYERS_A_LAUNCH;
    LayerPack pack{};
    for (int i = 0; i < n; ++i) pack.layer[i] = layers[first + i];
    // (eight pieces of sixteen bytes a thread)
    const long wanted = (l.size + 16 * 2048 - 1) / (16 * 2048);
    const dim3 grid = first == 0 ? dim3((unsigned)(wanted > 32 ? 32 : wanted), (unsigned)count) : dim3(1);
    hipLaunchKernelGGL(decode_layers_begin_kernel, grid, dim3(256), 0, stream, pack, first, n, held, control, first == 0 ? to_blank : Blank{},
                       first == 0 ? entry : Entry{});
  }
  Args a{};
  a.layers = held;
  a.control = control;
  a.exchange = exchange;
  a.residual = residual;
  a.table = table;
  a.block_table = block_table;
  a.per_layer = l.size;
  a.at_part = (int)l.part, a.at_ml = (int)l.ml, a.shares = shares;
  a.at_att = (int)l.att, a.at_mid = (int)l.mid, a.at_mid_sums = (int)l.mid_sums, a.at_hid = (int)l.hid;
  a.at_out = (int)l.out, a.at_out_sums = (int)l.out_sums;
  a.count = count, a.rows = rows, a.width = width, a.heads = heads, a.kv_heads = kv_heads, a.group = heads / kv_heads, a.inner = inner;
  a.norm_f32 = norm_dtype == Q3_F32;
  a.max_pos = max_pos, a.table_width = table_width, a.page = page, a.page_bits = __builtin_ctz(page), a.num_pages = num_pages;
  a.patience = patience, a.limit = limit;
  a.qk_eps = qk_eps;
  a.scale_log2 = make_score_scale(scale);
  auto kernel = qk_dtype == Q3_F32 ? kernel_of<float>(rows) : kernel_of<bf16_t>(rows);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(THREADS), 0, stream, a);
  return q3_launch_status();
}

}  // extern "C"
