// engine.cpp — replays recorded command lists on the device's HIP stream.
#include "engine.h"

#include <dlfcn.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <iterator>

#include "kernels.h"

namespace kz {

namespace {

template <class T>
hipError_t grow(T *&p, uint64_t count) {
    if (p) {
        hipError_t e = hipFree(p);
        p = nullptr;
        if (e != hipSuccess) return e;
    }
    return hipMalloc((void **)&p, std::max<uint64_t>(count, 1) * sizeof(T));
}

// gather binning: the most triangles and squares of a batch
constexpr uint32_t kGatherTris = 65536, kGatherSquares = 1024;
static_assert(kGatherTris <= KZ_GATHER_SEG * KZ_GATHER_SEGS, "segments of a batch");

// tiles whose state one thread of kz_bin_count clears, at least
constexpr uint32_t kInitTiles = 4;

// workgroups of kz_pair_scan that write the clip pieces' records (16 waves
// each, one triangle a wave at a time)
constexpr uint32_t kClipGrid = 64;

// striped partial counters followed by their totals
constexpr uint64_t kStatWords = (uint64_t)(KZ_STAT_STRIPES + 1) * KZ_STAT_COUNT;

#define KZ_TRY(x)                          \
    do {                                   \
        hipError_t e_ = (x);               \
        if (e_ != hipSuccess) return e_;   \
    } while (0)

}  // namespace

Engine::~Engine() {
    if (device_ < 0) return;
    hipSetDevice(device_);
    if (stream_) hipStreamSynchronize(stream_);
    hipFree(tile_counts_);
    hipFree(tile_offsets_);
    hipFree(tile_cursor_);
    hipFree(tile_lists_);
    hipFree(sort_tmp_);
    hipFree(tri_rect_);
    hipFree(tri_rec_);
    for (uint32_t *p : {tri_draw_, block_pairs_, chunk_offsets_, chunk_extra_, bin_ctrl_, tile_flag_, pair_keys_[0],
                        pair_keys_[1], pair_vals_[0], pair_vals_[1], radix_table_, radix_totals_, clip_of_, clip_tris_,
                        clip_rec_, gather_seg_, gather_list_, super_state_, zero_word_})
        hipFree(p);
    for (uint32_t *p : {tile_level_, split_slot_, split_info_, queue_, ctrl_, split_counts_, split_offsets_,
                        chunk_desc_, chunk_counts_, split_lists_, plan_table_, tile_acc_, tile_cycles_, tile_frags_, tri_z_})
        hipFree(p);
    hipFree(split_mask_);
    hipFree(list_mask_);
    hipFree(tile_feat_);
    hipFree(tile_pred_);
    hipFree(cost_model_d_);
    hipFree(stats_d_);
    if (stats_h_) hipHostFree(stats_h_);
    if (need_h_) hipHostFree(need_h_);
    for (hipEvent_t e : event_pool_) hipEventDestroy(e);
    if (ev_start_) hipEventDestroy(ev_start_);
    if (ev_end_) hipEventDestroy(ev_end_);
    if (stream_) hipStreamDestroy(stream_);
}

bool Engine::init(int hip_device, std::string &err) {
    device_ = hip_device;
    hipError_t e;
    if ((e = hipSetDevice(device_)) != hipSuccess || (e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking)) ||
        (e = hipEventCreate(&ev_start_)) || (e = hipEventCreate(&ev_end_)) ||
        (e = hipMalloc((void **)&stats_d_, kStatWords * sizeof(unsigned long long))) ||
        (e = hipHostMalloc((void **)&stats_h_, KZ_STAT_COUNT * sizeof(unsigned long long), hipHostMallocDefault)) ||
        (e = hipHostMalloc((void **)&need_h_, KZ_NEED_WORDS * sizeof(uint32_t), hipHostMallocCoherent))) {
        err = hipGetErrorString(e);
        return false;
    }
    std::memset(stats_h_, 0, KZ_STAT_COUNT * sizeof(unsigned long long));
    std::memset(need_h_, 0, KZ_NEED_WORDS * sizeof(uint32_t));
    // KAZAN_LIST_CAPACITY_LIMIT caps the per-tile list storage (entries);
    // tiles whose lists do not fit render through the in-order scan path
    if (const char *e = std::getenv("KAZAN_LIST_CAPACITY_LIMIT")) list_limit_ = std::strtoull(e, nullptr, 10);
    // KAZAN_CLIP_PIECES_LIMIT lowers the clip pieces kept per batch; triangles
    // past them are clipped again in every tile
    if (const char *e = std::getenv("KAZAN_CLIP_PIECES_LIMIT"))
        clip_limit_ = (uint32_t)std::min<uint64_t>(std::strtoull(e, nullptr, 10), clip_limit_);
    if (const char *e = std::getenv("KAZAN_PIPELINE")) balanced_ = std::strcmp(e, "plain") != 0;
    if (const char *e = std::getenv("KAZAN_AUTOTUNE")) autotune_ = std::strcmp(e, "0") != 0;
    if (const char *e = std::getenv("KAZAN_GRAPHS")) graphs_ = std::strcmp(e, "0") != 0;
    if (const char *e = std::getenv("KAZAN_SETUP_RECORDS")) setup_records_ = std::strcmp(e, "0") != 0;
    if (const char *e = std::getenv("KAZAN_BINNING")) {
        radix_ = std::strcmp(e, "sort") != 0;
        gather_ = radix_ && std::strcmp(e, "radix") != 0;
        gather_always_ = std::strcmp(e, "gather") == 0;
    }
    if (const char *e = std::getenv("KAZAN_GRID_DIVISOR")) {
        const int d = std::atoi(e);
        default_grid_div_ = d == 2 || d == 4 ? (uint32_t)d : 1u;
    }
    if (const char *e = std::getenv("KAZAN_SPLIT_LEVEL")) default_max_level_ = (uint32_t)std::min(std::max(std::atoi(e), 0), 2);
    if (radix_ &&
        ((e = hipMalloc((void **)&bin_ctrl_, KZ_BIN_WORDS * sizeof(uint32_t))) != hipSuccess ||
         (e = kz_launch_fill_u32(stream_, bin_ctrl_, KZ_BIN_WORDS, 0u)) != hipSuccess ||
         (e = hipMalloc((void **)&radix_totals_, kz_radix_digits_max() * sizeof(uint32_t))) != hipSuccess)) {
        err = hipGetErrorString(e);
        return false;
    }
    if ((e = hipMalloc((void **)&zero_word_, sizeof(uint32_t))) != hipSuccess ||
        (e = kz_launch_fill_u32(stream_, zero_word_, 1, 0u)) != hipSuccess) {
        err = hipGetErrorString(e);
        return false;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device_) == hipSuccess && cus > 0)
        split_grid_ = 4u * (uint32_t)cus;
    // the cost model: $KAZAN_COST_MODEL, else cost_model.bin beside this library
    std::string path;
    if (const char *e = std::getenv("KAZAN_COST_MODEL")) {
        path = e;
    } else {
        Dl_info info;
        if (dladdr((void *)&kz_launch_fill_u32, &info) && info.dli_fname) {
            path = info.dli_fname;
            const size_t slash = path.rfind('/');
            path = (slash == std::string::npos ? std::string(".") : path.substr(0, slash)) + "/cost_model.bin";
        }
    }
    if (!path.empty() && path != "none") {
        std::ifstream in(path, std::ios::binary);
        if (in) {
            std::vector<char> blob((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
            if (set_cost_model(blob.data(), blob.size())) cost_model_src_ = path;
        }
    }
    return true;
}

bool Engine::set_cost_model(const void *blob, size_t bytes) {
    KzCostModel m;
    if (!blob || bytes != sizeof m) return false;
    std::memcpy(&m, blob, sizeof m);
    if (m.magic != KZ_COST_MODEL_MAGIC || m.version != 1 || m.bytes != sizeof m) return false;
    if (!cost_model_d_ && hipMalloc((void **)&cost_model_d_, sizeof m) != hipSuccess) {
        cost_model_d_ = nullptr;
        return false;
    }
    if (hipStreamSynchronize(stream_) != hipSuccess ||
        hipMemcpy(cost_model_d_, &m, sizeof m, hipMemcpyHostToDevice) != hipSuccess)
        return false;
    frag_weight_ = m.frag_weight;
    ++generation_;  // captured graphs carry the old model's frag_weight
    cost_model_src_ = "memory";
    return true;
}

hipError_t Engine::ensure_model_scratch(uint32_t tiles, uint32_t tris) {
    if (tiles <= cap_model_tiles_ && tris <= cap_model_tris_) return hipSuccess;
    KZ_TRY(hipStreamSynchronize(stream_));
    if (tiles > cap_model_tiles_) {
        const uint32_t t = std::max(tiles, cap_model_tiles_ * 2);
        KZ_TRY(regrow(tile_acc_, (uint64_t)KZ_ACC * t));
        KZ_TRY(regrow(tile_feat_, (uint64_t)KZ_FEATURES * t));
        KZ_TRY(regrow(tile_pred_, t));
        KZ_TRY(regrow(tile_frags_, t));
        KZ_TRY(regrow(tile_cycles_, t));
        cap_model_tiles_ = t;
    }
    if (tris > cap_model_tris_) {
        const uint32_t t = std::max(tris, cap_model_tris_ + cap_model_tris_ / 2);
        KZ_TRY(regrow(tri_z_, t));
        cap_model_tris_ = t;
    }
    return hipSuccess;
}

namespace {
hipError_t copy_u32_as_float(float *dst, const uint32_t *src, uint32_t n) {
    std::vector<uint32_t> c(n);
    KZ_TRY(hipMemcpy(c.data(), src, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
    for (uint32_t i = 0; i < n; ++i) dst[i] = (float)c[i];
    return hipSuccess;
}
}  // namespace

hipError_t Engine::read_tile_profile(uint32_t *tiles, float *features, float *frags, float *cycles, float *pred) {
    KZ_TRY(hipSetDevice(device_));
    KZ_TRY(hipStreamSynchronize(stream_));
    const uint32_t n = tile_feat_ ? last_profile_tiles_ : 0;
    if (tiles) *tiles = n;
    if (n == 0) return hipSuccess;
    if (features)
        KZ_TRY(hipMemcpy(features, tile_feat_, (size_t)n * KZ_FEATURES * sizeof(float), hipMemcpyDeviceToHost));
    if (frags) {
        if (last_profile_labels_) KZ_TRY(copy_u32_as_float(frags, tile_frags_, n));
        else std::fill(frags, frags + n, 0.0f);
    }
    if (cycles) {
        if (last_profile_labels_) KZ_TRY(copy_u32_as_float(cycles, tile_cycles_, n));
        else std::fill(cycles, cycles + n, 0.0f);
    }
    if (pred) {
        if (last_profile_pred_) KZ_TRY(hipMemcpy(pred, tile_pred_, n * sizeof(float), hipMemcpyDeviceToHost));
        else std::fill(pred, pred + n, 0.0f);
    }
    return hipSuccess;
}

// Called after ensure_scratch (the chunk tables follow the list capacity).
hipError_t Engine::ensure_split_scratch(uint32_t tiles) {
    // a split tile's list fits the list storage, so its chunks number at
    // most list_capacity / KZ_SPLIT_CHUNK plus one partial chunk per tile
    const uint64_t want_chunks = (uint64_t)list_capacity_ / KZ_SPLIT_CHUNK + tiles;
    const uint32_t want_split = std::max(split_capacity_, list_capacity_);
    if (tiles <= cap_split_tiles_ && want_chunks <= max_chunks_ && want_split <= split_capacity_) return hipSuccess;
    KZ_TRY(hipStreamSynchronize(stream_));
    if (tiles > cap_split_tiles_) {
        const uint32_t t = std::max(tiles, cap_split_tiles_ * 2);
        KZ_TRY(regrow(tile_level_, t));
        KZ_TRY(regrow(split_slot_, t));
        KZ_TRY(regrow(split_info_, 2ull * t));
        KZ_TRY(regrow(queue_, 16ull * t));
        KZ_TRY(regrow(split_counts_, 16ull * t));
        KZ_TRY(regrow(split_offsets_, 16ull * t));
        KZ_TRY(regrow(plan_table_, kz_plan_table_words(t)));
        if (!ctrl_) {
            KZ_TRY(hipMalloc((void **)&ctrl_, KZ_CTRL_WORDS * sizeof(uint32_t)));
            KZ_TRY(kz_launch_fill_u32(stream_, ctrl_, KZ_CTRL_WORDS, 0u));
        }
        cap_split_tiles_ = t;
    }
    if (want_chunks > max_chunks_) {
        const uint64_t c = std::min<uint64_t>(std::max<uint64_t>(want_chunks, (uint64_t)max_chunks_ * 3 / 2),
                                              0x0FFFFFFFull);
        KZ_TRY(regrow(chunk_desc_, 4 * c));
        KZ_TRY(regrow(chunk_counts_, 16 * c));
        KZ_TRY(regrow(split_mask_, (uint64_t)KZ_SPLIT_CHUNK * c));
        max_chunks_ = (uint32_t)c;
    }
    if (want_split > split_capacity_) {
        KZ_TRY(regrow(split_lists_, want_split));
        split_capacity_ = want_split;
    }
    return hipSuccess;
}

hipError_t Engine::ensure_scratch(uint32_t tiles, uint32_t tris) {
    uint64_t want_list = std::max<uint64_t>(list_capacity_, 4ull * tris + 65536ull);
    if (list_limit_) want_list = std::min<uint64_t>(want_list, list_limit_);
    if (tiles <= cap_tiles_ && tris <= cap_tris_ && want_list <= list_capacity_) return hipSuccess;
    // buffers may still be in use by queued work
    KZ_TRY(hipStreamSynchronize(stream_));
    if (tiles > cap_tiles_) {
        const uint32_t t = std::max(tiles, cap_tiles_ * 2);
        KZ_TRY(regrow(tile_counts_, t));
        KZ_TRY(regrow(tile_offsets_, t));
        if (radix_) {
            KZ_TRY(regrow(tile_flag_, t));  // cleared with the counts before each batch
        } else {
            KZ_TRY(regrow(tile_cursor_, t));
        }
        cap_tiles_ = t;
    }
    if (tris > cap_tris_) {
        const uint32_t t = std::max(tris, cap_tris_ + cap_tris_ / 2);
        // (clip pieces: as many as there are triangles in a small batch; past
        // the limit the raster clips what is left tile by tile)
        cap_clip_ = radix_ && !setup_records_ ? std::min(std::max(t, 1024u), clip_limit_) : 0u;
        KZ_TRY(regrow(tri_rect_, (uint64_t)t + cap_clip_));
        KZ_TRY(regrow(tri_draw_, t));
        if (cap_clip_) {
            KZ_TRY(regrow(clip_of_, t));
            KZ_TRY(regrow(clip_tris_, cap_clip_));
        }
        if (radix_) {
            KZ_TRY(regrow(block_pairs_, (t + KZ_BIN_BLOCK - 1) / KZ_BIN_BLOCK));
            KZ_TRY(regrow(chunk_offsets_, (t + KZ_PAIR_CHUNK - 1) / KZ_PAIR_CHUNK));
            KZ_TRY(regrow(chunk_extra_, (t + KZ_PAIR_CHUNK - 1) / KZ_PAIR_CHUNK));
        }
        cap_tris_ = t;
    }
    if (want_list > list_capacity_) {
        const uint64_t c = std::min<uint64_t>(std::max<uint64_t>(want_list, (uint64_t)list_capacity_ * 3 / 2),
                                              0xFFFFFFF0ull);
        KZ_TRY(alloc_lists(c));
    }
    return hipSuccess;
}

namespace {
// The squares of gather binning over a w x h framebuffer
uint32_t squares(uint32_t px) { return (px + (1u << KZ_SUPER_PX_SHIFT) - 1) >> KZ_SUPER_PX_SHIFT; }

// entries of one square's coarse list: 32 per triangle over all squares (a
// square that needs more tests its segments' triangles one by one)
uint32_t gather_square_cap(uint32_t tris, uint32_t supers) {
    return (uint32_t)std::min<uint64_t>(tris, std::max<uint64_t>(4096, 32ull * tris / supers));
}
}  // namespace

// Gather binning's work, where radix binning's grows with the pairs only:
// - every segment is tested against every square (3 ns each);
// - a square's blocks of 8 tiles each read its list: ns per square by tile
//   size, between a grid's (all tiles busy) and a cluster's;
// - they do so the longer the denser the triangles, and at larger tiles a
//   wave walks more of them alone.
// The line is where the radix chain (eight launches, 40 to 50 us) has caught up
// over a grid, a cluster and 64 meshes drawn as one batch and as 64. Frames at
// one tile size and the plain raster, radix us / gather us of the four:
//   16 px tiles: 65,536 triangles at 720p 100/77, 81/73, 97/83, 2500/1442, at
//   1440p 153/158, 81/86, 117/119, 3047/1993, in 640x480 85/64, 112/124, 92/74,
//   2369/1378, and 8,192 at 4K 199/213, 86/77, 116/105, 3192/2445; past the
//   line at 4K 65,536 235/280, 95/126, 129/150 (as 64 batches each is within),
//   and in 256^2 67/71, 199/217, 68/64;
//   8 px: 8,192 in 640x480 83/76, 61/40, 74/57, 2241/1250, at 720p 104/129,
//   65/55, 85/70, 2445/1519 (a grid is 15 to 60 us faster at 16 px), 65,536 in
//   256^2 66/59, 114/116, 70/55, 2197/1226; past it at 1080p 139/213, 75/77,
//   103/97, at 4K 311/572, 128/163, 169/215, and 65,536 in 128^2 61/62, 92/138;
//   32 px: 32,768 at 720p 116/92, 93/83, 110/92; past it 65,536 129/122,
//   126/140, 126/116 and 32,768 in 640x480 126/117, 136/167;
//   64 px: 8,192 at 1080p 317/304, 91/83; past it 32,768 372/362, 144/150.
// With the tuner's choice of tiles and raster, gathering wherever the tables
// fit against this (grid, cluster, meshes): 65,536 triangles at 4K 274/237,
// 123/96, 132/112, in 256^2 59/59, 114/96, 42/41, in 128^2 50/50, 139/94, 38/45;
// within 4 % at 1440p, 1080p, 720p and in 640x480 and below.
bool gather_pays(uint32_t tris, uint32_t width, uint32_t height, uint32_t shift) {
    const uint64_t supers = (uint64_t)squares(width) * squares(height);
    const uint64_t segs = (tris + KZ_GATHER_SEG - 1) / KZ_GATHER_SEG;
    static constexpr uint32_t kSquareNs[] = {900, 96, 24, 8};  // 8 px tiles on
    static_assert(sizeof kSquareNs / sizeof *kSquareNs == kMaxTileShift - kMinTileShift + 1, "a cost per tile size");
    const uint32_t most = shift <= 4 ? kGatherTris : shift == 5 ? kGatherTris / 2 : kGatherTris / 4;
    const uint32_t density = shift > 4 ? 640u : shift == 3 ? 16384u : 4096u;
    return tris <= most && tris <= std::max<uint64_t>(supers * density, 2048) &&
           supers * (kSquareNs[shift - kMinTileShift] + 3 * segs) <= 56000;
}

// (squares: their totals are summed by every workgroup)
bool Engine::use_gather(const KzFrame &f, uint32_t shift) const {
    if (!gather_ || f.total_tris > kGatherTris || (uint64_t)squares(f.width) * squares(f.height) > kGatherSquares)
        return false;
    return gather_always_ || gather_pays(f.total_tris, f.width, f.height, shift);
}

hipError_t Engine::ensure_gather(const KzFrame &f) {
    const uint32_t supers = squares(f.width) * squares(f.height);
    const uint32_t segs = supers * ((f.total_tris + KZ_GATHER_SEG - 1) / KZ_GATHER_SEG);
    const uint64_t entries = (uint64_t)supers * gather_square_cap(f.total_tris, supers);
    if (supers <= cap_supers_ && segs <= cap_gather_segs_ && entries <= cap_gather_) return hipSuccess;
    KZ_TRY(hipStreamSynchronize(stream_));
    if (supers > cap_supers_) {
        KZ_TRY(regrow(super_state_, (uint64_t)supers * KZ_SUPER_WORDS));
        cap_supers_ = supers;
    }
    if (segs > cap_gather_segs_) {
        KZ_TRY(regrow(gather_seg_, 2ull * segs));
        cap_gather_segs_ = segs;
    }
    if (entries > cap_gather_) {
        KZ_TRY(regrow(gather_list_, 2 * entries));
        cap_gather_ = entries;
    }
    return hipSuccess;
}

hipError_t Engine::alloc_lists(uint64_t capacity) {
    list_capacity_ = 0;
    KZ_TRY(regrow(tile_lists_, capacity));
    if (radix_) {
        for (int i = 0; i < 2; ++i) {
            KZ_TRY(regrow(pair_keys_[i], capacity));
            KZ_TRY(regrow(pair_vals_[i], capacity));
        }
        KZ_TRY(regrow(radix_table_, (uint64_t)kz_radix_digits_max() * kz_radix_blocks(capacity)));
        if (balanced_) KZ_TRY(regrow(list_mask_, capacity));
    } else {
        KZ_TRY(regrow(sort_tmp_, capacity));
    }
    list_capacity_ = (uint32_t)capacity;
    return hipSuccess;
}

// Statistics accumulate over all submissions since the last collect_stats():
// a caller that queues K frames and then waits reads the K-frame totals and
// the GPU time from the first submission's start to the last one's end.
hipError_t Engine::begin_submit() {
    KZ_TRY(hipSetDevice(device_));
    if (!submit_open_) {
        KZ_TRY(kz_launch_fill_u32(stream_, (uint32_t *)stats_d_, kStatWords * 2, 0u));
        KZ_TRY(hipEventRecord(ev_start_, stream_));
        pending_batches_ = pending_launches_ = 0;
        submit_open_ = true;
    }
    return hipSuccess;
}

// All allocations a batch needs at tile size 1 << shift (so that a graph
// capture of the batch allocates nothing).
hipError_t Engine::prepare_batch(const Op &op, uint32_t shift) {
    const KzFrame &f = op.frame;
    if (f.total_tris == 0) return hipSuccess;
    const uint32_t ts = 1u << shift;
    const uint32_t ntiles = ((f.width + ts - 1) >> shift) * ((f.height + ts - 1) >> shift);
    KZ_TRY(ensure_scratch(ntiles, f.total_tris));
    if (setup_records_) {
        const uint64_t words = (uint64_t)f.total_tris * KZ_REC_WORDS_FOR(op.variants->fixed.num_varyings);
        if (words > cap_rec_words_) {
            KZ_TRY(hipStreamSynchronize(stream_));
            const uint64_t w = std::max(words, cap_rec_words_ + cap_rec_words_ / 2);
            KZ_TRY(regrow(tri_rec_, w));
            cap_rec_words_ = w;
        }
    }
    if (use_gather(f, shift)) KZ_TRY(ensure_gather(f));
    const uint64_t clip_words = (uint64_t)cap_clip_ * KZ_REC_WORDS_FOR(op.variants->fixed.num_varyings);
    if (clip_words > cap_clip_words_) {
        KZ_TRY(hipStreamSynchronize(stream_));
        KZ_TRY(regrow(clip_rec_, clip_words));
        cap_clip_words_ = clip_words;
    }
    if (balanced_) KZ_TRY(ensure_split_scratch(ntiles));
    if ((cost_model_d_ != nullptr && balanced_) || tile_profile_) KZ_TRY(ensure_model_scratch(ntiles, f.total_tris));
    return hipSuccess;
}

hipError_t Engine::run_batch(const Op &op, const BatchConfig &cfg) {
    KzFrame f = op.frame;
    if (f.total_tris == 0) return hipSuccess;
    const uint32_t shift = cfg.shift, grid_div = cfg.grid_div;
    // the balanced form's planned, persistent raster (else one workgroup per tile)
    const bool persistent = balanced_ && cfg.persistent;
    std::string err;
    const PipelineKernels *kern = op.variants->get(shift, &err);
    if (!kern) {
        std::fprintf(stderr, "kazan: tile size %u: %s\n", 1u << shift, err.c_str());
        return hipErrorInvalidValue;
    }
    const uint32_t ts = 1u << shift;
    f.tiles_x = (f.width + ts - 1) >> shift;
    f.tiles_y = (f.height + ts - 1) >> shift;
    const uint32_t ntiles = f.tiles_x * f.tiles_y;
    KZ_TRY(prepare_batch(op, shift));
    f.draws = op.d_draws;
    f.draw_begin = op.d_draw_begin;
    f.block_draw = op.d_block_draw;
    f.tile_counts = tile_counts_;
    f.tile_offsets = tile_offsets_;
    f.tile_cursor = tile_cursor_;
    f.tile_flag = radix_ ? tile_flag_ : nullptr;
    f.bin_ctrl = radix_ ? bin_ctrl_ : nullptr;
    f.tile_lists = tile_lists_;
    f.sort_tmp = sort_tmp_;
    f.list_capacity = list_capacity_;
    f.tri_rect = tri_rect_;
    f.tri_draw = f.ndraws > 1 ? tri_draw_ : nullptr;
    f.tri_rec = setup_records_ ? tri_rec_ : nullptr;
    f.stats = stats_d_;
    f.need = need_h_;
    f.tile_shift = shift;
    if (persistent) {
        f.balanced = 1;
        f.split_capacity = split_capacity_;
        f.queue = queue_;
        f.ctrl = ctrl_;
        f.tile_level = tile_level_;
        f.split_slot = split_slot_;
        f.split_info = split_info_;
        f.chunk_desc = chunk_desc_;
        f.chunk_counts = chunk_counts_;
        f.split_mask = split_mask_;
        f.split_counts = split_counts_;
        f.split_offsets = split_offsets_;
        f.split_lists = split_lists_;
        f.max_chunks = max_chunks_;
        f.raster_slots = std::max(1u, kern->persistent_blocks / std::max(grid_div, 1u));
        f.split_max_level = std::min(cfg.max_level, 2u);
        // the sub-tile masks travel in the pairs' keys (above 16 tile bits)
        // through the radix sort, so the split reads them beside the lists
        // instead of gathering pixel boxes
        if (radix_ && list_mask_ && f.split_max_level > 0 && shift >= 2 && ntiles < 65536u) f.list_mask = list_mask_;
    }
    // the cost model's inputs (and, in the static form, its labels) when a
    // model will run or tiles are being profiled
    // (predictions also run in a profiled static batch, to measure the
    // model's error against the fragments the rasteriser counts)
    const bool model = cost_model_d_ != nullptr && ((persistent && cfg.model) || tile_profile_);
    const bool acc = model || tile_profile_;
    const bool labels = tile_profile_ && !persistent;
    if (acc) {
        f.tri_z = tri_z_;
        f.tile_acc = tile_acc_;
        f.tile_feat = tile_feat_;
        if (model && persistent) {
            f.tile_pred = tile_pred_;
            f.frag_weight = frag_weight_ * (float)std::max(cfg.frag_scale, 1u);
        }
        if (labels) {
            f.tile_frags = tile_frags_;
            f.tile_cycles = tile_cycles_;
        }
    }
    void *args[] = {&f};
    // a thread per triangle, and enough of them to clear the tiles' state
    const uint32_t tri_blocks = std::max((f.total_tris + 255) / 256,
                                         std::min((ntiles + 256 * kInitTiles - 1) / (256 * kInitTiles), 4096u));
    uint32_t launches = 0;

    // binning: pixel boxes, then the per-tile lists in primitive order
    if (use_gather(f, shift)) {
        const uint32_t supers_x = squares(f.width), supers_y = squares(f.height);
        f.super_shift = KZ_SUPER_PX_SHIFT - shift;
        f.supers_x = supers_x;
        f.supers_y = supers_y;
        f.gather_segs = (f.total_tris + KZ_GATHER_SEG - 1) / KZ_GATHER_SEG;
        f.gather_cap = gather_square_cap(f.total_tris, supers_x * supers_y);
        f.gather_seg = gather_seg_;
        f.gather_list = gather_list_;
        f.super_state = super_state_;
        f.tile_flag = nullptr;  // (no cut: a list that does not fit is a scan)
        f.clip_cap = cap_clip_;
        f.clip_of = clip_of_;
        f.clip_tris = clip_tris_;
        f.clip_rec = clip_rec_;
        KZ_TRY(mark(KS_BIN_COUNT, false));
        KZ_TRY(hipModuleLaunchKernel(kern->bin_count, tri_blocks, 1, 1, KZ_BIN_BLOCK, 1, 1, 0, stream_, args,
                                     nullptr));
        KZ_TRY(mark(KS_BIN_COUNT, true));
        KZ_TRY(mark(KS_BIN_HIST, false));
        KZ_TRY(hipModuleLaunchKernel(kern->gather_coarse, supers_x * supers_y * f.gather_segs + kClipGrid, 1, 1, 256, 1,
                                     1, 0, stream_, args, nullptr));
        KZ_TRY(mark(KS_BIN_HIST, true));
        KZ_TRY(mark(KS_BIN_SCATTER, false));
        KZ_TRY(kz_launch_gather_lists(stream_, f));
        KZ_TRY(mark(KS_BIN_SCATTER, true));
        launches += 3;
    } else if (radix_) {
        // pairs in primitive order, a stable radix sort by tile whose last
        // pass writes the lists, counts and offsets
        f.block_pairs = block_pairs_;
        f.chunk_offsets = chunk_offsets_;
        f.chunk_extra = chunk_extra_;
        f.clip_cap = cap_clip_;
        f.clip_of = clip_of_;
        f.clip_tris = clip_tris_;
        f.clip_rec = clip_rec_;
        KzRadixScratch rs{bin_ctrl_, tile_flag_, {pair_keys_[0], pair_keys_[1]},
                          {pair_vals_[0], pair_vals_[1]}, radix_table_, radix_totals_,
                          kz_radix_blocks(list_capacity_)};
        KZ_TRY(mark(KS_BIN_COUNT, false));
        KZ_TRY(hipModuleLaunchKernel(kern->bin_count, tri_blocks, 1, 1, KZ_BIN_BLOCK, 1, 1, 0, stream_, args,
                                     nullptr));
        KZ_TRY(mark(KS_BIN_COUNT, true));
        KZ_TRY(mark(KS_BIN_HIST, false));
        KZ_TRY(hipModuleLaunchKernel(kern->pair_scan, 1 + kClipGrid, 1, 1, 1024, 1, 1, 0, stream_, args, nullptr));
        KZ_TRY(kz_launch_bin_pairs(stream_, f, rs));
        KZ_TRY(mark(KS_BIN_HIST, true));
        KZ_TRY(mark(KS_BIN_SCATTER, false));
        KZ_TRY(kz_launch_bin_radix(stream_, f, rs, ntiles));
        KZ_TRY(mark(KS_BIN_SCATTER, true));
        launches += 1 + 2 + 3 * kz_radix_passes(ntiles);
    } else {
        // per-tile counts, offsets, an unordered scatter, a sort of each list
        KZ_TRY(mark(KS_BIN_COUNT, false));
        KZ_TRY(hipModuleLaunchKernel(kern->bin_count, tri_blocks, 1, 1, KZ_BIN_BLOCK, 1, 1, 0, stream_, args,
                                     nullptr));
        KZ_TRY(mark(KS_BIN_COUNT, true));
        KZ_TRY(mark(KS_BIN_HIST, false));
        KZ_TRY(acc ? kz_launch_bin_hist_acc(stream_, f) : kz_launch_bin_hist(stream_, f));
        KZ_TRY(mark(KS_BIN_HIST, true));
        KZ_TRY(mark(KS_BIN_SCAN, false));
        KZ_TRY(kz_launch_scan(stream_, tile_counts_, tile_offsets_, tile_cursor_, ntiles, list_capacity_, stats_d_,
                              need_h_));
        KZ_TRY(mark(KS_BIN_SCAN, true));
        KZ_TRY(mark(KS_BIN_SCATTER, false));
        KZ_TRY(kz_launch_bin_scatter(stream_, f));
        KZ_TRY(mark(KS_BIN_SCATTER, true));
        KZ_TRY(mark(KS_BIN_SORT, false));
        KZ_TRY(kz_launch_sort_lists(stream_, f, ntiles));
        KZ_TRY(mark(KS_BIN_SORT, true));
        launches += 6;
    }

    if (!persistent) {
        if (acc) {
            KZ_TRY(kz_launch_tile_features(stream_, f, ntiles));
            launches += 1;
        }
        if (model) {
            KZ_TRY(kz_launch_cost_mlp(stream_, cost_model_d_, tile_feat_, ntiles, tile_pred_));
            launches += 1;
        }
        KZ_TRY(mark(KS_RASTER, false));
        KZ_TRY(hipModuleLaunchKernel(kern->raster, ntiles, 1, 1, 64, 1, 1, 0, stream_, args, nullptr));
        KZ_TRY(mark(KS_RASTER, true));
        launches += 1;
    } else {
        // predicted costs, split expensive tiles, cut their sub-tile lists,
        // order the items
        KZ_TRY(mark(KS_PLAN, false));
        if (model) {  // features, predictions and the plan's cost parts: one launch
            KZ_TRY(kz_launch_cost_plan(stream_, cost_model_d_, f, ntiles, plan_table_));
            launches += 1;
        } else if (acc) {
            KZ_TRY(kz_launch_tile_features(stream_, f, ntiles));
            launches += 1;
        }
        KZ_TRY(kz_launch_plan(stream_, f, ntiles, plan_table_, model));
        KZ_TRY(kz_launch_split(stream_, f, split_grid_, ntiles));
        KZ_TRY(mark(KS_PLAN, true));
        KZ_TRY(mark(KS_RASTER, false));
        const uint32_t grid = std::min(f.raster_slots, 16 * ntiles);
        KZ_TRY(hipModuleLaunchKernel(kern->raster_persistent, grid, 1, 1, 64, 1, 1, 0, stream_, args, nullptr));
        KZ_TRY(mark(KS_RASTER, true));
        // the plan (2, or 3 with its own cost pass), the split (4), the raster
        launches += (!model && !f.bin_ctrl) ? 8 : 7;
    }
    if (acc) {
        last_profile_tiles_ = ntiles;
        last_profile_pred_ = model;
        last_profile_labels_ = labels;
    }
    pending_batches_ += 1;
    pending_launches_ += launches;
    return hipSuccess;
}

hipError_t Engine::mark(int slot, bool end) {
    if (!kernel_timing_) return hipSuccess;
    if (events_used_ == event_pool_.size()) {
        hipEvent_t e;
        KZ_TRY(hipEventCreate(&e));
        event_pool_.push_back(e);
    }
    hipEvent_t e = event_pool_[events_used_++];
    KZ_TRY(hipEventRecord(e, stream_));
    timing_events_.push_back({end ? -1 - slot : slot, e});
    return hipSuccess;
}

BatchTuning::~BatchTuning() {
    if (trial) hipGraphExecDestroy(trial);
    for (hipEvent_t e : ev)
        if (e) hipEventDestroy(e);
}

void GraphCache::reset() {
    if (exec) hipGraphExecDestroy(exec);
    exec = nullptr;
    generation = 0;
}

template <class T>
hipError_t Engine::regrow(T *&p, uint64_t count) {
    ++generation_;
    return grow(p, count);
}

// The untuned configuration of a batch.
BatchConfig Engine::default_config(const Op &op) const {
    BatchConfig c;
    c.shift = op.tile_shift;
    c.grid_div = default_grid_div_;
    c.model = true;
    c.persistent = balanced_;
    c.max_level = default_max_level_;
    c.frag_scale = 1;
    return c;
}

namespace {
int fastest(const BatchTuning &t) {
    int best = -1;
    for (size_t i = 0; i < t.cand.size(); ++i)
        if (t.ms[i] >= 0 && (best < 0 || t.ms[i] < t.ms[best])) best = (int)i;
    return best;
}

// The choice: the finalist with the lowest median of its runs (one lucky
// run does not decide), else the fastest run.
int final_choice(const BatchTuning &t) {
    int best = -1;
    float best_ms = 0.0f;
    for (const std::vector<size_t> &runs : t.finals) {
        std::vector<float> v;
        for (size_t i : runs)
            if (t.ms[i] >= 0) v.push_back(t.ms[i]);
        if (v.empty()) continue;
        std::sort(v.begin(), v.end());
        const float med = v[v.size() / 2];
        if (best < 0 || med < best_ms) {
            best = (int)runs[0];
            best_ms = med;
        }
    }
    return best >= 0 ? best : fastest(t);
}
}  // namespace

// The first candidates: every tile size, the pipeline's own (which the first
// submission ran untimed) last.
void BatchTuning::begin(uint32_t own_shift, bool model) {
    for (uint32_t s = kMinTileShift; s <= kMaxTileShift; ++s)
        if (s != own_shift) cand.push_back({s, 1u, model, true, 2u});
    cand.push_back({own_shift, 1u, model, true, 2u});
    ms.assign(cand.size(), -1.0f);
}

// Candidates, one HIP-event-timed trial per submission from a recording's
// second on: every tile size (full grid, the plan with the cost model when
// there is one); at the fastest size, the model's plan with its fragment
// weight times 16 (without a model a half grid) and the plain raster (one
// workgroup per tile, no plan); at the fastest of those, the plan without the
// model and the plain raster of the next smaller tiles (the plain raster's
// neighbours when it is the fastest); at the fastest planned one, splits of at
// most 4 sub-tiles and none (many small triangles are set up once per sub-tile
// they touch); with a cost model, the model's plan with its fragment weight
// times 4, and times 16 with splits of at most 4 (a pipeline whose fragments
// cost more than the training pipelines'); at the fastest planned one, every
// other pair of tile size and grid size (both were chosen with the deepest
// splits and the model; with fewer splits smaller tiles on a larger grid may
// pay); then the three fastest, no two of them the same configuration, twice
// more each. The finalist with the lowest median of its three runs is kept.
// Candidates whose kernels do not build (tiles that do not fit LDS among
// them) are passed over. False when no trial is left: choice is then set, or
// left as it was if none could be timed.
bool BatchTuning::more(bool model, const std::function<bool(uint32_t shift)> &builds) {
    for (;; ++phase) {
        while (next < cand.size() && !builds(cand[next].shift)) ++next;
        if (next < cand.size()) return true;
        if (phase == 6) break;
        const int best = fastest(*this);
        if (best < 0) continue;
        const BatchConfig b = cand[best];
        if (phase == 0) {
            // (fragments weighted 16 times: where a frame has few tiles, of
            // many fragments each, its splits are what a plan is for, and it
            // has to be seen before the plain raster ends the search: 256
            // triangles in 64^2 83 us a frame, plain 89)
            if (b.model) cand.push_back({b.shift, 1u, true, true, 2u, 16u});
            else cand.push_back({b.shift, 2u, false, true, 2u, 1u});
            cand.push_back({b.shift, 1u, false, false, 2u, 1u});
        } else if (phase == 1) {
            // the plain raster has only its tiles to fill the chip with:
            // smaller ones often suit it better than the plan's best
            const uint32_t s = b.shift > kMinTileShift ? b.shift - 1 : b.shift + 1;
            if (b.persistent && b.model) cand.push_back({b.shift, b.grid_div, false, true, 2u, 1u});
            if (!b.persistent) cand.push_back({s > b.shift ? s + 1 : b.shift + 1, 1u, false, false, 2u, 1u});
            cand.push_back({s, 1u, false, false, 2u, 1u});
        } else if (phase == 2) {
            if (b.persistent) {
                cand.push_back({b.shift, b.grid_div, b.model, true, 1u, 1u});
                cand.push_back({b.shift, b.grid_div, b.model, true, 0u, 1u});
            }
        } else if (phase == 3) {
            if (b.persistent && model) {
                // (splitting by triangle counts may not have paid; by weighted
                // fragments it may)
                cand.push_back({b.shift, b.grid_div, true, true, 2u, 4u});
                cand.push_back({b.shift, b.grid_div, true, true, 1u, 16u});
            }
        } else if (phase == 4) {
            if (b.persistent)
                for (uint32_t s = kMinTileShift; s <= kMaxTileShift; ++s)
                    for (uint32_t d : {1u, 2u, 4u})
                        if (s != b.shift || d != b.grid_div)
                            cand.push_back({s, d, b.model, true, b.max_level, b.frag_scale});
        } else {
            // the three fastest twice more each (a near tie is decided by the
            // median of three runs, not by one run's noise)
            std::vector<size_t> order;
            for (size_t i = 0; i < cand.size(); ++i)
                if (ms[i] >= 0) order.push_back(i);
            std::sort(order.begin(), order.end(), [&](size_t x, size_t y) { return ms[x] < ms[y]; });
            for (size_t i : order) {
                const BatchConfig c = cand[i];
                const bool again = std::any_of(finals.begin(), finals.end(),
                                               [&](const std::vector<size_t> &f) { return cand[f[0]] == c; });
                if (again || finals.size() == 3) continue;
                finals.push_back({i, cand.size(), cand.size() + 1});
                cand.push_back(c);
                cand.push_back(c);
            }
        }
        ms.resize(cand.size(), -1.0f);
    }
    const int best = final_choice(*this);
    if (best >= 0) choice = cand[best];
    return false;
}

hipError_t Engine::advance_tuning(Op &op) {
    if (!autotune()) return hipSuccess;
    const bool model = cost_model_d_ != nullptr;
    if (!op.tuning) {
        op.tuning = std::make_shared<BatchTuning>();
        op.tuning->begin(op.tile_shift, model);
        op.tuning->choice = default_config(op);
        KZ_TRY(hipEventCreate(&op.tuning->ev[0]));
        KZ_TRY(hipEventCreate(&op.tuning->ev[1]));
    }
    BatchTuning &t = *op.tuning;
    if (t.done) return hipSuccess;
    if (t.pending >= 0) {  // the previous submission's trial
        KZ_TRY(hipEventSynchronize(t.ev[1]));
        float ms = -1.0f;
        if (hipEventElapsedTime(&ms, t.ev[0], t.ev[1]) == hipSuccess) t.ms[t.pending] = ms;
        t.pending = -1;
    }
    if (t.more(model, [&](uint32_t shift) { return op.variants->get(shift) != nullptr; })) return hipSuccess;
    t.done = true;
    if (t.trial) hipGraphExecDestroy(t.trial);
    t.trial = nullptr;
    last_tuned_ = t.choice;
    return hipSuccess;
}

// What a submission runs the batch with: the choice, the next trial, or (the
// recording's first submission, `tune` false) the untuned configuration, with
// the model if `model`.
void Engine::pick_config(Op &op, BatchConfig &cfg, bool &timed, bool tune, bool model) {
    cfg = default_config(op);
    timed = false;
    if (!autotune()) return;
    if (!tune) {
        cfg.model = model;
        return;
    }
    BatchTuning &t = *op.tuning;
    if (t.done) {
        cfg = t.choice;
    } else if (t.next < t.cand.size()) {
        cfg = t.cand[t.next];
        t.pending = (int)t.next++;
        timed = true;
    }
}

hipError_t Engine::execute(std::vector<Op> &ops, GraphCache *cache) {
    // Graphs pay off for command buffers that draw and are submitted again:
    // the first submission (and every tuning trial) runs eagerly. The first
    // is no trial: a command buffer recorded (or allocated) for every frame
    // would run the same one in all of them and never learn from it, and it
    // would load another tile size's kernels than the pipeline's creation did.
    bool graphable = cache != nullptr && graphs_ && !kernel_timing_;
    const bool first = cache && cache->eager_runs == 0;
    bool draws = false;
    for (Op &op : ops)
        if (op.kind == Op::Batch) {
            draws = true;
            if (!first) KZ_TRY(advance_tuning(op));
            if (autotune() && !(op.tuning && op.tuning->done)) graphable = false;
        }
    if (!graphable || !draws || first) {
        if (cache) ++cache->eager_runs;
        // (without the model in a recording for every frame: its statistics
        // and predictions cost more than its plan saves unless a trial has
        // shown otherwise)
        return execute_eager(ops, !first, !first || !cache->recorded_per_frame);
    }
    // every allocation before the capture
    for (Op &op : ops)
        if (op.kind == Op::Batch) {
            BatchConfig cfg;
            bool timed;
            pick_config(op, cfg, timed);
            if (!op.variants->get(cfg.shift)) return execute_eager(ops);
            KZ_TRY(prepare_batch(op, cfg.shift));
        }
    if (!cache->exec || cache->generation != generation_) {
        cache->reset();
        const uint32_t b0 = pending_batches_, l0 = pending_launches_;
        KZ_TRY(hipStreamBeginCapture(stream_, hipStreamCaptureModeRelaxed));
        const uint64_t gen = generation_;
        const hipError_t e = launch_ops(ops);
        hipGraph_t graph = nullptr;
        const hipError_t e2 = hipStreamEndCapture(stream_, &graph);
        cache->batches = pending_batches_ - b0;
        cache->launches = pending_launches_ - l0;
        pending_batches_ = b0;
        pending_launches_ = l0;
        if (e != hipSuccess || e2 != hipSuccess || gen != generation_) {
            if (graph) hipGraphDestroy(graph);
            if (e != hipSuccess) return e;
            if (e2 != hipSuccess) return e2;
            return execute_eager(ops);  // something was reallocated mid-capture
        }
        const hipError_t e3 = hipGraphInstantiate(&cache->exec, graph, nullptr, nullptr, 0);
        hipGraphDestroy(graph);
        if (e3 != hipSuccess) {
            cache->exec = nullptr;
            return e3;
        }
        cache->generation = generation_;
        ++graph_captures_;
    }
    KZ_TRY(hipGraphLaunch(cache->exec, stream_));
    pending_batches_ += cache->batches;
    pending_launches_ += cache->launches;
    ++graph_launches_;
    return hipSuccess;
}

// A first launch of the one-workgroup-per-tile raster, on one tile without
// triangles: the planned rasters of a tile size have theirs behind them in
// the trials before, it would have its only one timed.
hipError_t Engine::warm_raster(const PipelineKernels *kern) {
    KzFrame f{};
    f.tiles_x = f.tiles_y = 1;
    f.tile_counts = f.tile_offsets = zero_word_;
    f.list_capacity = 1;
    void *args[] = {&f};
    return hipModuleLaunchKernel(kern->raster, 1, 1, 1, 64, 1, 1, 0, stream_, args, nullptr);
}

// The batch as a timed trial, as a graph of its own where the choice will run
// in one: a kernel of a replayed graph takes at least 4.5 us, launched by
// itself half of that, so that trials of single launches favour plans of ten
// small kernels. The device waits first until the host has queued the rest.
// (With the plain raster tried at smaller tiles too, 131,072 Phong triangles
// at 720p and four samples 167 us a frame -> 130.)
hipError_t Engine::run_trial(const Op &op, const BatchConfig &cfg) {
    BatchTuning &t = *op.tuning;
    if (t.trial) hipGraphExecDestroy(t.trial);  // (the trial before has ended: its events were read)
    t.trial = nullptr;
    if (graphs_ && !kernel_timing_) {
        const uint32_t b0 = pending_batches_, l0 = pending_launches_;
        const uint64_t gen = generation_;
        hipGraph_t captured = nullptr;
        KZ_TRY(hipStreamBeginCapture(stream_, hipStreamCaptureModeRelaxed));
        const hipError_t e = run_batch(op, cfg);
        const hipError_t e2 = hipStreamEndCapture(stream_, &captured);
        if (e != hipSuccess || e2 != hipSuccess || gen != generation_ ||
            hipGraphInstantiate(&t.trial, captured, nullptr, nullptr, 0) != hipSuccess)
            t.trial = nullptr;
        else if (hipGraphUpload(t.trial, stream_) != hipSuccess) {
            hipGraphExecDestroy(t.trial);
            t.trial = nullptr;
        }
        if (captured) hipGraphDestroy(captured);
        if (!t.trial) {  // launched by itself instead
            pending_batches_ = b0;
            pending_launches_ = l0;
            if (e != hipSuccess) return e;
        }
    }
    KZ_TRY(kz_launch_wait(stream_));
    KZ_TRY(hipEventRecord(t.ev[0], stream_));
    KZ_TRY(t.trial ? hipGraphLaunch(t.trial, stream_) : run_batch(op, cfg));
    return hipEventRecord(t.ev[1], stream_);
}

hipError_t Engine::execute_eager(std::vector<Op> &ops, bool tune, bool model) {
    for (Op &op : ops)
        if (op.kind == Op::Batch) {
            BatchConfig cfg;
            bool timed;
            pick_config(op, cfg, timed, tune, model);
            if (timed) {
                // a trial times the batch, not the loading of a tile size's
                // kernels or the growth of its scratch (host work and syncs)
                if (const PipelineKernels *kern = op.variants->get(cfg.shift)) {
                    KZ_TRY(prepare_batch(op, cfg.shift));
                    if (!cfg.persistent) KZ_TRY(warm_raster(kern));
                }
                KZ_TRY(run_trial(op, cfg));
            } else {
                KZ_TRY(run_batch(op, cfg));
            }
        } else {
            KZ_TRY(launch_ops_one(op));
        }
    return hipSuccess;
}

hipError_t Engine::launch_ops(std::vector<Op> &ops) {
    for (Op &op : ops) {
        if (op.kind == Op::Batch) {
            const BatchTuning *t = op.tuning.get();
            KZ_TRY(run_batch(op, t && t->done ? t->choice : default_config(op)));
        } else {
            KZ_TRY(launch_ops_one(op));
        }
    }
    return hipSuccess;
}

hipError_t Engine::launch_ops_one(const Op &op) {
    {
        switch (op.kind) {
        case Op::Fill:
            KZ_TRY(kz_launch_fill_rect_u32(stream_, op.fill_ptr, op.fill_width, op.x0, op.y0, op.w, op.h, op.fill_spp,
                                           op.fill_value));
            ++pending_launches_;
            break;
        case Op::Batch: break;
        case Op::Copy:
            if (op.bytes) KZ_TRY(hipMemcpyAsync(op.dst, op.src, op.bytes, hipMemcpyDefault, stream_));
            break;
        case Op::Copy2D:
            if (op.rows && op.row_bytes)
                KZ_TRY(hipMemcpy2DAsync(op.dst, op.dst_pitch, op.src, op.src_pitch, op.row_bytes, op.rows,
                                        hipMemcpyDefault, stream_));
            break;
        case Op::Resolve:
            KZ_TRY(kz_launch_resolve4(stream_, op.rsrc, op.rdst, op.rwidth, op.x0, op.y0, op.w, op.h));
            ++pending_launches_;
            break;
        case Op::Dispatch: {
            size_t size = sizeof op.cframe;
            void *config[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, const_cast<KzComputeFrame *>(&op.cframe),
                              HIP_LAUNCH_PARAM_BUFFER_SIZE, &size, HIP_LAUNCH_PARAM_END};
            KZ_TRY(hipModuleLaunchKernel(op.cs_kernel, op.groups[0], op.groups[1], op.groups[2], op.block[0],
                                         op.block[1], op.block[2], 0, stream_, nullptr, config));
            ++pending_launches_;
            break;
        }
        }
    }
    return hipSuccess;
}

hipError_t Engine::end_submit(hipEvent_t fence_event) {
    ++submissions_;
    KZ_TRY(hipEventRecord(ev_end_, stream_));
    if (fence_event) KZ_TRY(hipEventRecord(fence_event, stream_));
    return hipSuccess;
}

bool Engine::outgrown() const {
    const volatile uint32_t *need = need_h_;
    return need[KZ_NEED_PAIRS] || need[KZ_NEED_SPLIT];
}

void Engine::collect_stats() {
    if (!submit_open_) return;
    // the striped counters are folded and read once per wait, not once per
    // submission (they accumulate over the submissions in between)
    if (kz_launch_stats_reduce(stream_, stats_d_) != hipSuccess ||
        hipMemcpyAsync(stats_h_, stats_d_ + (size_t)KZ_STAT_STRIPES * KZ_STAT_COUNT,
                       KZ_STAT_COUNT * sizeof(unsigned long long), hipMemcpyDeviceToHost, stream_) != hipSuccess)
        std::memset(stats_h_, 0, KZ_STAT_COUNT * sizeof(unsigned long long));
    hipEventSynchronize(ev_end_);
    hipStreamSynchronize(stream_);
    std::memcpy(last_.counters, stats_h_, sizeof(last_.counters));
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, ev_start_, ev_end_) == hipSuccess) last_.gpu_ms = ms;
    last_.batches = pending_batches_;
    last_.launches = pending_launches_;
    for (int k = 0; k < KS_COUNT; ++k) {
        last_.kernel_ms[k] = 0.0f;
        last_.kernel_launches[k] = 0;
    }
    for (size_t i = 0; i + 1 < timing_events_.size(); i += 2) {
        const int slot = timing_events_[i].first;
        float kms = 0.0f;
        if (hipEventElapsedTime(&kms, timing_events_[i].second, timing_events_[i + 1].second) == hipSuccess) {
            last_.kernel_ms[slot] += kms;
            last_.kernel_launches[slot] += 1;
        }
    }
    timing_events_.clear();
    events_used_ = 0;
    submit_open_ = false;
    // A batch whose lists overflowed rendered correctly through the in-order
    // scan fallback; size the lists for the largest such batch (the counters
    // hold the pairs of every batch since the last collection).
    const uint32_t pairs = need_h_[KZ_NEED_PAIRS];
    const bool split = need_h_[KZ_NEED_SPLIT] != 0;
    std::memset(need_h_, 0, KZ_NEED_WORDS * sizeof(uint32_t));
    if (pairs) {
        uint64_t need = (uint64_t)pairs + pairs / 4;
        if (list_limit_) need = std::min<uint64_t>(need, list_limit_);
        if (need > list_capacity_ && need < 0xFFFFFFF0ull) {
            hipStreamSynchronize(stream_);
            if (alloc_lists(need) != hipSuccess) list_capacity_ = 0, cap_tris_ = 0;  // next ensure_scratch reallocates
        }
    }
    // Likewise for sub-tile lists (their overflow fallback filters the
    // parent tile's list): the device keeps the largest batch total.
    if (ctrl_ && split) {
        uint32_t mx = 0;
        if (hipMemcpy(&mx, ctrl_ + KZ_CTRL_SPLIT_MAX, sizeof mx, hipMemcpyDeviceToHost) == hipSuccess &&
            mx > split_capacity_) {
            const uint64_t need = std::min<uint64_t>((uint64_t)mx + mx / 4, 0xFFFFFFF0ull);
            if (regrow(split_lists_, need) == hipSuccess)
                split_capacity_ = (uint32_t)need;
            else
                split_capacity_ = 0;  // next ensure_split_scratch reallocates
        }
    }
}

}  // namespace kz
