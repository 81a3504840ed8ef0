/*
 * esth_filter.hip - one island-model filter on one GPU: set-up and the step
 * of particle_filter() (src/partfilt/opencl/pf_generic.c:245-887) as a
 * sequence of kernels on the filter's stream, with no host synchronisation
 * inside a step (the reference blocks three times per step: pf_generic.c:231,
 * 614, 806).
 */
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "esth_internal.h"
#include "esth_dispatch.h"

/* MTGP32 words, three ways.  Where the step's sampling launch has 256-thread
 * work-groups (the fused sample+sort at m >= 512, or sample+weight alone) and
 * lasts longer than they need, the next step's words are generated by 96
 * extra work-groups of that launch (inline).  Where the step's launches
 * together last that long (the resampling has 256-thread work-groups but for
 * the alias at m = 1024), each of them carries a share of the next step's words
 * (carried).  Neither
 * needs a second stream or an event, whose waits cost the main stream 10 us
 * at every block of steps.  Otherwise a block of steps' words is generated
 * per launch on a second stream, one block ahead: ESTH_RNG_BLOCK_LONG steps,
 * or fewer where two blocks would pass ESTH_RNG_BLOCK_CACHED, but not fewer
 * than ESTH_RNG_BLOCK_DEFAULT (nor two blocks above ESTH_RNG_BLOCK_BYTES).
 * Whole runs with blocks of 2, 3 and 4 steps: randomwalk3 128 x 3001 (two
 * blocks of 4: 49 MB) 2.27, -, 2.03 ms; unicycle with 4 landmarks 512 x 2048
 * (134 MB) 9.13, 9.05, 8.93 ms; dh6 512 x 2048 (235 MB) 18.56, 18.21, 18.46;
 * unicycle 512 x 4096 (268 MB) 14.54, 14.33, 14.93: the words of two blocks
 * have to lie in the 256 MB Infinity Cache with what the step's launches
 * read.  Blocks of 8 gain 1-3 % more at 128 x 3001 for twice the memory. */
#define ESTH_RNG_BLOCK 8
#define ESTH_RNG_BLOCK_DEFAULT 2
#define ESTH_RNG_BLOCK_LONG 4
#define ESTH_RNG_BLOCK_CACHED (200ull << 20)
#define ESTH_RNG_BLOCK_BYTES (1ull << 30)
/* graph replay: one captured graph and one device frame slot per step of the
 * two word blocks */
#define ESTH_FRAME_RING (2 * ESTH_RNG_BLOCK)
#define ESTH_TIMING_STEPS 4096
#define ESTH_POLL_US 1000   /* a wait for an estimate polls this long */

struct esth_filter {
    esth_engine* e = nullptr;
    esth_filter_desc d{};
    int S = 0, V = 0, K = 0;
    uint32_t m = 0, G = 0, t = 0;
    size_t N = 0;
    uint64_t needed = 0, size = 0, words = 0;
    int dimx = 0, dimy = 0;
    unsigned char params[esth_max_model_params()];
    hipStream_t stream = nullptr;
    hipStream_t rng_stream = nullptr;   /* MTGP of the next step runs here, overlapped */
    /* device */
    float *state = nullptr, *tmp = nullptr, *w = nullptr, *bt_w = nullptr, *bt_s = nullptr,
          *part = nullptr, *frames = nullptr;
    /* random words in blocks of B steps: block b (steps bB .. bB + B - 1)
     * lives in R[b & 1], step bB + kk at R[b & 1] + kk words.  Its statuses
     * are slots of sring: slot (p, kk) = sring + (p (B + 1) + kk) K 351;
     * slot (b & 1, kk) is the status that generates step bB + kk, and the
     * block's last status, slot (b & 1, B), starts block b + 1 (the seed
     * sits in slot (1, B), the end of "block -1"). */
    int B = 1;
    float* R[2] = {nullptr, nullptr};
    uint32_t* sring = nullptr;
    int64_t ready_block = -1;           /* block whose words the RNG stream has been asked for */
    int64_t rest_block = -1;            /* block whose last words alone it has been asked for */
    uint64_t main_upto = 0;             /* the main stream has waited for or generated the words of steps below this */
    int64_t inline_block = -1;          /* block generated by the previous step's launch (B = 1) */
    bool inline_rng = false;            /* this filter generates its next step's words inline */
    bool carried = false;               /* ... in shares of all the step's launches (words kept in the same blocks) */
    uint64_t words_upto = 0;            /* carried: steps below this have their words */
    int words_room = 0;                 /* room that the fused launch leaves the second stream's words */
    bool prefetch = true;
    bool fuse_sample_sort = false;      /* sample+weight and sort in one launch (k_sample_sort) */
    hipEvent_t ev_rng_done[2], ev_consumed[2], ev_fork;
    bool consumed[2] = {};   /* ev_consumed recorded after that parity's last block */
    float2 *winner = nullptr, *result = nullptr;
    /* the posterior sums and best particle: pinned host memory that the argmax
     * writes across the bus (4 + 2 S doubles), so that reading an estimate is
     * a wait and no copy (a step and its estimate at 4096 particles 48 -> 32
     * us), and the wait is for the count of argmaxes that follows them, not
     * for the launch's resampling or the stream (4096 particles 29.6 -> 24.6
     * us, 256,000 with the alias resampler 52.6 -> 40.9, 2M 136 -> 128) */
    double* est = nullptr;
    uint64_t argmaxes = 0;   /* launches with an argmax enqueued so far */
    bool recount = false;    /* ... give or take one that failed and may have run */
    /* the cross-step launch (k_step_x): step n's resampling runs at the start
     * of step n + 1's launch.  Sorted-side buffers alternate by step parity
     * (winner/part/bt_w/bt_s for even steps, *2 for odd ones) and the words
     * rotate over three buffers (R[0], R[1], R3: step n's are R[n % 3]) */
    bool xstep = false;                 /* this filter takes the cross-step launch */
    bool xstep_on = true;               /* ... unless switched off */
    bool pending = false;               /* step steps - 1 is sorted, its resampling not yet run */
    float* R3 = nullptr;
    float2* winner2 = nullptr;
    float *part2 = nullptr, *bt_w2 = nullptr, *bt_s2 = nullptr;
    uint32_t* top = nullptr;
    esth_mtgp_stream* streams = nullptr;
    std::vector<std::pair<void*, size_t>> allocs;
    /* host */
    float* h_frames = nullptr;   /* pinned ring */
    hipEvent_t frame_ev[ESTH_FRAME_RING];   /* graph replay: the host slot's copy has run */
    bool frame_used[ESTH_FRAME_RING] = {};
    hipEvent_t ev[7];
    int timing = 0;   /* 0 off, 1 sample+weight only, 2 every stage */
    int timing_every = 1;   /* time one step in this many */
    uint64_t tcount = 0;
    /* per-step stage events while timing is on: 7 per step, up to ESTH_TIMING_STEPS steps */
    std::vector<hipEvent_t> tev;
    int tsteps = 0;
    uint64_t steps = 0;
    /* graph replay */
    bool use_graph = false;
    hipGraphExec_t gexec[ESTH_FRAME_RING] = {};
    bool gexec_inline[ESTH_FRAME_RING] = {};   /* the graph carries the next step's MTGP32 work-groups */
    int gexec_mode[ESTH_FRAME_RING] = {};      /* what the graph holds: ESTH_GRAPH_* */
};

/* status slot (p, kk) of the word blocks */
static uint32_t* status_slot(esth_filter* f, int p, int kk) {
    return f->sring + ((size_t)p * (size_t)(f->B + 1) + (size_t)kk) * (size_t)f->K * ESTH_MTGP_N;
}

/* How long the step's launches last by themselves (us), in stream order, for
 * the choice of where its words are made: a launch's latency, the sampling's
 * and the sort's VALU lane-instructions per particle at the rate they sustain,
 * the resampling's bytes, and the alias resampling's chain of pairings.
 * Figures of the models in the list, measured on MI355X; a model without one
 * counts as the lightest, whose launches hide the least. */
enum { ESTH_CARRY_SAMPLE, ESTH_CARRY_SORT, ESTH_CARRY_RESAMPLE, ESTH_CARRIERS };
static double sampling_us(const esth_filter* f) {
    double insts = 130.0;   /* the random walk */
    switch (f->d.model) {
    case ESTH_MODEL_UNICYCLE: insts = 200.0 + 47.0 * ((const esth_unicycle_params*)f->params)->num_landmarks; break;
    case ESTH_MODEL_UNICYCLE10: insts = 300.0; break;
    case ESTH_MODEL_ROBOTARM5:
    case ESTH_MODEL_ROBOTARM5_CAMERA:
    case ESTH_MODEL_DH6: insts = 800.0; break;
    default: break;
    }
    return (double)f->N * insts / 5.1e7;
}
static void launches(const esth_filter* f, bool fused_launch, double us[ESTH_CARRIERS]) {
    const double n = (double)f->N, launch = 6.0, sort = n * 340.0 / 5.1e7;
    us[ESTH_CARRY_SAMPLE] = launch + sampling_us(f) + (fused_launch ? sort : 0.0);
    us[ESTH_CARRY_SORT] = fused_launch ? 0.0 : launch + sort;
    us[ESTH_CARRY_RESAMPLE] = (launch + n * 8.0 * (f->S + 1) / 4.0e6) * (f->d.resampler == ESTH_RESAMPLE_ALIAS ? 1.4 : 1.0);
}
/* the same of those that can carry MTGP32 work-groups, 0 for the others */
static void carriers(const esth_filter* f, bool fused_launch, double us[ESTH_CARRIERS]) {
    launches(f, fused_launch, us);
    if (fused_launch && !esth_sample_sort_inline_rng(f->m)) us[ESTH_CARRY_SAMPLE] = 0.0;
    if (!esth_sort_carries_rng(f->m)) us[ESTH_CARRY_SORT] = 0.0;
    if (!esth_resample_carries_rng(f->d.resampler, f->m)) us[ESTH_CARRY_RESAMPLE] = 0.0;
}
/* A step's words, 768-word rounds of every stream side by side: 0.5 us a round
 * alone, 0.65 to 0.8 in work-groups beside a launch's own work */
static double rounds(const esth_filter* f) { return (double)(f->size / ESTH_MTGP_LARGE); }
static double mtgp_us(const esth_filter* f) { return 1.0 + 0.75 * rounds(f); }

/* The unicycle's sampling launch carries all of the next step's words (inline)
 * where its sampling alone lasts 0.585 us a round, the sort in the same launch
 * covering the rest: from 31 landmarks on (40 with the alias).  Around that
 * line the three ways are within 4 % of each other (26 to 48 landmarks, m = 64,
 * 512 and 1024, with and without the alias), but inline words bring the
 * cross-step launch where it applies: 512 x 4096 with 32 landmarks 95 us a step
 * inline, 101 carried, 102 by the second stream; 512 x 1024 32, 40 and 41.
 * With few landmarks and many particles they are the slower ones all the same
 * (512 x 4096 with 8: 71 and 69 us). */
static bool inline_rng_pays(const esth_filter* f) {
    return f->d.model == ESTH_MODEL_UNICYCLE && sampling_us(f) >= 0.585 * rounds(f);
}

/* Carried words cost what the generator's work-groups outlast their launches
 * by, the second stream's an event and a wait at each block of steps: carried
 * up to 4 us of the former.  Measured on 300 filters of five models, carried
 * against the second stream in blocks of 4, per step and, in brackets, with the
 * estimate read after each step, where the host's turn hides words that lie in
 * the launches but not a wait: randomwalk3 128 x 128 11.7 and 16.8 us, unicycle
 * 512 x 256 18.7 and 19.2, 512 x 512 23.1 and 22.5, 512 x 1024 32.4 and 28.3
 * (33.8 and 37.4), 512 x 2048 with 13 landmarks 50.5 and 47.6 (53.2 and 56.8),
 * randomwalk3 512 x 1024 30.9 and 25.9 (31.6 and 35.5); beyond the line 256 x
 * 1024 25.5 and 21.4, robotarm5 512 x 512 39.2 and 34.6, 256 x 1024 44.3 and
 * 30.0.  The line lies between the two uses. */
static bool carried_rng_pays(const esth_filter* f) {
    double us[ESTH_CARRIERS];
    carriers(f, f->fuse_sample_sort, us);
    return us[ESTH_CARRY_RESAMPLE] > 0.0 &&
           mtgp_us(f) <= us[ESTH_CARRY_SAMPLE] + us[ESTH_CARRY_SORT] + us[ESTH_CARRY_RESAMPLE] + 4.0;
}

/* Where the second stream's words (0.5 us a round by themselves) outlast the
 * step's launches, they bound the step, and the fused launch of models of many
 * dimensions leaves them room (esth_engine.hip, room_lds): some where they last
 * 1.15 times as long, more from 1.33 on, where the launches have the time.  Per
 * step, and in brackets with the estimate read after each, where the launches'
 * own time counts too; without, with some, with more room: robotarm5 256 x 4096
 * (1.28) 82.7 (79.2), 77.7 (81.8), 75.3 us (84.6); 512 x 2048 80.6 (71.6), 76.8
 * (73.0), 73.7 (78.8); 256 x 6144 (1.37) 122 (112), 115 (110), 110 (109); 512 x
 * 4096 (1.42) 157 (149), 152 (151), 147 (144).  Below 1.15 the launches bound
 * the step and only lose by it (256 x 2048, more room: 42 -> 46), as do those
 * of three dimensions, short of waves then, at any size (randomwalk3 512 x 4096
 * 62 -> 69, unicycle 512 x 8192 118 -> 148). */
static int words_room(const esth_filter* f) {
    if (f->inline_rng || f->carried || f->S < 9) return 0;
    double us[ESTH_CARRIERS];
    launches(f, true, us);
    const double ratio = (1.0 + 0.5 * rounds(f)) / (us[ESTH_CARRY_SAMPLE] + us[ESTH_CARRY_RESAMPLE]);
    return ratio >= 1.33 ? 2 : ratio >= 1.15 ? 1 : 0;
}

/* words of each stream that each launch generates: all in the resampling
 * where it lasts that long, else in proportion to what the launches last */
static void carried_shares(const esth_filter* f, bool fused_launch, uint32_t words[ESTH_CARRIERS]) {
    double us[ESTH_CARRIERS];
    carriers(f, fused_launch, us);
    if (mtgp_us(f) <= us[ESTH_CARRY_RESAMPLE]) us[ESTH_CARRY_SAMPLE] = us[ESTH_CARRY_SORT] = 0.0;
    const double sum = us[ESTH_CARRY_SAMPLE] + us[ESTH_CARRY_SORT] + us[ESTH_CARRY_RESAMPLE];
    const uint32_t rounds = (uint32_t)(f->size / ESTH_MTGP_LARGE);
    uint32_t left = rounds;
    for (int i = 0; i < ESTH_CARRY_RESAMPLE; ++i) {
        const uint32_t r = std::min(left, (uint32_t)(rounds * us[i] / sum + 0.5));
        words[i] = r * ESTH_MTGP_LARGE;
        left -= r;
    }
    words[ESTH_CARRY_RESAMPLE] = left * ESTH_MTGP_LARGE;
}

static int falloc(esth_filter* f, size_t bytes, void** p) {
    ESTH_TRY(esth_engine_alloc(f->e, bytes, p));
    f->allocs.push_back({*p, bytes});
    return ESTH_OK;
}

static void filter_free(esth_filter* f) {
    if (!f) return;
    hipSetDevice(f->e->device);
    if (f->stream) hipStreamSynchronize(f->stream);
    if (f->rng_stream) hipStreamSynchronize(f->rng_stream);   /* the next block may still be written */
    for (int i = 0; i < ESTH_FRAME_RING; ++i)
        if (f->gexec[i]) hipGraphExecDestroy(f->gexec[i]);
    for (auto& a : f->allocs) esth_engine_release(f->e, a.first, a.second);
    f->allocs.clear();
    if (f->h_frames) hipHostFree(f->h_frames);
    if (f->est) hipHostFree(f->est);
    for (int i = 0; i < ESTH_FRAME_RING; ++i) hipEventDestroy(f->frame_ev[i]);
    for (int i = 0; i < 7; ++i) hipEventDestroy(f->ev[i]);
    for (int i = 0; i < 2; ++i) { hipEventDestroy(f->ev_rng_done[i]); hipEventDestroy(f->ev_consumed[i]); }
    hipEventDestroy(f->ev_fork);
    if (f->rng_stream) hipStreamDestroy(f->rng_stream);
    for (auto ev : f->tev) hipEventDestroy(ev);
    if (f->stream) hipStreamDestroy(f->stream);
    delete f;
}

extern "C" int esth_filter_create(esth_engine* e, const esth_filter_desc* d, const void* params, size_t params_size,
                                  esth_filter** out) {
    if (!e || !out) return esth_fail(ESTH_ERR_INVALID, "null engine/out");
    int S, V;
    ESTH_TRY(esth_check_desc(d, &S, &V));
    size_t need = 0;
    ESTH_TRY(esth_params_size(d->model, &need));
    if (need && (!params || params_size != need))
        return esth_fail(ESTH_ERR_INVALID, "model %d needs %zu bytes of params, got %zu", d->model, need, params_size);
    ESTH_HIP(hipSetDevice(e->device));
    esth_filter* f = new esth_filter();
    f->e = e;
    f->d = *d;
    f->S = S;
    f->V = V;
    f->m = d->num_particles;
    f->G = d->num_blocks;
    f->t = (d->topology == ESTH_TOPO_NONE) ? 0 : d->num_transfer;
    f->N = (size_t)f->m * f->G;
    f->fuse_sample_sort = esth_sample_sort_pays(d->model, d->state_layout, f->m);
    memset(f->params, 0, sizeof(f->params));
    if (need) memcpy(f->params, params, need);
    f->needed = esth_rng_needed(V, d->resampler, d->adaptive, f->m, f->G);
    f->K = esth_rng_streams(d->rng, f->needed);
    f->size = esth_rng_stream_size(f->K, f->needed);
    f->words = f->size * (uint64_t)f->K;
    f->dimx = d->torus_dimx;
    f->dimy = d->torus_dimy;
    if (d->topology == ESTH_TOPO_TORUS && (f->dimx <= 0 || f->dimy <= 0)) esth_torus_dims(f->G, &f->dimx, &f->dimy);
    for (int i = 0; i < ESTH_FRAME_RING; ++i) hipEventCreateWithFlags(&f->frame_ev[i], hipEventDisableTiming);
    /* ESTH_RNG_BLOCK_STEPS (1..ESTH_RNG_BLOCK): the second stream in blocks of that length (1: inline words stay) */
    f->inline_rng = (!f->fuse_sample_sort || esth_sample_sort_inline_rng(f->m)) && inline_rng_pays(f);
    uint64_t blk = 0;
    if (const char* ev = getenv("ESTH_RNG_BLOCK_STEPS")) {
        const long v = strtol(ev, nullptr, 10);
        if (v >= 1 && v <= ESTH_RNG_BLOCK) blk = (uint64_t)v;
    }
    f->carried = !f->inline_rng && blk == 0 && carried_rng_pays(f);
    f->words_room = words_room(f);
    const uint64_t two = 2ull * sizeof(float) * f->words;   /* two blocks of one step */
    if (blk == 0)
        blk = f->inline_rng ? 1
              : f->carried  ? ESTH_RNG_BLOCK_DEFAULT
                            : std::min<uint64_t>(ESTH_RNG_BLOCK_LONG,
                                                 std::max<uint64_t>(ESTH_RNG_BLOCK_DEFAULT, ESTH_RNG_BLOCK_CACHED / two));
    f->B = (int)std::max<uint64_t>(1, std::min<uint64_t>(blk, ESTH_RNG_BLOCK_BYTES / two));
    f->xstep = f->inline_rng && f->B == 1 && f->fuse_sample_sort && f->m == 512 && d->model == ESTH_MODEL_UNICYCLE &&
               d->resampler != ESTH_RESAMPLE_ALIAS && f->t > 0 &&
               (d->topology == ESTH_TOPO_RING || d->topology == ESTH_TOPO_TORUS) && !d->carry_weights &&
               d->state_layout == ESTH_LAYOUT_SOA;
    for (int i = 0; i < 7; ++i) hipEventCreate(&f->ev[i]);
    /* These order launches of one device.  Without the system fence an event
     * does not make memory visible to the host and to other devices (neither
     * reads the words or statuses); launches of this device see what those
     * before them wrote by their own release and acquire, as on one stream.
     * With the fence, whole runs of 200 steps with two events per block of 2:
     * 4 landmarks, 2M particles 14.83 -> 14.54 ms, dh6 18.77 -> 18.52; with a
     * device-scope release in its place (hipEventReleaseToDevice) steps are 1
     * to 4 % longer (randomwalk3 128 x 3001 24.2 and 24.8 us, unicycle 512 x
     * 2048 38.1 and 39.6). */
    for (int i = 0; i < 2; ++i) {
        hipEventCreateWithFlags(&f->ev_rng_done[i], hipEventDisableTiming | hipEventDisableSystemFence);
        hipEventCreateWithFlags(&f->ev_consumed[i], hipEventDisableTiming | hipEventDisableSystemFence);
    }
    hipEventCreateWithFlags(&f->ev_fork, hipEventDisableTiming | hipEventDisableSystemFence);
    int rc = ESTH_OK;
    const size_t SN = (size_t)S * f->N;
    const size_t tG = (size_t)(f->t ? f->t : 1) * f->G;
#define FA(ptr, bytes) if (rc == ESTH_OK) rc = falloc(f, (bytes), (void**)&(ptr))
    FA(f->state, sizeof(float) * SN);
    FA(f->tmp, sizeof(float) * SN);
    FA(f->w, sizeof(float) * f->N);
    FA(f->R[0], sizeof(float) * f->words * (size_t)f->B);
    FA(f->R[1], sizeof(float) * f->words * (size_t)f->B);
    FA(f->bt_w, sizeof(float) * tG);
    FA(f->bt_s, sizeof(float) * tG * S);
    FA(f->part, sizeof(float) * (size_t)f->G * (2 + S));
    FA(f->frames, sizeof(float) * ESTH_FRAME_FLOATS * ESTH_FRAME_RING);
    FA(f->winner, sizeof(float2) * f->G);
    FA(f->result, sizeof(float2) + sizeof(uint64_t));   /* and the argmaxes' count */
    FA(f->sring, sizeof(uint32_t) * ESTH_MTGP_N * (size_t)f->K * (2 * (size_t)(f->B + 1) + ESTH_CARRIERS - 1));
    FA(f->top, sizeof(uint32_t) * 64);

    FA(f->streams, sizeof(esth_mtgp_stream) * (size_t)f->K);
    if (f->xstep) {
        FA(f->R3, sizeof(float) * f->words);
        FA(f->winner2, sizeof(float2) * f->G);
        FA(f->part2, sizeof(float) * (size_t)f->G * (2 + S));
        FA(f->bt_w2, sizeof(float) * tG);
        FA(f->bt_s2, sizeof(float) * tG * S);
    }
#undef FA
    if (rc != ESTH_OK) { filter_free(f); return rc; }
    hipError_t err = hipStreamCreateWithFlags(&f->stream, hipStreamNonBlocking);
    if (err == hipSuccess) err = hipStreamCreateWithFlags(&f->rng_stream, hipStreamNonBlocking);
    if (err == hipSuccess) err = hipHostMalloc((void**)&f->h_frames, sizeof(float) * ESTH_FRAME_FLOATS * ESTH_FRAME_RING, 0);
    const size_t est_bytes = sizeof(double) * ESTH_EST_DOUBLES;
    if (err == hipSuccess) err = hipHostMalloc((void**)&f->est, est_bytes, hipHostMallocMapped | hipHostMallocCoherent);
    if (err != hipSuccess) { filter_free(f); return esth_fail(ESTH_ERR_DEVICE, "stream/pinned: %s", hipGetErrorString(err)); }
    memset(f->est, 0, est_bytes);
    /* RNG status: make_kernel_data32 (mtgp32-opencl.c:31-60), stream j seeded seed + j + 1 */
    std::vector<uint32_t> st((size_t)ESTH_MTGP_N * f->K);
    std::vector<esth_mtgp_stream> sd(f->K);
    for (int j = 0; j < f->K; ++j) {
        esth_mtgp_seed_state(j, d->seed + (uint32_t)j + 1u, st.data() + (size_t)j * ESTH_MTGP_N);
        sd[j] = {(uint32_t)j, (uint32_t)f->size, (uint64_t)j * f->size, (uint64_t)j};
    }
    err = hipMemcpy(status_slot(f, 1, f->B), st.data(), st.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (err == hipSuccess) err = hipMemcpy(f->streams, sd.data(), sd.size() * sizeof(esth_mtgp_stream), hipMemcpyHostToDevice);
    if (err == hipSuccess) err = hipMemset(f->w, 0, sizeof(float) * f->N);
    /* the argmaxes' count: there when the copy returns, as the rest; a wait for
     * the device would stop at what other filters have queued */
    const unsigned char none[sizeof(float2) + sizeof(uint64_t)] = {};
    if (err == hipSuccess) err = hipMemcpy(f->result, none, sizeof(none), hipMemcpyHostToDevice);
    if (err != hipSuccess) { filter_free(f); return esth_fail(ESTH_ERR_DEVICE, "init upload: %s", hipGetErrorString(err)); }
    *out = f;
    return ESTH_OK;
}

extern "C" int esth_filter_destroy(esth_filter* f) {
    filter_free(f);
    return ESTH_OK;
}

extern "C" int esth_filter_init_uniform(esth_filter* f, const float* s) {
    if (!f || !s) return esth_fail(ESTH_ERR_INVALID, "null filter/state");
    std::vector<float> h((size_t)f->S * f->N);
    for (int c = 0; c < f->S; ++c) std::fill(h.begin() + (size_t)c * f->N, h.begin() + (size_t)(c + 1) * f->N, s[c]);
    return esth_filter_init(f, h.data());
}

/* the device state from / to host SOA planes, through the filter's layout */
static int upload_state(esth_filter* f, const float* soa) {
    const size_t n = (size_t)f->S * f->N;
    if (f->d.state_layout == ESTH_LAYOUT_SOA) {
        ESTH_HIP(hipMemcpy(f->state, soa, sizeof(float) * n, hipMemcpyHostToDevice));
        return ESTH_OK;
    }
    std::vector<float> h(n);
    ESTH_TRY(esth_state_convert(f->S, f->N, ESTH_LAYOUT_SOA, soa, f->d.state_layout, h.data()));
    ESTH_HIP(hipMemcpy(f->state, h.data(), sizeof(float) * n, hipMemcpyHostToDevice));
    return ESTH_OK;
}

static int download_state(esth_filter* f, float* soa) {
    const size_t n = (size_t)f->S * f->N;
    if (f->d.state_layout == ESTH_LAYOUT_SOA) {
        ESTH_HIP(hipMemcpy(soa, f->state, sizeof(float) * n, hipMemcpyDeviceToHost));
        return ESTH_OK;
    }
    std::vector<float> h(n);
    ESTH_HIP(hipMemcpy(h.data(), f->state, sizeof(float) * n, hipMemcpyDeviceToHost));
    return esth_state_convert(f->S, f->N, f->d.state_layout, h.data(), ESTH_LAYOUT_SOA, soa);
}

extern "C" int esth_filter_init(esth_filter* f, const float* soa) {
    if (!f || !soa) return esth_fail(ESTH_ERR_INVALID, "null filter/state");
    ESTH_HIP(hipSetDevice(f->e->device));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_TRY(upload_state(f, soa));
    f->pending = false;   /* a pending resampling would overwrite the new particles */
    if (f->d.carry_weights) {   /* a new particle set starts from equal weights */
        std::vector<float> w0(f->N, f->d.weights == ESTH_WEIGHTS_LOG ? 0.0f : 1.0f);
        ESTH_HIP(hipMemcpy(f->w, w0.data(), sizeof(float) * f->N, hipMemcpyHostToDevice));
    }
    return ESTH_OK;
}

/* the words of step n */
static float* step_words(esth_filter* f, uint64_t n) {
    if (f->xstep) {
        const uint64_t r = n % 3;
        return r == 0 ? f->R[0] : (r == 1 ? f->R[1] : f->R3);
    }
    return f->R[(n / f->B) & 1] + (size_t)(n % f->B) * f->words;
}

/* the sorted-side buffers of step n */
struct esth_xset {
    float2* winner;
    float *part, *bt_w, *bt_s;
};
static esth_xset xset(esth_filter* f, uint64_t n) {
    if (f->xstep && (n & 1)) return {f->winner2, f->part2, f->bt_w2, f->bt_s2};
    return {f->winner, f->part, f->bt_w, f->bt_s};
}

/* the status that generates step n */
static uint32_t* status_at(esth_filter* f, uint64_t n) {
    const uint64_t b = n / f->B, kk = n % f->B;
    return kk ? status_slot(f, (int)(b & 1), (int)kk) : status_slot(f, (int)((b + 1) & 1), f->B);
}

/* MTGP words of steps n .. n + steps - 1 of a block, in one launch; the
 * status after each step goes to its slot */
static int launch_rng(esth_filter* f, uint64_t n, int steps, hipStream_t s) {
    const uint64_t b = n / f->B;
    const int kk = (int)(n % f->B), p = (int)(b & 1);
    return esth_launch_mtgp(f->e->d_params, status_at(f, n), status_slot(f, p, kk + 1), f->streams, f->K,
                            step_words(f, n), 1, s, steps, f->words, (uint64_t)f->K * ESTH_MTGP_N);
}

/* the status between carrier i's share of a step's words and the next one's */
static uint32_t* status_between(esth_filter* f, int i) { return status_slot(f, 2, i); }

/* whether step n's sampling launch can carry the next step's MTGP32
 * work-groups: one-step blocks, prefetch on, a 256-thread sampling launch
 * (the fused one at m >= 512, or sample+weight alone), and nothing already
 * generating the next step on the RNG stream */
static bool inline_step(esth_filter* f, bool fused_launch) {
    if (!f->inline_rng || f->B != 1 || !f->prefetch) return false;
    if (fused_launch && !esth_sample_sort_inline_rng(f->m)) return false;
    return f->ready_block != (int64_t)f->steps + 1;
}

/* MTGP32 work carried by each of a step's launches */
struct esth_rng_work {
    esth_mtgp_inline mi[ESTH_CARRIERS];
};

/* the carried words of step n = f->steps: its own, where they are missing
 * (first step, after a restore, without prefetch), by a launch ahead of it,
 * and the next step's in shares */
static int rng_carried(esth_filter* f, bool fused_launch, esth_rng_work* work) {
    const uint64_t n = f->steps;
    if (f->words_upto <= n) {
        ESTH_TRY(esth_launch_mtgp(f->e->d_params, status_at(f, n), status_at(f, n + 1), f->streams, f->K,
                                  step_words(f, n), 1, f->stream));
        f->words_upto = n + 1;
    }
    if (!f->prefetch) return ESTH_OK;
    uint32_t words[ESTH_CARRIERS], first = 0;
    carried_shares(f, fused_launch, words);
    const uint32_t* in = status_at(f, n + 1);
    for (int i = 0; i < ESTH_CARRIERS; ++i) {
        if (!words[i]) continue;
        uint32_t* out = first + words[i] == f->size ? status_at(f, n + 2) : status_between(f, i);
        work->mi[i] = {f->e->d_params, in, out, f->streams, (uint32_t*)step_words(f, n + 1), esth_param_table()[3],
                       first, words[i], f->K};
        in = out;
        first += words[i];
    }
    f->words_upto = n + 2;
    return ESTH_OK;
}

/* RNG side of step n = f->steps, before its kernels.  At the first step of
 * a block the main stream uses the block's words generated inline by the
 * previous step's launch (already in stream order), waits for them
 * (prefetched on the RNG stream), or generates them itself (first step,
 * after a restore, without prefetch): those up to the end of a pair of steps,
 * so that this step does not wait for a long block's (a restored filter's
 * first step with its estimate, the 2M-particle unicycle with 4 landmarks at
 * the start of a block of 3: 228 us with the block generated whole, 133).  With `in`
 * (inline_step) the next step's words will be generated by this step's
 * sampling launch and *work receives that launch's MTGP32 work; otherwise,
 * with prefetch on, the rest of this block and the next one are generated on
 * the RNG stream while this one's steps run, once the block before this one
 * (whose buffer the next one reuses) has been consumed. */
static int rng_before_step(esth_filter* f, bool in, bool fused_launch, esth_rng_work* work) {
    hipStream_t s = f->stream;
    const uint64_t n = f->steps;
    const int64_t b = (int64_t)(n / f->B);
    const int p = (int)(b & 1);
    *work = esth_rng_work{};
    if (f->carried) return rng_carried(f, fused_launch, work);
    esth_mtgp_inline* mi = &work->mi[ESTH_CARRY_SAMPLE];
    const uint64_t end = (uint64_t)(b + 1) * f->B;
    bool cold = false;
    if (n >= f->main_upto) {
        if (f->inline_block == b) {
            f->main_upto = end;   /* generated by the previous launch on this stream */
        } else if (f->ready_block == b || f->rest_block == b) {
            ESTH_HIP(hipStreamWaitEvent(s, f->ev_rng_done[p], 0));
            f->main_upto = end;
        } else {
            const uint64_t pair = (n / ESTH_RNG_BLOCK_DEFAULT + 1) * ESTH_RNG_BLOCK_DEFAULT;
            const int steps = (int)(std::min(end, pair) - n);
            ESTH_TRY(launch_rng(f, n, steps, s));
            f->main_upto = n + steps;
            cold = true;
        }
    }
    if (in) {
        mi->params = f->e->d_params;
        mi->status_in = status_at(f, n + 1);
        mi->status_out = status_slot(f, (int)((n + 1) & 1), 1);
        mi->streams = f->streams;
        mi->out = (uint32_t*)step_words(f, n + 1);
        mi->mask = esth_param_table()[3];
        mi->first = mi->count = 0;   /* all */
        mi->n = f->K;
        f->inline_block = b + 1;
        f->ready_block = b + 1;
        return ESTH_OK;
    }
    if (f->prefetch && f->ready_block != b + 1) {
        const bool rest = f->main_upto < end && f->rest_block != b;
        if (cold || rest || (b > 0 && !f->consumed[p ^ 1])) {
            /* words follow a status that the main stream left, or a block generated inline: behind everything up to here */
            ESTH_HIP(hipEventRecord(f->ev_fork, s));
            ESTH_HIP(hipStreamWaitEvent(f->rng_stream, f->ev_fork, 0));
        } else if (b > 0) {
            ESTH_HIP(hipStreamWaitEvent(f->rng_stream, f->ev_consumed[p ^ 1], 0));
        }
        if (rest) {
            ESTH_TRY(launch_rng(f, f->main_upto, (int)(end - f->main_upto), f->rng_stream));
            ESTH_HIP(hipEventRecord(f->ev_rng_done[p], f->rng_stream));
            f->rest_block = b;
        }
        ESTH_TRY(launch_rng(f, end, f->B, f->rng_stream));
        ESTH_HIP(hipEventRecord(f->ev_rng_done[p ^ 1], f->rng_stream));
        f->ready_block = b + 1;
    }
    return ESTH_OK;
}

/* after the last step of a block its buffer may be refilled.  A step that
 * generates the next one's words inline needs no event: the refill follows
 * on the same stream, and an event between two launches holds the second one
 * back (the 2M-particle unicycle with 32 landmarks: 2.5 us a step, 112.5 ->
 * 110.0) */
static int rng_after_step(esth_filter* f, bool in) {
    const uint64_t n = f->steps;
    if (f->carried || n % f->B != (uint64_t)(f->B - 1)) return ESTH_OK;
    const int p = (int)((n / f->B) & 1);
    f->consumed[p] = !in;
    if (!in) ESTH_HIP(hipEventRecord(f->ev_consumed[p], f->stream));
    return ESTH_OK;
}

/* The main-stream kernels of step n, reading the step's words and its frame:
 * by value from h_frame (eager steps) or, when h_frame is null, at d_frame
 * (graph capture).  ev (optional): timing events.  The first half samples,
 * weights and sorts (into step n's sorted-side buffers), the second runs the
 * argmax, the exchange and the resampling from them. */
static int enqueue_sample(esth_filter* f, uint64_t n, const float* d_frame, const float* h_frame, hipEvent_t* ev,
                          const esth_rng_work* work) {
    const esth_mtgp_inline* mi = &work->mi[ESTH_CARRY_SAMPLE];
    const bool timing = ev != nullptr;
    const bool all = timing && f->timing >= 2;
    hipStream_t s = f->stream;
    const esth_filter_desc& d = f->d;
    const int log_w = d.weights == ESTH_WEIGHTS_LOG;
    const uint32_t N = (uint32_t)f->N;
    float* R = step_words(f, n);
    const esth_xset x = xset(f, n);
    if (timing) ESTH_HIP(hipEventRecord(ev[1], s));
    if (!all && f->fuse_sample_sort) {
        /* sampling_importance (pf_generic.c:521-533) and block_sort
         * (pf_generic.c:572-585) in one launch: the propagated state stays in
         * LDS between them.  Per-stage timing keeps the two launches below
         * (their results are bit-identical). */
        /* a sub-filter the resampling skips keeps its propagated state unless
         * weights are carried (then it takes the sorted one): the scan and
         * the plain alias gate on the uniform rnd[N + g] (pf_generic.cl:403),
         * the adaptive alias on the weights themselves */
        const bool carry = d.carry_weights != 0;
        const int keep_all = !carry && d.resampler == ESTH_RESAMPLE_ALIAS && d.adaptive;
        const float keep_thr = carry ? INFINITY : d.resampling_threshold;
        ESTH_TRY(esth_launch_sample_sort(d.model, f->m, f->state, N, f->G, R, d_frame, log_w, f->w, d.carry_weights,
                                         d.state_layout, f->tmp, x.winner, f->t, x.bt_w, x.bt_s, x.part,
                                         R + (size_t)N * f->V + N, keep_thr, keep_all, s, h_frame, mi, f->words_room));
        if (timing) ESTH_HIP(hipEventRecord(ev[2], s));
    } else {
        /* sampling_importance with Box-Muller fused (pf_generic.c:521-533) */
        ESTH_TRY(esth_launch_sample_weight(d.model, f->state, N, R, d_frame, log_w, f->w, d.carry_weights,
                                           d.state_layout, s, h_frame, mi));
        if (timing) ESTH_HIP(hipEventRecord(ev[2], s));
        /* block_sort (pf_generic.c:572-585) */
        ESTH_TRY(esth_launch_sort(f->S, f->m, f->w, f->state, f->tmp, N, f->G, x.winner, nullptr, f->t, x.bt_w,
                                  x.bt_s, x.part, log_w, d.state_layout, s, &work->mi[ESTH_CARRY_SORT]));
    }
    if (all) ESTH_HIP(hipEventRecord(ev[3], s));
    return ESTH_OK;
}

static int enqueue_resample(esth_filter* f, uint64_t n, hipEvent_t* ev, const esth_mtgp_inline* mi = nullptr) {
    const bool all = ev != nullptr && f->timing >= 2;
    hipStream_t s = f->stream;
    const esth_filter_desc& d = f->d;
    const int log_w = d.weights == ESTH_WEIGHTS_LOG;
    const uint32_t N = (uint32_t)f->N;
    float* R = step_words(f, n);
    const esth_xset x = xset(f, n);
    /* reduce (pf_generic.c:604-615), result kept on the device.  With a scan
     * resampler, or the one-wave alias (m >= 64), it rides in the resampling
     * launch (below); its best particle is rank 0 of the winning sub-filter,
     * read from the sort's compact best-t copy, which the exchange does not
     * touch. */
    const bool fused = d.resampler != ESTH_RESAMPLE_ALIAS || f->m >= 64;   /* one wave per sub-filter */
    if (!fused) ESTH_TRY(esth_launch_argmax(f->S, x.winner, f->G, log_w, x.part, f->tmp, N, f->m, f->result, f->est, true, s));
    if (all) ESTH_HIP(hipEventRecord(ev[4], s));
    /* exchange (pf_generic.c:702-715): in the fused launches its receiving
     * side is applied by the resampling as it reads each sub-filter */
    if (!fused)
        ESTH_TRY(esth_launch_exchange(f->tmp, f->w, f->S, N, f->m, f->G, f->t, d.topology, f->dimx, f->dimy, x.bt_w,
                                      x.bt_s, f->top, s));
    if (all) ESTH_HIP(hipEventRecord(ev[5], s));
    /* resampling (pf_generic.c:732-757), uniforms at rand_offset = N*V */
    if (fused) {
        const bool bt = f->t > 0 && d.topology != ESTH_TOPO_NONE;
        if (d.resampler == ESTH_RESAMPLE_ALIAS)
            ESTH_TRY(esth_launch_alias_argmax(f->S, f->state, f->tmp, f->w, R + (size_t)N * f->V, N, f->m, f->G,
                                              d.resampling_threshold, d.adaptive, log_w, x.winner, x.part,
                                              bt ? x.bt_s : f->tmp, bt ? (size_t)f->G * f->t : (size_t)N,
                                              bt ? f->t : f->m, f->result, f->est, f->t, d.topology, f->dimx,
                                              f->dimy, x.bt_w, x.bt_s, f->top, d.carry_weights, d.state_layout,
                                              s, mi));
        else
            ESTH_TRY(esth_launch_resample_argmax(d.resampler, f->S, f->state, f->tmp, f->w, R + (size_t)N * f->V, N,
                                                 f->m, f->G, d.resampling_threshold, log_w, x.winner, x.part,
                                                 bt ? x.bt_s : f->tmp, bt ? (size_t)f->G * f->t : (size_t)N,
                                                 bt ? f->t : f->m, f->result, f->est, f->t, d.topology, f->dimx,
                                                 f->dimy, x.bt_w, x.bt_s, f->top, d.carry_weights,
                                                 d.state_layout, s, mi));
    } else {
        ESTH_TRY(esth_launch_resample(d.resampler, f->S, f->state, f->tmp, f->w, R + (size_t)N * f->V, N, f->m, f->G,
                                      d.resampling_threshold, d.adaptive, log_w, nullptr, d.carry_weights,
                                      d.state_layout, s));
    }
    if (all) ESTH_HIP(hipEventRecord(ev[6], s));
    return ESTH_OK;
}

static int enqueue_step(esth_filter* f, uint64_t n, const float* d_frame, const float* h_frame, hipEvent_t* ev,
                        const esth_rng_work* work) {
    ESTH_TRY(enqueue_sample(f, n, d_frame, h_frame, ev, work));
    return enqueue_resample(f, n, ev, &work->mi[ESTH_CARRY_RESAMPLE]);
}

/* step n - 1's resampling, argmax and posterior, then step n's sampling and
 * sort, in one launch */
static int enqueue_cross(esth_filter* f, uint64_t n, const float* d_frame, const float* h_frame, hipEvent_t* ev,
                         const esth_rng_work* work) {
    const esth_mtgp_inline* mi = &work->mi[ESTH_CARRY_SAMPLE];
    hipStream_t s = f->stream;
    const esth_filter_desc& d = f->d;
    const uint32_t N = (uint32_t)f->N;
    const float* Rk = step_words(f, n - 1);
    const float* Rk1 = step_words(f, n);
    const esth_xset xk = xset(f, n - 1), xk1 = xset(f, n);
    if (ev) ESTH_HIP(hipEventRecord(ev[1], s));
    ESTH_TRY(esth_launch_step_x(d.model, f->m, f->tmp, f->w, Rk + (size_t)N * f->V, d.resampling_threshold,
                                d.resampler == ESTH_RESAMPLE_SYSTEMATIC ? 1 : 0, xk.bt_w, xk.bt_s, xk.winner, xk.part,
                                f->result, f->est, f->state, N, f->G, f->t, d.topology, f->dimx, f->dimy, Rk1, d_frame,
                                h_frame, d.weights == ESTH_WEIGHTS_LOG, xk1.winner, xk1.bt_w, xk1.bt_s, xk1.part,
                                Rk1 + (size_t)N * f->V + N, mi, s));
    if (ev) ESTH_HIP(hipEventRecord(ev[2], s));
    return ESTH_OK;
}

/* rc of enqueuing a launch with an argmax: it is counted once it is known to
 * run.  A failed one may have run all the same (an error left by an earlier
 * call is reported by the next launch): the next estimate takes the count
 * from the device. */
static int counted(esth_filter* f, int rc) {
    if (rc == ESTH_OK) f->argmaxes++;
    else f->recount = true;
    return rc;
}

/* run the resampling the last step left pending */
static int flush(esth_filter* f) {
    if (!f->pending) return ESTH_OK;
    ESTH_HIP(hipSetDevice(f->e->device));
    f->pending = false;
    return counted(f, enqueue_resample(f, f->steps - 1, nullptr));
}

/* Capture the kernels of a step that reads word block parity p, position kk
 * (graph slot p B + kk; with the cross-step layout, step mod 6): its words,
 * its device frame slot and, with inline generation, the next step's words
 * and statuses are fixed by the slot.  The frame reaches its slot by a copy
 * ahead of each replay.  mode: ESTH_GRAPH_STEP the whole step,
 * ESTH_GRAPH_SAMPLE its sample+weight and sort (the resampling left
 * pending), ESTH_GRAPH_CROSS the cross-step launch. */
enum { ESTH_GRAPH_STEP = 0, ESTH_GRAPH_SAMPLE = 1, ESTH_GRAPH_CROSS = 2 };
static int capture_graph(esth_filter* f, uint64_t n, int slot, const esth_rng_work* work, int mode,
                         hipGraphExec_t* out) {
    hipGraph_t g = nullptr;
    ESTH_HIP(hipStreamBeginCapture(f->stream, hipStreamCaptureModeThreadLocal));
    const float* dfr = f->frames + (size_t)slot * ESTH_FRAME_FLOATS;
    int rc = mode == ESTH_GRAPH_CROSS    ? enqueue_cross(f, n, dfr, nullptr, nullptr, work)
             : mode == ESTH_GRAPH_SAMPLE ? enqueue_sample(f, n, dfr, nullptr, nullptr, work)
                                         : enqueue_step(f, n, dfr, nullptr, nullptr, work);
    hipError_t e2 = hipStreamEndCapture(f->stream, &g);
    if (rc != ESTH_OK) { if (g) hipGraphDestroy(g); return rc; }
    if (e2 != hipSuccess) return esth_fail(ESTH_ERR_DEVICE, "end capture: %s", hipGetErrorString(e2));
    hipError_t e3 = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (e3 != hipSuccess) return esth_fail(ESTH_ERR_DEVICE, "instantiate: %s", hipGetErrorString(e3));
    return ESTH_OK;
}

extern "C" int esth_filter_step(esth_filter* f, const void* control, const void* measurement, float dt) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_HIP(hipSetDevice(f->e->device));
    const uint64_t n = f->steps;
    /* eager steps pass the frame by value; graph replays copy it to the
     * device slot their graph reads (one slot per step of the two blocks; with
     * the cross-step layout, per step mod 6: three word buffers, two
     * sorted-side sets) */
    const int slot = f->xstep ? (int)(n % 6) : (int)(((n / f->B) & 1) * (uint64_t)f->B + n % f->B);
    float frame[ESTH_FRAME_FLOATS];
    float* hf = frame;
    if (f->use_graph) {
        if (f->frame_used[slot]) ESTH_HIP(hipEventSynchronize(f->frame_ev[slot]));
        hf = f->h_frames + (size_t)slot * ESTH_FRAME_FLOATS;
    }
    if (esth_build_frame_impl(f->d.model, f->params, control, measurement, dt, hf))
        return esth_fail(ESTH_ERR_INVALID, "bad control/measurement for model %d", f->d.model);
    hipEvent_t* ev = nullptr;
    if (!f->use_graph && f->timing && f->tsteps < ESTH_TIMING_STEPS && (f->tcount++ % (uint64_t)f->timing_every) == 0) {
        if ((size_t)(f->tsteps + 1) * 7 > f->tev.size()) {
            for (int i = 0; i < 7; ++i) {
                /* timing only: no system-scope release at each event (its
                 * cache write-back would be timed with the kernel) */
                hipEvent_t e;
                ESTH_HIP(hipEventCreateWithFlags(&e, hipEventDisableSystemFence));
                f->tev.push_back(e);
            }
        }
        ev = &f->tev[(size_t)f->tsteps * 7];
        f->tsteps++;
    }
    /* per-stage timing (level 2) runs sample+weight and the sort as two launches */
    const bool level2 = ev && f->timing >= 2;
    const bool fused_launch = f->fuse_sample_sort && !level2;
    /* the cross-step launch: steps without per-stage timing */
    const bool cross = f->xstep && f->xstep_on && f->fuse_sample_sort && !level2;
    if (f->pending && !cross) ESTH_TRY(flush(f));
    const bool in = f->carried ? f->prefetch : inline_step(f, fused_launch);
    if (level2) ESTH_HIP(hipEventRecord(ev[0], f->stream));
    esth_rng_work work;
    ESTH_TRY(rng_before_step(f, in, fused_launch, &work));
    if (f->use_graph) {
        const int mode = !cross ? ESTH_GRAPH_STEP : f->pending ? ESTH_GRAPH_CROSS : ESTH_GRAPH_SAMPLE;
        if (f->gexec[slot] && (f->gexec_inline[slot] != in || f->gexec_mode[slot] != mode)) {
            hipGraphExecDestroy(f->gexec[slot]);
            f->gexec[slot] = nullptr;
        }
        if (!f->gexec[slot]) {
            ESTH_TRY(capture_graph(f, n, slot, &work, mode, &f->gexec[slot]));
            f->gexec_inline[slot] = in;
            f->gexec_mode[slot] = mode;
        }
        float* dfr = f->frames + (size_t)slot * ESTH_FRAME_FLOATS;
        ESTH_HIP(hipMemcpyAsync(dfr, hf, sizeof(float) * ESTH_FRAME_FLOATS, hipMemcpyHostToDevice, f->stream));
        ESTH_HIP(hipEventRecord(f->frame_ev[slot], f->stream));
        f->frame_used[slot] = true;
        const hipError_t err = hipGraphLaunch(f->gexec[slot], f->stream);
        const int rc = err == hipSuccess ? ESTH_OK : esth_fail(ESTH_ERR_DEVICE, "graph launch: %s", hipGetErrorString(err));
        ESTH_TRY(mode != ESTH_GRAPH_SAMPLE ? counted(f, rc) : rc);
        if (cross) f->pending = true;
    } else if (cross) {
        if (f->pending) {
            ESTH_TRY(counted(f, enqueue_cross(f, n, nullptr, hf, ev, &work)));
        } else {
            ESTH_TRY(enqueue_sample(f, n, nullptr, hf, ev, &work));
        }
        f->pending = true;
    } else {
        ESTH_TRY(counted(f, enqueue_step(f, n, nullptr, hf, ev, &work)));
    }
    ESTH_TRY(rng_after_step(f, in));
    f->steps++;
    return ESTH_OK;
}

extern "C" int esth_filter_set_cross_step(esth_filter* f, int enable, int* active) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_TRY(flush(f));
    f->xstep_on = enable != 0;
    if (active) *active = (f->xstep && f->xstep_on && f->fuse_sample_sort) ? 1 : 0;
    return ESTH_OK;
}

extern "C" int esth_filter_rng_mode(esth_filter* f, int* inline_words, int* block_steps) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    if (inline_words) *inline_words = inline_step(f, f->fuse_sample_sort) ? 1 : 0;
    if (block_steps) *block_steps = f->B;
    return ESTH_OK;
}

extern "C" int esth_filter_use_graph(esth_filter* f, int enable) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_HIP(hipStreamSynchronize(f->rng_stream));
    f->use_graph = enable != 0;
    return ESTH_OK;
}

/* Overlap the next step's MTGP words with the current step (default on). */
extern "C" int esth_filter_set_fusion(esth_filter* f, int enable, int* active) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_HIP(hipSetDevice(f->e->device));
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    for (int i = 0; i < ESTH_FRAME_RING; ++i)
        if (f->gexec[i]) { hipGraphExecDestroy(f->gexec[i]); f->gexec[i] = nullptr; }
    f->fuse_sample_sort = enable != 0 && esth_sample_sort_pays(f->d.model, f->d.state_layout, f->m);
    if (active) *active = f->fuse_sample_sort ? 1 : 0;
    return ESTH_OK;
}

extern "C" int esth_filter_set_prefetch(esth_filter* f, int enable) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_HIP(hipStreamSynchronize(f->rng_stream));
    for (int i = 0; i < ESTH_FRAME_RING; ++i)
        if (f->gexec[i]) { hipGraphExecDestroy(f->gexec[i]); f->gexec[i] = nullptr; }
    f->prefetch = enable != 0;
    return ESTH_OK;
}

extern "C" int esth_filter_sync(esth_filter* f) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_HIP(hipStreamSynchronize(f->rng_stream));
    return ESTH_OK;
}

int esth_filter_time_steps(esth_filter* f, int n, const void* control, const void* measurement, float dt,
                           float* us_per_step) {
    if (!f || n <= 0 || !us_per_step) return esth_fail(ESTH_ERR_INVALID, "time steps: bad arguments");
    ESTH_HIP(hipSetDevice(f->e->device));
    hipEvent_t ev[2];
    ESTH_HIP(hipEventCreate(&ev[0]));
    if (hipEventCreate(&ev[1]) != hipSuccess) {
        hipEventDestroy(ev[0]);
        return esth_fail(ESTH_ERR_DEVICE, "time steps: event");
    }
    int rc = esth_filter_sync(f);
    if (rc == ESTH_OK && hipEventRecord(ev[0], f->stream) != hipSuccess) rc = esth_fail(ESTH_ERR_DEVICE, "event");
    for (int i = 0; rc == ESTH_OK && i < n; ++i) rc = esth_filter_step(f, control, measurement, dt);
    if (rc == ESTH_OK && hipEventRecord(ev[1], f->stream) != hipSuccess) rc = esth_fail(ESTH_ERR_DEVICE, "event");
    float ms = 0.0f;
    if (rc == ESTH_OK && hipEventSynchronize(ev[1]) != hipSuccess) rc = esth_fail(ESTH_ERR_DEVICE, "event sync");
    if (rc == ESTH_OK && hipEventElapsedTime(&ms, ev[0], ev[1]) != hipSuccess) rc = esth_fail(ESTH_ERR_DEVICE, "elapsed");
    hipEventDestroy(ev[0]);
    hipEventDestroy(ev[1]);
    if (rc == ESTH_OK) *us_per_step = ms * 1000.0f / (float)n;
    return rc;
}

extern "C" int esth_filter_stream(esth_filter* f, void** s) {
    if (!f || !s) return esth_fail(ESTH_ERR_INVALID, "null");
    *s = (void*)f->stream;
    return ESTH_OK;
}

extern "C" int esth_filter_set_timing(esth_filter* f, int on) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null filter");
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    f->timing = on < 0 ? 0 : (on > 2 ? 2 : on);
    f->tsteps = 0;
    f->tcount = 0;
    return ESTH_OK;
}

extern "C" int esth_filter_set_timing_every(esth_filter* f, int every) {
    if (!f || every < 1) return esth_fail(ESTH_ERR_INVALID, "timing stride must be >= 1");
    f->timing_every = every;
    f->tcount = 0;
    return ESTH_OK;
}

/* mean per-stage device time over the steps recorded since timing was switched on */
extern "C" int esth_filter_stage_times(esth_filter* f, float us[6]) {
    if (!f || !us) return esth_fail(ESTH_ERR_INVALID, "null");
    if (f->tsteps == 0) return esth_fail(ESTH_ERR_STATE, "no timed steps (timing off, or graph replay)");
    ESTH_HIP(hipStreamSynchronize(f->stream));
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int k = 0; k < f->tsteps; ++k) {
        hipEvent_t* ev = &f->tev[(size_t)k * 7];
        for (int i = 0; i < 6; ++i) {
            if (f->timing < 2 && i != 1) continue;
            float ms = 0.0f;
            ESTH_HIP(hipEventElapsedTime(&ms, ev[i], ev[i + 1]));
            acc[i] += ms;
        }
    }
    for (int i = 0; i < 6; ++i)
        us[i] = (f->timing < 2 && i != 1) ? NAN : (float)(acc[i] * 1000.0 / f->tsteps);
    return ESTH_OK;
}

/* until the last argmax enqueued has published its estimate: its count,
 * polled for up to ESTH_POLL_US, beyond that (long queues) the stream's end */
static int wait_estimate(esth_filter* f) {
    const std::atomic<uint64_t>* count = reinterpret_cast<const std::atomic<uint64_t>*>(f->est + ESTH_EST_COUNT);
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 1; !f->recount; ++i) {
        if (count->load(std::memory_order_acquire) >= f->argmaxes) return ESTH_OK;
        if (i % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(ESTH_POLL_US)) break;
#if !defined(__HIP_DEVICE_COMPILE__)
        __builtin_ia32_pause();
#endif
    }
    ESTH_HIP(hipStreamSynchronize(f->stream));
    const uint64_t done = count->load(std::memory_order_acquire);
    const bool lost = !f->recount && done < f->argmaxes;
    f->argmaxes = done;
    f->recount = false;
    return lost ? esth_fail(ESTH_ERR_DEVICE, "the step's estimate was not written") : ESTH_OK;
}

extern "C" int esth_filter_estimate(esth_filter* f, esth_estimate* out) {
    if (!f || !out) return esth_fail(ESTH_ERR_INVALID, "null");
    ESTH_TRY(flush(f));
    ESTH_TRY(wait_estimate(f));
    const double* h = f->est;
    memset(out, 0, sizeof(*out));
    const int S = f->S;
    out->state_dim = S;
    out->log_weight_max = h[0];
    out->weight_sum = h[1];
    for (int c = 0; c < S; ++c) {
        out->mean[c] = h[1] > 0.0 ? h[2 + c] / h[1] : NAN;
        out->best[c] = (float)h[4 + S + c];
    }
    out->best_weight = (float)h[2 + S];
    out->best_block = (int)h[3 + S];
    out->step = f->steps;
    return ESTH_OK;
}

extern "C" int esth_filter_read_particles(esth_filter* f, float* soa, float* w) {
    if (!f) return esth_fail(ESTH_ERR_INVALID, "null");
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    if (soa) ESTH_TRY(download_state(f, soa));
    if (w) ESTH_HIP(hipMemcpy(w, f->w, sizeof(float) * f->N, hipMemcpyDeviceToHost));
    return ESTH_OK;
}

/* snapshot: magic, S, N, K, steps, model, m, G | state (SOA planes, whatever
 * the filter's layout) | w | status */
#define ESTH_SNAP_MAGIC 0x45535448u
extern "C" int esth_filter_snapshot_size(esth_filter* f, size_t* bytes) {
    if (!f || !bytes) return esth_fail(ESTH_ERR_INVALID, "null");
    *bytes = 8 * sizeof(uint64_t) + sizeof(float) * ((size_t)f->S * f->N + f->N) + sizeof(uint32_t) * ESTH_MTGP_N * (size_t)f->K;
    return ESTH_OK;
}

extern "C" int esth_filter_snapshot(esth_filter* f, void* buf, size_t bytes) {
    size_t need = 0;
    ESTH_TRY(esth_filter_snapshot_size(f, &need));
    if (!buf || bytes < need) return esth_fail(ESTH_ERR_INVALID, "snapshot buffer %zu < %zu", bytes, need);
    ESTH_TRY(flush(f));
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_HIP(hipStreamSynchronize(f->rng_stream));
    uint64_t* hdr = (uint64_t*)buf;
    hdr[0] = ESTH_SNAP_MAGIC; hdr[1] = (uint64_t)f->S; hdr[2] = f->N; hdr[3] = (uint64_t)f->K; hdr[4] = f->steps;
    hdr[5] = f->d.model; hdr[6] = f->m; hdr[7] = f->G;
    char* p = (char*)buf + 8 * sizeof(uint64_t);
    ESTH_TRY(download_state(f, (float*)p));
    p += sizeof(float) * (size_t)f->S * f->N;
    ESTH_HIP(hipMemcpy(p, f->w, sizeof(float) * f->N, hipMemcpyDeviceToHost));
    p += sizeof(float) * f->N;
    /* the status that generates the next step's words (words generated ahead are regenerated on restore) */
    ESTH_HIP(hipMemcpy(p, status_at(f, f->steps), sizeof(uint32_t) * ESTH_MTGP_N * (size_t)f->K, hipMemcpyDeviceToHost));
    return ESTH_OK;
}

extern "C" int esth_filter_restore(esth_filter* f, const void* buf, size_t bytes) {
    size_t need = 0;
    ESTH_TRY(esth_filter_snapshot_size(f, &need));
    if (!buf || bytes < need) return esth_fail(ESTH_ERR_INVALID, "snapshot buffer %zu < %zu", bytes, need);
    const uint64_t* hdr = (const uint64_t*)buf;
    if (hdr[0] != ESTH_SNAP_MAGIC || hdr[1] != (uint64_t)f->S || hdr[2] != f->N || hdr[3] != (uint64_t)f->K ||
        hdr[5] != (uint64_t)f->d.model || hdr[6] != f->m || hdr[7] != f->G)
        return esth_fail(ESTH_ERR_INVALID, "snapshot does not match this filter");
    ESTH_HIP(hipStreamSynchronize(f->stream));
    ESTH_HIP(hipStreamSynchronize(f->rng_stream));
    const char* p = (const char*)buf + 8 * sizeof(uint64_t);
    ESTH_TRY(upload_state(f, (const float*)p));
    p += sizeof(float) * (size_t)f->S * f->N;
    ESTH_HIP(hipMemcpy(f->w, p, sizeof(float) * f->N, hipMemcpyHostToDevice));
    p += sizeof(float) * f->N;
    f->steps = hdr[4];
    f->pending = false;
    ESTH_HIP(hipMemcpy(status_at(f, f->steps), p, sizeof(uint32_t) * ESTH_MTGP_N * (size_t)f->K, hipMemcpyHostToDevice));
    f->ready_block = -1;
    f->rest_block = -1;
    f->main_upto = 0;
    f->inline_block = -1;
    f->words_upto = 0;
    return ESTH_OK;
}

/* ================================================= trace I/O, reference */
/* read_trace, pf_model_host.h:30-54: 20 whitespace-separated floats per row */
extern "C" int esth_trace_load_robotarm(const char* path, int max_rows, esth_robotarm5_measurement* meas,
                                        esth_robotarm5_control* ctrl, float* dt, float* truth, int* rows) {
    if (!path || !rows) return esth_fail(ESTH_ERR_INVALID, "null");
    FILE* fh = fopen(path, "r");
    if (!fh) return esth_fail(ESTH_ERR_IO, "could not open %s", path);
    int n = 0;
    while (n < max_rows) {
        float v[20];
        int k = 0;
        for (; k < 20; ++k)
            if (fscanf(fh, "%f", &v[k]) != 1) break;
        if (k < 20) break;   /* a short or garbled row ends the trace, as read_trace's -1 */
        if (meas) {
            meas[n].x = v[0]; meas[n].y = v[1];
            for (int i = 0; i < 5; ++i) meas[n].angles[i] = v[2 + i];
        }
        if (ctrl) for (int i = 0; i < 5; ++i) ctrl[n].angles[i] = v[7 + i];
        if (dt) dt[n] = v[12];
        if (truth) {
            float* tr = truth + (size_t)n * 9;
            for (int i = 0; i < 5; ++i) tr[i] = v[15 + i];
            tr[5] = v[13]; tr[6] = v[14]; tr[7] = 0.0f; tr[8] = 0.0f;
        }
        ++n;
    }
    fclose(fh);
    *rows = n;
    return ESTH_OK;
}

static void write_floats(FILE* fh, const float* v, int n) {
    for (int k = 0; k < n; ++k) fprintf(fh, k ? " %.9g" : "%.9g", (double)v[k]);
    fputc('\n', fh);
}

extern "C" int esth_trace_write_robotarm(const char* path, int rows, const esth_robotarm5_measurement* meas,
                                         const esth_robotarm5_control* ctrl, const float* dt, const float* truth) {
    if (!path || rows < 0 || (rows > 0 && (!meas || !ctrl || !dt || !truth))) return esth_fail(ESTH_ERR_INVALID, "null");
    FILE* fh = fopen(path, "w");
    if (!fh) return esth_fail(ESTH_ERR_IO, "could not open %s", path);
    for (int n = 0; n < rows; ++n) {
        const float* tr = truth + (size_t)n * 9;
        float v[20];
        v[0] = meas[n].x; v[1] = meas[n].y;
        for (int i = 0; i < 5; ++i) { v[2 + i] = meas[n].angles[i]; v[7 + i] = ctrl[n].angles[i]; v[15 + i] = tr[i]; }
        v[12] = dt[n]; v[13] = tr[5]; v[14] = tr[6];
        write_floats(fh, v, 20);
    }
    if (fclose(fh)) return esth_fail(ESTH_ERR_IO, "could not write %s", path);
    return ESTH_OK;
}

/* estimate_error, pf_model_host.h:56-69 */
extern "C" float esth_robotarm5_estimate_error(const float* est, const float* act) {
    float error = 0.0f;
    error += (est[5] - act[5]) * (est[5] - act[5]) * ESTH_RA5_NOISE_CAMERA_X;
    error += (est[6] - act[6]) * (est[6] - act[6]) * ESTH_RA5_NOISE_CAMERA_Y;
    for (int i = 0; i < 5; ++i) error += (est[i] - act[i]) * (est[i] - act[i]) * ESTH_RA5_NOISE_ANGLE_MEASUREMENTS;
    return error;
}

static int count_lines(const char* path, int* lines);

/* particle_filter() for the robot arm over a trace (pf_generic.c:245-887) */
extern "C" int esth_particle_filter(uint32_t m, uint32_t G, uint32_t t, float thr, const char* trace, uint32_t seed,
                                    int resampler, double* mean_error, int* steps) {
    const int max_rows = 1 << 20;
    std::vector<esth_robotarm5_measurement> meas;
    std::vector<esth_robotarm5_control> ctrl;
    std::vector<float> dt, truth;
    int rows = 0;
    ESTH_TRY(count_lines(trace, &rows));
    rows = std::min(rows, max_rows);
    meas.resize(rows); ctrl.resize(rows); dt.resize(rows); truth.resize((size_t)rows * 9);
    ESTH_TRY(esth_trace_load_robotarm(trace, rows, meas.data(), ctrl.data(), dt.data(), truth.data(), &rows));
    esth_engine* e = nullptr;
    ESTH_TRY(esth_engine_create(0, 0, &e));
    esth_filter_desc d;
    esth_filter_desc_default(&d, ESTH_MODEL_ROBOTARM5);
    d.num_particles = m; d.num_blocks = G; d.num_transfer = t; d.resampling_threshold = thr;
    d.resampler = resampler; d.seed = seed; d.topology = t ? ESTH_TOPO_RING : ESTH_TOPO_NONE;
    esth_filter* f = nullptr;
    int rc = esth_filter_create(e, &d, nullptr, 0, &f);
    if (rc != ESTH_OK) { esth_engine_destroy(e); return rc; }
    /* initial particles, pf_generic.c:346-361 */
    const float a0 = (float)(0.75f * M_PI);
    float init[9] = {a0, a0, a0, a0, a0, 7.0f, 0.0f, 0.0f, 0.0f};
    rc = esth_filter_init_uniform(f, init);
    double err_sum = 0.0;
    for (int i = 0; rc == ESTH_OK && i < rows; ++i) {
        rc = esth_filter_step(f, &ctrl[i], &meas[i], dt[i]);
        esth_estimate est;
        if (rc == ESTH_OK) rc = esth_filter_estimate(f, &est);
        if (rc == ESTH_OK) {
            float best[9];
            for (int c = 0; c < 9; ++c) best[c] = est.best[c];
            best[7] = 0.0f; best[8] = 0.0f;
            err_sum += esth_robotarm5_estimate_error(best, &truth[(size_t)i * 9]);
        }
    }
    esth_filter_destroy(f);
    esth_engine_destroy(e);
    if (rc != ESTH_OK) return rc;
    if (mean_error) *mean_error = rows ? err_sum / rows : 0.0;
    if (steps) *steps = rows;
    return ESTH_OK;
}

extern "C" int esth_trace_write_unicycle10(const char* path, int rows, const esth_unicycle10_measurement* meas,
                                           const esth_unicycle_control* ctrl, const float* dt, const float* truth) {
    if (!path || rows < 0 || (rows > 0 && (!meas || !ctrl || !dt || !truth))) return esth_fail(ESTH_ERR_INVALID, "null");
    FILE* fh = fopen(path, "w");
    if (!fh) return esth_fail(ESTH_ERR_IO, "could not open %s", path);
    for (int n = 0; n < rows; ++n) {
        float v[16];
        for (int i = 0; i < 10; ++i) v[i] = meas[n].range[i];
        v[10] = ctrl[n].v; v[11] = ctrl[n].omega; v[12] = dt[n];
        for (int i = 0; i < 3; ++i) v[13 + i] = truth[(size_t)n * 3 + i];
        write_floats(fh, v, 16);
    }
    if (fclose(fh)) return esth_fail(ESTH_ERR_IO, "could not write %s", path);
    return ESTH_OK;
}

/* the reference unicycle's input rows (particle_filter.cu:756-772): 16 floats */
extern "C" int esth_trace_load_unicycle10(const char* path, int max_rows, esth_unicycle10_measurement* meas,
                                          esth_unicycle_control* ctrl, float* dt, float* truth, int* rows) {
    if (!path || !rows) return esth_fail(ESTH_ERR_INVALID, "null");
    FILE* fh = fopen(path, "r");
    if (!fh) return esth_fail(ESTH_ERR_IO, "could not open %s", path);
    int n = 0;
    while (n < max_rows) {
        float v[16];
        int k = 0;
        for (; k < 16; ++k)
            if (fscanf(fh, "%f", &v[k]) != 1) break;
        if (k < 16) break;   /* the reference loop runs while fscanf reads all 16 */
        if (meas) for (int i = 0; i < 10; ++i) meas[n].range[i] = v[i];
        if (ctrl) { ctrl[n].v = v[10]; ctrl[n].omega = v[11]; }
        if (dt) dt[n] = v[12];
        if (truth) { truth[(size_t)n * 3] = v[13]; truth[(size_t)n * 3 + 1] = v[14]; truth[(size_t)n * 3 + 2] = v[15]; }
        ++n;
    }
    fclose(fh);
    *rows = n;
    return ESTH_OK;
}

static int count_lines(const char* path, int* lines) {
    FILE* fh = fopen(path, "r");
    if (!fh) return esth_fail(ESTH_ERR_IO, "could not open %s", path);
    int n = 0, ch;
    while ((ch = fgetc(fh)) != EOF) n += ch == '\n';
    fclose(fh);
    *lines = n + 1;
    return ESTH_OK;
}

/* particle_filter.cu:729-1157 with the engine's step: one filter over the
 * trace, error = |best particle - truth| in the plane, averaged over steps */
extern "C" int esth_unicycle10_filter(uint32_t m, uint32_t G, uint32_t t, float thr, const char* trace, uint32_t seed,
                                      int resampler, double* mean_error, int* steps) {
    if (!trace) return esth_fail(ESTH_ERR_INVALID, "null trace");
    int rows = 0;
    ESTH_TRY(count_lines(trace, &rows));
    rows = std::min(rows, 1 << 20);
    std::vector<esth_unicycle10_measurement> meas(rows);
    std::vector<esth_unicycle_control> ctrl(rows);
    std::vector<float> dt(rows), truth((size_t)rows * 3);
    ESTH_TRY(esth_trace_load_unicycle10(trace, rows, meas.data(), ctrl.data(), dt.data(), truth.data(), &rows));
    esth_unicycle10_params prm;
    esth_unicycle10_params_default(&prm);
    esth_engine* e = nullptr;
    ESTH_TRY(esth_engine_create(0, 0, &e));
    esth_filter_desc d;
    esth_filter_desc_default(&d, ESTH_MODEL_UNICYCLE10);
    d.num_particles = m; d.num_blocks = G; d.num_transfer = t; d.resampling_threshold = thr;
    d.resampler = resampler; d.seed = seed; d.topology = t ? ESTH_TOPO_RING : ESTH_TOPO_NONE;
    esth_filter* f = nullptr;
    int rc = esth_filter_create(e, &d, &prm, sizeof(prm), &f);
    if (rc != ESTH_OK) { esth_engine_destroy(e); return rc; }
    const float init[3] = {20.0f, 40.0f, (float)(-M_PI / 2)};
    rc = esth_filter_init_uniform(f, init);
    double err_sum = 0.0;
    for (int i = 0; rc == ESTH_OK && i < rows; ++i) {
        rc = esth_filter_step(f, &ctrl[i], &meas[i], dt[i]);
        esth_estimate est;
        if (rc == ESTH_OK) rc = esth_filter_estimate(f, &est);
        if (rc == ESTH_OK) {
            const double ex = (double)est.best[0] - truth[(size_t)i * 3], ey = (double)est.best[1] - truth[(size_t)i * 3 + 1];
            err_sum += std::sqrt(ex * ex + ey * ey);
        }
    }
    esth_filter_destroy(f);
    esth_engine_destroy(e);
    if (rc != ESTH_OK) return rc;
    if (mean_error) *mean_error = rows ? err_sum / rows : 0.0;
    if (steps) *steps = rows;
    return ESTH_OK;
}

/* ============================================================ scenarios
 * Seeded host generators: splitmix64 words, uniform doubles in [0,1), normals
 * by the polar-free Box-Muller in double. */
struct esth_hostrng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }
    double uniform() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); }
    double normal() {
        double u1 = 1.0 - uniform(), u2 = uniform();
        return sqrt(-2.0 * log(u1)) * cos(2.0 * M_PI * u2);
    }
};

static double wrap_pi(double a) {
    a = fmod(a + M_PI, 2.0 * M_PI);
    if (a <= 0.0) a += 2.0 * M_PI;
    return a - M_PI;
}

extern "C" int esth_unicycle_scenario(uint32_t seed, int L, float box, int steps, float dt, esth_unicycle_params* p,
                                      esth_unicycle_control* ctrl, esth_unicycle_measurement* meas, float* truth) {
    if (!p || L < 0 || L > ESTH_UNICYCLE_MAX_LANDMARKS || steps < 0) return esth_fail(ESTH_ERR_INVALID, "scenario args");
    esth_hostrng rng{0x5eed000000000000ull ^ (uint64_t)seed};
    memset(p, 0, sizeof(*p));
    p->num_landmarks = L;
    p->sigma_x = 0.05f; p->sigma_y = 0.05f; p->sigma_theta = 0.01f;
    p->sigma_range = 0.1f; p->sigma_bearing = 0.02f;
    if (L == 4 && box == 0.0f) {
        const float lx[4] = {10.0f, -10.0f, -10.0f, 10.0f}, ly[4] = {10.0f, 10.0f, -10.0f, -10.0f};
        for (int j = 0; j < 4; ++j) { p->lx[j] = lx[j]; p->ly[j] = ly[j]; }
    } else {
        for (int j = 0; j < L; ++j) {
            p->lx[j] = (float)(-box + 2.0 * box * rng.uniform());
            p->ly[j] = (float)(-box + 2.0 * box * rng.uniform());
        }
    }
    double x = 0.0, y = 0.0, th = 0.0;
    for (int k = 0; k < steps; ++k) {
        const double v = 1.0, om = 0.2 * sin(0.05 * (double)k);
        double nth = th;
        x += v * dt * cos(nth) + p->sigma_x * rng.normal();
        y += v * dt * sin(nth) + p->sigma_y * rng.normal();
        th += om * dt + p->sigma_theta * rng.normal();
        if (ctrl) { ctrl[k].v = (float)v; ctrl[k].omega = (float)om; }
        if (truth) { truth[3 * k] = (float)x; truth[3 * k + 1] = (float)y; truth[3 * k + 2] = (float)th; }
        if (meas) {
            memset(&meas[k], 0, sizeof(meas[k]));
            for (int j = 0; j < L; ++j) {
                double dx = p->lx[j] - x, dy = p->ly[j] - y;
                meas[k].range[j] = (float)(sqrt(dx * dx + dy * dy) + p->sigma_range * rng.normal());
                meas[k].bearing[j] = (float)wrap_pi(atan2(dy, dx) - th + p->sigma_bearing * rng.normal());
            }
        }
    }
    return ESTH_OK;
}

extern "C" int esth_dh6_scenario(uint32_t seed, int steps, float dt, esth_dh6_params* p, esth_dh6_measurement* meas,
                                 float* truth) {
    if (!p || steps < 0) return esth_fail(ESTH_ERR_INVALID, "scenario args");
    esth_hostrng rng{0xd6a0000000000000ull ^ (uint64_t)seed};
    memset(p, 0, sizeof(*p));
    const double alpha[6] = {M_PI / 2, 0.0, 0.0, M_PI / 2, -M_PI / 2, 0.0};
    for (int i = 0; i < 6; ++i) {
        p->a[i] = (float)(0.2 + 0.4 * rng.uniform());
        p->d[i] = (float)(-0.1 + 0.2 * rng.uniform());
        p->alpha[i] = (float)alpha[i];
    }
    p->sigma_acc = 0.5f; p->sigma_pos = 0.01f; p->sigma_enc = 0.005f;
    double q[6], qd[6];
    for (int i = 0; i < 6; ++i) { q[i] = -0.5 + rng.uniform(); qd[i] = -0.5 + rng.uniform(); }
    /* truth row 0 holds the initial state; rows 1..steps the states after each step */
    if (truth) for (int i = 0; i < 6; ++i) { truth[i] = (float)q[i]; truth[6 + i] = (float)qd[i]; }
    for (int k = 0; k < steps; ++k) {
        for (int i = 0; i < 6; ++i) {
            double a = p->sigma_acc * rng.normal();
            q[i] += qd[i] * dt + 0.5 * dt * dt * a;
            qd[i] += a * dt;
        }
        double T[4][4] = {{1, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 1, 0}, {0, 0, 0, 1}};
        for (int i = 0; i < 6; ++i) {
            double cq = cos(q[i]), sq = sin(q[i]), ca = cos((double)p->alpha[i]), sa = sin((double)p->alpha[i]);
            double A[4][4] = {{cq, -sq * ca, sq * sa, p->a[i] * cq}, {sq, cq * ca, -cq * sa, p->a[i] * sq}, {0, sa, ca, p->d[i]}, {0, 0, 0, 1}};
            double R[4][4];
            for (int r = 0; r < 4; ++r)
                for (int c = 0; c < 4; ++c) {
                    double acc = 0;
                    for (int kk = 0; kk < 4; ++kk) acc += T[r][kk] * A[kk][c];
                    R[r][c] = acc;
                }
            memcpy(T, R, sizeof(T));
        }
        if (meas) {
            for (int i = 0; i < 3; ++i) meas[k].p[i] = (float)(T[i][3] + p->sigma_pos * rng.normal());
            for (int i = 0; i < 6; ++i) meas[k].q[i] = (float)(q[i] + p->sigma_enc * rng.normal());
        }
        if (truth) {
            float* tr = truth + (size_t)(k + 1) * 12;
            for (int i = 0; i < 6; ++i) { tr[i] = (float)q[i]; tr[6 + i] = (float)qd[i]; }
        }
    }
    return ESTH_OK;
}

/* the base's pixel position for an arm state (pinhole + distortion of the
 * robotarm5_camera model), in double */
static void camera_project(const double* q, double x, double y, const esth_camera_params* p, double* u, double* v) {
    double cx = x * cos(q[0]) + y * sin(q[0]);
    double cy = -x * sin(q[0]) + y * cos(q[0]);
    double cz = 0.0;
    for (int i = 1; i < 5; ++i) {
        const double nb = cy * cos(q[i]) - cz * sin(q[i]);
        const double nc = cy * sin(q[i]) + cz * cos(q[i]);
        cy = nb;
        cz = nc - 3.0;
    }
    const double xn = cx / cz, yn = cy / cz, r2 = xn * xn + yn * yn;
    const double radial = 1.0 + p->kc[0] * r2 + p->kc[1] * r2 * r2;
    const double xd = xn * radial + 2.0 * p->kc[2] * xn * yn + p->kc[3] * (r2 + 2.0 * xn * xn);
    const double yd = yn * radial + p->kc[2] * (r2 + 2.0 * yn * yn) + 2.0 * p->kc[3] * xn * yn;
    *u = p->fc[0] * xd + p->cc[0];
    *v = p->fc[1] * yd + p->cc[1];
}

extern "C" int esth_robotarm5_camera_scenario(uint32_t seed, int steps, float dt, const esth_camera_params* params,
                                              esth_robotarm5_control* ctrl, esth_robotarm5_measurement* meas,
                                              float* truth) {
    if (steps < 0 || !(dt > 0.0f)) return esth_fail(ESTH_ERR_INVALID, "scenario args");
    esth_camera_params dflt;
    esth_camera_params_default(&dflt);
    const esth_camera_params* p = params ? params : &dflt;
    esth_hostrng rng{0xca3e000000000000ull ^ (uint64_t)seed};
    double q[5], x = 0.0, y = 0.0, vx = 0.0, vy = 0.0, ph[5];
    for (int i = 0; i < 5; ++i) { q[i] = 0.75 * M_PI; ph[i] = 2.0 * M_PI * rng.uniform(); }
    if (truth) {
        for (int i = 0; i < 5; ++i) truth[i] = (float)q[i];
        truth[5] = truth[6] = truth[7] = truth[8] = 0.0f;
    }
    for (int k = 0; k < steps; ++k) {
        for (int i = 0; i < 5; ++i) {
            const double rate = 0.2 * sin(0.05 * (double)k + ph[i]);
            if (ctrl) ctrl[k].angles[i] = (float)rate;
            q[i] += rate * dt + 0.01 * rng.normal();
        }
        vx = fmin(0.5, fmax(-0.5, vx + 0.1 * rng.normal()));
        vy = fmin(0.5, fmax(-0.5, vy + 0.1 * rng.normal()));
        x += vx * dt;
        y += vy * dt;
        if (fabs(x) > 1.0) { x = copysign(2.0, x) - x; vx = -vx; }
        if (fabs(y) > 1.0) { y = copysign(2.0, y) - y; vy = -vy; }
        if (meas) {
            double u, v;
            camera_project(q, x, y, p, &u, &v);
            for (int i = 0; i < 5; ++i) meas[k].angles[i] = (float)(q[i] + 0.05 * rng.normal());
            meas[k].x = (float)(u + rng.normal());
            meas[k].y = (float)(v + rng.normal());
        }
        if (truth) {
            float* tr = truth + (size_t)(k + 1) * 9;
            for (int i = 0; i < 5; ++i) tr[i] = (float)q[i];
            tr[5] = (float)x; tr[6] = (float)y; tr[7] = (float)vx; tr[8] = (float)vy;
        }
    }
    return ESTH_OK;
}
