// context.hip -- lifecycle, host exchange and dispatch of the C-ABI.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>

#include "ctx.hpp"

using namespace sphgpu;

namespace sphgpu {

int fail(sphgpu_ctx *c, int code, const std::string &msg)
{
    if (c) c->err = msg;
    return code;
}

// the kernel groups that timing mode 2 keeps
static bool pair_kernel(const char *name)
{
    static const char *const keep[] = {"search_pre", "search_force", "pre_interaction", "fluid_force", "gravity"};
    for (const char *k : keep)
        if (std::strcmp(name, k) == 0) return true;
    return false;
}

void time_begin(sphgpu_ctx *c, const char *name)
{
    c->timing_open = false;
    if (!c->timing || (c->timing == 2 && !pair_kernel(name))) return;
    c->timing_open = true;
    Timer t;
    if (c->event_pool.size() >= 2) {
        t.a = c->event_pool.back(); c->event_pool.pop_back();
        t.b = c->event_pool.back(); c->event_pool.pop_back();
    } else {
        hipEventCreate(&t.a);
        hipEventCreate(&t.b);
    }
    t.name = name;
    hipEventRecord(t.a, c->stream);
    c->pending.push_back(t);
}

void time_end(sphgpu_ctx *c)
{
    if (!c->timing_open || c->pending.empty()) return;
    c->timing_open = false;
    hipEventRecord(c->pending.back().b, c->stream);
}

void collect_times(sphgpu_ctx *c)
{
    if (c->pending.empty()) return;
    hipEventSynchronize(c->pending.back().b);
    for (auto &t : c->pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, t.a, t.b) == hipSuccess) {
            auto &e = c->ktimes[t.name];
            e.first += ms;
            e.second += 1;
        }
        c->event_pool.push_back(t.a);
        c->event_pool.push_back(t.b);
    }
    c->pending.clear();
}

template <> RecView<float> rec_view<float>(sphgpu_ctx *c)
{
    RecView<float> v;
    for (int r = 0; r < R_NREC; ++r) v.r[r] = c->rec32[r];
    return v;
}

template <> RecView<double> rec_view<double>(sphgpu_ctx *c)
{
    RecView<double> v;
    for (int r = 0; r < R_NREC; ++r) v.r[r] = c->rec64[r];
    return v;
}

} // namespace sphgpu

// --------------------------------------------------------------------------
// plain copy of known size (counter calibration and attainable bandwidth)
__global__ __launch_bounds__(256) void k_copy_probe(const float4 *__restrict__ src, float4 *__restrict__ dst,
                                                   long long n16)
{
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n16; k += (long long)gridDim.x * blockDim.x)
        dst[k] = src[k];
}

// --------------------------------------------------------------------------
// host-exchange kernels: the masked rows, one after the other, in id order
struct FieldPtrs {
    double *p[SPHGPU_NFIELDS];
    int *ip[SPHGPU_NFIELDS];
};

__global__ void k_gather_fields(FieldPtrs dst, const double *__restrict__ stage, const int *__restrict__ id,
                                int n, unsigned long long mask)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int src = id[k];
    for (int f = 0; f < SPHGPU_NFIELDS; ++f) {
        if (!(mask & (1ull << f))) continue;
        const double v = *(stage + src);
        stage += n;
        if (dst.p[f]) dst.p[f][k] = v;
        else if (dst.ip[f]) dst.ip[f][k] = (int)v;
    }
}

__global__ void k_scatter_fields(FieldPtrs src, double *__restrict__ stage, const int *__restrict__ id, int n,
                                 unsigned long long mask)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int dst = id[k];
    for (int f = 0; f < SPHGPU_NFIELDS; ++f) {
        if (!(mask & (1ull << f))) continue;
        double v = 0.0;
        if (src.p[f]) v = src.p[f][k];
        else if (src.ip[f]) v = (double)src.ip[f][k];
        stage[dst] = v;
        stage += n;
    }
}

__global__ void k_iota(int *a, int n)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) a[k] = k;
}

static FieldPtrs field_ptrs(sphgpu_ctx *c)
{
    FieldPtrs f;
    for (int i = 0; i < SPHGPU_NFIELDS; ++i) { f.p[i] = nullptr; f.ip[i] = nullptr; }
    for (int k = 0; k < c->dim; ++k) {
        f.p[SPHGPU_F_POS + k] = c->pos[k];
        f.p[SPHGPU_F_VEL + k] = c->vel[k];
        f.p[SPHGPU_F_VEL_P + k] = c->vel_p[k];
        f.p[SPHGPU_F_ACC + k] = c->acc[k];
        f.p[SPHGPU_F_GRAD_D + k] = c->grad[k];
        f.p[SPHGPU_F_GRAD_P + k] = c->grad[3 + k];
        for (int a = 0; a < c->dim; ++a) f.p[SPHGPU_F_GRAD_V + 3 * a + k] = c->grad[6 + 3 * a + k];
    }
    const int smap[S_NSCALAR] = {SPHGPU_F_MASS, SPHGPU_F_DENS, SPHGPU_F_PRES, SPHGPU_F_ENE, SPHGPU_F_ENE_P,
                                 SPHGPU_F_DENE, SPHGPU_F_SML, SPHGPU_F_SOUND, SPHGPU_F_BALSARA, SPHGPU_F_ALPHA,
                                 SPHGPU_F_GRADH, SPHGPU_F_PHI};
    for (int s = 0; s < S_NSCALAR; ++s) f.p[smap[s]] = c->sc[s];
    f.ip[SPHGPU_F_NEIGHBOR] = c->neighbor;
    return f;
}

// --------------------------------------------------------------------------
// Pinned memory of the host exchange, two halves, shared by the contexts of the
// process: one exchange has it at a time and another one that comes meanwhile
// copies its rows directly.  It is set up when a context exchanges rows for the
// third time and freed with the last context: pinned pages cost 0.4 us per KB
// when they are first written and 0.3 ms to have (memory of each context's own
// made the first upload of 65k particles 1.0 ms instead of 0.25 and the creation
// of a context up to twice as long), which a program that uploads, runs and
// downloads once does not get back.  4 MB a half: with 2 MB the rows of 1M
// particles came back as fast, but the program's 16 threads that converted them
// right after took 10 to 45 ms in a third of the passes instead of 1 to 3.
constexpr size_t kBounceHalf = 4u << 20;
constexpr int kBounceAfter = 2;  // exchanges of a context without it

namespace {
struct Bounce {
    std::mutex lock;
    char *mem = nullptr;
    int users = 0;
} g_bounce;

void bounce_enter()
{
    std::lock_guard<std::mutex> l(g_bounce.lock);
    ++g_bounce.users;
}

void bounce_leave()
{
    std::lock_guard<std::mutex> l(g_bounce.lock);
    if (--g_bounce.users > 0 || !g_bounce.mem) return;
    hipHostFree(g_bounce.mem);
    g_bounce.mem = nullptr;
}

// the halves for one exchange of a context, given back when its stream is idle
class BounceHold {
    std::unique_lock<std::mutex> l;
    hipStream_t stream = nullptr;

public:
    bool take(sphgpu_ctx *c)
    {
        l = std::unique_lock<std::mutex>(g_bounce.lock, std::try_to_lock);
        if (!l.owns_lock()) return false;
        stream = c->stream;
        if (!g_bounce.mem && c->exchanges++ >= kBounceAfter &&
            hipHostMalloc((void **)&g_bounce.mem, 2 * kBounceHalf, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            g_bounce.mem = nullptr;
            c->exchanges = 0;
        }
        if (!g_bounce.mem) l.unlock();
        return l.owns_lock();
    }
    char *mem() const { return g_bounce.mem; }
    // after the stream was waited for (a call that fails before leaves that here)
    void give_back()
    {
        if (l.owns_lock()) l.unlock();
    }
    ~BounceHold()
    {
        if (l.owns_lock()) hipStreamSynchronize(stream);
    }
};
} // namespace

extern "C" {

void sphgpu_params_default(sphgpu_params *p, int dim)
{
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->dim = dim;
    p->sph_type = SPHGPU_SSPH;
    p->kernel = SPHGPU_CUBIC_SPLINE;
    p->riemann_solver = SPHGPU_RIEMANN_HLL;
    p->neighbor_number = 50;
    p->leaf_particle_num = 1;
    p->max_tree_level = 20;
    p->iterative_sml = 1;
    p->use_balsara_switch = 1;
    p->use_time_dependent_av = 0;
    p->use_ac = 0;
    p->periodic = 0;
    p->use_gravity = 0;
    p->gsph_2nd_order = 1;
    p->pair_precision = SPHGPU_PAIR_FP32;
    p->riemann_guess = SPHGPU_GUESS_PLAIN;
    p->gamma = 1.6666666666666667;
    p->cfl_sound = 0.3;
    p->cfl_force = 0.125;
    p->av_alpha = 1.0;
    p->alpha_max = 2.0;
    p->alpha_min = 0.1;
    p->epsilon_av = 0.2;
    p->alpha_ac = 1.0;
    p->gravity_constant = 1.0;
    p->theta = 0.5;
}

int sphgpu_device_info(char *name, int name_len, int *cu_count, double *hbm_gb)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return SPHGPU_E_HIP;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return SPHGPU_E_HIP;
    if (name && name_len > 0) {
        std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (cu_count) *cu_count = prop.multiProcessorCount;
    if (hbm_gb) *hbm_gb = (double)prop.totalGlobalMem / (1024.0 * 1024.0 * 1024.0);
    return 0;
}

static int check_params(const sphgpu_params *p, std::string &why)
{
    if (p->dim < 1 || p->dim > 3) { why = "dim must be 1, 2 or 3"; return 0; }
    if (p->sph_type < SPHGPU_SSPH || p->sph_type > SPHGPU_GDISPH) { why = "unsupported SPHType"; return 0; }
    if (p->kernel < SPHGPU_CUBIC_SPLINE || p->kernel > SPHGPU_GAUSSIAN) { why = "unknown kernel"; return 0; }
    if (p->kernel == SPHGPU_WENDLAND && p->dim == 1) { why = "Wendland C4 is undefined in 1D"; return 0; }
    const int bits = p->dim;
    if (p->max_tree_level < 1 || p->max_tree_level * bits > 63) { why = "maxTreeLevel too deep for 64-bit keys"; return 0; }
    if (p->leaf_particle_num < 1 || p->leaf_particle_num > 4096) { why = "leafParticleNumber out of range"; return 0; }
    if (p->neighbor_number < 1) { why = "neighborNumber must be positive"; return 0; }
    return 1;
}

int sphgpu_create(const sphgpu_params *p, int n, sphgpu_ctx **out)
{
    if (!p || !out || n <= 0) return SPHGPU_E_ARG;
    std::string why;
    if (!check_params(p, why)) { *out = nullptr; return SPHGPU_E_ARG; }
    sphgpu_ctx *c = new sphgpu_ctx;
    bounce_enter();
    c->prm = *p;
    c->n = n;
    c->dim = p->dim;
    c->box.periodic = p->periodic;
    for (int k = 0; k < 3; ++k) {
        c->box.lo[k] = p->range_min[k];
        c->box.hi[k] = p->range_max[k];
        c->box.range[k] = p->range_max[k] - p->range_min[k];
        c->box.rangef[k] = (float)c->box.range[k];
        c->box.rinvf[k] = c->box.range[k] > 0.0 ? (float)(1.0 / c->box.range[k]) : 0.f;
    }
    auto alloc = [&](void **ptr, size_t bytes) -> bool {
        if (hipMalloc(ptr, bytes) != hipSuccess) return false;
        return hipMemset(*ptr, 0, bytes) == hipSuccess;
    };
    bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess;
    const size_t dn = sizeof(double) * (size_t)n;
    for (int k = 0; k < 3 && ok; ++k) {
        ok = ok && alloc((void **)&c->pos[k], dn) && alloc((void **)&c->vel[k], dn) &&
             alloc((void **)&c->vel_p[k], dn) && alloc((void **)&c->acc[k], dn);
    }
    for (int s = 0; s < S_NSCALAR && ok; ++s) ok = alloc((void **)&c->sc[s], dn);
    for (int g = 0; g < kNGrad && ok; ++g) ok = alloc((void **)&c->grad[g], dn);
    for (int a = 0; a < kAlt && ok; ++a) ok = hipMalloc((void **)&c->alt[a], dn) == hipSuccess;  // written before read
    ok = ok && alloc((void **)&c->id, sizeof(int) * n) && alloc((void **)&c->id_alt, sizeof(int) * n) &&
         alloc((void **)&c->neighbor, sizeof(int) * n);
    for (int r = 0; r < R_NREC && ok; ++r) ok = alloc((void **)&c->rec32[r], sizeof(float4) * (size_t)n);
    if (p->pair_precision == SPHGPU_PAIR_FP64)
        for (int r = 0; r < R_NREC && ok; ++r) ok = alloc((void **)&c->rec64[r], sizeof(double4) * (size_t)n);
    ok = ok && alloc((void **)&c->hs, dn) && hipMalloc((void **)&c->stage, dn * SPHGPU_NFIELDS) == hipSuccess;
    for (auto &e : c->bounce_moved) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (p->use_time_dependent_av) ok = ok && alloc((void **)&c->alpha_snap, dn);
    c->red_blocks = 1024;
    ok = ok && alloc((void **)&c->red, sizeof(double) * 8 * c->red_blocks);
    ok = ok && alloc((void **)&c->dscal, sizeof(double) * 16) && alloc((void **)&c->dmin, sizeof(unsigned long long) * kStatCopies) &&
         alloc((void **)&c->dstats, sizeof(long long) * kStatSlots * kStatCopies) && alloc((void **)&c->dflag, sizeof(int) * 8);
    ok = ok && hipHostMalloc((void **)&c->hscal, sizeof(double) * 16, hipHostMallocDefault) == hipSuccess;
    ok = ok && hipHostMalloc((void **)&c->hflag, sizeof(int) * 8, hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess &&
         hipHostGetDevicePointer((void **)&c->hflag_dev, c->hflag, 0) == hipSuccess &&
         hipEventCreateWithFlags(&c->flag_ready, hipEventDisableTiming) == hipSuccess;
    ok = ok && tree_alloc(c) == 0;
    // neighbour lists: about 5x the expected candidate count nn * 1.2^D
    // (a shock compresses the gas ahead of the smoothing lengths, and a list
    // that overflows costs a second search in that step; the slot-major
    // layout touches only the slots a particle fills, so capacity costs
    // memory, 4 B per slot and particle, not traffic)
    const double kap = p->iterative_sml ? std::pow(1.2, p->dim) : 1.0;
    int cap = (int)std::ceil(p->neighbor_number * kap * 5.0 / 64.0) * 64;
    cap = std::max(cap, 64);
    ok = ok && lists_alloc(c, c->lpre, cap) == 0 && lists_alloc(c, c->lforce, cap) == 0;
    ok = ok && mlp_create(c) == 0;
    if (!ok) {
        sphgpu_destroy(c);
        *out = nullptr;
        return SPHGPU_E_NOMEM;
    }
    hipLaunchKernelGGL(k_iota, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, c->id, n);
    hipStreamSynchronize(c->stream);
    *out = c;
    return 0;
}

int sphgpu_destroy(sphgpu_ctx *c)
{
    if (!c) return SPHGPU_E_ARG;
    if (c->stream) hipStreamSynchronize(c->stream);
    for (int k = 0; k < 3; ++k) {
        hipFree(c->pos[k]); hipFree(c->vel[k]); hipFree(c->vel_p[k]); hipFree(c->acc[k]);
    }
    for (int s = 0; s < S_NSCALAR; ++s) hipFree(c->sc[s]);
    for (int g = 0; g < kNGrad; ++g) hipFree(c->grad[g]);
    for (int a = 0; a < kAlt; ++a) hipFree(c->alt[a]);
    hipFree(c->id); hipFree(c->id_alt); hipFree(c->neighbor);
    for (int r = 0; r < R_NREC; ++r) {
        hipFree(c->rec32[r]);
        hipFree(c->rec64[r]);
    }
    hipFree(c->hs); hipFree(c->alpha_snap); hipFree(c->stage); hipFree(c->red);
    hipFree(c->dscal); hipFree(c->dmin); hipFree(c->dstats); hipFree(c->dflag);
    bounce_leave();
    for (auto e : c->bounce_moved)
        if (e) hipEventDestroy(e);
    if (c->hscal) hipHostFree(c->hscal);
    if (c->hflag) hipHostFree(c->hflag);
    if (c->flag_ready) hipEventDestroy(c->flag_ready);
    tree_free(c);
    lists_free(c->lpre);
    lists_free(c->lforce);
    mlp_destroy(c);
    if (c->rlog) hipFree(c->rlog);
    if (c->rlog_count) hipFree(c->rlog_count);
    for (auto &t : c->pending) { hipEventDestroy(t.a); hipEventDestroy(t.b); }
    for (auto e : c->event_pool) hipEventDestroy(e);
    if (c->stream) hipStreamDestroy(c->stream);
    delete c;
    return 0;
}

const char *sphgpu_last_error(const sphgpu_ctx *c) { return c ? c->err.c_str() : "null context"; }

int sphgpu_get_params(const sphgpu_ctx *c, sphgpu_params *p, int32_t *n)
{
    if (!c) return SPHGPU_E_ARG;
    if (p) *p = c->prm;
    if (n) *n = c->n;
    return 0;
}

// Masked rows between the user's memory and the front of the staging block.
// A copy of pageable memory costs a pinning or a staging of its own per row, one
// after the other: the rows go through two halves of pinned memory instead, the
// DMA of one running while the other is copied.  Download of 14 rows of 1M
// particles 6.1 -> 3.9 ms, 7 rows of 133k 510 -> 310 us, of 16k 134 -> 68; upload
// of 14 rows of 133k 560 -> 445 us, of 16k 178 -> 95 (1M the same, 3.8 ms).
// Copying with three helper threads took half of that at 1M and 10 ms more at
// 133k where the process shares its cores: one thread does it.
namespace {
struct RowRange {
    double *row[SPHGPU_NFIELDS];
    size_t row_bytes;
    // bytes [a, b) of the rows taken one after the other, at buf + (a - base)
    void copy(char *buf, size_t base, size_t a, size_t b, bool up) const
    {
        while (a < b) {
            const size_t r = a / row_bytes, off = a % row_bytes;
            const size_t len = std::min(b - a, row_bytes - off);
            char *const user = reinterpret_cast<char *>(row[r]) + off;
            if (up) std::memcpy(buf + (a - base), user, len);
            else std::memcpy(user, buf + (a - base), len);
            a += len;
        }
    }
};

// One row gains nothing from the pinned halves but the shorter wait of a small
// download (500 particles 23 -> 16 us) and the copies of a large one (400k 205 ->
// 170 us); between them, and for uploads, HIP's own copy is the faster: upload
// 21 us against 25 at 500, 29 / 32 at 16k, 150 / 167 at 400k; download 25 / 30 at
// 5000, 36 / 42 at 40k, 84 / 80 at 133k.  Two large rows up are like one (133k 112 /
// 119, 400k 240 / 275) and so are two of 16 KB (25 / 31), others not (5000 37 / 30).
constexpr size_t kRowTiny = 16u << 10, kRowSmall = 32u << 10, kRowLarge = 512u << 10;
bool copy_rows_directly(int count, size_t row_bytes, bool up)
{
    if (up) return count == 1 || (count == 2 && (row_bytes <= kRowTiny || row_bytes >= kRowLarge));
    return count == 1 && row_bytes > kRowSmall && row_bytes < kRowLarge;
}

// memory that HIP knows (pinned, managed or device) is copied as it is
bool known_to_hip(const void *p)
{
    if (hipPeekAtLastError() != hipSuccess) return true;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// `hold` has the pinned halves when they are in use; the caller keeps it until
// its stream is idle
int exchange_rows(sphgpu_ctx *c, double *fields, uint64_t mask, bool up, BounceHold &hold)
{
    RowRange rows;
    rows.row_bytes = sizeof(double) * (size_t)c->n;
    int count = 0;
    for (int f = 0; f < SPHGPU_NFIELDS; ++f)
        if (mask & SPHGPU_MASK(f)) rows.row[count++] = fields + (size_t)f * c->n;
    if (count == 0) return 0;
    const size_t total = rows.row_bytes * count;
    if (copy_rows_directly(count, rows.row_bytes, up) || known_to_hip(fields) || !hold.take(c)) {
        for (int r = 0; r < count; ++r) {
            double *const dev = c->stage + (size_t)r * c->n;
            HIPCHK(c, up ? hipMemcpyAsync(dev, rows.row[r], rows.row_bytes, hipMemcpyHostToDevice, c->stream)
                         : hipMemcpyAsync(rows.row[r], dev, rows.row_bytes, hipMemcpyDeviceToHost, c->stream));
        }
        return 0;
    }
    // up 16 rounds, of 2 MB at least, down 8, of 1 MB: what the first and the last
    // round do alone is not hidden, and a round costs some 10 us itself (7 rows of
    // 133k up 290 us in rounds of 1 MB, 243 of 2; down 300 and 312, 336 of 4)
    const size_t least = up ? 2u << 20 : 1u << 20, part = (total / (up ? 16 : 8) + 4095) & ~(size_t)4095;
    const size_t chunk = std::min(kBounceHalf, std::max(least, part));
    const int rounds = (int)((total + chunk - 1) / chunk);
    char *const dev = reinterpret_cast<char *>(c->stage);
    auto dma = [&](int r) {
        const size_t a = (size_t)r * chunk, len = std::min(chunk, total - a);
        char *const host = hold.mem() + (r & 1) * kBounceHalf;
        const hipError_t e = up ? hipMemcpyAsync(dev + a, host, len, hipMemcpyHostToDevice, c->stream)
                                : hipMemcpyAsync(host, dev + a, len, hipMemcpyDeviceToHost, c->stream);
        return e == hipSuccess ? hipEventRecord(c->bounce_moved[r & 1], c->stream) : e;
    };
    if (!up) HIPCHK(c, dma(0));
    auto copy = [&](int r) {
        const size_t a = (size_t)r * chunk;
        rows.copy(hold.mem() + (r & 1) * kBounceHalf, a, a, std::min(total, a + chunk), up);
    };
    for (int r = 0; r < rounds; ++r) {
        if (up) {
            if (r >= 2) HIPCHK(c, hipEventSynchronize(c->bounce_moved[r & 1]));
            copy(r);
            HIPCHK(c, dma(r));
        } else {
            if (r + 1 < rounds) HIPCHK(c, dma(r + 1));
            HIPCHK(c, hipEventSynchronize(c->bounce_moved[r & 1]));
            copy(r);
        }
    }
    return 0;
}
} // namespace

int sphgpu_upload(sphgpu_ctx *c, const double *fields, uint64_t mask)
{
    if (!c || !fields) return SPHGPU_E_ARG;
    mask &= SPHGPU_MASK_ALL & ~SPHGPU_MASK(SPHGPU_F_ID);
    BounceHold hold;
    int rc = exchange_rows(c, const_cast<double *>(fields), mask, true, hold);
    if (rc) return rc;
    FieldPtrs fp = field_ptrs(c);
    hipLaunchKernelGGL(k_gather_fields, dim3(grid_for(c->n, 256)), dim3(256), 0, c->stream, fp,
                       (const double *)c->stage, (const int *)c->id, c->n, (unsigned long long)mask);
    HIPCHK(c, hipGetLastError());
    if (mask & SPHGPU_MASK(SPHGPU_F_MASS)) {
        // masses are inputs only: whether they are all equal is decided here
        const double *m = fields + (size_t)SPHGPU_F_MASS * c->n;
        bool same = c->n > 0;
        for (int p = 0; same && p < c->n; p += 4096) {
            int differ = 0;
            for (int q = p; q < std::min(p + 4096, c->n); ++q) differ |= m[q] != m[0];
            same = !differ;
        }
        c->mass_uniform = same;
        c->mass_u = c->n > 0 ? m[0] : 0.0;
    }
    // new positions make the tree stale (BHTree::make runs again before the
    // next search); any host change of inputs invalidates the FP32 mirrors
    // and with them a derived force list
    const uint64_t pos_rows = SPHGPU_MASK(SPHGPU_F_POS) | SPHGPU_MASK(SPHGPU_F_POS + 1) | SPHGPU_MASK(SPHGPU_F_POS + 2);
    if (mask & pos_rows) c->tree.valid = false;
    const bool ok = refresh_mirrors(c) == 0;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    hold.give_back();
    return ok ? 0 : SPHGPU_E_HIP;
}

int sphgpu_download(sphgpu_ctx *c, double *fields, uint64_t mask)
{
    if (!c || !fields) return SPHGPU_E_ARG;
    mask &= SPHGPU_MASK_ALL;
    FieldPtrs fp = field_ptrs(c);
    fp.ip[SPHGPU_F_ID] = c->id;
    hipLaunchKernelGGL(k_scatter_fields, dim3(grid_for(c->n, 256)), dim3(256), 0, c->stream, fp, c->stage,
                       (const int *)c->id, c->n, (unsigned long long)mask);
    HIPCHK(c, hipGetLastError());
    BounceHold hold;
    int rc = exchange_rows(c, fields, mask, false, hold);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    hold.give_back();
    return 0;
}

static int get_scalar(sphgpu_ctx *c, int idx, double *v)
{
    if (!c || !v) return SPHGPU_E_ARG;
    HIPCHK(c, hipMemcpyAsync(c->hscal + idx, c->dscal + idx, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    *v = c->hscal[idx];
    return 0;
}

static int set_scalar(sphgpu_ctx *c, int idx, double v)
{
    if (!c) return SPHGPU_E_ARG;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->hscal[idx] = v;
    HIPCHK(c, hipMemcpyAsync(c->dscal + idx, c->hscal + idx, sizeof(double), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int sphgpu_set_dt(sphgpu_ctx *c, double dt) { return set_scalar(c, 0, dt); }
int sphgpu_get_dt(sphgpu_ctx *c, double *dt) { return get_scalar(c, 0, dt); }
int sphgpu_set_time(sphgpu_ctx *c, double t) { return set_scalar(c, 1, t); }
int sphgpu_get_time(sphgpu_ctx *c, double *t) { return get_scalar(c, 1, t); }
int sphgpu_get_h_per_v_sig(sphgpu_ctx *c, double *v) { return get_scalar(c, 2, v); }
int sphgpu_set_h_per_v_sig(sphgpu_ctx *c, double v) { return set_scalar(c, 2, v); }

#define CTX_CALL(expr)                                   \
    do {                                                 \
        if (!c) return SPHGPU_E_ARG;                     \
        int rc_ = (expr);                                \
        if (rc_) return rc_;                             \
        HIPCHK(c, hipStreamSynchronize(c->stream));      \
        collect_times(c);                                \
        return 0;                                        \
    } while (0)

int sphgpu_build_tree(sphgpu_ctx *c) { CTX_CALL(tree_build(c)); }
int sphgpu_set_kernel(sphgpu_ctx *c) { CTX_CALL(tree_set_kernel(c)); }
int sphgpu_pre_interaction(sphgpu_ctx *c) { CTX_CALL(pre_interaction(c)); }
int sphgpu_fluid_force(sphgpu_ctx *c) { CTX_CALL(fluid_force(c)); }
int sphgpu_gravity(sphgpu_ctx *c) { CTX_CALL(gravity(c)); }
int sphgpu_timestep(sphgpu_ctx *c) { CTX_CALL(timestep(c)); }
int sphgpu_predict(sphgpu_ctx *c) { CTX_CALL(predict(c)); }
int sphgpu_correct(sphgpu_ctx *c) { CTX_CALL(correct(c)); }

static int initialize_impl(sphgpu_ctx *c)
{
    int rc;
    if ((rc = init_fields(c))) return rc;
    if ((rc = tree_build(c))) return rc;
    if ((rc = pre_interaction(c))) return rc;
    if ((rc = fluid_force(c))) return rc;
    return gravity(c);
}

int sphgpu_initialize(sphgpu_ctx *c) { CTX_CALL(initialize_impl(c)); }

static int integrate_impl(sphgpu_ctx *c, int nsteps)
{
    int rc;
    for (int s = 0; s < nsteps; ++s) {
        if ((rc = timestep(c))) return rc;
        if ((rc = predict(c))) return rc;
        c->in_step = true;
        rc = tree_build(c);
        c->in_step = false;
        if (rc) return rc;
        if ((rc = pre_interaction_deferred(c))) return rc;
        if ((rc = fluid_force(c))) return rc;  // settles the deferred search first
        if ((rc = gravity(c))) return rc;
        if ((rc = correct(c, true))) return rc;
    }
    return 0;
}

int sphgpu_integrate(sphgpu_ctx *c, int nsteps) { CTX_CALL(integrate_impl(c, nsteps)); }

int sphgpu_energy_momentum(sphgpu_ctx *c, double out[7])
{
    if (!c || !out) return SPHGPU_E_ARG;
    return energy_momentum(c, out);
}

int sphgpu_get_stats(sphgpu_ctx *c, sphgpu_stats *out)
{
    if (!c || !out) return SPHGPU_E_ARG;
    std::vector<long long> all((size_t)kStatSlots * kStatCopies);
    HIPCHK(c, hipMemcpyAsync(all.data(), c->dstats, sizeof(long long) * all.size(), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    // sum the copies (slot 12, the tree depth, is a maximum)
    long long h[kStatSlots] = {};
    for (int k = 0; k < kStatCopies; ++k)
        for (int s = 0; s < kStatSlots; ++s) {
            const long long v = all[(size_t)k * kStatSlots + s];
            h[s] = (s == 12) ? std::max(h[s], v) : h[s] + v;
        }
    std::memset(out, 0, sizeof(*out));
    out->pre_candidates = h[0];
    out->pre_newton_iters = h[1];
    out->pre_newton_fail = h[2];
    out->force_pairs = h[3];
    out->force_candidates = h[4];
    out->riemann_iters = h[5];
    out->riemann_wave_max_iters = h[6];
    out->riemann_calls = h[7];
    out->riemann_fallbacks = h[8];
    out->riemann_learned = h[9];
    out->gravity_interactions = h[10];
    out->nodes = c->tree.n_nodes;
    out->leaves = h[11];
    out->max_depth = (int32_t)h[12];
    out->search_node_visits = h[13];
    out->search_member_tests = h[14];
    out->search_windows = h[15];
    out->search_leaves = h[16];
    out->search_exact = h[17];
    out->flist_h_beyond = h[18];
    out->flist_other = h[19];
    out->flist_searches = c->flist_searches;
    out->search_reach_tests = h[20];
    return 0;
}

int sphgpu_reset_stats(sphgpu_ctx *c)
{
    if (!c) return SPHGPU_E_ARG;
    HIPCHK(c, hipMemsetAsync(c->dstats, 0, sizeof(long long) * kStatSlots * kStatCopies, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->flist_searches = 0;
    return 0;
}

int sphgpu_neighbor_sets(sphgpu_ctx *c, const double *h, int is_ij, int cap, int32_t *counts, int32_t *lists)
{
    if (!c || !counts || !lists || cap <= 0 || is_ij < 0 || is_ij > 2 || (is_ij != 2 && !h)) return SPHGPU_E_ARG;
    if (!c->tree.valid) return fail(c, SPHGPU_E_STATE, "neighbor_sets needs a built tree");
    int rc;
    if (is_ij == 2) {
        // the force pair lists the last pre-interaction derived
        if ((rc = flist_check(c)) < 0) return rc;
        if (rc) return fail(c, SPHGPU_E_STATE, "neighbor_sets: no force pair list from a pre-interaction");
    } else {
        // smoothing lengths in id order -> sorted order
        std::vector<double> stage((size_t)c->n * SPHGPU_NFIELDS, 0.0);
        std::memcpy(stage.data() + (size_t)SPHGPU_F_SML * c->n, h, sizeof(double) * c->n);
        if ((rc = sphgpu_upload(c, stage.data(), SPHGPU_MASK(SPHGPU_F_SML)))) return rc;
        if ((rc = tree_set_kernel(c))) return rc;
        // pre-interaction radius: h itself (r2 < h^2, src/bhtree.cpp:280-299)
        HIPCHK(c, hipMemcpyAsync(c->hs, c->sc[S_SML], sizeof(double) * c->n, hipMemcpyDeviceToDevice, c->stream));
        if ((rc = search(c, is_ij ? c->lforce : c->lpre, is_ij, c->hs))) return rc;
    }
    Lists &l = is_ij ? c->lforce : c->lpre;
    const size_t list_len = (size_t)l.cap * (((size_t)c->n + 63) / 64) * 64;
    std::vector<int> ids(c->n), cnt(c->n), idx(list_len);
    HIPCHK(c, hipMemcpyAsync(ids.data(), c->id, sizeof(int) * c->n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipMemcpyAsync(cnt.data(), l.cnt, sizeof(int) * c->n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipMemcpyAsync(idx.data(), l.idx, sizeof(int) * list_len, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (int k = 0; k < c->n; ++k) {
        const int i = ids[k];
        const int m = cnt[k];
        if (m > cap) return fail(c, SPHGPU_E_NEIGHBOR_OVERFLOW, "neighbor_sets: cap too small");
        counts[i] = m;
        for (int s = 0; s < m; ++s) lists[(size_t)i * cap + s] = ids[idx[list_slot(k, s, l.cap)]];
    }
    return 0;
}

int sphgpu_tree_dump(sphgpu_ctx *c, int64_t *n_nodes, int32_t *level, int32_t *count, int32_t *first,
                     int32_t *is_leaf, double *center, double *edge, double *mass, double *com,
                     double *kernel_size, int32_t *members)
{
    if (!c || !n_nodes) return SPHGPU_E_ARG;
    return tree_dump(c, n_nodes, level, count, first, is_leaf, center, edge, mass, com, kernel_size, members);
}

int sphgpu_riemann_batch(sphgpu_ctx *c, int solver, int precision, int n, const double *left, const double *right,
                         double *pstar, double *vstar, int32_t *iters, int32_t *learned_used)
{
    if (!c || n < 0 || (n > 0 && (!left || !right || !pstar || !vstar))) return SPHGPU_E_ARG;
    if (n == 0) return 0;
    return riemann_batch(c, solver, precision, n, left, right, pstar, vstar, iters, learned_used);
}

int sphgpu_riemann_batch_static(sphgpu_ctx *c, int solver, int precision, int n, const double *left,
                                const double *right, double *pstar, double *vstar, int32_t *iters,
                                int32_t *learned_used)
{
    if (!c || n < 0 || (n > 0 && (!left || !right || !pstar || !vstar))) return SPHGPU_E_ARG;
    if (n == 0) return 0;
    return riemann_batch_static(c, solver, precision, n, left, right, pstar, vstar, iters, learned_used);
}

int sphgpu_enable_timing(sphgpu_ctx *c, int on)
{
    if (!c) return SPHGPU_E_ARG;
    collect_times(c);
    c->timing = on < 0 ? 0 : on > 2 ? 1 : on;
    c->ktimes.clear();
    return 0;
}

int sphgpu_kernel_times(sphgpu_ctx *c, char *name_buf, int buf_len, double *avg_ms, int64_t *count, int max_kernels,
                        int *n_kernels)
{
    if (!c || !name_buf || buf_len <= 0 || !n_kernels) return SPHGPU_E_ARG;
    collect_times(c);
    std::string names;
    int k = 0;
    for (auto &kv : c->ktimes) {
        if (k >= max_kernels) break;
        if (avg_ms) avg_ms[k] = kv.second.first / (double)std::max(1LL, kv.second.second);
        if (count) count[k] = kv.second.second;
        names += kv.first;
        names += ";";
        ++k;
    }
    std::snprintf(name_buf, buf_len, "%s", names.c_str());
    *n_kernels = k;
    return 0;
}

int sphgpu_copy_probe(sphgpu_ctx *c, int64_t nbytes, double *ms)
{
    if (!c || !ms || nbytes < 16) return SPHGPU_E_ARG;
    const long long n16 = nbytes / 16;
    float4 *src = nullptr, *dst = nullptr;
    HIPCHK(c, hipMalloc((void **)&src, 16ull * n16));
    HIPCHK(c, hipMalloc((void **)&dst, 16ull * n16));
    HIPCHK(c, hipMemsetAsync(src, 0, 16ull * n16, c->stream));
    hipEvent_t e0, e1;
    HIPCHK(c, hipEventCreate(&e0));
    HIPCHK(c, hipEventCreate(&e1));
    const int blocks = 4096;
    hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, c->stream, (const float4 *)src, dst, n16);
    HIPCHK(c, hipEventRecord(e0, c->stream));
    hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, c->stream, (const float4 *)src, dst, n16);
    HIPCHK(c, hipEventRecord(e1, c->stream));
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventSynchronize(e1));
    float t = 0.f;
    HIPCHK(c, hipEventElapsedTime(&t, e0, e1));
    *ms = t;
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipFree(src);
    hipFree(dst);
    return 0;
}

} // extern "C"
