// The launches the C ABI makes, recorded on the CPU (tests/test_launch_geometry.py builds and runs
// this; it holds no device code). The program exports the HIP runtime functions that
// libluminav_hip.so imports, so a call runs the library's whole host path and ends in the recorder
// below instead of on a device. The kernel of a launch is known by the name its function was
// registered under, whose template arguments fix its threads per block, work unit and option word.
// For every mode, dtype, option, pass, entry point and launch kind the recorded launch must be the
// one its kernel was built for.
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "luminav_hip.h"
#include "lv_device.h"

struct Kernel {
    int mode = 0, pt = 0, st = 0, pass = 0, table = 0;
    uint32_t fl = 0;
    bool unit = false;  // a unit kernel (else a fold, fill or step record kernel)
};

struct Launch {
    Kernel k;
    uint32_t grid = 0, threads = 0, lds = 0;
    lv::Args args;
};

static std::map<const void *, std::string> g_names;
static std::vector<Launch> g_launches;
static std::vector<void *> g_buffers;  // pretended device and pinned memory
alignas(256) static char g_symbol[4 << 20];
static dim3 g_grid, g_block;

// ------------------------------------------------------------------ the HIP runtime, recorded

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 8; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(1, n); g_buffers.push_back(*p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void *) { return hipSuccess; }  // kept: recorded launches may point into it
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)(uintptr_t)1; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = g_symbol; return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *h = nullptr; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    g_names[fn] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { g_grid = g; g_block = b; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = g_grid; *b = g_block; *s = 0; *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t) {
    Launch l;
    const std::string &name = g_names[fn];
    l.k.unit = std::sscanf(name.c_str(), "_ZN2lv11unit_kernelILi%dELi%dELi%dELi%dELj%uELb%dE", &l.k.mode, &l.k.pt, &l.k.st,
                           &l.k.pass, &l.k.fl, &l.k.table) == 6;
    l.grid = grid.x;
    l.threads = block.x;
    l.lds = (uint32_t)lds;
    if (l.k.unit) l.args = *static_cast<const lv::Args *>(args[0]);
    g_launches.push_back(l);
    return hipSuccess;
}
}

// ------------------------------------------------------------------ calls and checks

using MultiFn = int (*)(const lv_config *, const lv_tensor *, int, void *, size_t, void *);
using NoAllocFn = int (*)(const lv_config *, const lv_tensor *, int, void *);
using GraphFn = int (*)(const lv_config *, const lv_tensor *, int, lv_step_record *, void *, size_t, void *);
using BytesFn = size_t (*)(const lv_config *, const lv_tensor *, int);
using ErrFn = const char *(*)(void);
static MultiFn f_multi;
static NoAllocFn f_noalloc;
static GraphFn f_graph;
static BytesFn f_bytes;
static ErrFn f_error;

enum Entry { kMulti, kNoAlloc, kGraph };
static long g_calls, g_checked, g_bad, g_large, g_one_wave;
static std::string g_case;

static bool check(bool ok, const char *what, const Launch *l = nullptr) {
    if (ok) return true;
    if (g_bad++ < 20) {
        std::printf("MISMATCH %s: %s", g_case.c_str(), what);
        if (l)
            std::printf(" (kernel mode %d params %d state %d pass %d flags 0x%x %s, %u threads, grid %u)", l->k.mode, l->k.pt,
                        l->k.st, l->k.pass, l->k.fl, l->k.table ? "table" : "inline", l->threads, l->grid);
        std::printf("\n");
    }
    return false;
}

static int bytes_of(int dt) { return dt == LV_DTYPE_F32 ? 4 : 2; }

// The option word of a pass's arithmetic, from the call's config and a tensor of the class.
static uint32_t wanted_word(const lv_config &c, const lv_tensor &t, int bound, bool master) {
    uint32_t f = (uint32_t)t.grad_dtype << 8;
    if (c.cautious) f |= lv::kFCautious;
    if (c.stochastic_rounding) f |= lv::kFSR;
    if (master) f |= lv::kFMaster;
    if (c.weight_decay != 0.0f) f |= lv::kFWeightDecay;
    if (t.param_dtype == LV_DTYPE_F16) f |= lv::kFClampV;
    if (bound == LV_BOUND_COORDINATE) f |= lv::kFCoordinate;
    if (bound == LV_BOUND_RADIAL) f |= lv::kFRadial;
    return f;
}

// One tensor's buffers: disjoint pretended addresses, `off` elements into an aligned start.
static lv_tensor tensor(int i, uint64_t n, int pt, int gt, int st, bool dual, bool master, uint64_t off, uint64_t goff) {
    lv_tensor t;
    std::memset(&t, 0, sizeof t);
    const uintptr_t base = (uintptr_t)(i + 1) << 34;
    auto at = [&](int k, int dt, uint64_t o) { return (void *)(base + ((uintptr_t)k << 30) + o * (uintptr_t)bytes_of(dt)); };
    t.param = at(0, pt, off);
    t.grad = at(1, gt, goff);
    t.exp_avg = at(2, st, off);
    t.exp_avg_sq = dual ? at(3, st, off) : nullptr;
    t.master_param = master ? (float *)at(4, LV_DTYPE_F32, off) : nullptr;
    t.scratch = (float *)at(5, LV_DTYPE_F32, 0);
    t.numel = n;
    t.param_index = (uint64_t)i;
    t.param_dtype = pt;
    t.grad_dtype = gt;
    t.state_dtype = st;
    return t;
}

static void check_call(const lv_config &c, std::vector<lv_tensor> &T, Entry entry, uint64_t step, uint64_t radial_limit) {
    static std::vector<char> ws_mem;
    for (lv_tensor &t : T) t.step = step;
    const size_t need = f_bytes(&c, T.data(), (int)T.size());
    if (ws_mem.size() < need + 512) ws_mem.assign(need + 512, 0);
    char *ws = (char *)(((uintptr_t)ws_mem.data() + 255) & ~(uintptr_t)255);
    size_t ws_bytes = need;
    static lv_step_record rec;
    g_launches.clear();
    g_calls++;
    int rc;
    if (entry == kMulti) rc = f_multi(&c, T.data(), (int)T.size(), ws, need, nullptr);
    else if (entry == kGraph) rc = f_graph(&c, T.data(), (int)T.size(), &rec, ws, need, nullptr);
    else {
        rc = f_noalloc(&c, T.data(), (int)T.size(), nullptr);
        ws = g_symbol;
        ws_bytes = sizeof g_symbol;
    }
    const int bound = (c.bound && c.bound_ratio > 0.0f) ? c.bound_type : LV_BOUND_NONE;
    uint64_t all = 0;
    for (const lv_tensor &t : T) all += t.numel;
    if (entry == kNoAlloc && bound == LV_BOUND_RADIAL && all / 1024 >= radial_limit) {
        check(rc == LV_STATUS_INVALID_CONFIG || rc == LV_STATUS_SUCCESS, "a radial call above the no-allocation limit");
        if (rc != LV_STATUS_SUCCESS) return;
    }
    if (!check(rc == LV_STATUS_SUCCESS, f_error())) return;
    const bool two = c.fused_single_pass == 0 || (entry != kGraph && step < 2);
    const int first = (!c.cautious && bound != LV_BOUND_RADIAL) ? lv::kSingle : two ? lv::kCount : lv::kFused;
    std::map<const void *, int> seen[4];  // per pass: how often each param was stepped
    uint32_t next = 0, counted = 0;
    for (const Launch &l : g_launches) {
        if (!l.k.unit) continue;
        g_checked++;
        const lv::Args &a = l.args;
        const Kernel &k = l.k;
        const uint32_t threads = (uint32_t)lv::unit_threads(k.mode, k.pt, k.st, k.pass, k.fl, k.table);
        const uint32_t unit = lv::unit_elems(k.mode, k.pt, k.st, k.pass, k.fl, k.table);
        if (!check(l.threads == threads, "threads per block are not the kernel's", &l)) continue;
        check((uint64_t)l.grid * l.threads < (1ull << 32), "grid x threads", &l);
        check(l.grid <= lv::kMaxGrid || a.xcds == 1, "grid above the block mapping's range", &l);
        check(l.lds + 256u <= 65536u, "dynamic LDS", &l);
        // pieces cover the unit space in order
        check(a.unit_base == next, "pieces do not follow each other", &l);
        next = a.unit_base + l.grid;
        check(next <= a.total_units, "blocks past the last unit", &l);
        if (next == a.total_units) next = 0;
        uint64_t units = 0, slots = 0, elems = 0;
        bool ok = true;
        for (int i = 0; i < a.ndesc && ok; i++) {
            const lv::Desc &D = k.table ? a.dtab[i].d : a.d[i];
            const lv_tensor &t = T[D.pidx];
            const bool master = c.master_weights && t.master_param;
            ok = ok && check(D.p == t.param && D.n == t.numel && (const void *)D.mp == (master ? t.master_param : nullptr),
                             "descriptor of another tensor", &l);
            ok = ok && check(k.pt == t.param_dtype && (k.st == LV_DTYPE_F32) == (t.state_dtype == LV_DTYPE_F32) && k.mode == c.buffer,
                             "kernel of other dtypes", &l);
            // whole units from the head on, every stream aligned there
            if (D.vec) {
                const uintptr_t h = D.head();
                ok = ok && check(threads == 64 || h < 64, "a 256-thread kernel reads six bits of the head", &l);
                bool al = ((uintptr_t)D.p + h * bytes_of(t.param_dtype)) % 16 == 0 || bytes_of(t.param_dtype) == 2;
                al = al && ((uintptr_t)D.p + h * bytes_of(t.param_dtype)) % 16 == 0;
                al = al && ((uintptr_t)D.g + h * bytes_of(t.grad_dtype)) % 16 == 0;
                al = al && ((uintptr_t)D.m + h * bytes_of(t.state_dtype)) % 16 == 0;
                if (D.v) al = al && ((uintptr_t)D.v + h * bytes_of(t.state_dtype)) % 16 == 0;
                if (D.mp) al = al && ((uintptr_t)D.mp + h * 4) % 16 == 0;
                ok = ok && check(al && h < t.numel, "vector layout from an unaligned element", &l);
                // one-wave kernels: whole units of every stream, where the streams agree on an offset and the
                // tensor reaches that far
                const uintptr_t e = (uintptr_t)D.p / bytes_of(t.param_dtype) % 256;
                bool same = (uintptr_t)D.g / bytes_of(t.grad_dtype) % 256 == e && (uintptr_t)D.m / bytes_of(t.state_dtype) % 256 == e;
                same = same && (!D.v || (uintptr_t)D.v / bytes_of(t.state_dtype) % 256 == e) && (!D.mp || (uintptr_t)D.mp / 4 % 256 == e);
                if (unit == 256 && same && (256 - e) % 256 < t.numel)
                    ok = ok && check(h == (256 - e) % 256, "a one-wave kernel's units do not start at whole units", &l);
            }
            const uint64_t u = (t.numel - (D.vec ? D.head() : 0) + unit - 1) / unit;
            ok = ok && check(D.unit_begin == units, "units are not the kernel's", &l);
            units += u;
            elems += t.numel;
            if (k.table) {  // the count slots and the fold slot the kernel will use
                ok = ok && check(a.dtab[i].unit_end == units, "unit end", &l);
                ok = ok && check(a.dtab[i].slot_base >= slots, "count slots of two tensors overlap", &l);
                slots = a.dtab[i].slot_base + (uint64_t)lv::launch_count_slots((uint32_t)u, unit, true) + 1;
            }
            // the arithmetic the call asked for
            const uint32_t want = wanted_word(c, t, bound, master);
            const uint32_t word = (k.fl & lv::kFDynamic) ? a.flags & ~(uint32_t)lv::kFLarge : k.fl & ~(uint32_t)lv::kFLarge;
            uint32_t mask = ~0u;  // a non-radial counting pass reads only the mask's options and the grad dtype
            if (k.pass == lv::kCount && bound != LV_BOUND_RADIAL) mask = lv::kFCautious | lv::kFClampV | lv::kFRadial | 0x300u;
            ok = ok && check((word & mask) == (want & mask), "kernel of another option word", &l);
            ok = ok && check((a.flags & (lv::kFCautious | lv::kFRadial)) == (want & (lv::kFCautious | lv::kFRadial)), "launch flags", &l);
            if (a.unit_base == 0) seen[k.pass][t.param]++;
        }
        if (!ok) continue;
        check(units == a.total_units, "total units", &l);
        // a small two-pass launch cuts its tensors (and uploads its table) once for both passes
        if (k.pass == lv::kCount) counted = unit;
        if (k.pass == lv::kApply && elems < lv::kLargeElems) check(unit == counted, "the passes' units differ", &l);
        const char *s0 = (const char *)a.slots;
        const uint64_t nslots = k.table ? slots : (uint64_t)a.ndesc * lv::kSlotWords;
        check(s0 >= ws && s0 + nslots * lv::kSlotStride * 8 <= ws + ws_bytes, "count slots outside the workspace", &l);
        // the form for large launches exactly where the kernel has one
        const uint32_t base = k.fl & ~(uint32_t)lv::kFLarge;
        const bool master = c.master_weights && T[0].master_param;
        const bool lanes = lv::unit_lanes(k.mode, k.pt, k.st, k.pass, base | lv::kFLarge);
        const uint32_t wanted = base & lv::kFDynamic ? a.flags : base;  // a dynamic kernel may stand in for a large form
        bool take = lv::unit_large(k.mode, k.pt, k.st, k.pass, wanted) && elems >= lv::kLargeElems;
        if (k.table && lv::unit_threads(k.mode, k.pt, k.st, k.pass, wanted | lv::kFLarge, true) == 64)
            take = take && elems >= (uint64_t)a.ndesc * lv::wave_table_mean(k.mode, k.pt, k.pass, master);
        // lanes take no launch whose steps would mostly fall below their range
        if (lanes) take = take && c.lr >= 0x1p-30f;
        const bool large = (k.fl & lv::kFLarge) != 0;
        check(large == take, "the large form is taken on other launches", &l);
        g_large += large;
        g_one_wave += l.threads == 64;
    }
    for (const lv_tensor &t : T) {
        int want[4] = {0, 0, 0, 0};
        want[first] = 1;
        if (first == lv::kCount) want[lv::kApply] = 1;
        for (int p = 0; p < 4; p++) check(seen[p][t.param] == want[p], "a tensor is not stepped exactly once per pass");
    }
}

static lv_config defaults(int mode, float lr, bool master) {
    lv_config c;
    std::memset(&c, 0, sizeof c);
    c.lr = lr; c.beta1 = 0.9f; c.beta2 = 0.999f; c.eps = 1e-8f; c.tau = 0.8f; c.lam = 0.3f;
    c.cautious_clamp_min = 0.5f; c.bound_ratio = 0.05f; c.ema_decay = 0.8f;
    c.buffer = mode;
    c.master_weights = master ? 2 : 0;
    c.seed = 1337;
    return c;
}

// route MODE PARAMS STATE MASTER SIZE...: the kernels of one fused step with the default options over
// tensors of these sizes, one "flags threads" line per launch.
static int route(int argc, char **argv) {
    const int mode = std::atoi(argv[3]), pt = std::atoi(argv[4]), st = std::atoi(argv[5]);
    const bool master = std::atoi(argv[6]) != 0;
    lv_config c = defaults(mode, 1e-3f, master);
    c.cautious = c.stochastic_rounding = c.bound = c.fused_single_pass = 1;
    c.weight_decay = 0.1f;
    c.bound_type = LV_BOUND_COORDINATE;
    std::vector<lv_tensor> T;
    for (int i = 7; i < argc; i++)
        T.push_back(tensor(i - 7, std::strtoull(argv[i], nullptr, 10), pt, pt, st, mode == LV_BUFFER_DUAL || mode == LV_BUFFER_T2,
                           master, 0, 0));
    check_call(c, T, kMulti, 2, ~0ull);
    for (const Launch &l : g_launches)
        if (l.k.unit) std::printf("%u %u\n", l.k.fl, l.threads);
    return g_bad ? 1 : 0;
}

int main(int argc, char **argv) {
    if (argc < 2) return 2;
    void *h = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL);
    if (!h) {
        std::printf("%s\n", dlerror());
        return 2;
    }
    f_multi = (MultiFn)dlsym(h, "lv_step_multi");
    f_noalloc = (NoAllocFn)dlsym(h, "lv_step_multi_noalloc");
    f_graph = (GraphFn)dlsym(h, "lv_step_multi_graph");
    f_bytes = (BytesFn)dlsym(h, "lv_workspace_bytes_for");
    f_error = (ErrFn)dlsym(h, "lv_last_error");
    if (g_names.empty()) {
        std::printf("the library's kernels were not registered with this program\n");
        return 2;
    }
    if (argc > 6 && !std::strcmp(argv[2], "route")) return route(argc, argv);
    const uint64_t kRadialLimit = 1u << 16;
    struct Shape {
        const char *name;
        int count;
        uint64_t last;
        const char *max_grid;
    } shapes[] = {
        {"inline", 5, 0, nullptr},
        {"table", 60, 0, nullptr},
        {"inline large", 5, (1u << 25) + 7, nullptr},
        {"table large", 60, (1u << 27) + 7, nullptr},
        {"table of small tensors", 60, (1u << 25) + 7, nullptr},
        {"table of many small tensors", 150, (1u << 25) + 7, nullptr},
        {"table split", 60, 0, "50"},
    };
    static const uint64_t sizes[] = {1, 300, 1025, 4097, 70001, 64 * 1024 + 1};
    for (const Shape &sh : shapes) {
        if (sh.max_grid) setenv("LV_MAX_GRID_BLOCKS", sh.max_grid, 1);
        else unsetenv("LV_MAX_GRID_BLOCKS");
        for (int mode = 1; mode <= 4; mode++)
        for (int pt = 0; pt < 3; pt++)
        for (int gt = 0; gt < 3; gt++)
        for (int st = 0; st < 3; st++)
        for (int master = 0; master < 2; master++) {
            const bool dual = mode == LV_BUFFER_DUAL || mode == LV_BUFFER_T2;
            std::vector<lv_tensor> T;
            for (int i = 0; i < sh.count; i++) {
                // views: aligned, +1, +33 and +130 elements, and a grad that disagrees
                static const uint64_t offs[] = {0, 1, 33, 130, 0}, goffs[] = {0, 1, 33, 130, 1};
                const uint64_t n = sh.last && i == sh.count - 1 ? sh.last : sizes[(size_t)i % 6];
                T.push_back(tensor(i, n, pt, gt, st, dual, master, offs[i % 5], goffs[i % 5]));
            }
            for (float lr : {1e-3f, 9.5e-10f, 9e-10f, 0.0f})
            for (int opt = lr == 1e-3f && sh.count < 100 ? 0 : 6; opt < 8; opt++)
            for (int bound = 0; bound < 3; bound++)
            for (int when = 0; when < 3; when++)
            for (int entry = 0; entry < 3; entry++) {
                lv_config c = defaults(mode, lr, master);
                c.cautious = opt & 1;
                c.stochastic_rounding = (opt >> 1) & 1;
                c.weight_decay = (opt & 4) ? 0.1f : 0.0f;
                c.bound = bound != LV_BOUND_NONE;
                c.bound_type = bound;
                c.fused_single_pass = when != 2;
                g_case = std::string(sh.name) + " mode " + std::to_string(mode) + " params " + std::to_string(pt) + " grads " +
                         std::to_string(gt) + " state " + std::to_string(st) + " master " + std::to_string(master) +
                         " lr " + std::to_string(lr) + " options " + std::to_string(opt) + " bound " + std::to_string(bound) + " when " +
                         std::to_string(when) + " entry " + std::to_string(entry);
                check_call(c, T, (Entry)entry, when == 0 ? 1 : 2, kRadialLimit);
            }
        }
    }
    std::printf("%ld calls, %ld unit launches checked, %ld of large forms, %ld of one-wave blocks, %ld mismatches\n", g_calls, g_checked,
                g_large, g_one_wave, g_bad);
    return g_bad ? 1 : 0;
}
