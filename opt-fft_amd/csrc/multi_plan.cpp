// Host side of the mixed-batch persistent launch (include/fft3d_mi355x.h, multi.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "claims_hip.hpp"
#include "fft3d_mi355x.h"
#include "multi.hpp"
#include "multi_tasks.hpp"
#include "plan_internal.hpp"
#include "race_hip.hpp"

using namespace fx;

struct fft3d_mx_multi {
    int nitems, prec;
    int code[kMultiMaxItems], batch[kMultiMaxItems], conj[kMultiMaxItems];
    double scale[kMultiMaxItems];
    const MultiDesc* k;
    int2* tasks;   // device
    int ntasks;
    void* bank;    // device
    unsigned* work;  // device: the claim counters `claims` hands out (claims.hpp)
    ClaimSlots claims;
    int device;
};

template <typename T>
static void fill_args(const fft3d_mx_multi* m, const void* const* in, void* const* out,
                      MultiArgs<T>& a)
{
    std::memset(&a, 0, sizeof a);
    for (int i = 0; i < m->nitems; ++i) {
        a.item[i].in = (const cx<T>*)in[i];
        a.item[i].out = (cx<T>*)out[i];
        a.item[i].nvol = m->batch[i];
        a.item[i].code = m->code[i];
        a.item[i].conj = m->conj[i];
        a.item[i].scale = (T)m->scale[i];
    }
}

// One launch with claim counter `work` (the race passes the first counter directly; user
// launches take theirs from m->claims).
static hipError_t multi_launch(fft3d_mx_multi* m, const MultiDesc* k, const int2* tasks,
                               int ntasks, const void* const* in, void* const* out,
                               unsigned* work, hipStream_t s)
{
    if (m->prec == kC128) {
        MultiArgs<double> a;
        fill_args(m, in, out, a);
        return k->launch(&a, tasks, ntasks, m->bank, work, s);
    }
    MultiArgs<float> a;
    fill_args(m, in, out, a);
    return k->launch(&a, tasks, ntasks, m->bank, work, s);
}

static int upload_tasks(const std::vector<int2>& t, int2** dev)
{
    *dev = nullptr;
    if (t.empty()) return FFT3D_MX_OK;
    hipError_t e = hipMalloc((void**)dev, t.size() * sizeof(int2));
    if (e == hipSuccess) e = hipMemcpy(*dev, t.data(), t.size() * sizeof(int2), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(*dev);
        *dev = nullptr;
        return fail(FFT3D_MX_ENOMEM, "fft3d_mx_multi_create: task table: %s", hipGetErrorString(e));
    }
    return FFT3D_MX_OK;
}

// Time every preset on the items (batches capped at 256 MiB of input).
static const MultiDesc* multi_race(fft3d_mx_multi* m, const std::vector<const MultiDesc*>& cands)
{
    const size_t elem = elem_bytes(m->prec);
    size_t total = 0;
    int rb[kMultiMaxItems];
    for (int i = 0; i < m->nitems; ++i) {
        const int g = m->code[i];
        total += (size_t)kMultiShape[g][0] * kMultiShape[g][1] * kMultiShape[g][2] * elem * m->batch[i];
    }
    const double shrink = total > (256ull << 20) ? (double)(256ull << 20) / (double)total : 1.0;
    // Sets of buffers in turn, 256 MiB of input in all and at least two, 16 at most, and as much
    // output: stores of part of a line cost little while the line is in a cache and much otherwise
    // (6^3 x 200, 8^3 x 800, 12^3 x 300 as multi_c128_t192: 8.4 us over 256 MB, 10.3 over 384), and
    // one set of 256 MiB leaves parts of itself there (the complex64 mix 6^3 x 65536, 8^3 x 32768,
    // 12^3 x 8192, 17^3 x 2048: multi_c64_t320_fill_lin 85 us to .._lin_mix's 108 over one set, 102
    // to 100 over two; executed it takes 164 to 161).
    const size_t one = std::max<size_t>(1, std::min<size_t>(total, 256ull << 20));
    int sets = (int)std::max<size_t>(2, std::min<size_t>(16, (256ull << 20) / one));
    std::vector<void*> bufs;
    std::vector<std::vector<const void*>> ins(sets, std::vector<const void*>(m->nitems));
    std::vector<std::vector<void*>> outs(sets, std::vector<void*>(m->nitems));
    auto alloc = [&](int sets) {
        for (int i = 0; i < m->nitems; ++i) {
            const int g = m->code[i];
            rb[i] = std::max(m->batch[i] > 0 ? 1 : 0, (int)(m->batch[i] * shrink));
            const size_t bytes = std::max<size_t>(1, (size_t)kMultiShape[g][0] * kMultiShape[g][1] *
                                                         kMultiShape[g][2] * elem * rb[i]);
            const size_t pitch = (bytes + 255) / 256 * 256;
            void *a = nullptr, *b = nullptr;
            const bool got = hipMalloc(&a, pitch * sets) == hipSuccess &&
                             hipMalloc(&b, pitch * sets) == hipSuccess;
            if (a) bufs.push_back(a);
            if (b) bufs.push_back(b);
            if (!got) {
                for (void* p : bufs) (void)hipFree(p);
                bufs.clear();
                return false;
            }
            (void)hipMemsetD32((hipDeviceptr_t)a, 0x3F800000u, pitch * sets / 4);
            for (int w = 0; w < sets; ++w) {
                ins[w][i] = (char*)a + w * pitch;
                outs[w][i] = (char*)b + w * pitch;
            }
        }
        return true;
    };
    sets = fit_sets(sets, alloc);   // fewer where memory is short
    const MultiDesc* win = cands[0];
    if (sets > 0) {
        int saved[kMultiMaxItems];
        std::memcpy(saved, m->batch, sizeof saved);
        std::memcpy(m->batch, rb, sizeof(int) * m->nitems);
        std::vector<int2*> tasks(cands.size(), nullptr);
        std::vector<int> ntasks(cands.size(), -1);
        for (size_t i = 0; i < cands.size(); ++i) {
            std::vector<int2> t;
            multi_tasks(*cands[i], m->code, m->batch, m->nitems, elem, t);
            if (upload_tasks(t, &tasks[i]) == FFT3D_MX_OK) ntasks[i] = (int)t.size();
        }
        hipStream_t s;
        if (hipStreamCreate(&s) == hipSuccess) {
            {
                RaceEvents ev(cands.size());
                int w = 0;
                auto launch = [&](size_t k, int n) {
                    for (int i = 0; i < n; ++i) {
                        const int c = w++ % sets;
                        if (ntasks[k] < 0 || multi_launch(m, cands[k], tasks[k], ntasks[k], ins[c].data(),
                                                          outs[c].data(), m->work, s) != hipSuccess)
                            return false;
                    }
                    return true;
                };
                std::vector<Trial> ts(cands.size());
                if (ev.ok) {
                    run_trials(ts, kMultiRace, sets * one >= (128ull << 20) ? sets : 1, launch,
                               [&](const std::vector<Trial>& c, std::vector<double>& t) {
                                   return ev.round(c, t, s, launch);
                               });
                    const int best = race_winner(ts);
                    if (best >= 0) win = cands[best];
                }
                (void)hipStreamSynchronize(s);
            }
            (void)hipStreamDestroy(s);
        }
        for (int2* t : tasks) (void)hipFree(t);
        std::memcpy(m->batch, saved, sizeof saved);
    }
    for (void* b : bufs) (void)hipFree(b);
    (void)hipGetLastError();
    return win;
}

extern "C" fft3d_mx_multi* fft3d_mx_multi_create(const fft3d_mx_item* items, int nitems,
                                                 int precision, unsigned flags)
{
    if (!items || nitems < 1 || nitems > kMultiMaxItems) {
        fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_create: need 1..%d items, got %d", kMultiMaxItems,
             nitems);
        return nullptr;
    }
    if (precision != kC128 && precision != kC64) {
        fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_create: unknown precision %d", precision);
        return nullptr;
    }
    if ((flags & FFT3D_MX_MFMA_BF16) && (flags & FFT3D_MX_MFMA_FP16)) {
        fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_create: MFMA_BF16 and MFMA_FP16 are exclusive");
        return nullptr;
    }
    fft3d_mx_multi* m = new (std::nothrow) fft3d_mx_multi();
    if (!m) {
        fail(FFT3D_MX_ENOMEM, "fft3d_mx_multi_create: out of host memory");
        return nullptr;
    }
    m->nitems = nitems;
    m->prec = precision;
    for (int i = 0; i < nitems; ++i) {
        const fft3d_mx_item& it = items[i];
        const int g = multi_code(it.n0, it.n1, it.n2);
        if (g < 0 || it.batch < 0 || (it.direction != -1 && it.direction != 1)) {
            fail(g < 0 ? FFT3D_MX_EUNSUPPORTED : FFT3D_MX_EINVAL,
                 "fft3d_mx_multi_create: item %d (%dx%dx%d, batch %d, direction %d) is not "
                 "supported in a mixed launch", i, it.n0, it.n1, it.n2, it.batch, it.direction);
            delete m;
            return nullptr;
        }
        m->code[i] = g;
        m->batch[i] = it.batch;
        m->conj[i] = it.direction > 0;
        m->scale[i] = (flags & FFT3D_MX_NORMALIZE) ? 1.0 / ((double)it.n0 * it.n1 * it.n2) : 1.0;
    }
    if (hipGetDevice(&m->device) != hipSuccess) m->device = 0;
    const int algo = (flags & FFT3D_MX_MFMA_BF16) ? 1 : (flags & FFT3D_MX_MFMA_FP16) ? 2 : 0;
    std::vector<unsigned char> img;
    bank_device_image(precision, algo, img);
    hipError_t e = hipMalloc(&m->bank, img.size());
    if (e == hipSuccess) e = hipMemcpy(m->bank, img.data(), img.size(), hipMemcpyHostToDevice);
    const size_t work_bytes = ClaimSlots::bytes();
    if (e == hipSuccess) e = hipMalloc((void**)&m->work, work_bytes);
    if (e == hipSuccess) e = hipMemset(m->work, 0, work_bytes);
    if (e != hipSuccess) {
        fail(FFT3D_MX_ENOMEM, "fft3d_mx_multi_create: bank: %s", hipGetErrorString(e));
        (void)hipFree(m->bank);
        (void)hipFree(m->work);
        delete m;
        return nullptr;
    }
    m->claims.attach(m->work);
    std::vector<const MultiDesc*> cands;
    const char* forced = getenv("FFT3D_MX_MULTI_KERNEL");
    for (const MultiDesc& d : multi_registry())
        if (d.prec == precision && d.algo == algo &&
            (!forced || !*forced || !strcmp(forced, d.name)))
            cands.push_back(&d);
    if (cands.empty()) {
        fail(FFT3D_MX_EUNSUPPORTED, "fft3d_mx_multi_create: no %smixed kernel%s%s for %s",
             algo ? "matrix-core " : "", forced && *forced ? " named " : "",
             forced && *forced ? forced : "", precision == kC128 ? "complex128" : "complex64");
        (void)hipFree(m->bank);
        (void)hipFree(m->work);
        delete m;
        return nullptr;
    }
    m->k = (cands.size() > 1 && !(flags & FFT3D_MX_NO_TUNE)) ? multi_race(m, cands) : cands[0];
    std::vector<int2> t;
    multi_tasks(*m->k, m->code, m->batch, nitems, elem_bytes(precision), t);
    m->ntasks = (int)t.size();
    if (upload_tasks(t, &m->tasks) != FFT3D_MX_OK) {
        (void)hipFree(m->bank);
        (void)hipFree(m->work);
        delete m;
        return nullptr;
    }
    return m;
}

extern "C" int fft3d_mx_multi_execute(fft3d_mx_multi* m, const void* const* in, void* const* out,
                                      void* stream)
{
    if (!m || !in || !out) return fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_execute: NULL argument");
    for (int i = 0; i < m->nitems; ++i) {
        if (m->batch[i] == 0) continue;
        if (!in[i] || !out[i] || in[i] == (const void*)out[i])
            return fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_execute: item %d needs distinct buffers", i);
        if (!elem_aligned(in[i], m->prec) || !elem_aligned(out[i], m->prec))
            return fail(FFT3D_MX_EINVAL,
                        "fft3d_mx_multi_execute: item %d buffers must be aligned to %zu bytes", i,
                        elem_bytes(m->prec));
    }
    int cur = m->device;
    (void)hipGetDevice(&cur);
    if (cur != m->device) (void)hipSetDevice(m->device);
    const hipStream_t s = (hipStream_t)stream;
    const hipError_t e = m->claims.run(s, [&](unsigned* w) {
        return multi_launch(m, m->k, m->tasks, m->ntasks, in, out, w, s);
    });
    if (cur != m->device) (void)hipSetDevice(cur);
    if (e == HipClaimRT::busy)
        return fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_execute: %d launches of this plan were "
                    "already captured into graphs; no claim counter is left",
                    ClaimSlots::kSlots);
    if (e != hipSuccess)
        return fail(FFT3D_MX_EHIP, "fft3d_mx_multi_execute: %s: %s", m->k->name, hipGetErrorString(e));
    return FFT3D_MX_OK;
}

extern "C" int fft3d_mx_multi_get_info(const fft3d_mx_multi* m, char* kernel, size_t cap,
                                       int* ntasks, int* grid)
{
    if (!m) return fail(FFT3D_MX_EINVAL, "fft3d_mx_multi_get_info: NULL plan");
    if (kernel && cap) snprintf(kernel, cap, "%s", m->k->name);
    if (ntasks) *ntasks = m->ntasks;
    if (grid) {
        int cur = m->device;
        (void)hipGetDevice(&cur);
        if (cur != m->device) (void)hipSetDevice(m->device);
        bool g17 = false;
        for (int i = 0; i < m->nitems; ++i) g17 |= m->code[i] == 3 && m->batch[i] > 0;
        *grid = m->k->launch_grid && m->ntasks > 0 ? (int)m->k->launch_grid(m->ntasks, g17) : 0;
        if (cur != m->device) (void)hipSetDevice(cur);
    }
    return FFT3D_MX_OK;
}

extern "C" void fft3d_mx_multi_destroy(fft3d_mx_multi* m)
{
    if (!m) return;
    m->claims.release_events();
    (void)hipFree(m->tasks);
    (void)hipFree(m->bank);
    (void)hipFree(m->work);
    delete m;
}
