// resident.hip -- host side of the resident Jacobi launches (resident.h):
// the division of a cell grid into tiles, the outboxes, and the order of a
// device's resident launches and grid barriers.
#include "resident.h"

#include <algorithm>
#include <mutex>

namespace {

struct DeviceOrder {
    std::mutex m;
    hipEvent_t last = nullptr;
    bool any = false;
    uint32_t barriers = 0;  // BarrierUses held
};
constexpr int MAX_DEVICES = 64;
DeviceOrder g_order[MAX_DEVICES];

int ceil_div(int a, int b) { return (a + b - 1) / b; }

}  // namespace

// At most one tile per compute unit and 2 cells per thread.  Among the
// divisions that fit, the one with the fewest rounds of waves over a compute
// unit's four SIMDs (256 cells each), then few tiles and a small halo: on 16 x
// 16 x 32 cells 256 tiles of 32 cells took 1.79 us per iteration, 32 tiles of
// 256 cells 1.6 us; one to a few cells per thread and the tile's shape made
// less than 10% on 48 x 48 x 96 cells.
void resident_plan(Resident &r, int device, int nx, int ny, int nz, int wrap)
{
    r.planned = true;
    r.usable = false;
    if (nx < 3 || ny < 3 || nz < 3 || device < 0 || device >= MAX_DEVICES) return;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return;
    const int n[3] = {nx, ny, nz};
    double best = 1e300;
    for (int a = 1; a <= std::max(1, nx / 2) && a <= cus; ++a)
        for (int b = 1; b <= std::max(1, ny / 2) && a * b <= cus; ++b)
            for (int c = 1; c <= std::max(1, nz / 2) && a * b * c <= cus; ++c) {
                const int T[3] = {a, b, c};
                int e[3];
                for (int k = 0; k < 3; ++k) e[k] = ceil_div(n[k], T[k]);
                const long long cells = (long long)e[0] * e[1] * e[2];
                if (cells > 2 * RES_CELL_THREADS) continue;
                long long halo = 0;
                for (int k = 0; k < 3; ++k)
                    if (T[k] > 1 || ((wrap >> k) & 1)) halo += 2 * (cells / e[k]);
                const long long items = std::max(cells, halo);
                const int per = items > RES_CELL_THREADS ? 2 : 1;
                const long long nth = ceil_div((int)items, per * 64) * 64ll;
                if (nth > RES_CELL_THREADS) continue;
                const long long lds = 2ll * (e[0] + 2) * (e[1] + 2) * (e[2] + 2) * (long long)sizeof(double);
                if (lds > 60 * 1024) continue;
                const double cost = (double)(ceil_div((int)cells, 256) * 4) + (double)halo / 256.0 +
                                    (double)(a * b * c) / 64.0;
                if (cost >= best) continue;
                best = cost;
                for (int k = 0; k < 3; ++k) r.T[k] = T[k];
                r.tiles = (uint32_t)(a * b * c);
                r.threads = (uint32_t)nth + 64u;
                r.per_thread = (uint32_t)per;
                r.lds = (uint32_t)lds;
                r.box = (uint32_t)res_shell(e);
            }
    if (best >= 1e300) return;
    r.wrap = wrap;
    r.words = 4u * (size_t)r.tiles * (r.box + 1u);
    r.usable = true;
}

void resident_free(Resident &r)
{
    if (r.words_d) (void)hipFree(r.words_d);
    r = Resident{};
}

bool resident_ready(Resident &r)
{
    if (!r.usable) return false;
    if (r.rest == 0) return true;
    --r.rest;
    return false;
}

void resident_gave_up(Resident &r)
{
    r.repeated++;
    r.pause = r.pause ? std::min(2u * r.pause, 65536u) : 16u;
    r.rest = r.pause;
}

bool resident_args(Resident &r, hipStream_t s, int nx, int ny, int nz, uint32_t it0, uint32_t it1,
                   const ResidentWait &wait, ResidentArgs &out)
{
    const uint32_t its = it1 - it0;
    if (!r.words_d) {
        if (hipMalloc((void **)&r.words_d, r.words * 8) != hipSuccess) {
            r.words_d = nullptr;
            (void)hipGetLastError();
            return false;
        }
        if (hipMemsetAsync(r.words_d, 0, r.words * 8, s) != hipSuccess) return false;
        r.tag = 1;
    } else if (r.tag > 0xffffffffu - its) {
        // no tag is used twice on the same words
        if (hipMemsetAsync(r.words_d, 0, r.words * 8, s) != hipSuccess) return false;
        r.tag = 1;
    }
    out.n[0] = nx;
    out.n[1] = ny;
    out.n[2] = nz;
    for (int k = 0; k < 3; ++k) out.T[k] = r.T[k];
    out.wrap = r.wrap;
    out.it0 = it0;
    out.it1 = it1;
    out.tag0 = r.tag;
    out.box = r.box;
    out.spin = wait.polls && it0 >= wait.from ? wait.polls : RES_SPIN;
    out.mail = r.words_d;
    out.slots = r.words_d + 4u * (size_t)r.tiles * r.box;
    r.tag += its;
    return true;
}

bool resident_begin(int device, hipStream_t s, uint32_t held)
{
    DeviceOrder &o = g_order[device];
    o.m.lock();
    if (o.barriers > held) {
        o.m.unlock();
        return false;
    }
    if (o.any) (void)hipStreamWaitEvent(s, o.last, 0);
    return true;
}

void resident_end(int device, hipStream_t s)
{
    DeviceOrder &o = g_order[device];
    if (!o.last && hipEventCreateWithFlags(&o.last, hipEventDisableTiming) != hipSuccess) o.last = nullptr;
    o.any = o.last && hipEventRecord(o.last, s) == hipSuccess;
    o.m.unlock();
}

void BarrierUse::open(int device, hipStream_t s)
{
    close();
    if (device < 0 || device >= MAX_DEVICES) return;  // no resident launches there
    DeviceOrder &o = g_order[device];
    std::lock_guard<std::mutex> lock(o.m);
    ++o.barriers;
    if (o.any) (void)hipStreamWaitEvent(s, o.last, 0);
    device_ = device;
    stream_ = s;
}

void BarrierUse::close()
{
    if (device_ < 0) return;
    (void)hipStreamSynchronize(stream_);
    DeviceOrder &o = g_order[device_];
    std::lock_guard<std::mutex> lock(o.m);
    --o.barriers;
    device_ = -1;
}
