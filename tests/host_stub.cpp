// Stand-in for libarhip that keeps "device" memory on the host, runs nothing and writes down what the host layer asks for, in
// order: "launch <handle> <entry>", with " foreign" behind it if a buffer is another handle's, and "sync <handle>" (test_host_order.py compiles it with csrc/host/).
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "../include/arhip.h"

struct arhip_device {
    int id;
};

static std::string g_log;
static int g_handles = 0;
static std::map<void *, int> g_owner;  // handle of an allocation

static void note(const std::string &what, arhip_device *d, const char *name = "")
{
    g_log += what + " " + std::to_string(d->id) + (*name ? " " : "") + name + "\n";
}

extern "C" {

const char *stub_log(void) { return g_log.c_str(); }
void stub_clear(void) { g_log.clear(); }

const char *arhip_last_error(void) { return ""; }
int arhip_open(int, arhip_device **out)
{
    *out = new arhip_device{g_handles++};
    return ARHIP_OK;
}
int arhip_close(arhip_device *d)
{
    delete d;
    return ARHIP_OK;
}
int arhip_compute_units(arhip_device *) { return 256; }
void *arhip_stream(arhip_device *d) { return d; }
int arhip_sync(arhip_device *d)
{
    note("sync", d);
    return ARHIP_OK;
}
int arhip_alloc(arhip_device *d, size_t bytes, void **p)
{
    *p = std::calloc(1, bytes);
    g_owner[*p] = d->id;
    return ARHIP_OK;
}
int arhip_free(arhip_device *, void *p)
{
    std::free(p);
    return ARHIP_OK;
}
int arhip_copyin(arhip_device *, void *dst, const void *src, size_t n)
{
    std::memcpy(dst, src, n);
    return ARHIP_OK;
}
int arhip_copyout(arhip_device *, void *dst, const void *src, size_t n)
{
    std::memcpy(dst, src, n);
    return ARHIP_OK;
}
int arhip_cast_bf16(arhip_device *, const float *, uint16_t *, int64_t, int, double *) { return ARHIP_OK; }
int arhip_attn_supported(int, int64_t, int64_t, int) { return 1; }
int arhip_module_load(arhip_device *d, const void *, size_t, void **m)
{
    *m = d;
    return ARHIP_OK;
}
int arhip_launch(arhip_device *d, void *, const char *name, const unsigned *, const unsigned *, void *const *bufs, int nbufs,
                 const int64_t *, const int *, int, int wait, double *)
{
    bool foreign = false;
    for (int i = 0; i < nbufs; ++i) foreign = foreign || g_owner[bufs[i]] != d->id;
    note("launch", d, (std::string(name) + (foreign ? " foreign" : "")).c_str());
    if (wait) note("sync", d);
    return ARHIP_OK;
}

}  // extern "C"
