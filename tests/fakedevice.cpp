// A device made of host memory behind the few entry points of the kernel library that blobs need on their way in and out:
// preloaded in front of it, so that what the host library enqueues, and when it waits, is seen without a GPU.
// Work on a stream runs when somebody waits for the stream (as late as the rules allow); under capture it is recorded, and
// waiting or allocating breaks the capture, as it does on the device.
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <vector>

typedef std::function<void()> Op;

struct Stream
{
    std::deque<Op> ops;
    std::vector<Op> recorded;
    bool capturing = false, broken = false;
};
struct Event
{
    Stream* stream = 0;
    bool captured = false;
    std::shared_ptr<bool> passed;
};

static Stream* g_capturing = 0;
static std::vector<Stream*> g_streams;

static int run(Stream* s)
{
    if (s->capturing)
    {
        s->broken = true;
        return -1;
    }
    while (!s->ops.empty())
    {
        Op op = s->ops.front();
        s->ops.pop_front();
        op();
    }
    return 0;
}
static int enqueue(void* stream, Op op)
{
    Stream* s = (Stream*)stream;
    if (s->capturing)
        s->recorded.push_back(op);
    else
        s->ops.push_back(op);
    return 0;
}
static int allocate(void** p, size_t bytes)
{
    if (g_capturing)
    {
        g_capturing->broken = true;
        return -1;
    }
    *p = calloc(1, bytes + 64);
    return 0;
}

extern "C" {
int fake_pending()
{
    size_t n = 0;
    for (Stream* s : g_streams) n += s->ops.size();
    return (int)n;
}
int ncnnhip_init(int) { return 0; }
const char* ncnnhip_last_error() { return "fake device"; }
int ncnnhip_stream_create(void** s)
{
    g_streams.push_back(new Stream);
    *s = g_streams.back();
    return 0;
}
int ncnnhip_stream_destroy(void* s) { return run((Stream*)s); }
int ncnnhip_stream_synchronize(void* s) { return run((Stream*)s); }
int ncnnhip_device_synchronize()
{
    if (g_capturing) return run(g_capturing);
    for (Stream* s : g_streams) run(s);
    return 0;
}
int ncnnhip_stream_begin_capture(void* s)
{
    g_capturing = (Stream*)s;
    g_capturing->capturing = true;
    g_capturing->broken = false;
    g_capturing->recorded.clear();
    return 0;
}
int ncnnhip_stream_is_capturing(void* s, int* capturing)
{
    *capturing = ((Stream*)s)->capturing;
    return 0;
}
int ncnnhip_stream_end_capture(void* stream, void** exec)
{
    Stream* s = (Stream*)stream;
    s->capturing = false;
    g_capturing = 0;
    *exec = s->broken ? 0 : new std::vector<Op>(s->recorded);
    return s->broken ? -1 : 0;
}
int ncnnhip_graph_launch(void* exec, void* s)
{
    for (Op& op : *(std::vector<Op>*)exec) enqueue(s, op);
    return 0;
}
int ncnnhip_graph_destroy(void* exec)
{
    delete (std::vector<Op>*)exec;
    return 0;
}
int ncnnhip_malloc(void** p, size_t bytes) { return allocate(p, bytes); }
int ncnnhip_free(void* p)
{
    free(p);
    return 0;
}
int ncnnhip_host_malloc(void** p, size_t bytes) { return allocate(p, bytes); }
int ncnnhip_host_free(void* p)
{
    free(p);
    return 0;
}
int ncnnhip_event_create(void** e)
{
    *e = new Event;
    return 0;
}
int ncnnhip_event_destroy(void* e)
{
    delete (Event*)e;
    return 0;
}
int ncnnhip_event_record(void* e, void* s)
{
    Event* event = (Event*)e;
    event->stream = (Stream*)s;
    event->captured = event->stream->capturing;
    event->passed.reset(new bool(false));
    const std::shared_ptr<bool> passed = event->passed;
    return enqueue(s, [=] { *passed = true; });
}
int ncnnhip_event_synchronize(void* e)
{
    Event* event = (Event*)e;
    if (event->captured) return -1;
    while (event->passed && !*event->passed) // up to the event, not what lies behind it
    {
        Op op = event->stream->ops.front();
        event->stream->ops.pop_front();
        op();
    }
    return 0;
}
int ncnnhip_copy(void* dst, const void* src, size_t bytes, void* s)
{
    return enqueue(s, [=] { memcpy(dst, src, bytes); });
}
int ncnnhip_memcpy_d2d(void* dst, const void* src, size_t bytes, void* s) { return ncnnhip_copy(dst, src, bytes, s); }
int ncnnhip_memcpy_d2h(void* dst, const void* src, size_t bytes, void* s) { return ncnnhip_copy(dst, src, bytes, s); }
int ncnnhip_memcpy_h2d(void* dst, const void* src, size_t bytes, void* s)
{
    // pageable memory has been read when the call returns
    std::vector<unsigned char> held((const unsigned char*)src, (const unsigned char*)src + bytes);
    return enqueue(s, [=] { memcpy(dst, held.data(), bytes); });
}
int ncnnhip_chw_to_nhwc(const void* src, int elemsize, int c, int hw, int batch, size_t cstep, size_t nstep, void* dst, void* s)
{
    const int cp = (c + 15) / 16 * 16;
    return enqueue(s, [=] {
        memset(dst, 0, (size_t)batch * hw * cp * elemsize);
        for (int b = 0; b < batch; b++)
            for (int i = 0; i < hw; i++)
                for (int q = 0; q < c; q++)
                    memcpy((char*)dst + (((size_t)b * hw + i) * cp + q) * elemsize, (const char*)src + (nstep * b + cstep * q + i) * elemsize, elemsize);
    });
}
int ncnnhip_relu(const void* src, void* dst, int elemsize, size_t count, float, void* s)
{
    if (elemsize != 4) return -1;
    return enqueue(s, [=] { for (size_t i = 0; i < count; i++) ((float*)dst)[i] = ((const float*)src)[i] > 0.f ? ((const float*)src)[i] : 0.f; });
}
}
