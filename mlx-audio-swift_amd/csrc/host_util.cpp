// host_util.cpp - error plumbing, minimal JSON reader, safetensors mmap reader.
// Replaces (host side) MLX.loadArrays + JSONDecoder use in SNACDecoder.swift:156-189 and
// LlamaTTS.swift:942-993.  Format: 8-byte LE header length, JSON header
// {name: {dtype, shape, data_offsets:[b,e]}, "__metadata__": {...}}, raw little-endian data.
#include "common.h"

#include <dirent.h>
#include <fcntl.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <fstream>
#include <memory>
#include <mutex>
#include <sstream>
#include <thread>

static std::atomic<int64_t> g_device_held{0}, g_device_limit{INT64_MAX};
hipError_t mis_device_malloc(void** p, size_t bytes) {
    *p = nullptr;
    if (g_device_held.fetch_add((int64_t)bytes) + (int64_t)bytes > g_device_limit.load()) { g_device_held -= (int64_t)bytes; return hipErrorOutOfMemory; }
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) { g_device_held -= (int64_t)bytes; *p = nullptr; }
    return e;
}
void mis_device_free(void* p, size_t bytes) {
    (void)hipFree(p);
    g_device_held -= (int64_t)bytes;
}
extern "C" int64_t mis_debug_device_limit(int64_t more) {
    const int64_t held = g_device_held.load();
    g_device_limit = more < 0 ? INT64_MAX : held + more;
    return held;
}

static thread_local std::string g_last_error;

void mis_set_error(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}
mis_status mis_fail(mis_status code, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

extern "C" const char* mis_last_error(void) { return g_last_error.c_str(); }
extern "C" int mis_abi_version(void) { return MIS_ABI_VERSION; }
extern "C" void mis_free(void* p) {
    if (p) (void)hipHostFree(p);
}
extern "C" int mis_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

// ---------------------------------------------------------------------------- JSON
namespace {
struct JsonParser {
    const std::string& s;
    size_t i = 0;
    explicit JsonParser(const std::string& t) : s(t) {}
    void ws() { while (i < s.size() && (s[i] == ' ' || s[i] == '\n' || s[i] == '\t' || s[i] == '\r')) i++; }
    [[noreturn]] void fail(const char* what) {
        throw MisError(MIS_ERR_INVALID_INPUT, std::string("json: ") + what + " at offset " + std::to_string(i));
    }
    JsonValue parse() {
        ws();
        if (i >= s.size()) fail("unexpected end");
        char c = s[i];
        JsonValue v;
        if (c == '{') {
            v.type = JsonValue::OBJ;
            i++;
            ws();
            if (i < s.size() && s[i] == '}') { i++; return v; }
            for (;;) {
                ws();
                if (i >= s.size() || s[i] != '"') fail("expected key");
                std::string k = str();
                ws();
                if (i >= s.size() || s[i] != ':') fail("expected ':'");
                i++;
                JsonValue val = parse();
                v.obj.emplace_back(std::move(k), std::move(val));
                ws();
                if (i < s.size() && s[i] == ',') { i++; continue; }
                if (i < s.size() && s[i] == '}') { i++; break; }
                fail("expected ',' or '}'");
            }
        } else if (c == '[') {
            v.type = JsonValue::ARR;
            i++;
            ws();
            if (i < s.size() && s[i] == ']') { i++; return v; }
            for (;;) {
                v.arr.push_back(parse());
                ws();
                if (i < s.size() && s[i] == ',') { i++; continue; }
                if (i < s.size() && s[i] == ']') { i++; break; }
                fail("expected ',' or ']'");
            }
        } else if (c == '"') {
            v.type = JsonValue::STR;
            v.str = str();
        } else if (s.compare(i, 4, "true") == 0) { v.type = JsonValue::BOOL; v.b = true; i += 4; }
        else if (s.compare(i, 5, "false") == 0) { v.type = JsonValue::BOOL; v.b = false; i += 5; }
        else if (s.compare(i, 4, "null") == 0) { v.type = JsonValue::NUL; i += 4; }
        else {
            size_t j = i;
            while (j < s.size() && (isdigit((unsigned char)s[j]) || s[j] == '-' || s[j] == '+' || s[j] == '.' ||
                                    s[j] == 'e' || s[j] == 'E')) j++;
            if (j == i) fail("unexpected character");
            v.type = JsonValue::NUM;
            v.num = strtod(s.substr(i, j - i).c_str(), nullptr);
            i = j;
        }
        return v;
    }
    std::string str() {
        std::string out;
        i++;   // opening quote
        while (i < s.size() && s[i] != '"') {
            if (s[i] == '\\' && i + 1 < s.size()) {
                char e = s[i + 1];
                if (e == 'n') out += '\n';
                else if (e == 't') out += '\t';
                else if (e == 'u') { out += '?'; i += 4; }
                else out += e;
                i += 2;
            } else out += s[i++];
        }
        if (i >= s.size()) fail("unterminated string");
        i++;
        return out;
    }
};
}   // namespace

JsonValue json_parse(const std::string& text) {
    JsonParser p(text);
    return p.parse();
}

std::string read_text_file(const std::string& path) {
    std::ifstream f(path, std::ios::binary);
    if (!f) throw MisError(MIS_ERR_NOT_INITIALIZED, "cannot open " + path);
    std::stringstream ss;
    ss << f.rdbuf();
    return ss.str();
}

// ---------------------------------------------------------------------------- safetensors
SafeTensorFile::~SafeTensorFile() {
    if (map) munmap(map, map_len);
}

void SafeTensorFile::open(const std::string& path) {
    int fd = ::open(path.c_str(), O_RDONLY);
    if (fd < 0) throw MisError(MIS_ERR_NOT_INITIALIZED, "cannot open " + path);
    struct stat st;
    if (fstat(fd, &st) != 0) { ::close(fd); throw MisError(MIS_ERR_NOT_INITIALIZED, "cannot stat " + path); }
    map_len = (size_t)st.st_size;
    map = mmap(nullptr, map_len, PROT_READ, MAP_PRIVATE, fd, 0);
    ::close(fd);
    if (map == MAP_FAILED) { map = nullptr; throw MisError(MIS_ERR_NOT_INITIALIZED, "mmap failed for " + path); }
    if (map_len < 8) throw MisError(MIS_ERR_INVALID_INPUT, "safetensors file too small: " + path);
    const uint8_t* base = (const uint8_t*)map;
    uint64_t hlen = 0;
    memcpy(&hlen, base, 8);
    if (8 + hlen > map_len) throw MisError(MIS_ERR_INVALID_INPUT, "bad safetensors header length in " + path);
    std::string header((const char*)base + 8, (size_t)hlen);
    JsonValue root = json_parse(header);
    if (root.type != JsonValue::OBJ) throw MisError(MIS_ERR_INVALID_INPUT, "safetensors header is not an object");
    const uint8_t* data0 = base + 8 + hlen;
    size_t data_len = map_len - 8 - (size_t)hlen;
    for (auto& kv : root.obj) {
        if (kv.first == "__metadata__") continue;
        const JsonValue& t = kv.second;
        const JsonValue* dt = t.get("dtype");
        const JsonValue* sh = t.get("shape");
        const JsonValue* off = t.get("data_offsets");
        if (!dt || !sh || !off || off->arr.size() != 2)
            throw MisError(MIS_ERR_INVALID_INPUT, "malformed safetensors entry " + kv.first);
        SafeTensorEntry e;
        e.name = kv.first;
        e.dtype = dt->str;
        for (auto& d : sh->arr) e.shape.push_back((int64_t)d.num);
        size_t b = (size_t)off->arr[0].num, en = (size_t)off->arr[1].num;
        if (en < b || en > data_len) throw MisError(MIS_ERR_INVALID_INPUT, "safetensors offsets out of range: " + kv.first);
        e.data = data0 + b;
        e.nbytes = en - b;
        entries.push_back(std::move(e));
    }
}

std::vector<std::string> list_safetensors(const std::string& dir) {
    std::vector<std::string> out;
    DIR* d = opendir(dir.c_str());
    if (!d) throw MisError(MIS_ERR_NOT_INITIALIZED, "cannot open model directory " + dir);
    while (struct dirent* e = readdir(d)) {
        std::string n = e->d_name;
        if (n.size() > 12 && n.substr(n.size() - 12) == ".safetensors") out.push_back(dir + "/" + n);
    }
    closedir(d);
    std::sort(out.begin(), out.end());
    return out;
}

mis_dtype dtype_from_safetensors(const std::string& s) {
    if (s == "F32") return MIS_F32;
    if (s == "F16") return MIS_F16;
    if (s == "BF16") return MIS_BF16;
    if (s == "I32") return MIS_I32;
    throw MisError(MIS_ERR_INVALID_INPUT, "unsupported safetensors dtype " + s);
}

// ---------------------------------------------------------------------------- calls on a device
namespace {
struct DeviceUse {
    std::mutex m;
    std::condition_variable given;
    int calls = 0;
    uint64_t came = 0;
    const DeviceTurn* holder = nullptr;
    std::thread::id holder_thread;
    bool resting = false;
};
constexpr int DEVICES = 64;                                                // (past them: no call is alone)
DeviceUse g_use[DEVICES];
thread_local int t_depth[DEVICES];
bool known(int device) { return device >= 0 && device < DEVICES; }
}
DeviceCall::DeviceCall(int d) : device(d) {
    if (!known(d) || t_depth[d]++) return;
    std::lock_guard<std::mutex> g(g_use[d].m);
    ++g_use[d].calls;
    ++g_use[d].came;
}
DeviceCall::~DeviceCall() {
    if (!known(device) || --t_depth[device]) return;
    std::lock_guard<std::mutex> g(g_use[device].m);
    --g_use[device].calls;
}
bool DeviceTurn::take(int d) {
    give();
    if (!known(d)) return false;
    DeviceUse& u = g_use[d];
    std::lock_guard<std::mutex> g(u.m);
    device = d;
    seen = u.came;
    since = std::chrono::steady_clock::now();
    if (u.calls != 1 || u.holder || !t_depth[d]) return false;
    u.holder = this; u.holder_thread = std::this_thread::get_id(); u.resting = false;
    return held = true;
}
void DeviceTurn::rest() {
    if (!held) return;
    DeviceUse& u = g_use[device];
    { std::lock_guard<std::mutex> g(u.m); u.resting = true; }
    u.given.notify_all();
}
bool DeviceTurn::at_poll() {
    if (device < 0) return false;
    DeviceUse& u = g_use[device];
    std::lock_guard<std::mutex> g(u.m);
    const auto now = std::chrono::steady_clock::now();
    if (u.came != seen || u.calls != 1) {
        seen = u.came;
        since = now;
        if (held) { u.holder = nullptr; held = false; u.given.notify_all(); }
        return false;
    }
    if (!held && !u.holder && now - since >= std::chrono::milliseconds(QUIET_MS)) {
        u.holder = this; u.holder_thread = std::this_thread::get_id();
        held = true;
    }
    if (held) u.resting = false;
    return held;
}
void DeviceTurn::give() {
    if (!held) return;
    DeviceUse& u = g_use[device];
    std::lock_guard<std::mutex> g(u.m);
    u.holder = nullptr;
    held = false;
    u.given.notify_all();
}
void device_settle(int d) {
    if (!known(d)) return;
    DeviceUse& u = g_use[d];
    std::unique_lock<std::mutex> g(u.m);
    const auto me = std::this_thread::get_id();
    u.given.wait_for(g, std::chrono::milliseconds(DeviceTurn::SETTLE_MS), [&] { return !u.holder || u.resting || u.holder_thread == me; });
}
extern "C" int32_t mis_debug_device_turn(int device, int op) {
    static thread_local std::vector<std::unique_ptr<DeviceCall>> calls;
    static thread_local DeviceTurn turn;
    switch (op) {
        case 0: calls.emplace_back(new DeviceCall(device)); return 0;
        case 1: if (!calls.empty()) calls.pop_back(); return 0;
        case 2: return turn.take(device);
        case 3: turn.rest(); return 0;
        case 4: return turn.at_poll();
        case 5: turn.give(); return 0;
        default: device_settle(device); return 0;
    }
}

// ---------------------------------------------------------------------------- large host copies
HostRing::~HostRing() {
    for (auto& e : ev) if (e) (void)hipEventDestroy(e);
}
void HostRing::reserve(bool large) {
    if (buf.p) return;
    if (large) for (auto& e : ev) if (!e) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    const size_t n = (large ? SLOTS * SLOT : 0) + SMALL + INPUT;
    buf.alloc(n);
    held = n;
}
// block x, x + gridDim.x, ..: 16 bytes a thread; the last bytes one by one
struct CopyPieces { HostRing::Piece p[HostRing::PIECES]; };
static __global__ void __launch_bounds__(256) k_copy_pieces(CopyPieces c) {
    const HostRing::Piece p = c.p[blockIdx.y];
    const size_t units = p.bytes / 16, i0 = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (size_t i = i0; i < units; i += (size_t)gridDim.x * 256) reinterpret_cast<uint4*>(p.to)[i] = reinterpret_cast<const uint4*>(p.from)[i];
    if (i0 < p.bytes % 16) reinterpret_cast<uint8_t*>(p.to)[units * 16 + i0] = reinterpret_cast<const uint8_t*>(p.from)[units * 16 + i0];
}
static void copy_pieces(const CopyPieces& c, int n, hipStream_t s) {
    size_t most = 0;
    for (int i = 0; i < n; ++i) most = std::max(most, c.p[i].bytes);
    hipLaunchKernelGGL(k_copy_pieces, dim3((unsigned)std::min<size_t>(64, (most / 16 + 255) / 256 + 1), n), dim3(256), 0, s, c);
    HIP_CHECK(hipGetLastError());
}
// waits for results on their way to the caller's memory (diagnostics, tests)
static std::atomic<int64_t> g_result_waits{0};
extern "C" int64_t mis_debug_result_waits(void) { return g_result_waits.load(); }
static void wait_for_results(hipStream_t s) {
    g_result_waits.fetch_add(1, std::memory_order_relaxed);
    HIP_CHECK(hipStreamSynchronize(s));
}
bool HostRing::out_together(const Piece* p, int n, hipStream_t s) {
    size_t total = 0;
    if (!buf.p || n < 1 || n > PIECES) return false;
    bool by_kernel = true;
    for (int i = 0; i < n; ++i) {
        total += round_up(p[i].bytes, 16);
        if (!p[i].bytes || total >= MIN || !pageable(p[i].to)) return false;
        by_kernel = by_kernel && ((uintptr_t)p[i].from & 15) == 0;
    }
    by_kernel = by_kernel && total <= SMALL;
    if (!by_kernel && !ev[0]) return false;
    CopyPieces c;
    uint8_t* at = by_kernel ? buf.p + held - INPUT - SMALL : buf.p;
    for (int i = 0; i < n; ++i) { c.p[i] = {at, p[i].from, p[i].bytes}; at += round_up(p[i].bytes, 16); }
    if (by_kernel) copy_pieces(c, n, s);
    else for (int i = 0; i < n; ++i) HIP_CHECK(hipMemcpyAsync(c.p[i].to, c.p[i].from, c.p[i].bytes, hipMemcpyDeviceToHost, s));
    wait_for_results(s);
    for (int i = 0; i < n; ++i) memcpy(p[i].to, c.p[i].to, p[i].bytes);
    return true;
}
bool HostRing::in_small(const Piece* p, int n, hipStream_t s) {
    size_t total = 0;
    if (!buf.p || n < 1 || n > PIECES) return false;
    for (int i = 0; i < n; ++i) {
        total += round_up(p[i].bytes, 16);
        if (!p[i].bytes || total > INPUT || ((uintptr_t)p[i].to & 15) || !pageable(p[i].from)) return false;
    }
    CopyPieces c;
    uint8_t* at = buf.p + held - INPUT;
    for (int i = 0; i < n; ++i) {
        memcpy(at, p[i].from, p[i].bytes);
        c.p[i] = {p[i].to, at, p[i].bytes};
        at += round_up(p[i].bytes, 16);
    }
    copy_pieces(c, n, s);
    return true;
}
bool HostRing::pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) { (void)hipGetLastError(); return true; }
    return a.type == hipMemoryTypeUnregistered;
}
void HostRing::out(void* host, const void* dev, size_t n, hipStream_t s) {
    if (n == 0) { HIP_CHECK(hipStreamSynchronize(s)); return; }
    const Piece p{host, dev, n};
    if (n <= SMALL && ((uintptr_t)dev & 15) == 0 && out_together(&p, 1, s)) return;
    if (ev[0] && buf.p && n >= MIN && pageable(host)) { run((uint8_t*)host, (uint8_t*)const_cast<void*>(dev), n, true, s); return; }
    HIP_CHECK(hipMemcpyAsync(host, dev, n, hipMemcpyDefault, s));
    wait_for_results(s);
}
void HostRing::in(void* dev, const void* host, size_t n, hipStream_t s) {
    if (n == 0) return;
    if (ev[0] && buf.p && n >= MIN && pageable(host)) { run((uint8_t*)const_cast<void*>(host), (uint8_t*)dev, n, false, s); return; }
    HIP_CHECK(hipMemcpyAsync(dev, host, n, hipMemcpyDefault, s));
    HIP_CHECK(hipStreamSynchronize(s));
}
// Chunk i uses slot i % SLOTS.  The calling thread queues the copies in order; worker w moves chunks w, w + SLOTS, ... between slot w and the caller's
// memory.  turn[w] counts the hand-overs of slot w: even - the worker's, odd - the queue's (to the device), the other way round from it.
void HostRing::run(uint8_t* host, uint8_t* dev, size_t n, bool to_host, hipStream_t s) {
    const size_t chunks = (n + SLOT - 1) / SLOT;
    const int workers = (int)std::min<size_t>(SLOTS, chunks);
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    std::atomic<size_t> turn[SLOTS];
    std::atomic<int> bad{(int)hipSuccess};
    for (auto& t : turn) t.store(0);
    auto bytes = [&](size_t i) { return std::min(SLOT, n - i * SLOT); };
    auto wait_turn = [&](int w, size_t t) {
        while (turn[w].load(std::memory_order_acquire) < t) {
            if (bad.load(std::memory_order_relaxed) != (int)hipSuccess) return false;
            std::this_thread::yield();
        }
        return true;
    };
    auto worker = [&](int w) {
        hipError_t e = hipSetDevice(device);
        for (size_t i = w, k = 0; i < chunks && e == hipSuccess; i += SLOTS, ++k) {
            if (to_host) {
                if (!wait_turn(w, 2 * k + 1)) return;                 // the copy of this chunk is queued
                if ((e = hipEventSynchronize(ev[w])) != hipSuccess) break;
                memcpy(host + i * SLOT, buf.p + w * SLOT, bytes(i));
            } else {
                if (!wait_turn(w, 2 * k)) return;
                if (k > 0 && (e = hipEventSynchronize(ev[w])) != hipSuccess) break;      // the slot's last copy has left it
                memcpy(buf.p + w * SLOT, host + i * SLOT, bytes(i));
            }
            turn[w].fetch_add(1, std::memory_order_release);
        }
        if (e != hipSuccess) bad.store((int)e);
    };
    std::vector<std::thread> th;
    auto join = [&] { for (auto& t : th) t.join(); th.clear(); };
    try {
        for (int w = 0; w < workers; ++w) th.emplace_back(worker, w);
    } catch (...) {                                                   // no threads to be had: the plain copy
        bad.store((int)hipErrorUnknown);
        join();
        HIP_CHECK(hipMemcpyAsync(to_host ? host : dev, to_host ? dev : host, n, hipMemcpyDefault, s));
        HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    for (size_t i = 0; i < chunks; ++i) {
        const int w = (int)(i % SLOTS);
        const size_t k = i / SLOTS;
        if (!wait_turn(w, to_host ? 2 * k : 2 * k + 1)) break;
        hipError_t e = to_host ? hipMemcpyAsync(buf.p + w * SLOT, dev + i * SLOT, bytes(i), hipMemcpyDeviceToHost, s)
                               : hipMemcpyAsync(dev + i * SLOT, buf.p + w * SLOT, bytes(i), hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(ev[w], s);
        if (e != hipSuccess) { bad.store((int)e); break; }
        turn[w].fetch_add(1, std::memory_order_release);
    }
    join();
    const hipError_t e = hipStreamSynchronize(s);
    if (bad.load() != (int)hipSuccess) HIP_CHECK((hipError_t)bad.load());
    HIP_CHECK(e);
}
