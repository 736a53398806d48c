// HostStage (gopf_amd/csrc/hostcopy.h) on the stand-in runtime beside this file: exit code 0 when
// every transfer gave the right bytes.
#include <cstdint>
#include <cstdio>
#include <stdexcept>
#include <vector>

#include "../../include/gpf.h"
#include "hostcopy.h"

using gpf::HostStage;
using Bytes = std::vector<char>;

static int bad = 0;
static const size_t kDirect = 3584u << 10;  // HostStage's line between one copy and chunks

static Bytes pattern(size_t n, unsigned seed) {
    Bytes b(n);
    uint32_t x = seed * 2654435761u + 1u;
    for (auto& c : b) {
        x = x * 1664525u + 1013904223u;
        c = (char)(x >> 24);
    }
    return b;
}

static void put(HostStage& h, FakeStream& st, Bytes& dev, const Bytes& from) {
    h.upload(dev.data(), from.size(), &st, [&](char* to, size_t off, size_t len) { std::memcpy(to, &from[off], len); });
}

static void get(HostStage& h, FakeStream& st, const Bytes& dev, Bytes& to) {
    h.download(dev.data(), to.size(), &st, [&](const char* from, size_t off, size_t len) { std::memcpy(&to[off], from, len); });
}

static void check(bool ok, const char* what, size_t n) {
    if (ok) return;
    std::printf("wrong: %s, %zu bytes\n", what, n);
    bad = 1;
}

int main() {
    const size_t sizes[] = {1, 4096, 300000, kDirect, kDirect + 16, 4u << 20, 5000000, 9000016, 40000000};
    HostStage h;  // one object over all sizes: its buffers grow and its slots change
    FakeStream st;
    unsigned seed = 1;
    for (size_t n : sizes) {
        for (int rep = 0; rep < 2; ++rep) {
            const Bytes a = pattern(n, ++seed), b = pattern(n, ++seed);
            Bytes dev(n), dev2(n), out(n);
            put(h, st, dev, a);
            put(h, st, dev2, b);  // the first upload's copies may still be pending
            get(h, st, dev, out);
            check(out == a, "upload, download", n);
            get(h, st, dev2, out);
            check(out == b, "second upload, download", n);
        }
        // a download that ends in an error, before its first use or as a copy is refused, then an
        // upload through the same buffers
        for (int kind = 0; kind < 4; ++kind) {
            HostStage fresh;
            HostStage& o = (kind & 2) ? fresh : h;
            const Bytes old = pattern(n, ++seed), a = pattern(n, ++seed);
            Bytes dev = old, out(n);
            bool threw = false;
            try {
                auto use = [&](const char* from, size_t off, size_t len) { std::memcpy(&out[off], from, len); };
                if ((kind & 1) == 0) {
                    o.download(dev.data(), n, &st, use, [] { throw std::runtime_error("not valid"); });
                } else {
                    st.fail_after = n > kDirect ? 3 : 0;
                    o.download(dev.data(), n, &st, use);
                }
            } catch (const std::exception&) {
                threw = true;
            }
            st.fail_after = -1;
            check(threw, "an error passed on", n);
            Bytes dev2(n);
            put(o, st, dev2, a);
            get(o, st, dev2, out);
            check(out == a, "upload after a failed download", n);
        }
    }
    return bad;
}
