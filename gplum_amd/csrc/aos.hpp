// aos.hpp -- gplum_particle arrays (the ABI's layout) <-> the device's one array per field.
#pragma once
#include <vector>

#include "engine.hpp"

namespace gplum {

constexpr int AOS_WORDS = sizeof(gplum_particle) / 8;
static_assert(sizeof(gplum_particle) == 8 * AOS_WORDS, "gplum_particle is made of 8-byte words");

// Where word w of particle i lives: a[stride i] (8 bytes), or, of two 32-bit fields, a[i] and
// b[i].  A null source leaves the word (half) as it is; so does a null destination.
struct AosWord {
    void *a, *b;
    int stride, pair;
};
struct AosTable {
    AosWord w[AOS_WORDS] = {};
    void set(size_t off, double *p) { w[off / 8] = AosWord{p, nullptr, 1, 0}; }
    void set(size_t off, int64_t *p) { w[off / 8] = AosWord{p, nullptr, 1, 0}; }
    void set3(size_t off, double *p) {
        for (int k = 0; k < 3; k++) w[off / 8 + k] = AosWord{p + k, nullptr, 3, 0};
    }
    void set(size_t off, int32_t *p) {
        AosWord &q = w[off / 8];
        q.stride = q.pair = 1;
        (off % 8 ? q.b : q.a) = p;
    }
};
#define AOS_SET(T, field, p) (T).set(offsetof(gplum_particle, field), p)
#define AOS_SET3(T, field, p) (T).set3(offsetof(gplum_particle, field), p)

// particles [i0, i0 + n) of the arrays -> / <- aos[0 .. n)
int aos_pack(const AosTable &t, int i0, int n, gplum_particle *aos, hipStream_t st);
int aos_unpack(const AosTable &t, int i0, int n, const gplum_particle *aos, hipStream_t st);

}  // namespace gplum
