// Driver of the excitation's normals (mtrack_amd/csrc/qe_dev.h) for
// tests/test_gpu_qe_normals.py, argument: the oracle's library.  Prints the number of
// inputs, of all 2^24, whose radius, sine or cosine differ in a bit from the oracle's,
// and of macroparticle-turns whose five normals do.
#include <dlfcn.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "qe_dev.h"

#define ALL (1 << 24)
#define TURNS (1 << 20)

#define CK(x)                                                                    \
  do {                                                                           \
    const hipError_t e_ = (x);                                                   \
    if (e_ != hipSuccess) {                                                      \
      fprintf(stderr, "%s: %s\n", #x, hipGetErrorString(e_));                    \
      return 1;                                                                  \
    }                                                                            \
  } while (0)

// inputs differ in their upper 24 bits; the lower eight are not looked at
__global__ void k_parts(float *r, float *s, float *c)
{
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= ALL) return;
  const uint32_t x = i << 8 | (i * 0x9E3779B9u >> 24);
  r[i] = qe_radius(x);
  qe_sincos(x, s + i, c + i);
}

__host__ __device__ static inline void key_of(uint32_t i, uint32_t &seed, uint32_t &bucket, unsigned long long &rev,
                                              uint32_t &j)
{
  seed = 1u + 0x9E3779B9u * (i & 15u);
  bucket = (i >> 4) & 511u;
  rev = i % 3u ? (unsigned long long)(i % 20000u) : 0x100000000ULL + i;
  j = i * 2654435761u % 1000003u;
}

__global__ void k_normals(double *n)
{
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= TURNS) return;
  uint32_t seed, bucket, j;
  unsigned long long rev;
  key_of(i, seed, bucket, rev, j);
  qe_normals(seed, bucket, rev, j, n + 5 * (size_t)i);
}

typedef float (*logf_t)(float);
typedef void (*sincos_t)(float, float *, float *);
typedef void (*normals_t)(unsigned, unsigned, unsigned long long, unsigned, double *);

int main(int argc, char **argv)
{
  void *lib = argc > 1 ? dlopen(argv[1], RTLD_NOW) : NULL;
  if (!lib) return 1;
  const logf_t lf = (logf_t)dlsym(lib, "orc_logf");
  const sincos_t sc = (sincos_t)dlsym(lib, "orc_sincos2pif");
  const normals_t nm = (normals_t)dlsym(lib, "orc_qe_normals");
  if (!lf || !sc || !nm) return 1;
  float *d, *h = (float *)malloc(sizeof(float) * 3 * (size_t)ALL);
  double *dn, *hn = (double *)malloc(sizeof(double) * 5 * (size_t)TURNS);
  CK(hipMalloc(&d, sizeof(float) * 3 * (size_t)ALL));
  CK(hipMalloc(&dn, sizeof(double) * 5 * (size_t)TURNS));
  hipLaunchKernelGGL(k_parts, dim3(ALL / 256), dim3(256), 0, 0, d, d + ALL, d + 2 * (size_t)ALL);
  CK(hipGetLastError());
  hipLaunchKernelGGL(k_normals, dim3(TURNS / 256), dim3(256), 0, 0, dn);
  CK(hipGetLastError());
  CK(hipMemcpy(h, d, sizeof(float) * 3 * (size_t)ALL, hipMemcpyDeviceToHost));
  CK(hipMemcpy(hn, dn, sizeof(double) * 5 * (size_t)TURNS, hipMemcpyDeviceToHost));
  long rad = 0, sin_ = 0, cos_ = 0, norm = 0;
  for (uint32_t i = 0; i < ALL; i++) {
    const float u = ((float)(i + 1u)) * 5.9604645e-8f, r = sqrtf(-2.0f * lf(u));
    float s, c;
    sc(u, &s, &c);
    rad += memcmp(&r, h + i, 4) != 0;
    sin_ += memcmp(&s, h + ALL + i, 4) != 0;
    cos_ += memcmp(&c, h + 2 * (size_t)ALL + i, 4) != 0;
  }
  for (uint32_t i = 0; i < TURNS; i++) {
    uint32_t seed, bucket, j;
    unsigned long long rev;
    double n[5];
    key_of(i, seed, bucket, rev, j);
    nm(seed, bucket, rev, j, n);
    norm += memcmp(n, hn + 5 * (size_t)i, sizeof n) != 0;
  }
  printf("radius %ld sine %ld cosine %ld normals %ld\n", rad, sin_, cos_, norm);
  (void)hipFree(d);
  (void)hipFree(dn);
  return 0;
}
