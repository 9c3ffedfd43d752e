/*
 * The host layer's kernel launches without a GPU: the HIP entry points that it needs are defined here, so a launch is
 * printed instead of made. Commands on standard input, one a line:
 *   process TYPE M N K S                      libsmm_acc_process of S entries
 *   config  TYPE M N K S <configuration>      libsmm_acc_process_config
 *   set     TYPE M N K <configuration>        libsmm_acc_config_set
 *   get     TYPE M N K                        libsmm_acc_config_get
 *   clear                                     libsmm_acc_learned_set(NULL)
 * <configuration>: variant tm tn nt bs kt flush s split bs_short split_short. Output: for every launch
 *   launch <groups> <threads> <bs> <k> <kt> <tsplit> <atomic> <byte offset of A> <byte offset of B> <piece>
 * for get "config <source> <configuration>", then "rc <result>" for every command.
 */
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>
#include "acc_libsmm.h"
#include "libxstream_amd.h"

static char *const apool = (char*)0x100000, *const bpool = (char*)0x200000, *const cpool = (char*)0x300000;

hipError_t hipGetDeviceCount(int* count) {
  *count = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int device) {
  (void)device;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* props, int device) { /* a macro names the versioned symbol */
  (void)device;
  memset(props, 0, sizeof(*props));
  strcpy(props->name, "AMD Instinct MI355X");
  strcpy(props->gcnArchName, "gfx950");
  props->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t stream) {
  (void)fn;
  (void)lds;
  (void)stream;
  printf("launch %u %u %d %d %d %d %d %ld %ld %d\n", grid.x, block.x, *(int*)args[5], *(int*)args[8], *(int*)args[9],
    *(int*)args[13], *(int*)args[10], (long)(*(char**)args[1] - apool), (long)(*(char**)args[2] - bpool),
    *(int*)args[14]);
  return hipSuccess;
}

static int read_config(const char* text, libsmm_acc_smm_config_t* c) {
  memset(c, 0, sizeof(*c));
  return 11 == sscanf(text, "%d %d %d %d %d %d %d %d %d %d %d", &c->variant, &c->tm, &c->tn, &c->nt, &c->bs, &c->kt,
                 &c->flush, &c->s, &c->split, &c->bs_short, &c->split_short);
}

int main(void) {
  char line[512], cmd[16];
  if (0 != libsmm_acc_init()) return 2;
  while (NULL != fgets(line, sizeof(line), stdin)) {
    libsmm_acc_smm_config_t c;
    int t, m, n, k, s, at = 0, rc = -99, src = -1;
    if (1 != sscanf(line, "%15s%n", cmd, &at)) continue;
    if (0 == strcmp(cmd, "clear")) {
      rc = libsmm_acc_learned_set(NULL, 0.0);
    }
    else if (0 == strcmp(cmd, "process") && 5 == sscanf(line + at, "%d %d %d %d %d", &t, &m, &n, &k, &s)) {
      rc = libsmm_acc_process(NULL, (const int*)cpool, s, (libsmm_acc_data_t)t, apool, bpool, cpool, m, n, k, 80, 1, NULL, NULL);
    }
    else if (0 == strcmp(cmd, "get") && 4 == sscanf(line + at, "%d %d %d %d", &t, &m, &n, &k)) {
      rc = libsmm_acc_config_get((libsmm_acc_data_t)t, m, n, k, &c, &src);
      printf("config %d %d %d %d %d %d %d %d %d %d %d %d\n", src, c.variant, c.tm, c.tn, c.nt, c.bs, c.kt, c.flush, c.s,
        c.split, c.bs_short, c.split_short);
    }
    else if (0 == strcmp(cmd, "set") && 4 == sscanf(line + at, "%d %d %d %d%n", &t, &m, &n, &k, &s) &&
             read_config(line + at + s, &c)) {
      rc = libsmm_acc_config_set((libsmm_acc_data_t)t, m, n, k, &c);
    }
    else if (0 == strcmp(cmd, "config")) {
      int skip = 0;
      if (5 == sscanf(line + at, "%d %d %d %d %d%n", &t, &m, &n, &k, &s, &skip) && read_config(line + at + skip, &c)) {
        rc = libsmm_acc_process_config(&c, (const int*)cpool, s, (libsmm_acc_data_t)t, apool, bpool, cpool, m, n, k, NULL);
      }
    }
    printf("rc %d\n", rc);
    fflush(stdout);
  }
  libsmm_acc_finalize();
  return 0;
}
