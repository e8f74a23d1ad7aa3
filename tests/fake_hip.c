/* A libamdhip64.so that launches nothing: it writes down what a program would launch, so that the host library's choices
 * can be looked at without a GPU (tests/launches.py).  Kernels are looked up in the code object that hipModuleLoad was given:
 * a name that is not one of its symbols is refused, as the runtime refuses it. */
#define _GNU_SOURCE
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static char* code;
static size_t code_len;
static char names[4096][64];
static int n_names;
static char record[1 << 20];
static size_t record_len;

static void note(const char* line)
{
    const size_t n = strlen(line);
    if (record_len + n < sizeof record) memcpy(record + record_len, line, n + 1), record_len += n;
}
const char* fake_hip_record(void) { return record; }
void fake_hip_clear(void) { record[record_len = 0] = 0; }

int hipModuleLoad(void** m, const char* path)
{
    FILE* f = fopen(path, "rb");
    if (!f) return 301;
    fseek(f, 0, SEEK_END);
    code_len = (size_t)ftell(f);
    rewind(f);
    code = malloc(code_len);
    const size_t got = fread(code, 1, code_len, f);
    fclose(f);
    *m = code;
    return got == code_len ? 0 : 301;
}
int hipModuleGetFunction(void** fn, void* m, const char* name)
{
    (void)m;
    char symbol[96];
    const int n = snprintf(symbol, sizeof symbol, "%c%s.kd", 0, name) + 1;      /* as it stands in the string table */
    if (!code || !memmem(code, code_len, symbol, (size_t)n)) return 500;
    int i = 0;
    while (i < n_names && strcmp(names[i], name) != 0) i++;
    if (i == 4096) return 500;
    if (i == n_names) snprintf(names[n_names++], sizeof names[0], "%s", name);
    *fn = names[i];
    return 0;
}
int hipModuleLaunchKernel(void* fn, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned shmem, void* s,
                          void** args, void** extra)
{
    (void)s, (void)args, (void)extra;
    char line[192];
    snprintf(line, sizeof line, "%s %u %u %u %u %u %u %u\n", (const char*)fn, gx, gy, gz, bx, by, bz, shmem);
    note(line);
    return 0;
}
const char* hipGetErrorString(int e) { return e == 500 ? "named symbol not found" : "error of the fake runtime"; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { (void)d, (void)s, (void)n, (void)kind, (void)st; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }

#define REFUSED(name) int name(void) { return 100; }
REFUSED(hipGetDeviceCount) REFUSED(hipSetDevice) REFUSED(hipDeviceCanAccessPeer) REFUSED(hipDeviceEnablePeerAccess)
REFUSED(hipDeviceGetName) REFUSED(hipDeviceTotalMem) REFUSED(hipMemGetInfo) REFUSED(hipMalloc) REFUSED(hipFree) REFUSED(hipMemcpy)
REFUSED(hipMemcpyPeerAsync) REFUSED(hipStreamCreate) REFUSED(hipStreamDestroy) REFUSED(hipStreamSynchronize) REFUSED(hipStreamWaitEvent)
REFUSED(hipDeviceSynchronize) REFUSED(hipModuleUnload) REFUSED(hipStreamBeginCapture) REFUSED(hipStreamEndCapture)
REFUSED(hipGraphInstantiate) REFUSED(hipGraphLaunch) REFUSED(hipGraphDestroy) REFUSED(hipGraphExecDestroy) REFUSED(hipEventCreate)
REFUSED(hipEventRecord) REFUSED(hipEventSynchronize) REFUSED(hipEventElapsedTime) REFUSED(hipEventDestroy)
