/* The streamer's SVD workspace where device or page-locked memory runs out:
 * host_stream.c with the allocators of this file in the place of HIP's. */
#include "../../butterfly_amd/csrc/host_stream.c"

#include <assert.h>

static size_t devMost, hostMost, devLive, lockedLive;

void *bfk_malloc(size_t n) {
  if (n > devMost) return NULL;
  ++devLive;
  return malloc(n);
}
void bfk_free(void *p) {
  if (p) --devLive;
  free(p);
}
void *bfk_host_malloc(size_t n) {
  if (n > hostMost) return NULL;
  ++lockedLive;
  return malloc(n);
}
void bfk_host_free(void *p) {
  if (p) --lockedLive;
  free(p);
}

int main(void) {
  SvdWork w;
  memset(&w, 0, sizeof(w));
  w.lock = 1;
  devMost = hostMost = 1 << 20;
  assert(svd_work(&w, 1000, 2000) == 0 && w.dev && w.host && w.devBytes >= 1000 && w.hostBytes >= 2000);
  assert(w.locked && lockedLive == 1 && devLive == 1);
  /* no page-locked memory any more: ordinary memory serves */
  hostMost = 0;
  assert(svd_work(&w, 1000, 30000) == 0 && w.host && w.hostBytes >= 30000 && !w.locked && lockedLive == 0);
  memset(w.host, 1, 30000);
  /* and page-locked memory again for a larger round */
  hostMost = 1 << 20;
  assert(svd_work(&w, 1000, 60000) == 0 && w.locked && lockedLive == 1);
  /* the device has room for what is asked, not for more */
  devMost = 5000;
  assert(svd_work(&w, 5000, 100) == 0 && w.dev && w.devBytes >= 5000 && devLive == 1);
  /* not even that: refused, and usable afterwards */
  assert(svd_work(&w, 5001, 100) == -2 && !w.dev && w.devBytes == 0 && devLive == 0);
  assert(svd_work(&w, 4000, 100) == 0 && devLive == 1);
  svd_work_free(&w);
  assert(devLive == 0 && lockedLive == 0);
  puts("ok");
  return 0;
}
