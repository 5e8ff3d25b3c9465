/* seph_run_jobs at an atom count for which it starts threads: every job is run
 * once, on a helper with all signals blocked but those its own instructions
 * raise, or on the caller with the caller's own mask, which is the same after
 * the call (tests/test_host_layer.py). */
#include <pthread.h>
#include <signal.h>
#include <stdio.h>
#include <unistd.h>

#include "sephost.h"

#define JOBS 64
#define FIRST_RT 34 /* the signals below it that a program may use are 1 .. 31 */

static pthread_t caller;
static int runs[JOBS], helper_jobs, bad;

static int own(int sig)
{
	return sig == SIGSEGV || sig == SIGBUS || sig == SIGFPE || sig == SIGILL;
}

static int job(void *arg, int k)
{
	const sigset_t *mine = arg;
	const int helper = !pthread_equal(pthread_self(), caller);
	sigset_t now;
	__atomic_fetch_add(&runs[k], 1, __ATOMIC_SEQ_CST);
	__atomic_fetch_add(&helper_jobs, helper, __ATOMIC_SEQ_CST);
	pthread_sigmask(SIG_BLOCK, NULL, &now);
	for (int sig = 1; sig <= SIGRTMAX; sig++) {
		if (sig == SIGKILL || sig == SIGSTOP || (sig > 31 && sig < FIRST_RT))
			continue;
		const int want = helper ? !own(sig) || sigismember(mine, sig) : sigismember(mine, sig);
		if (sigismember(&now, sig) != want)
			__atomic_store_n(&bad, sig, __ATOMIC_SEQ_CST);
	}
	usleep(2000); /* the others get their turn */
	return 0;
}

int main(void)
{
	sigset_t mine, after;
	caller = pthread_self();
	sigemptyset(&mine);
	sigaddset(&mine, SIGUSR2);
	pthread_sigmask(SIG_SETMASK, &mine, NULL);
	if (seph_run_jobs(JOBS, 1000000, job, &mine))
		return 2;
	pthread_sigmask(SIG_BLOCK, NULL, &after);
	for (int sig = 1; sig <= 31; sig++)
		if (sigismember(&after, sig) != sigismember(&mine, sig))
			bad = 100 + sig;
	for (int k = 0; k < JOBS; k++)
		if (runs[k] != 1)
			bad = 200 + k;
	printf("bad %d helper jobs %d\n", bad, helper_jobs);
	return bad || !helper_jobs;
}
